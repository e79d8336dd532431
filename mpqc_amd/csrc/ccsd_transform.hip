// Integral preparation on the GPU: the AO -> MO transform that produces the
// cc::Integrals blocks of the CCSD residual.
//
// Reference: LCAOFactory::compute4 (src/mpqc/chemistry/qc/lcao/factory/
// lcao_factory.h:378-497).  Without density fitting it transforms the AO
// integrals one index at a time (quarter transforms, :421-493) and reads
// physical-notation blocks <pq|rs> = (pr|qs); with density fitting (:386-406)
// a four-index block is the product of two three-index factors over the fitting
// index, result("i,k,j,l") = left("q,i,j") * right("q,k,l").  The Fock blocks
// are <p|F|q> = C_p^T F C_q.
//
// Both entry points write the context's integral buffers exactly as
// set_integral would; temporaries come from the context's scratch cache.
#include <stdexcept>

#include "ccsd_ctx.hpp"

namespace mpqc_hip {

namespace {

// out[a,b,c,d] (extents n) = src[off + a*s0 + b*s1 + c*s2 + d*s3]
void strided_copy(double* out, const long n[4], const double* src, long off, const long s[4], long src_vol,
                  hipStream_t stream) {
  TTerm t;
  t.p = src + off;
  for (int d = 0; d < 4; ++d) t.s[d] = s[d];
  t.alpha = 1.0;
  t.vol = src_vol - off;
  // every read stays inside the source
  long last = off;
  for (int d = 0; d < 4; ++d) last += (n[d] - 1) * s[d];
  if (off < 0 || last >= src_vol) throw std::logic_error("strided_copy reads past its source");
  tadd(out, n, 0.0, &t, 1, stream);
}

}  // namespace

// C_act = [C_occ | C_vir] (nbf x (o+v), row-major) on the device.
static void gather_coefficients(double* Cact, int nbf, int o, int v, const double* c_occ, const double* c_vir,
                                int memspace, hipStream_t s) {
  const hipMemcpyKind kind = memspace ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
  const size_t pitch = (size_t)(o + v) * sizeof(double);
  MPQC_HIP_CHECK(hipMemcpy2DAsync(Cact, pitch, c_occ, (size_t)o * sizeof(double), (size_t)o * sizeof(double), nbf,
                                  kind, s));
  MPQC_HIP_CHECK(hipMemcpy2DAsync(Cact + o, pitch, c_vir, (size_t)v * sizeof(double), (size_t)v * sizeof(double),
                                  nbf, kind, s));
}

// Fia, Fij, Fab = blocks of C_act^T F C_act  (<i|F|a>, <i|F|j>, <a|F|b>)
void CCSDContext::transform_fock(int nbf, const double* fock, const double* Cact, int memspace) {
  const int o = o_, v = v_, nmo = o_ + v_;
  ScratchBuf Fdev(scratch_, memspace ? 0 : (size_t)nbf * nbf), T(scratch_, (size_t)nbf * nmo), Fmo(scratch_, (size_t)nmo * nmo);
  const double* F = fock;
  if (!memspace) {
    MPQC_HIP_CHECK(hipMemcpyAsync(Fdev.p, fock, (size_t)nbf * nbf * sizeof(double), hipMemcpyHostToDevice, stream_));
    F = Fdev.p;
  }
  mpqc_hip::gemm(make_gemm(false, false, nbf, nmo, nbf, 1.0, F, nbf, Cact, nmo, 0.0, T.p, nmo),
                 GemmPrecision::F64, ws_, stream_);
  mpqc_hip::gemm(make_gemm(true, false, nmo, nmo, nbf, 1.0, Cact, nmo, T.p, nmo, 0.0, Fmo.p, nmo),
                 GemmPrecision::F64, ws_, stream_);
  const size_t d = sizeof(double), pitch = (size_t)nmo * d;
  MPQC_HIP_CHECK(hipMemcpy2DAsync(Fia_, v * d, Fmo.p + o, pitch, v * d, o, hipMemcpyDeviceToDevice, stream_));
  MPQC_HIP_CHECK(hipMemcpy2DAsync(Fij_, o * d, Fmo.p, pitch, o * d, o, hipMemcpyDeviceToDevice, stream_));
  MPQC_HIP_CHECK(hipMemcpy2DAsync(Fab_, v * d, Fmo.p + (size_t)o * nmo + o, pitch, v * d, v,
                                  hipMemcpyDeviceToDevice, stream_));
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  have_ints_ |= 0x7u;
}

// compute4 without density fitting (lcao_factory.h:421-493): quarter transforms of
// (mu nu|la si), each one GEMM that contracts an index and appends the new one, in the
// order mu -> p, la -> r, nu -> q, si -> s.  In that order a block <pr|qs> = (pq|rs) with
// p, r, q, s occupied or virtual comes out of the last GEMM in its own layout:
//   (mu nu la si) -> Y1 (nu la si p) -> Y2 (nu si p r) -> Y3 (si p r q) -> <pr|qs>,
// and the tree of occupied / virtual choices stops at the six blocks that are needed:
// p = i: r = j: q = k: <ij|kl>, <ij|ka>; q = a: <ij|ab>; r = a: q = j: <ia|jb>; q = b: <ia|bc>;
// p = a: r = b: q = c: <ab|cd>.  (All of (pq|rs) and six strided copies took 2.5e11 multiply-adds
// and 9 GB at 144 functions and 30 + 114 orbitals; the tree takes 1.95e11 and 5 GB.)  p goes in
// blocks and nu in slabs, so that Y1 to Y3 fit the scratch cache and calls after the first
// allocate nothing.  Bound: the matrix cores (at
// those sizes 15.0 -> 9.8 ms of kernels, 40 TFLOP/s, and 101-219 -> 10.6 ms for the call).  Up to
// kFullTransform functions either form is a chain of short launches, 18 in the tree and 13 with all of
// (pq|rs) and copies: the call with the blocks read back takes, us, all : tree, 205 : 240 at 15 functions,
// 210 : 246 at 24, 300 : 352 at 48, 455 : 490 at 60, 558 : 541 at 64, 1030 : 980 at 80 (with all functions active).
constexpr long kFullTransform = 60;

void CCSDContext::transform_ao(int nbf, const double* eri, const double* fock, const double* c_occ,
                               const double* c_vir, int memspace) {
  if (nbf <= 0 || !eri || !fock || !c_occ || !c_vir) throw std::invalid_argument("transform_ao: null or empty input");
  if (memspace != 0 && memspace != 1) throw std::invalid_argument("memspace must be host or device");
  if (memspace) MPQC_HIP_CHECK(hipDeviceSynchronize());  // the caller's pending work on its buffers
  const long n = nbf, nmo = (long)o_ + v_, O = o_, V = v_;
  if (nmo > n) throw std::invalid_argument("more active orbitals than basis functions");
  if (n * n * n >= (1L << 31) || n * n * n * n >= (1L << 40))
    throw std::invalid_argument("nbf too large for the dense AO transform");
  const long n4 = n * n * n * n;
  ScratchBuf Cact(scratch_, (size_t)n * nmo);
  gather_coefficients(Cact.p, nbf, o_, v_, c_occ, c_vir, memspace, stream_);
  ScratchBuf up(scratch_, memspace ? 0 : (size_t)n4);
  const double* x0 = eri;
  if (!memspace) {
    MPQC_HIP_CHECK(hipMemcpyAsync(up.p, eri, n4 * sizeof(double), hipMemcpyHostToDevice, stream_));
    x0 = up.p;
  }
  if (!Gabcd_) Gabcd_ = alloc((size_t)V * V * V * V);
  // out[m, c] = sum_k x[k, m] Cact[k, c0 + c], c < nc, for each of `batch` x and out
  auto quarter = [&](const double* x, long rows, long ldx, long c0, long nc, double* out, long batch, long sx, long so) {
    GemmDesc g = make_gemm(true, false, (int)rows, (int)nc, nbf, 1.0, x, ldx, Cact.p + c0, nmo, 0.0, out, nc);
    g.sA = sx; g.sC = so; g.batch = (int)batch;
    mpqc_hip::gemm(g, GemmPrecision::F64, ws_, stream_);
  };
  auto full = [&] {
    // all of (pq|rs), the leading index contracted four times, and the blocks as strided copies
    ScratchBuf a(scratch_, (size_t)(n * n * n * nmo)), b(scratch_, (size_t)(n * n * nmo * nmo));
    const double* x = x0;
    long rows = n * n * n;
    for (int k = 0; k < 4; ++k) {
      double* const y = k % 2 ? b.p : a.p;
      quarter(x, rows, rows, 0, nmo, y, 1, 0, 0);
      x = y;
      rows = rows / n * nmo;
    }
    struct Blk { double* dst; long P0, Q0, R0, S0, nP, nQ, nR, nS; };
    const Blk blocks[] = {{Gijab_, 0, 0, O, O, O, O, V, V}, {Gijkl_, 0, 0, 0, 0, O, O, O, O},
                          {Giajb_, 0, O, 0, O, O, V, O, V}, {Giabc_, 0, O, O, O, O, V, V, V},
                          {Gijka_, 0, 0, 0, O, O, O, O, V}, {Gabcd_, O, O, O, O, V, V, V, V}};
    const long m2 = nmo * nmo, s[4] = {m2 * nmo, nmo, m2, 1};
    for (const Blk& q : blocks) {  // <PQ|RS>[a,b,c,d] = (P0+a, R0+c | Q0+b, S0+d)
      const long ext[4] = {q.nP, q.nQ, q.nR, q.nS};
      strided_copy(q.dst, ext, x, q.P0 * m2 * nmo + q.R0 * m2 + q.Q0 * nmo + q.S0, s, m2 * m2, stream_);
    }
  };
  auto tree = [&] {
    // Y1 to Y3 take 2 GiB (every p block reads the AO integrals again, but a new context's first
    // call pays 20 to 90 ms per GB for the allocation), 128 MiB of them for Y1
    const long kSlab = 16L << 20, budget = (256L << 20) - kSlab;
    struct Part { long nP, nR, nRQ, pb, slab; };  // p occupied, p virtual
    Part part[2];
    size_t words = 0;
    for (int virt = 0; virt < 2; ++virt) {
      Part& t = part[virt];
      t.nP = virt ? V : O;
      t.nR = virt ? V : nmo;  // r: all of Y2's last index (occupied first); only virtual ones for <ab|cd>
      t.nRQ = virt ? V * V : std::max(O, V) * std::max(O, V);
      const long per_p = n * n * t.nR + n * t.nRQ;
      t.pb = ceil_div(t.nP, ceil_div(t.nP, std::max(1L, budget / per_p)));
      t.slab = std::max(1L, std::min(n, kSlab / (n * n * t.pb)));
      words = std::max<size_t>(words, (size_t)(t.slab * n * n * t.pb + t.pb * per_p));
    }
    ScratchBuf Y(scratch_, words);
    for (int virt = 0; virt < 2; ++virt) {
      const Part& t = part[virt];
      const long nP = t.nP, c0 = virt ? O : 0, pb = t.pb, slab = t.slab;
      double* const Y1 = Y.p;
      double* const Y2 = Y1 + slab * n * n * pb;
      double* const Y3 = Y2 + n * n * pb * t.nR;
      for (long p0 = 0; p0 < nP; p0 += pb) {
        const long np = std::min(pb, nP - p0);
        double* Y2o = Y2;                                  // r occupied (p occupied only)
        double* Y2v = Y2 + (virt ? 0 : n * n * np * O);    // r virtual
        for (long m0 = 0; m0 < n; m0 += slab) {
          const long ns = std::min(slab, n - m0);
          quarter(x0 + m0 * n * n, ns * n * n, n * n * n, c0 + p0, np, Y1, 1, 0, 0);
          if (!virt) quarter(Y1, n * np, n * np, 0, O, Y2o + m0 * n * np * O, ns, n * n * np, n * np * O);
          quarter(Y1, n * np, n * np, O, V, Y2v + m0 * n * np * V, ns, n * n * np, n * np * V);
        }
        // the last two quarters of one choice of r and q, to the block(s) <pr|q.>
        auto finish = [&](const double* y2, long R, long q0, long Q, double* dst_o, double* dst_v) {
          quarter(y2, n * np * R, n * np * R, q0, Q, Y3, 1, 0, 0);
          const long rows = np * R * Q;
          if (dst_o) quarter(Y3, rows, rows, 0, O, dst_o + p0 * R * Q * O, 1, 0, 0);
          quarter(Y3, rows, rows, O, V, dst_v + p0 * R * Q * V, 1, 0, 0);
        };
        if (virt) {
          finish(Y2v, V, O, V, nullptr, Gabcd_);
        } else {
          finish(Y2o, O, 0, O, Gijkl_, Gijka_);
          finish(Y2o, O, O, V, nullptr, Gijab_);
          finish(Y2v, V, 0, O, nullptr, Giajb_);
          finish(Y2v, V, O, V, nullptr, Giabc_);
        }
      }
    }
  };
  if (n <= kFullTransform) full();
  else tree();
  check_launch("transform_ao");
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  have_ints_ |= 0x1f8u;
  transform_fock(nbf, fock, Cact.p, memspace);
  prepared_ = false;
}

// compute4 with density fitting (lcao_factory.h:386-406) for the "df" method:
// X(K,p,q) = sum_L metric(L,K) (L|mu nu) C(mu,p) C(nu,q) gives Xai, Xij, Xab
// (ccsd.h:481-493), then every four-index block the df residual reads is a
// product of two factors over K, e.g. <ij|ab> = (ia|jb) = X(K,i,a) X(K,j,b).
void CCSDContext::transform_df(int nbf, const double* B3, const double* metric, const double* fock,
                               const double* c_occ, const double* c_vir, int memspace) {
  if (naux_ == 0) throw std::logic_error("transform_df needs set_df_basis first");
  if (nbf <= 0 || !B3 || !fock || !c_occ || !c_vir) throw std::invalid_argument("transform_df: null or empty input");
  if (memspace != 0 && memspace != 1) throw std::invalid_argument("memspace must be host or device");
  if (memspace) MPQC_HIP_CHECK(hipDeviceSynchronize());  // the caller's pending work on its buffers
  const long n = nbf, Q = naux_, nmo = (long)o_ + v_, O = o_, V = v_;
  if (nmo > n) throw std::invalid_argument("more active orbitals than basis functions");
  if (Q * n * n >= (1L << 31)) throw std::invalid_argument("naux * nbf^2 too large");
  const hipMemcpyKind kind = memspace ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
  ScratchBuf Cact(scratch_, (size_t)n * nmo);
  gather_coefficients(Cact.p, nbf, o_, v_, c_occ, c_vir, memspace, stream_);
  // fitted AO factors X(K, mu nu) = sum_L metric(L,K) B(L, mu nu)
  ScratchBuf Xao(scratch_, (size_t)Q * n * n), Bup(scratch_, metric ? (size_t)Q * n * n : 0),
      Mup(scratch_, metric ? (size_t)Q * Q : 0);
  if (metric) {
    MPQC_HIP_CHECK(hipMemcpyAsync(Bup.p, B3, Q * n * n * sizeof(double), kind, stream_));
    MPQC_HIP_CHECK(hipMemcpyAsync(Mup.p, metric, Q * Q * sizeof(double), kind, stream_));
    mpqc_hip::gemm(make_gemm(true, false, (int)Q, (int)(n * n), (int)Q, 1.0, Mup.p, Q, Bup.p, n * n, 0.0, Xao.p,
                             n * n), GemmPrecision::F64, ws_, stream_);
  } else {
    MPQC_HIP_CHECK(hipMemcpyAsync(Xao.p, B3, Q * n * n * sizeof(double), kind, stream_));
  }
  // Y(K,mu,q) = X(K,mu,nu) C(nu,q);  Z(K,p,q) = C(mu,p) Y(K,mu,q)
  ScratchBuf Y(scratch_, (size_t)Q * n * nmo), Z(scratch_, (size_t)Q * nmo * nmo);
  mpqc_hip::gemm(make_gemm(false, false, (int)(Q * n), (int)nmo, nbf, 1.0, Xao.p, n, Cact.p, nmo, 0.0, Y.p, nmo),
                 GemmPrecision::F64, ws_, stream_);
  {
    GemmDesc d = make_gemm(true, false, (int)nmo, (int)nmo, nbf, 1.0, Cact.p, nmo, Y.p, nmo, 0.0, Z.p, nmo);
    d.sA = 0; d.sB = n * nmo; d.sC = nmo * nmo; d.batch = (int)Q;
    mpqc_hip::gemm(d, GemmPrecision::F64, ws_, stream_);
  }
  const long zvol = Q * nmo * nmo;
  const long zs[4] = {0, nmo * nmo, nmo, 1};
  {
    const long e_ai[4] = {1, Q, V, O}, e_ij[4] = {1, Q, O, O}, e_ab[4] = {1, Q, V, V};
    strided_copy(Xai_, e_ai, Z.p, O * nmo, zs, zvol, stream_);
    strided_copy(Xij_, e_ij, Z.p, 0, zs, zvol, stream_);
    strided_copy(Xab_, e_ab, Z.p, O * nmo + O, zs, zvol, stream_);
  }
  // Xia(K,i,a) contiguous, then the four-index blocks as X^T X GEMMs over K and one
  // permutation each
  ScratchBuf Xia(scratch_, (size_t)Q * O * V);
  {
    const long e_ia[4] = {1, Q, O, V};
    strided_copy(Xia.p, e_ia, Z.p, O, zs, zvol, stream_);
  }
  const bool full = !reduced_abcd_;
  const long tmp_n = full ? std::max(V * V * V * V, O * V * V * V) : std::max(O * O * V * V, O * O * O * V);
  ScratchBuf T(scratch_, (size_t)std::max(tmp_n, O * O * O * O));
  // dst[perm(x,y,z,w)] = sum_K A(K,x,y) B(K,z,w): T[(x,y)][(z,w)] = A^T B, then dst = permute(T)
  auto block = [&](double* dst, const double* A, long nx, long ny, const double* Bm, long nz, long nw,
                   std::array<int, 4> perm) {
    mpqc_hip::gemm(make_gemm(true, false, (int)(nx * ny), (int)(nz * nw), (int)Q, 1.0, A, nx * ny, Bm, nz * nw,
                             0.0, T.p, nz * nw), GemmPrecision::F64, ws_, stream_);
    const long in_ext[4] = {nx, ny, nz, nw};
    long out_ext[4];
    const int pm[4] = {perm[0], perm[1], perm[2], perm[3]};
    for (int d = 0; d < 4; ++d) out_ext[d] = in_ext[pm[d]];
    TTerm t;
    t.p = T.p;
    permuted_strides(in_ext, pm, t.s);
    t.alpha = 1.0;
    t.vol = nx * ny * nz * nw;
    tadd(dst, out_ext, 0.0, &t, 1, stream_);
  };
  block(Gijab_, Xia.p, O, V, Xia.p, O, V, {0, 2, 1, 3});  // (ia|jb) -> <ij|ab>
  block(Gijkl_, Xij_, O, O, Xij_, O, O, {0, 2, 1, 3});    // (ik|jl) -> <ij|kl>
  block(Giajb_, Xij_, O, O, Xab_, V, V, {0, 2, 1, 3});    // (ij|ab) -> <ia|jb>
  block(Gijka_, Xij_, O, O, Xia.p, O, V, {0, 2, 1, 3});   // (ik|ja) -> <ij|ka>
  unsigned bits = 0x0b8u | 0xe00u;                        // Gijab Gijkl Giajb Gijka, Xai Xij Xab
  if (full) {
    if (!Gabcd_) Gabcd_ = alloc((size_t)V * V * V * V);
    block(Giabc_, Xia.p, O, V, Xab_, V, V, {0, 2, 1, 3});  // (ib|ac) -> <ia|bc>
    block(Gabcd_, Xab_, V, V, Xab_, V, V, {0, 2, 1, 3});   // (ac|bd) -> <ab|cd>
    bits |= 0x140u;
  }
  check_launch("transform_df");
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  have_ints_ |= bits;
  transform_fock(nbf, fock, Cact.p, memspace);
  prepared_ = false;
}

}  // namespace mpqc_hip
