// The residual of a small molecule as a few launches of independent ops.
//
// Water in cc-pVDZ (o = 5, v = 19) runs about 80 dependent kernels of 4 to 8 us per residual,
// nearly all of it load latency and launch overhead.  The op tape of the residual (the list
// the adjoint sweeps) is scheduled instead: an op goes into the first level that comes
// after the ops it depends on, and a level is one launch of every small op in it, a workgroup
// per output tile, followed by the contractions that fill the chip by themselves.  Sums into one
// tensor may enter in any order (the order is fixed when the plan is made, so results do
// not vary); contractions over a long K leave partial sums that the next level adds.
//
// One residual with its amplitudes in and residuals out, op by op -> by levels (us):
//   o, v:  3, 16  341 -> 162;  5, 19  374 -> 174;  8, 40  427 -> 273;  10, 50  497 -> 374;
//   8, 70  619 -> 469;  13, 61  769 -> 679;  10, 90  1004 -> 963;  16, 70  1136 -> 1286.
// With more than about a million doubles the ops fill the chip one at a time, and their own
// kernels (the combinations of amplitude layouts above all) are the better ones: kLevelMaxDoubles.
#include <algorithm>
#include <functional>
#include <stdexcept>

#include "ccsd_ctx.hpp"
#include "gemm_f64_tile.hpp"
#include "permute.hpp"

namespace mpqc_hip {

namespace {

constexpr int kLvThreads = 1024;
constexpr int kLvElems = 4096;   // output elements of a workgroup of an element-wise op
constexpr int kLvSplit = 512;    // K of a workgroup where K is split
constexpr long kLvTarget = 1024; // no K split beyond this many workgroups of an op
constexpr double kLvWideWork = 3.0e7;  // multiply-adds from which an op gets 64-column tiles
// A contraction is a launch of its own (gemm(), its shape's kernel) from this many
// multiply-adds, or if its tiles alone fill the chip:
constexpr double kLvOwnWork = 2.0e8;
constexpr long kLvOwnGroups = 300;

}  // namespace

struct LevelOp {
  enum Kind : int { kGemm = 0, kTAdd = 1, kReduce = 2, kPerm = 3, kGemv = 4 };
  int kind;
  int first;  // first workgroup of the op in its level's launch
  // kGemm (and kReduce: C, ldc, sC, M, N, nsplit, beta, W; nsplit_batch: batch entries)
  KParams p;
  int trans;  // 1 A^T, 2 B^T
  int wide;   // kGemm: 64-column tiles instead of 16-column ones; kReduce: a wave per output
  // kTAdd: out[e] = beta out[e] + sum_t alpha_t p_t[strides . e] (+ x[.] y[.])
  double* out;
  double beta;
  int n[4];
  int nterms;
  struct Term {
    const double* p;
    int s[4];
    double alpha;
  } t[kMaxTerms];
  const double *px, *py;  // product term, or null
  int sx[4], sy[4];
  // kPerm: the same through LDS tiles (out, beta as above)
  PermGeom g;
};

namespace {

template <int CB, int U>
constexpr int lv_lds() {
  return std::max({F64Shared<1, CB, 4, U, false, false>::kDoubles, F64Shared<1, CB, 4, U, false, true>::kDoubles,
                   F64Shared<1, CB, 4, U, true, false>::kDoubles});
}

// One level: workgroup w belongs to the last op whose first workgroup is <= w.  A
// contraction tile is run by four K groups of four waves (dgemm_f64_tile), which is the
// shortest chain of load latencies per tile; an element-wise op gathers (the operands of these sizes stay in L2).
__global__ __launch_bounds__(kLvThreads, 4) void level_kernel(const LevelOp* __restrict__ ops, int nops) {
  __shared__ __attribute__((aligned(16))) double smem[std::max(lv_lds<1, 2>(), lv_lds<4, 1>())];
  const int w = blockIdx.x;
  int q = 0;
  while (q + 1 < nops && ops[q + 1].first <= w) ++q;
  const LevelOp& op = ops[q];
  const int local = w - op.first;
  if (op.kind == LevelOp::kGemm) {
    const KParams& p = op.p;
    const int ntiles = p.tiles_m * p.tiles_n;
    const int z = local / ntiles, tile = local - z * ntiles;
    if (op.wide) {
      if (op.trans == 0) dgemm_f64_tile<1, 4, 4, 1, false, false>(p, tile, z, smem);
      else if (op.trans == 1) dgemm_f64_tile<1, 4, 4, 1, true, false>(p, tile, z, smem);
      else dgemm_f64_tile<1, 4, 4, 1, false, true>(p, tile, z, smem);
    } else {
      if (op.trans == 0) dgemm_f64_tile<1, 1, 4, 2, false, false>(p, tile, z, smem);
      else if (op.trans == 1) dgemm_f64_tile<1, 1, 4, 2, true, false>(p, tile, z, smem);
      else dgemm_f64_tile<1, 1, 4, 2, false, true>(p, tile, z, smem);
    }
  } else if (op.kind == LevelOp::kTAdd) {
    const int n1 = op.n[1], n2 = op.n[2], n3 = op.n[3], total = op.n[0] * n1 * n2 * n3;
    int e[4], i[4][4];
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[k] = local * kLvElems + k * kLvThreads + (int)threadIdx.x;
      const int ek = min(e[k], total - 1);
      const int a = ek / n3, b = a / n2;
      i[k][3] = ek - a * n3;
      i[k][2] = a - b * n2;
      i[k][0] = b / n1;
      i[k][1] = b - i[k][0] * n1;
      v[k] = 0.0;
    }
    for (int t = 0; t < op.nterms; ++t) {
      const LevelOp::Term& T = op.t[t];
      double x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = T.p[i[k][0] * T.s[0] + i[k][1] * T.s[1] + i[k][2] * T.s[2] + i[k][3] * T.s[3]];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] += T.alpha * x[k];
    }
    if (op.px) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] += op.px[i[k][0] * op.sx[0] + i[k][1] * op.sx[1] + i[k][2] * op.sx[2] + i[k][3] * op.sx[3]] *
                op.py[i[k][0] * op.sy[0] + i[k][1] * op.sy[1] + i[k][2] * op.sy[2] + i[k][3] * op.sy[3]];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (e[k] < total) op.out[e[k]] = op.beta == 0.0 ? v[k] : v[k] + op.beta * op.out[e[k]];
  } else if (op.kind == LevelOp::kGemv) {  // a wave per row of A
    const KParams& p = op.p;
    const int lane = threadIdx.x & 63, m = local * (kLvThreads / 64) + (int)(threadIdx.x >> 6);
    if (m < p.M) {
      const double* a = p.A + (long)m * p.lda;
      double s = 0.0;
#pragma unroll 8
      for (int k = lane; k < p.K; k += 64) s = fma(a[k], p.B[(long)k * p.ldb], s);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
      if (lane == 0) {
        double* y = p.C + (long)m * p.ldc;
        *y = p.beta == 0.0 ? p.alpha * s : fma(p.beta, *y, p.alpha * s);
      }
    }
  } else if (op.kind == LevelOp::kPerm) {
    const int gx = op.g.tiles3 * op.g.tilesq, gy = (int)op.g.nr1;
    const int rest = local / gx;
    permute_block<1, kLvThreads>(
        op.g, local - rest * gx, rest % gy, rest / gy,
        [&](long e, double v) { op.out[e] = op.beta == 0.0 ? v : v + op.beta * op.out[e]; }, smem);
  } else {  // kReduce: C[b] = beta C[b] + sum_s W[b, s] in split order
    const KParams& p = op.p;
    const long MN = (long)p.M * p.N, total = MN * p.nsplit_batch;
    if (op.wide) {  // a wave per output: lane l adds the partials l, l + 64, ... in turn
      const long el = (long)local * (kLvThreads / 64) + (threadIdx.x >> 6);
      if (el < total) {
        const int lane = threadIdx.x & 63;
        const long b = el / MN, mn = el - b * MN;
        const double* ws = p.W + b * p.nsplit * MN + mn;
        double acc = 0.0;
        for (int s = lane; s < p.nsplit; s += 64) acc += ws[(long)s * MN];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (lane == 0) {
          const long m = mn / p.N;
          double* c = p.C + b * p.sC + m * p.ldc + (mn - m * p.N);
          *c = p.beta == 0.0 ? acc : acc + p.beta * (*c);
        }
      }
      return;
    }
    for (int k = 0; k < kLvElems / kLvThreads; ++k) {
      const long el = (long)local * kLvElems + k * kLvThreads + threadIdx.x;
      if (el >= total) break;
      const long b = el / MN, mn = el - b * MN;
      const double* ws = p.W + b * p.nsplit * MN + mn;
      double acc = 0.0;
      for (int s = 0; s < p.nsplit; ++s) acc += ws[(long)s * MN];
      const long m = mn / p.N;
      double* c = p.C + b * p.sC + m * p.ldc + (mn - m * p.N);
      *c = p.beta == 0.0 ? acc : acc + p.beta * (*c);
    }
  }
}

}  // namespace

// Whether the scheduled form is the faster one: the table above; o^4 arrays too large for it, from
// o = 54 or so ((o, v), op by op : by levels, us: (48, 21) 1029 : 1067, (56, 18) 1212 : 1320, (53, 8) 636 :
// 525, (80, 6) 1329 : 1575, (100, 10) 3413 : 4225, (120, 4) 4466 : 5902); and one occupied orbital beside
// many virtual ones, whose matrix-vector products are whole passes over HBM ((1, 150) 893 : 813, (1, 180)
// 1330 : 1330, (1, 256) 3651 : 4103; (2, 256) 5380 : 4910).
bool CCSDContext::levels_usable() const {
  const long O = o_, V = v_;
  return levels_mode_ && prec_ == GemmPrecision::F64 && !df_ && !direct_ && !tape_ && !kernel_timing_ &&
         V * V * O * O <= kLevelMaxDoubles && O * O * O * O <= kLevelMaxOoccDoubles && (O > 1 || V <= 180);
}

void CCSDContext::plan_levels() {
  if (levels_gen_ == gen_) return;
  std::vector<TapeOp> tape;
  const bool fresh = tau_fresh_;
  tape_ = &tape;
  tape_execute_ = false;
  try {
    residual_ops();
  } catch (...) {
    tape_ = nullptr;
    tape_execute_ = true;
    throw;
  }
  tape_ = nullptr;
  tape_execute_ = true;
  tau_fresh_ = fresh;

  const bool psym = (double)v_ * v_ * v_ * v_ * o_ * o_ >= kPairWork && pp_symmetric_usable();
  if (psym && !pp_packed_) pack_pp_symmetric();

  // ---- ops with the buffers they read and write (buffers: allocation numbers; partial
  // sums get numbers of their own past them)
  struct Node {
    LevelOp op;
    std::vector<int> reads;
    int write = -1;
    bool accumulates = false;
    int groups = 0;         // workgroups
    std::vector<int> deps;  // earlier nodes
    int height = 0, level = -1;
    int own = -1;           // launched by itself: number of its LevelCall
  };
  std::vector<Node> nodes;
  level_calls_.clear();
  size_t ws_doubles = 0;
  int next_buffer = (int)allocations_.size();
  std::vector<std::pair<size_t, size_t>> ws_of;  // node -> workspace offset
  auto buf = [&](const double* p) {
    const int k = alloc_index(p);
    if (k < 0) throw std::logic_error("level plan: operand not owned by the context");
    return k;
  };
  auto elementwise = [&](Node& nd, long total) { nd.groups = (int)ceil_div(total, kLvElems); };
  // a transposing combination with whole tiles runs through LDS, any other gathers
  auto tiled = [&](Node& nd, const long n[4], const TTerm* terms, int nterms, const TProd* prod) {
    const PermGeom g = make_perm_geom(n, terms, nterms, prod);
    if (!g.tiled || g.t3 * g.tq < kLvThreads) return;
    nd.op.kind = LevelOp::kPerm;
    nd.op.g = g;
    nd.groups = (int)((long)g.tiles3 * g.tilesq * g.nr0 * g.nr1);
  };
  auto terms_of = [&](LevelOp& op, const Src& s, double alpha) {
    LevelOp::Term& t = op.t[op.nterms++];
    long ext[4] = {s.ext[0], s.ext[1], s.ext[2], s.ext[3]}, st[4];
    int perm[4] = {s.perm[0], s.perm[1], s.perm[2], s.perm[3]};
    permuted_strides(ext, perm, st);
    t.p = s.p;
    t.alpha = alpha;
    for (int d = 0; d < 4; ++d) t.s[d] = (int)st[d];
  };
  if (psym) {
    Node nd;
    nd.op = LevelOp{};
    nd.reads = {buf(tau_)};
    nd.write = buf(Spk_);
    nd.own = (int)level_calls_.size();
    level_calls_.push_back([this] { pack_tau_pairs(); });
    nodes.push_back(nd);
  }
  for (const TapeOp& o : tape) {
    Node nd;
    nd.op = LevelOp{};
    switch (o.kind) {
      case TapeOp::kCopy: {
        nd.op.kind = LevelOp::kTAdd;
        nd.op.out = o.dst;
        nd.op.n[0] = nd.op.n[1] = nd.op.n[2] = 1;
        nd.op.n[3] = (int)o.n;
        nd.op.nterms = 1;
        nd.op.t[0] = LevelOp::Term{o.src, {0, 0, 0, 1}, 1.0};
        nd.reads = {buf(o.src)};
        nd.write = buf(o.dst);
        elementwise(nd, o.n);
        break;
      }
      case TapeOp::kTAdd: {
        nd.op.kind = LevelOp::kTAdd;
        nd.op.out = o.dst;
        nd.op.beta = o.beta;
        long total = 1;
        for (int d = 0; d < 4; ++d) {
          nd.op.n[d] = (int)o.ext[d];
          total *= o.ext[d];
        }
        for (int t = 0; t < o.nterms; ++t) {
          terms_of(nd.op, o.terms[t], o.terms[t].alpha);
          nd.reads.push_back(buf(o.terms[t].p));
        }
        nd.write = buf(o.dst);
        nd.accumulates = o.beta == 1.0;
        if (o.beta != 0.0 && o.beta != 1.0) nd.reads.push_back(nd.write);
        elementwise(nd, total);
        {
          TTerm tt[kMaxTerms];
          long n[4];
          for (int t = 0; t < o.nterms; ++t) {
            tt[t].p = o.terms[t].p;
            long ext[4] = {o.terms[t].ext[0], o.terms[t].ext[1], o.terms[t].ext[2], o.terms[t].ext[3]};
            int perm[4] = {o.terms[t].perm[0], o.terms[t].perm[1], o.terms[t].perm[2], o.terms[t].perm[3]};
            permuted_strides(ext, perm, tt[t].s);
            tt[t].alpha = o.terms[t].alpha;
            tt[t].vol = total;
          }
          for (int d = 0; d < 4; ++d) n[d] = o.ext[d];
          tiled(nd, n, tt, o.nterms, nullptr);
        }
        break;
      }
      case TapeOp::kTP: {  // TP(a,i,l,d) = 0.5 t2(d,a,i,l) + t1(d,i) t1(a,l)
        const long O = o_, V = v_;
        nd.op.kind = LevelOp::kTAdd;
        nd.op.out = o.dst;
        const long n[4] = {V, O, O, V};
        for (int d = 0; d < 4; ++d) nd.op.n[d] = (int)n[d];
        terms_of(nd.op, Src{o.src, {V, V, O, O}, {1, 2, 3, 0}, 0.5}, 0.5);
        const TProd pr = tp_product();
        nd.op.px = pr.x;
        nd.op.py = pr.y;
        for (int d = 0; d < 4; ++d) {
          nd.op.sx[d] = (int)pr.sx[d];
          nd.op.sy[d] = (int)pr.sy[d];
        }
        nd.reads = {buf(o.src), buf(o.src2)};
        nd.write = buf(o.dst);
        elementwise(nd, V * O * O * V);
        {
          TTerm tt;
          tt.p = o.src;
          const long ext[4] = {V, V, O, O};
          const int perm[4] = {1, 2, 3, 0};
          permuted_strides(ext, perm, tt.s);
          tt.alpha = 0.5;
          tt.vol = V * V * O * O;
          tiled(nd, n, &tt, 1, &pr);
        }
        break;
      }
      case TapeOp::kGemm: {
        const GemmDesc& g = o.g;
        const double work = (double)g.M * g.N * g.K * g.batch;
        const long narrow = ceil_div(g.M, 64) * ceil_div(g.N, 16) * g.batch;
        nd.reads = {buf(g.A), buf(g.B)};
        nd.write = buf(g.C);
        nd.accumulates = g.beta == 1.0;
        if (g.beta != 0.0 && g.beta != 1.0) nd.reads.push_back(nd.write);
        if (psym && o.tag == "r2:pp_ladder") {  // on the packed pairs (pack_tau_pairs above)
          nd.reads = {buf(Spk_)};
          nd.own = (int)level_calls_.size();
          level_calls_.push_back([this] { pp_ladder_symmetric(r2_); });
          break;
        }
        if (g.N == 1 && !g.transA && g.batch == 1 && work < kLvOwnWork) {
          nd.op.kind = LevelOp::kGemv;
          nd.op.p.A = g.A; nd.op.p.B = g.B; nd.op.p.C = g.C;
          nd.op.p.lda = g.lda; nd.op.p.ldb = g.transB ? 1 : g.ldb; nd.op.p.ldc = g.ldc;
          nd.op.p.M = g.M; nd.op.p.N = 1; nd.op.p.K = g.K; nd.op.p.nsplit = 1;
          nd.op.p.alpha = g.alpha; nd.op.p.beta = g.beta;
          nd.groups = (int)ceil_div(g.M, kLvThreads / 64);
          break;
        }
        nd.op.wide = work >= kLvWideWork && g.N > 16;
        if (work >= kLvOwnWork || (nd.op.wide ? ceil_div(narrow, 4) : narrow) > kLvOwnGroups) {
          nd.own = (int)level_calls_.size();
          level_calls_.push_back([this, g] { mpqc_hip::gemm(g, GemmPrecision::F64, ws_, stream_); });
          break;
        }
        if (g.transA && g.transB) throw std::logic_error("level plan: no A^T B^T contractions expected");
        KParams& p = nd.op.p;
        nd.op.kind = LevelOp::kGemm;
        nd.op.trans = g.transA ? 1 : g.transB ? 2 : 0;
        p.A = g.A; p.B = g.B; p.C = g.C;
        p.lda = g.lda; p.ldb = g.ldb; p.ldc = g.ldc; p.sA = g.sA; p.sB = g.sB; p.sC = g.sC;
        p.M = g.M; p.N = g.N; p.K = g.K; p.batch0 = 0; p.per_xcd = 0; p.nsplit_batch = g.batch;
        p.alpha = g.alpha; p.beta = g.beta; p.W = nullptr;
        const int bn = nd.op.wide ? 64 : 16, slice = nd.op.wide ? 16 : 32;
        p.tiles_m = (int)ceil_div(g.M, 64);
        p.tiles_n = (int)ceil_div(g.N, bn);
        const long tiles = (long)p.tiles_m * p.tiles_n * g.batch;
        const long ns = std::max(1L, std::min<long>(ceil_div(g.K, kLvSplit), kLvTarget / std::max(1L, tiles)));
        p.kchunk = (int)(ceil_div(ceil_div(g.K, ns), slice) * slice);
        p.nsplit = (int)ceil_div(g.K, p.kchunk);
        nd.groups = (int)(tiles * p.nsplit);
        if (p.nsplit > 1) {
          const size_t off = ws_doubles;
          ws_doubles += (size_t)p.nsplit * g.batch * g.M * g.N;
          p.W = reinterpret_cast<double*>(off);  // (resolved below)
          nd.write = next_buffer++;
          nd.accumulates = false;
          nd.reads = {buf(g.A), buf(g.B)};
          nodes.push_back(nd);
          Node rd;
          rd.op = LevelOp{};
          rd.op.kind = LevelOp::kReduce;
          rd.op.p = p;
          rd.reads = {nd.write};
          rd.write = buf(g.C);
          rd.accumulates = g.beta == 1.0;
          if (g.beta != 0.0 && g.beta != 1.0) rd.reads.push_back(rd.write);
          rd.op.wide = p.nsplit >= 16;
          if (rd.op.wide) rd.groups = (int)ceil_div((long)g.batch * g.M * g.N, kLvThreads / 64);
          else elementwise(rd, (long)g.batch * g.M * g.N);
          nodes.push_back(rd);
          continue;
        }
        break;
      }
      case TapeOp::kTau: throw std::logic_error("level plan: tau is built before the residual");
    }
    nodes.push_back(nd);
  }

  // ---- dependencies.  Per buffer: `base` is what any further sum into it has to wait for
  // (the write that started it, or the readers of an earlier state), `sums` the sums since.
  struct State {
    std::vector<int> base, sums, readers;
  };
  std::vector<State> state(next_buffer);
  auto add = [](std::vector<int>& to, const std::vector<int>& from) { to.insert(to.end(), from.begin(), from.end()); };
  for (int k = 0; k < (int)nodes.size(); ++k) {
    Node& nd = nodes[k];
    for (int r : nd.reads) {
      add(nd.deps, state[r].base);
      add(nd.deps, state[r].sums);
    }
    State& st = state[nd.write];
    if (nd.accumulates && st.readers.empty()) {
      add(nd.deps, st.base);
    } else {  // a new state of the buffer: after everything that saw the old one
      add(nd.deps, st.base);
      add(nd.deps, st.sums);
      add(nd.deps, st.readers);
      st.base = {k};
      st.sums.clear();
      st.readers.clear();
    }
    if (st.base.empty() || st.base[0] != k) st.sums.push_back(k);
    for (int r : nd.reads)
      if (r != nd.write) state[r].readers.push_back(k);
  }
  for (int k = (int)nodes.size() - 1; k >= 0; --k)
    for (int d : nodes[k].deps) nodes[d].height = std::max(nodes[d].height, nodes[k].height + 1);

  // ---- levels: ready ops, those on the longest remaining chain first; one op per written
  // buffer and level
  std::vector<std::vector<int>> levels;
  std::vector<int> todo(nodes.size());
  for (size_t k = 0; k < nodes.size(); ++k) todo[k] = (int)k;
  while (!todo.empty()) {
    const int lv = (int)levels.size();
    std::vector<int> ready, taken, left;
    for (int k : todo) {
      bool ok = true;
      for (int d : nodes[k].deps) ok = ok && nodes[d].level >= 0 && nodes[d].level < lv;
      (ok ? ready : left).push_back(k);
    }
    std::stable_sort(ready.begin(), ready.end(), [&](int a, int b) { return nodes[a].height > nodes[b].height; });
    std::vector<char> written(next_buffer, 0);
    for (int k : ready) {
      if (written[nodes[k].write]) {
        left.push_back(k);
        continue;
      }
      written[nodes[k].write] = 1;
      nodes[k].level = lv;
      taken.push_back(k);
    }
    if (taken.empty()) throw std::logic_error("level plan: cyclic dependencies");
    levels.push_back(taken);
    std::sort(left.begin(), left.end());
    todo.swap(left);
  }

  // ---- device records
  if (ws_doubles > levels_ws_n_) {
    levels_ws_ = alloc(ws_doubles);
    levels_ws_n_ = ws_doubles;
  }
  std::vector<LevelOp> host;
  levels_.clear();
  for (const std::vector<int>& lv : levels) {
    Level L;
    L.first_op = (int)host.size();
    L.nops = 0;
    L.groups = 0;
    for (int k : lv) {
      if (nodes[k].own >= 0) {
        L.calls.push_back(nodes[k].own);
        continue;
      }
      ++L.nops;
      LevelOp op = nodes[k].op;
      if (op.p.nsplit > 1 && (op.kind == LevelOp::kGemm || op.kind == LevelOp::kReduce))
        op.p.W = levels_ws_ + reinterpret_cast<size_t>(op.p.W);
      op.first = L.groups;
      L.groups += nodes[k].groups;
      host.push_back(op);
    }
    levels_.push_back(L);
  }
  const size_t words = ceil_div((long)(host.size() * sizeof(LevelOp)), (long)sizeof(double));
  if (words > levels_ops_n_) {
    levels_ops_ = alloc(words);
    levels_ops_n_ = words;
  }
  MPQC_HIP_CHECK(hipMemcpyAsync(levels_ops_, host.data(), host.size() * sizeof(LevelOp), hipMemcpyHostToDevice, stream_));
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  levels_gen_ = gen_;
}

void CCSDContext::run_levels() {
  const LevelOp* ops = reinterpret_cast<const LevelOp*>(levels_ops_);
  for (const Level& L : levels_) {
    if (L.nops > 0) {
      hipLaunchKernelGGL(level_kernel, dim3((unsigned)L.groups), dim3(kLvThreads), 0, stream_, ops + L.first_op, L.nops);
      check_launch("level");
    }
    for (int c : L.calls) level_calls_[c]();
  }
}

}  // namespace mpqc_hip
