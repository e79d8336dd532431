// Perturbative triples correction (T) on the GPU from the converged CCSD
// amplitudes held by the context.
//
// Reference: CCSD_T::compute_ccsd_t_straight (src/mpqc/chemistry/qc/lcao/cc/
// ccsd_t.h:1127-1167) with CCSD_T_Reduce (:2274-2335):
//   t3(a,b,c,i,j,k) = <id|ab> t2(d,c,j,k) - <jk|lc> t2(a,b,i,l)        (raw W)
//   t3s = sum of the six simultaneous permutations of (a,i), (b,j), (c,k)
//   v3s = <ij|ab> t1(c,k) + <jk|bc> t1(a,i) + <ik|ac> t1(b,j)
//   E(T) = 1/3 sum (t3s + v3s)(4 t3s + t3s(abckij) + t3s(abcjki)
//                   - 2 (t3s(abckji) + t3s(abcikj) + t3s(abcjik))) / D
// The reference stores t3 over all (a,b,c,i,j,k).  Here the occupied triples
// are visited as multisets {i <= j <= k}.
//
// FP64: t3s(a,b,c) of a block of triples is summed where it is formed, so that v^3 values
// a triple go through HBM instead of the 6 v^3 of its orderings: three launches, each of
// the two orderings that share a row pair, (a,b), (a,c) or (b,c)
// (triples_sum_kernel), then the energy.
//
// Split-precision forms of a large K = v + o: for a pair (j,k) and a block of i,
// five GEMMs build the raw W of the six orderings of each triple.  The
// particle and hole terms are one GEMM with K = v + o: A_i = [<id|ab>^T | t2(a,b,i,:)]
// ((a,b) x (v+o), built once) and B_jk = [t2(:,c,j,k) ; -<jk|:c>] ((v+o) x c).
// The orderings (i,j,k), (i,k,j) stack the block's i along M and the two B's
// along N; the four orderings led by j or k share A and put the block's i
// along N (N = nb v), so every GEMM has long M and N.
//
// Energy: t3s and v3s are invariant under the simultaneous permutation of
// (a,b,c) and (i,j,k), and the coefficients (4, 1, 1, -2, -2, -2) depend only
// on the conjugacy class of the occupied permutation, so the 36 energy terms
// of the orbit pair {a,b,c} x {i,j,k} collapse to 6 x sum_u F(u) with
//   T_u = t3s(x, y_u) = t3s(x_{u^-1}, y) = sum_r W_{u o r}(x_r),  F(u) = (T_u + V_u) sum_m c_m T_{u o m},
// x = (a >= b >= c), y = (i <= j <= k), weighted by 1/(|stab x| |stab y|) so
// that every ordered (a,b,c,i,j,k) counts once.  In the split-precision forms
// the W GEMMs read 16-bit planes of A and B (split once per call) and write
// FP64 W; the energy is FP64 throughout.  A workgroup owns a multiset
// of 8^3 cubes of (a,b,c) space and stages the six permuted cubes of t3s (of W_s, ordering
// by ordering) through LDS, so they are read with coalesced rows once.
#include <cmath>
#include <memory>
#include <stdexcept>

#include "ccsd_ctx.hpp"

namespace mpqc_hip {

namespace {

// S3 as position maps: 0 (0,1,2) 1 (0,2,1) 2 (1,0,2) 3 (1,2,0) 4 (2,0,1) 5 (2,1,0)
__constant__ int kPerm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
// kComp[p][r] = index of the map n -> p[r[n]];  kInv[r] = index of r^-1
__constant__ int kComp[6][6];
__constant__ int kInv[6];
// energy terms: t3s at occupied order (y'[m[0]], y'[m[1]], y'[m[2]]) with coefficient
// (i,j,k):4  (k,i,j):1  (j,k,i):1  (k,j,i):-2  (i,k,j):-2  (j,i,k):-2
__constant__ int kTermPerm[6] = {0, 4, 3, 5, 1, 2};
__constant__ double kTermCoef[6] = {4.0, 1.0, 1.0, -2.0, -2.0, -2.0};

// the same maps for code unrolled over them
constexpr int kPermC[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
constexpr int kInvC[6] = {0, 1, 2, 4, 3, 5};

constexpr int kT = 8;                        // cube edge
constexpr int kS2 = kT + 1, kS1 = kT * kS2 + 1;  // padded LDS strides (odd: no bank conflicts)
constexpr int kCube = kT * kS1;
constexpr int kTThreads = 256;
static_assert(6 * kT * kT * kT % kTThreads == 0 && 6 * kT * kT * kT / kTThreads <= 32, "cube staging layout");

void upload_s3_tables(hipStream_t s) {
  static const int P[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  auto index_of = [&](const int m[3]) {
    for (int q = 0; q < 6; ++q)
      if (P[q][0] == m[0] && P[q][1] == m[1] && P[q][2] == m[2]) return q;
    return -1;
  };
  int comp[6][6], inv[6];
  for (int p = 0; p < 6; ++p) {
    for (int r = 0; r < 6; ++r) {
      const int m[3] = {P[p][P[r][0]], P[p][P[r][1]], P[p][P[r][2]]};
      comp[p][r] = index_of(m);
    }
    int m[3];
    for (int n = 0; n < 3; ++n) m[P[p][n]] = n;
    inv[p] = index_of(m);
  }
  MPQC_HIP_CHECK(hipMemcpyToSymbolAsync(HIP_SYMBOL(kComp), comp, sizeof(comp), 0, hipMemcpyHostToDevice, s));
  MPQC_HIP_CHECK(hipMemcpyToSymbolAsync(HIP_SYMBOL(kInv), inv, sizeof(inv), 0, hipMemcpyHostToDevice, s));
}

__device__ inline long tet(long a) { return a * (a + 1) * (a + 2) / 6; }

// multiset number e -> (a >= b >= c)
__device__ inline void unrank3(long e, int& a, int& b, int& c) {
  long x = (long)cbrt(6.0 * (double)e);
  while (x > 0 && tet(x) > e) --x;
  while (tet(x + 1) <= e) ++x;
  const long rem = e - tet(x);
  long y = (long)((sqrt(8.0 * (double)rem + 1.0) - 1.0) * 0.5);
  while (y > 0 && y * (y + 1) / 2 > rem) --y;
  while ((y + 1) * (y + 2) / 2 <= rem) ++y;
  a = (int)x;
  b = (int)y;
  c = (int)(rem - y * (y + 1) / 2);
}

struct TriplesArgs {
  // W of ordering s for triple z of the block at (a,b,c):
  //   Wb[s] + z * Wz[s] + (a v + b) * Wr[s] + c
  const double* Wb[6];
  long Wz[6], Wr[6];
  const double* G;  // Gijab (i,j,a,b)
  const double* t1; // (a,i)
  const double* eo;
  const double* ev;
  int o, v, i0, j, k;
};

__global__ __launch_bounds__(kTThreads) void triples_energy_kernel(TriplesArgs g, double* partials) {
  __shared__ double tile[6 * kCube];
  __shared__ double red[kTThreads];
  const int z = blockIdx.y;
  const int v = g.v, o = g.o;
  int X[3];
  unrank3(blockIdx.x, X[0], X[1], X[2]);  // cube multiset A >= B >= C
  const int y[3] = {g.i0 + z, g.j, g.k};
  // this thread's two points of cube (A,B,C): local coordinates and validity
  int l[2][3];
  bool ok[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int q = threadIdx.x + h * kTThreads;
    l[h][0] = q / (kT * kT);
    l[h][1] = (q / kT) % kT;
    l[h][2] = q % kT;
    const int a = X[0] * kT + l[h][0], b = X[1] * kT + l[h][1], c = X[2] * kT + l[h][2];
    ok[h] = a < v && b < v && c < v && a >= b && b >= c;
  }
  double T[2][6];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < 6; ++u) T[h][u] = 0.0;
  // W_s cubes: every thread owns kPerThr elements of the six permuted cubes; the
  // loads of ordering s + 1 are issued before the products of ordering s, from
  // clamped addresses (out-of-range elements are zeroed at the LDS store), so they
  // stay in flight across the compute
  constexpr int kCubeEl = kT * kT * kT, kPerThr = 6 * kCubeEl / kTThreads;
  double pre[kPerThr];
  uint32_t okmask = 0;
  auto gload = [&](int s) {
    const double* Ws = g.Wb[s] + (long)z * g.Wz[s];
    const long rs = g.Wr[s];
#pragma unroll
    for (int k = 0; k < kPerThr; ++k) {
      const int e = threadIdx.x + k * kTThreads;
      const int r = e / kCubeEl, rem = e - r * kCubeEl;
      const int u = rem / (kT * kT), w = (rem / kT) % kT, zz = rem % kT;
      const int ga = X[kPerm[r][0]] * kT + u, gb = X[kPerm[r][1]] * kT + w, gc = X[kPerm[r][2]] * kT + zz;
      const bool in = ga < v && gb < v && gc < v;
      okmask = in ? (okmask | (1u << k)) : (okmask & ~(1u << k));
      pre[k] = Ws[((long)min(ga, v - 1) * v + min(gb, v - 1)) * rs + min(gc, v - 1)];
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int k = 0; k < kPerThr; ++k) {
      const int e = threadIdx.x + k * kTThreads;
      const int r = e / kCubeEl, rem = e - r * kCubeEl;
      const int u = rem / (kT * kT), w = (rem / kT) % kT, zz = rem % kT;
      tile[r * kCube + u * kS1 + w * kS2 + zz] = ((okmask >> k) & 1u) ? pre[k] : 0.0;
    }
  };
  gload(0);
  for (int s = 0; s < 6; ++s) {
    lstore();
    __syncthreads();
    if (s + 1 < 6) gload(s + 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!ok[h]) continue;
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        // x_r lies in cube r at local (l[r0], l[r1], l[r2]); W_s(x_r) adds to T_{s o r^-1}
        const double val = tile[r * kCube + l[h][kPerm[r][0]] * kS1 + l[h][kPerm[r][1]] * kS2 + l[h][kPerm[r][2]]];
        T[h][kComp[s][kInv[r]]] += val;
      }
    }
    __syncthreads();
  }
  double acc = 0.0;
  const int sy = (y[0] == y[1] && y[1] == y[2]) ? 6 : (y[0] == y[1] || y[1] == y[2]) ? 2 : 1;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (!ok[h]) continue;
    const int x[3] = {X[0] * kT + l[h][0], X[1] * kT + l[h][1], X[2] * kT + l[h][2]};
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      const int i0 = y[kPerm[u][0]], i1 = y[kPerm[u][1]], i2 = y[kPerm[u][2]];
      // v3s(x, y_u) with g_abij(a,b,i,j) = Gijab(i,j,a,b)
      const double vs = g.G[(((long)i0 * o + i1) * v + x[0]) * v + x[1]] * g.t1[(long)x[2] * o + i2] +
                        g.G[(((long)i1 * o + i2) * v + x[1]) * v + x[2]] * g.t1[(long)x[0] * o + i0] +
                        g.G[(((long)i0 * o + i2) * v + x[0]) * v + x[2]] * g.t1[(long)x[1] * o + i1];
      double Xm = 0.0;
#pragma unroll
      for (int m = 0; m < 6; ++m) Xm += kTermCoef[m] * T[h][kComp[u][kTermPerm[m]]];
      sum += (T[h][u] + vs) * Xm;
    }
    const int sx = (x[0] == x[1] && x[1] == x[2]) ? 6 : (x[0] == x[1] || x[1] == x[2]) ? 2 : 1;
    const double D = g.eo[y[0]] + g.eo[y[1]] + g.eo[y[2]] - g.ev[x[0]] - g.ev[x[1]] - g.ev[x[2]];
    acc += 2.0 * sum / (D * (double)(sx * sy));  // 6 sum_u F(u) / (3 D |stab x| |stab y|)
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kTThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[(long)blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// The same energies from t3s, for the block's triples z0 + z: a workgroup owns a cube multiset,
// t3s(x_r) of its six permuted cubes is T_{r^-1}.  Bound: HBM, v^3 reads a triple, if the vector
// ALU is kept off it: cubes and triples come from tables, a thread's offset inside a cube is one
// for all six (cubes past the edge aside) and the V terms' 18 factors of a point are read once.
// o = 20, v = 76, 119 triples: 323 us without these three, 138 us with.
struct TripleEnergyArgs {
  const double* t;         // t3s of triple z at t + z v^3
  const uint64_t* cubes;   // A | B << 21 | C << 42, A >= B >= C
  const uint64_t* triples; // i | j << 21 | k << 42, i <= j <= k, the block's first on
  const double* G;         // Gijab (i,j,a,b)
  const double* t1;        // (a,i)
  const double* eo;
  const double* ev;
  int o, v, ncube, n;  // n: triples of the block
};

__global__ __launch_bounds__(kTThreads) void triples_energy_sum_kernel(TripleEnergyArgs g, double* partials) {
  __shared__ double tile[6 * kCube];
  __shared__ double Gs[18 * 64], t1s[3][kT][3], evs[3][kT], red[kTThreads / 64];
  static_assert(kTThreads == 256 && kT == 8, "two half cubes a thread");
  const int v = g.v, o = g.o;
  // workgroup w runs on XCD w % 8: a triple's cubes all on one, whose L2 then serves the second
  // halves of the 128-byte lines that a cube's 64-byte rows use
  const int q8 = blockIdx.x / 8, zq = q8 / g.ncube, cube = q8 - zq * g.ncube, z = 8 * zq + (int)(blockIdx.x % 8);
  if (z >= g.n) return;
  const uint64_t cu = g.cubes[cube], tr = g.triples[z];
  const int X[3] = {(int)(cu & 0x1fffff), (int)(cu >> 21 & 0x1fffff), (int)(cu >> 42)};
  const int y[3] = {(int)(tr & 0x1fffff), (int)(tr >> 21 & 0x1fffff), (int)(tr >> 42)};
  const double* const t = g.t + (long)z * v * v * v;
  // this thread's points (lu, lw, lz) and (lu + 4, lw, lz) of a cube
  const int lu = threadIdx.x >> 6, lw = threadIdx.x >> 3 & 7, lz = threadIdx.x & 7;
  double pre[6][2];
  if ((X[0] + 1) * kT <= v) {  // (X[0] is the largest)
    const long off = ((long)lu * v + lw) * v + lz, half = 4l * v * v;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      const double* p = t + (((long)X[kPermC[r][0]] * v + X[kPermC[r][1]]) * v + X[kPermC[r][2]]) * kT;
      pre[r][0] = p[off];
      pre[r][1] = p[off + half];
    }
  } else {
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      const int a = X[kPermC[r][0]] * kT + lu, b = X[kPermC[r][1]] * kT + lw, c = X[kPermC[r][2]] * kT + lz;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool in = a + 4 * h < v && b < v && c < v;
        const double x = t[((long)min(a + 4 * h, v - 1) * v + min(b, v - 1)) * v + min(c, v - 1)];
        pre[r][h] = in ? x : 0.0;
      }
    }
  }
  // Gs[6 q + p][8x8]: Gijab(y_n, y_m) for the p-th ordered pair n != m, at (x_0, x_1), (x_1, x_2) or
  // (x_0, x_2) for q = 0, 1, 2; t1s[n][.][m] = t1(x_n, y_m)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  double gpre[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const int s = wave + 4 * k, q = s / 6, p = s - 6 * q;
    if (s >= 18) break;
    const int n = p >> 1, m = n == 0 ? 1 + (p & 1) : n == 1 ? 2 * (p & 1) : (p & 1);
    const int yn = n == 0 ? y[0] : n == 1 ? y[1] : y[2], ym = m == 0 ? y[0] : m == 1 ? y[1] : y[2];
    const int xr = min((q == 1 ? X[1] : X[0]) * kT + (lane >> 3), v - 1);
    const int xc = min((q == 0 ? X[1] : X[2]) * kT + (lane & 7), v - 1);
    gpre[k] = g.G[((long)yn * o + ym) * v * v + xr * v + xc];
  }
  if (threadIdx.x < 24) {
    const int n = threadIdx.x >> 3, xn = min((n == 0 ? X[0] : n == 1 ? X[1] : X[2]) * kT + (int)(threadIdx.x & 7), v - 1);
    evs[n][threadIdx.x & 7] = g.ev[xn];
#pragma unroll
    for (int m = 0; m < 3; ++m) t1s[n][threadIdx.x & 7][m] = g.t1[xn * o + y[m]];
  }
#pragma unroll
  for (int k = 0; k < 5; ++k)
    if (wave + 4 * k < 18) Gs[(wave + 4 * k) * 64 + lane] = gpre[k];
  const int dst = lu * kS1 + lw * kS2 + lz;
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int h = 0; h < 2; ++h) tile[r * kCube + dst + 4 * h * kS1] = pre[r][h];
  __syncthreads();
  const int sy = (y[0] == y[1] && y[1] == y[2]) ? 6 : (y[0] == y[1] || y[1] == y[2]) ? 2 : 1;
  const double e_occ = g.eo[y[0]] + g.eo[y[1]] + g.eo[y[2]];
  double acc = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int l[3] = {lu + 4 * h, lw, lz};
    const int x[3] = {X[0] * kT + l[0], X[1] * kT + l[1], X[2] * kT + l[2]};
    if (x[0] >= v || x[1] > x[0] || x[2] > x[1]) continue;
    double T[6];
#pragma unroll
    for (int r = 0; r < 6; ++r)
      T[kInvC[r]] = tile[r * kCube + l[kPermC[r][0]] * kS1 + l[kPermC[r][1]] * kS2 + l[kPermC[r][2]]];
    // sum_m c_m T_{u o m} = 3 T_u + (sum of u's class) - 2 (sum of the other class): the
    // coefficients are 4, 1, 1 on the even maps from u and -2 on the odd ones
    const double even = T[0] + T[3] + T[4], odd = T[1] + T[2] + T[5];
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      constexpr bool kEven[6] = {true, false, false, true, true, false};
      const int i0 = kPermC[u][0], i1 = kPermC[u][1], i2 = kPermC[u][2];
      auto G = [&](int q, int n, int m, int a, int b) {  // pair (n, m) is the 2 n + (m > n ? m - 1 : m)-th
        return Gs[(6 * q + 2 * n + (m > n ? m - 1 : m)) * 64 + 8 * a + b];
      };
      const double vs = G(0, i0, i1, l[0], l[1]) * t1s[2][l[2]][i2] + G(1, i1, i2, l[1], l[2]) * t1s[0][l[0]][i0] +
                        G(2, i0, i2, l[0], l[2]) * t1s[1][l[1]][i1];
      sum += (T[u] + vs) * (3.0 * T[u] + (kEven[u] ? even - 2.0 * odd : odd - 2.0 * even));
    }
    const int sx = (x[0] == x[1] && x[1] == x[2]) ? 6 : (x[0] == x[1] || x[1] == x[2]) ? 2 : 1;
    const double D = e_occ - evs[0][l[0]] - evs[1][l[1]] - evs[2][l[2]];
    acc += 2.0 * sum / (D * (double)(sx * sy));  // 6 sum_u F(u) / (3 D |stab x| |stab y|)
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) acc += __shfl_down(acc, w);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partials[(long)z * g.ncube + cube] = red[0] + red[1] + red[2] + red[3];
}

// t3s of the block's triples: the two orderings of PART that share the row pair,
//   0  t(a,b,c)  = A_i[(a,b)] B_jk[c] + A'_j[(a,b)] B_ik[c]
//   1  t(a,b,c) += A_i[(a,c)] B_kj[b] + A'_k[(a,c)] B_ij[b]
//   2  t(a,b,c) += A_j[(b,c)] B_ki[a] + A'_k[(b,c)] B_ji[a]
// with A_i[(x,y)][K] = [<id|xy> | t2(x,y,i,:)], A'_i[(x,y)] = A_i[(y,x)] and
// B_jk[z][K] = [t2(:,z,j,k) | -<jk|:z>], rows of pitch K = v + o padded with zeros to a
// multiple of 16, so that no slice of K is partial.  A workgroup's tile: 64 RB rows (x,y),
// 16 CB columns z of one triple; the FP64 tile of the general contraction (A fragments
// straight from global memory one slice ahead, B double buffered in LDS, products of a step
// on fragments read a step ahead) with a second pair of operands after the first.  PART 1
// and 2 run the products transposed, so that 16 lanes hold consecutive rows and store to
// consecutive addresses of t.
// Bound: the matrix cores (2 x 2 v^3 (v + o) flops a triple and part) with the v^3 values
// written, or read and written, behind them.  Workgroups of one XCD take a run of row tiles,
// triples fastest: the o A's of a row tile stay in that XCD's L2 (2 MB at o = 20, v = 76).
// o = 20, v = 76: 360, 385 and 413 us a part of 119 triples (2.0e10 flops each, 55 to 48 TFLOP/s); all
// of (T) 40.2 ms with a GEMM and a stored W an ordering, 17.2 ms so.  Tried and dropped: 128
// rows a tile (383 to 477 us), blocks of 64 MB that stay in the last-level cache (8 % slower).
struct TripleSumArgs {
  const double* A;
  const double* As;
  const double* B;
  double* t;
  int o, v, pitch;
  const uint64_t* list;  // the block's triples, as in TripleEnergyArgs
  int triples, tiles_m, tiles_n;
  long per_xcd;
};

template <int PART, int RB, int CB>
__global__ __launch_bounds__(256, 2) void triples_sum_kernel(TripleSumArgs g) {
  typedef double vec2 __attribute__((ext_vector_type(2)));
  constexpr int BK = 16, BN = 16 * CB, PITCH = BK + 2, STAGE = BN * PITCH;
  constexpr int kStep = 32, PER = (BN + kStep - 1) / kStep;  // 8 threads of 16 bytes a row of B
  __shared__ __attribute__((aligned(16))) double Bs[2 * STAGE];
  const long idx = (long)(blockIdx.x % 8) * g.per_xcd + blockIdx.x / 8;
  if (idx >= (long)g.triples * g.tiles_m * g.tiles_n) return;
  const int z = (int)(idx % g.triples), tile = (int)(idx / g.triples);
  const int tm = tile / g.tiles_n, tn = tile - tm * g.tiles_n;
  const int v = g.v, o = g.o, vv = v * v, K = g.pitch;
  const uint64_t tr = g.list[z];
  const int i = (int)(tr & 0x1fffff), j = (int)(tr >> 21 & 0x1fffff), k = (int)(tr >> 42);
  const long sa = (long)vv * K, sb = (long)v * K;
  const double* const A1 = g.A + (PART == 2 ? j : i) * sa;
  const double* const A2 = g.As + (PART == 0 ? j : k) * sa;
  const double* const B1 = g.B + (PART == 0 ? j * o + k : PART == 1 ? k * o + j : k * o + i) * sb;
  const double* const B2 = g.B + (PART == 0 ? i * o + k : PART == 1 ? i * o + j : j * o + i) * sb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int m0 = tm * 64 * RB + wave * RB * 16, n0 = tn * BN;

  long aoff[RB];  // rows and columns past the edge read the last ones
#pragma unroll
  for (int q = 0; q < RB; ++q) aoff[q] = (long)min(m0 + 16 * q + lr, vv - 1) * K + 4 * lk;
  long boff[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) boff[r] = (long)min(n0 + tid / 8 + kStep * r, v - 1) * K + 2 * (tid % 8);
  double* const bdst = Bs + (tid / 8) * PITCH + 2 * (tid % 8);

  // where this lane's accumulators [q][jn][r] go: row m, column n of the tile
  long base[RB];
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    const int m = m0 + 16 * q + (PART == 0 ? lk : lr), n = n0 + (PART == 0 ? lr : lk), x = m / v;
    base[q] = (long)z * vv * v + (PART == 0   ? (long)m * v + n                           // (a,b),c
                                  : PART == 1 ? (long)x * vv + (m - x * v) + (long)n * v  // a,b,c from (a,c),b
                                              : m + (long)n * vv);                        // a,(b,c)
  }
  auto inside = [&](int q, int jn, int r) {
    return PART == 0 ? m0 + 16 * q + 4 * r + lk < vv && n0 + 16 * jn + lr < v
                     : m0 + 16 * q + lr < vv && n0 + 16 * jn + 4 * r + lk < v;
  };
  auto step = [&](int jn, int r) -> long {
    return PART == 0 ? 4l * r * v + 16 * jn : (16l * jn + 4 * r) * (PART == 1 ? v : vv);
  };
  double4_t acc[RB][CB];
#pragma unroll
  for (int q = 0; q < RB; ++q)
#pragma unroll
    for (int jn = 0; jn < CB; ++jn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[q][jn][r] = 0.0;
        // (the sum so far is on its way while the first slices are)
        if (PART > 0 && inside(q, jn, r)) acc[q][jn][r] = g.t[base[q] + step(jn, r)];
      }

  double an[RB][4], a[RB][4], fb[2][CB][2];
  vec2 bn[PER];
  const double *ap = A1, *bp = B1;
  auto load = [&]() {
#pragma unroll
    for (int q = 0; q < RB; ++q) {
      const vec2 x = *reinterpret_cast<const vec2*>(ap + aoff[q]);
      const vec2 y = *reinterpret_cast<const vec2*>(ap + aoff[q] + 2);
      an[q][0] = x[0];
      an[q][1] = x[1];
      an[q][2] = y[0];
      an[q][3] = y[1];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) bn[r] = *reinterpret_cast<const vec2*>(bp + boff[r]);
    ap += BK;
    bp += BK;
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int r = 0; r < PER; ++r)
      if (BN % kStep == 0 || tid / 8 + kStep * r < BN)
        *reinterpret_cast<vec2*>(bdst + buf * STAGE + kStep * r * PITCH) = bn[r];
  };
  auto read_b = [&](int buf, int step, double (&f)[CB][2]) {
    const double* bs = Bs + buf * STAGE + lr * PITCH + 4 * lk + 2 * step;
#pragma unroll
    for (int jn = 0; jn < CB; ++jn) {
      const vec2 x = *reinterpret_cast<const vec2*>(bs + 16 * jn * PITCH);
      f[jn][0] = x[0];
      f[jn][1] = x[1];
    }
  };
  auto products = [&](int step) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < RB; ++q)
#pragma unroll
        for (int jn = 0; jn < CB; ++jn) {
          const double x = a[q][2 * step + h], y = fb[step][jn][h];
          acc[q][jn] = __builtin_amdgcn_mfma_f64_16x16x4f64(PART == 0 ? x : y, PART == 0 ? y : x, acc[q][jn], 0, 0, 0);
        }
  };
  const int half = K / BK, nslices = 2 * half;
  load();
  store_b(0);
  __syncthreads();
  read_b(0, 0, fb[0]);
#pragma unroll
  for (int q = 0; q < RB; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) a[q][e] = an[q][e];
  int buf = 0;
  for (int s = 0; s < nslices; ++s) {
    const bool has_next = s + 1 < nslices;
    if (s + 1 == half) {
      ap = A2;
      bp = B2;
    }
    if (has_next) load();
    read_b(buf, 1, fb[1]);
    __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the products
    products(0);
    if (has_next) store_b(buf ^ 1);
    __syncthreads();
    buf ^= 1;
    if (has_next) read_b(buf, 0, fb[0]);
    __builtin_amdgcn_sched_barrier(0);
    products(1);
#pragma unroll
    for (int q = 0; q < RB; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[q][e] = an[q][e];
  }
#pragma unroll
  for (int q = 0; q < RB; ++q)
#pragma unroll
    for (int jn = 0; jn < CB; ++jn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (inside(q, jn, r)) g.t[base[q] + step(jn, r)] = acc[q][jn][r];
}

template <int RB, int CB>
void launch_triples_sum(const TripleSumArgs& args, hipStream_t s) {
  TripleSumArgs g = args;
  g.tiles_m = (int)ceil_div((long)g.v * g.v, 64 * RB);
  g.tiles_n = (int)ceil_div(g.v, 16 * CB);
  g.per_xcd = ceil_div((long)g.triples * g.tiles_m * g.tiles_n, 8);
  const dim3 grid((unsigned)(8 * g.per_xcd));
  hipLaunchKernelGGL((triples_sum_kernel<0, RB, CB>), grid, dim3(256), 0, s, g);
  hipLaunchKernelGGL((triples_sum_kernel<1, RB, CB>), grid, dim3(256), 0, s, g);
  hipLaunchKernelGGL((triples_sum_kernel<2, RB, CB>), grid, dim3(256), 0, s, g);
  check_launch("triples_sum");
}

// Columns in equal tiles of at most 144, so that v is not padded to a power of two
void triples_sum(const TripleSumArgs& g, hipStream_t s) {
  const int blocks = (int)ceil_div(g.v, 16), tiles = (int)ceil_div(blocks, 9);
  switch (ceil_div(blocks, tiles)) {
    case 1: return launch_triples_sum<1, 1>(g, s);
    case 2: return launch_triples_sum<1, 2>(g, s);
    case 3: return launch_triples_sum<1, 3>(g, s);
    case 4: return launch_triples_sum<1, 4>(g, s);
    case 5: return launch_triples_sum<1, 5>(g, s);
    case 6: return launch_triples_sum<1, 6>(g, s);
    case 7: return launch_triples_sum<1, 7>(g, s);
    case 8: return launch_triples_sum<1, 8>(g, s);
    default: return launch_triples_sum<1, 9>(g, s);
  }
}

// Whether the split-precision forms' (T) takes the FP64 sums too: planes cut the products' time,
// which grows with K = v + o (in steps of 16), but every ordering's W still goes through HBM.  From
// K = 145 to 160 the two are within 10 %, and planes are the faster where their blocks are long
// (o > 20), tiles are filled (v >= 96) and rows of W start on 32 bytes (v a multiple of 4).  FP64 sums
// against W from fp16 planes, ms, (o, v) = (20, 76) 17 : 38, (24, 110) 113 : 146, (40, 104) 439 : 492, (56, 88)
// 747 : 829, (16, 144) 90 : 94, (20, 140) 157 : 163, (31, 129) 477 : 517, (50, 110) 1097 : 1165, (100, 60) 1450 :
// 1786; (24, 136) 250 : 240, (32, 120) 398 : 380, (40, 120) 764 : 696, (60, 100) 1504 : 1441; (12, 190) 115 : 104,
// (40, 152) 1750 : 1360.  bf16x6, with twice the plane products: (30, 130) 441 : 616, (60, 100) 1472 : 2048.
bool summed_faster(long o, long v, GemmPrecision prec) {
  const long K = v + o;
  if (K <= 144) return true;
  return K <= 160 && (prec == GemmPrecision::BF16X6 || !(o > 20 && v >= 96 && v % 4 == 0));
}

// acc[slot + block] = the block's run of partials[0..n), each summed in a fixed order
constexpr int kSumBlocks = 32;
__global__ __launch_bounds__(256) void sum_to_slot(const double* partials, long n, double* acc, long slot) {
  __shared__ double sh[256];
  double s = 0.0;
  const long run = (n + gridDim.x - 1) / gridDim.x, end = min(n, run * (blockIdx.x + 1));
  for (long e = run * blockIdx.x + threadIdx.x; e < end; e += 256) s += partials[e];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) acc[slot + blockIdx.x] = sh[0];
}

// planes of one (T) operand, owned for the duration of the call
struct TPlanes {
  Planes P;
  std::vector<std::unique_ptr<ScratchBuf>> owned;
  TPlanes(ScratchCache& scratch, PlaneKind kind, long rows, long row, hipStream_t stream) {
    if (plane_pitch(row) != row) {
      P.row = row;
      P.pitch = plane_pitch(row);
    }
    const long n = rows * plane_pitch(row);
    P.n = n;
    for (int q = 0; q < plane_count(kind); ++q) {
      owned.emplace_back(new ScratchBuf(scratch, (size_t)ceil_div(std::max<long>(n, 8), 4)));
      P.p[q] = (uint16_t*)owned.back()->p;
      if (P.row) MPQC_HIP_CHECK(hipMemsetAsync(P.p[q], 0, (size_t)n * sizeof(uint16_t), stream));  // the gaps stay 0
    }
    owned.emplace_back(new ScratchBuf(scratch, 1));
    P.scale = owned.back()->p;
  }
  // the same planes starting at element `off` (a whole number of rows)
  Planes at(long off) const {
    Planes q = P;
    off = P.at(off);
    for (int k = 0; k < 3; ++k)
      if (q.p[k]) q.p[k] += off;
    q.n = P.n - off;
    return q;
  }
};

long energy_cubes(long v) {
  const long nB = ceil_div(v, kT);
  return nB * (nB + 1) * (nB + 2) / 6;
}

// out (dense, extents out_ext) = alpha * input permuted (out axis d reads input axis perm[d])
void permute_into(double* out, const long out_ext[4], const double* in, const long in_ext[4], const int perm[4],
                  double alpha, hipStream_t s) {
  TTerm t;
  t.p = in;
  permuted_strides(in_ext, perm, t.s);
  t.alpha = alpha;
  t.vol = in_ext[0] * in_ext[1] * in_ext[2] * in_ext[3];
  tadd(out, out_ext, 0.0, &t, 1, s);
}

}  // namespace

// Giabc(i,a,b,c) = <ia|bc> = (ib|ac) = sum_K Xai(K,b,i) Xab(K,a,c) for the df
// method without a stored Giabc (the reference's get_abci with "[df]",
// ccsd_t.h:2224-2234, through compute4's density-fitted branch)
void CCSDContext::ensure_iabc_for_triples() {
  if ((have_ints_ >> 6) & 1u) return;
  if (!df_) throw std::logic_error("(T) needs Giabc");
  const long Q = naux_, O = o_, V = v_;
  ScratchBuf T(scratch_, (size_t)(O * V * V * V));
  // T[(i,b)][(a,c)] = Xia(K,(i,b))^T Xab(K,(a,c)) ; Giabc(i,a,b,c) = T(i,b,a,c)
  mpqc_hip::gemm(make_gemm(true, false, (int)(O * V), (int)(V * V), (int)Q, 1.0, Xia_, O * V, Xab_, V * V, 0.0,
                           T.p, V * V), GemmPrecision::F64, ws_, stream_);
  const long ext[4] = {O, V, V, V};
  const int pm[4] = {0, 2, 1, 3};
  permute_into(Giabc_, ext, T.p, ext, pm, 1.0, stream_);
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  have_ints_ |= 1u << 6;
}

// The FP64 sums: energies of the blocks' partial sums, in order
std::vector<double> CCSDContext::triples_summed(double block_bytes) {
  const long O = o_, V = v_, v3 = V * V * V, VK = V + O, pitch = ceil_div(VK, 16) * 16;
  const long ncube = energy_cubes(V), total = O * (O + 1) * (O + 2) / 6;
  // triples a block: as many t3s as fit (at most the memory of one (j,k)'s six orderings, beyond
  // which the launches are long enough), in blocks of equal size within the energy's 2^24 workgroups
  // (2^32 threads of a launch)
  long T = std::max(1L, std::min({(long)(block_bytes / (sizeof(double) * (double)v3)), 6 * O, total,
                                  (1L << 24) / ncube - 8}));
  const long nchunks = ceil_div(total, T);
  T = ceil_div(total, nchunks);
  const size_t d = sizeof(double);
  ScratchBuf A(scratch_, (size_t)(O * V * V * pitch)), As(scratch_, (size_t)(O * V * V * pitch)),
      B(scratch_, (size_t)(O * O * V * pitch)), W(scratch_, (size_t)(T * v3));
  {
    // The operands' parts go through a temporary a few occupied orbitals at a time: with one for
    // all of o v^3, the two A's would take more memory than one A and the W of every ordering,
    // and fewer orbitals would fit the device.  128 MiB of it cost no time (at o = 20, v = 76 it holds
    // all orbitals).
    const long per = V * std::max(V, O) * std::max(V, O), step = std::max(1L, std::min(O, (16L << 20) / per));
    ScratchBuf tmp(scratch_, (size_t)(step * per));
    if (pitch != VK) {
      fill(A.p, O * V * V * pitch, 0.0, stream_);
      fill(B.p, O * O * V * pitch, 0.0, stream_);
    }
    auto rows = [&](double* dst, long n, long width) {  // dst rows of `pitch` take tmp's rows of `width`
      MPQC_HIP_CHECK(hipMemcpy2DAsync(dst, pitch * d, tmp.p, width * d, width * d, n, hipMemcpyDeviceToDevice, stream_));
    };
    const long e_iabc[4] = {O, V, V, V}, e_t2[4] = {V, V, O, O}, e_ijka[4] = {O, O, O, V};
    const int pa1[4] = {0, 2, 3, 1}, pa2[4] = {2, 0, 1, 3}, pb1[4] = {2, 3, 1, 0}, pb2[4] = {0, 1, 3, 2};
    for (long i0 = 0; i0 < O; i0 += step) {
      const long n = std::min(step, O - i0);
      // A[i][(a,b)][d] = Giabc(i,d,a,b), [v + l] = t2(a,b,i,l)
      const long e_a1[4] = {n, V, V, V}, e_a2[4] = {n, V, V, O};
      double* const a = A.p + i0 * V * V * pitch;
      permute_into(tmp.p, e_a1, Giabc_ + i0 * v3, e_iabc, pa1, 1.0, stream_);
      rows(a, n * V * V, V);
      permute_into(tmp.p, e_a2, t2_ + i0 * O, e_t2, pa2, 1.0, stream_);
      rows(a + V, n * V * V, O);
      // B[j][k][c][d] = t2(d,c,j,k), [v + l] = -Gijka(j,k,l,c)
      const long e_b1[4] = {n, O, V, V}, e_b2[4] = {n, O, V, O};
      double* const b = B.p + i0 * O * V * pitch;
      permute_into(tmp.p, e_b1, t2_ + i0 * O, e_t2, pb1, 1.0, stream_);
      rows(b, n * O * V, V);
      permute_into(tmp.p, e_b2, Gijka_ + i0 * O * O * V, e_ijka, pb2, -1.0, stream_);
      rows(b + V, n * O * V, O);
    }
    const long e_a[4] = {O, V, V, pitch};
    const int psw[4] = {0, 2, 1, 3};
    permute_into(As.p, e_a, A.p, e_a, psw, 1.0, stream_);
  }
  // tables of the cube and triple multisets
  const long nB = ceil_div(V, kT);
  std::vector<uint64_t> table((size_t)(ncube + total));
  size_t e = 0;
  for (long a = 0; a < nB; ++a)
    for (long b = 0; b <= a; ++b)
      for (long c = 0; c <= b; ++c) table[e++] = (uint64_t)(a | b << 21 | c << 42);
  for (long k = 0; k < O; ++k)
    for (long j = 0; j <= k; ++j)
      for (long i = 0; i <= j; ++i) table[e++] = (uint64_t)(i | j << 21 | k << 42);
  ScratchBuf tables(scratch_, table.size());
  uint64_t* const cubes = reinterpret_cast<uint64_t*>(tables.p);
  MPQC_HIP_CHECK(hipMemcpyAsync(cubes, table.data(), table.size() * sizeof(uint64_t), hipMemcpyHostToDevice, stream_));
  ScratchBuf partials(scratch_, (size_t)(ncube * T)), acc(scratch_, (size_t)(nchunks * kSumBlocks));
  for (long c = 0; c < nchunks; ++c) {
    const long z0 = c * T, n = std::min(T, total - z0);
    if (n <= 0) {  // (equal blocks can leave the last ones empty)
      fill(acc.p + c * kSumBlocks, kSumBlocks, 0.0, stream_);
      continue;
    }
    const uint64_t* list = cubes + ncube + z0;
    TripleSumArgs w{A.p, As.p, B.p, W.p, o_, v_, (int)pitch, list, (int)n, 0, 0, 0};
    triples_sum(w, stream_);
    const TripleEnergyArgs g{W.p, cubes, list, Gijab_, t1_, eo_, ev_, o_, v_, (int)ncube, (int)n};
    hipLaunchKernelGGL(triples_energy_sum_kernel, dim3((unsigned)(ncube * ceil_div(n, 8) * 8)), dim3(kTThreads), 0, stream_, g,
                       partials.p);
    hipLaunchKernelGGL(sum_to_slot, dim3(kSumBlocks), dim3(256), 0, stream_, partials.p, ncube * n, acc.p,
                       c * kSumBlocks);
    check_launch("triples_energy");
  }
  std::vector<double> h((size_t)(nchunks * kSumBlocks));
  MPQC_HIP_CHECK(hipMemcpyAsync(h.data(), acc.p, h.size() * d, hipMemcpyDeviceToHost, stream_));
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  return h;
}

// The split-precision forms of a large K: the same, from the W of every ordering
std::vector<double> CCSDContext::triples_orderings(double block_bytes) {
  const int o = o_, v = v_;
  const long O = o, V = v, v3 = V * V * V, VK = V + O;
  const long ncube = energy_cubes(V);
  upload_s3_tables(stream_);
  long nbmax = (long)(block_bytes / (6.0 * sizeof(double) * (double)v3));
  nbmax = std::max(1L, std::min(nbmax, O));
  // GEMM operands with K = v + o:
  //   Acat(i, (a,b), K)   = [<id|ab> for K = d < v | t2(a,b,i,l) for K = v + l]
  //   Bcat(j, k, K, c)    = [t2(d,c,j,k)           | -<jk|lc>]
  // and three layouts of Bcat that make the N dimension of each GEMM long:
  //   Bt (K, j, k, c), Bt2 (K, k, j, c) = Bcat(j, k, K, c), Bp (j, k, K, 2, c) = [Bcat(j,k) | Bcat(k,j)]
  const size_t d = sizeof(double);
  ScratchBuf Acat(scratch_, (size_t)(O * V * V * VK)), Bt(scratch_, (size_t)(VK * O * O * V)),
      Bt2(scratch_, (size_t)(VK * O * O * V)), Bp(scratch_, (size_t)(2 * O * O * VK * V)),
      W(scratch_, (size_t)(6 * nbmax * v3));
  {
    ScratchBuf tmp(scratch_, (size_t)(O * V * V * std::max(V, O)));
    // Acat[i][(a,b)][d] = Giabc(i,d,a,b); Acat[i][(a,b)][v + l] = t2(a,b,i,l)
    const long e_iabc[4] = {O, V, V, V};
    const int p1[4] = {0, 2, 3, 1};
    permute_into(tmp.p, e_iabc, Giabc_, e_iabc, p1, 1.0, stream_);
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Acat.p, VK * d, tmp.p, V * d, V * d, O * V * V, hipMemcpyDeviceToDevice,
                                    stream_));
    const long e_t2[4] = {V, V, O, O};
    const int p2[4] = {2, 0, 1, 3};
    const long ext2[4] = {O, V, V, O};
    permute_into(tmp.p, ext2, t2_, e_t2, p2, 1.0, stream_);
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Acat.p + V, VK * d, tmp.p, O * d, O * d, O * V * V, hipMemcpyDeviceToDevice,
                                    stream_));
    // Bcat[j][k][d][c] = t2(d,c,j,k); Bcat[j][k][v + l][c] = -Gijka(j,k,l,c)
    ScratchBuf Bcat(scratch_, (size_t)(O * O * VK * V)), tmp2(scratch_, (size_t)(O * O * std::max(V, O) * V));
    const int p3[4] = {2, 3, 0, 1};
    const long ext3[4] = {O, O, V, V};
    permute_into(tmp2.p, ext3, t2_, e_t2, p3, 1.0, stream_);
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Bcat.p, VK * V * d, tmp2.p, V * V * d, V * V * d, O * O,
                                    hipMemcpyDeviceToDevice, stream_));
    const long e_ijka[4] = {O, O, O, V};
    const int pid[4] = {0, 1, 2, 3};
    permute_into(tmp2.p, e_ijka, Gijka_, e_ijka, pid, -1.0, stream_);
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Bcat.p + V * V, VK * V * d, tmp2.p, O * V * d, O * V * d, O * O,
                                    hipMemcpyDeviceToDevice, stream_));
    const long e_b[4] = {O, O, VK, V};
    const int pt[4] = {2, 0, 1, 3}, pt2[4] = {2, 1, 0, 3}, psw[4] = {1, 0, 2, 3};
    const long e_bt[4] = {VK, O, O, V};
    permute_into(Bt.p, e_bt, Bcat.p, e_b, pt, 1.0, stream_);
    permute_into(Bt2.p, e_bt, Bcat.p, e_b, pt2, 1.0, stream_);
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Bp.p, 2 * V * d, Bcat.p, V * d, V * d, O * O * VK, hipMemcpyDeviceToDevice,
                                    stream_));
    ScratchBuf BcatT(scratch_, (size_t)(O * O * VK * V));
    permute_into(BcatT.p, e_b, Bcat.p, e_b, psw, 1.0, stream_);  // BcatT(j,k) = Bcat(k,j)
    MPQC_HIP_CHECK(hipMemcpy2DAsync(Bp.p + V, 2 * V * d, BcatT.p, V * d, V * d, O * O * VK,
                                    hipMemcpyDeviceToDevice, stream_));
  }
  // split-precision forms: the W GEMMs read 16-bit planes of the operands in
  // k-contiguous layout (A as is; B transposed to [c][K] rows), split once here
  const PlaneKind kind = plane_kind();
  const long VKp = plane_pitch(VK);
  TPlanes Ap(scratch_, kind, O * V * V, VK, stream_), BTp(scratch_, kind, O * O * V, VK, stream_),
      BT2p(scratch_, kind, O * O * V, VK, stream_), BPp(scratch_, kind, O * O * 2 * V, VK, stream_);
  size_t wsP_bytes = 0;
  {
    auto split1 = [&](const Planes& out, const long out_ext[4], const double* src, const long in_ext[4],
                      const int perm[4]) {
      TTerm t;
      t.p = src;
      permuted_strides(in_ext, perm, t.s);
      t.alpha = 1.0;
      t.vol = in_ext[0] * in_ext[1] * in_ext[2] * in_ext[3];
      split_to_planes(kind, out, out_ext, &t, 1, partials_, stream_);
    };
    const long e_a[4] = {1, O, V * V, VK};
    const int pid[4] = {0, 1, 2, 3};
    split1(Ap.P, e_a, Acat.p, e_a, pid);
    const long e_bt[4] = {VK, O, O, V}, e_bto[4] = {O, O, V, VK};
    const int p_bt[4] = {1, 2, 3, 0}, p_bt2[4] = {2, 1, 3, 0};
    split1(BTp.P, e_bto, Bt.p, e_bt, p_bt);    // [o2][o3][c][K]
    split1(BT2p.P, e_bto, Bt.p, e_bt, p_bt2);  // [o3][o2][c][K]
    const long e_bp[4] = {O, O, VK, 2 * V}, e_bpo[4] = {O, O, 2 * V, VK};
    const int p_bp[4] = {0, 1, 3, 2};
    split1(BPp.P, e_bpo, Bp.p, e_bp, p_bp);    // [j][k][(t,c)][K]
    for (long nb = 1; nb <= nbmax; ++nb) {
      wsP_bytes = std::max(wsP_bytes, gemm_planes_workspace_bytes((int)(nb * V * V), (int)(2 * V), (int)VKp, 1));
      wsP_bytes = std::max(wsP_bytes, gemm_planes_workspace_bytes((int)(V * V), (int)(nb * V), (int)VKp, 1));
    }
  }
  ScratchBuf wsP(scratch_, (wsP_bytes + sizeof(double) - 1) / sizeof(double));
  auto plane_gemm = [&](int M, int N, const Planes& A, const Planes& B, double* C, long ldc) {
    PlaneGemmDesc dg;
    dg.kind = kind;
    dg.M = M; dg.N = N; dg.K = (int)VKp; dg.alpha = 1.0; dg.beta = 0.0;
    dg.A = A; dg.lda = VKp; dg.sA = 0; dg.B = B; dg.ldb = VKp; dg.sB = 0;
    dg.C = C; dg.ldc = ldc; dg.sC = 0; dg.batch = 1;
    gemm_planes(dg, wsP.p, wsP_bytes, stream_);
  };
  // W buffers: orderings (i,j,k), (i,k,j) interleaved as [(i,a,b)][2][c]; the other four as
  // [(a,b)][i][c] with row stride nbmax v
  double* W1 = W.p;                       // 2 nbmax v^3
  double* Wg[4];                          // (j,k,i), (j,i,k), (k,j,i), (k,i,j)
  for (int q = 0; q < 4; ++q) Wg[q] = W.p + (2 + q) * nbmax * v3;
  const long ldw = nbmax * V;
  long nchunks = 0;
  for (int k = 0; k < o; ++k)
    for (int j = 0; j <= k; ++j) nchunks += ceil_div(j + 1, nbmax);
  ScratchBuf partials(scratch_, (size_t)(ncube * nbmax)), acc(scratch_, (size_t)nchunks);
  long slot = 0;
  for (int k = 0; k < o; ++k)
    for (int j = 0; j <= k; ++j)
      for (int i0 = 0; i0 <= j; i0 += (int)nbmax) {
        const int nb = (int)std::min<long>(nbmax, j + 1 - i0);
        // (i,j,k) and (i,k,j): C[(i,a,b)][(t,c)] = Acat[(i,a,b)][K] Bp[j][k][K][(t,c)]
        plane_gemm((int)(nb * V * V), (int)(2 * V), Ap.at((long)i0 * V * V * VK),
                   BPp.at(((long)j * O + k) * 2 * V * VK), W1, 2 * V);
        // fixed first index o1 in {j, k}: C[(a,b)][(i,c)] = Acat[o1][(a,b)][K] B[K][(i,c)]
        // (j,k,i): Bcat(k, i), (j,i,k): Bcat(i, k), (k,j,i): Bcat(j, i), (k,i,j): Bcat(i, j)
        for (int q = 0; q < 4; ++q)
          plane_gemm((int)(V * V), (int)(nb * V), Ap.at((long)(q < 2 ? j : k) * V * V * VK),
                     (q % 2 == 0 ? BTp : BT2p).at(((long)(q < 2 ? k : j) * O + i0) * V * VK), Wg[q], ldw);
        TriplesArgs g;
        // orderings by S3 index: 0 (i,j,k) 1 (i,k,j) 2 (j,i,k) 3 (j,k,i) 4 (k,i,j) 5 (k,j,i)
        g.Wb[0] = W1;     g.Wz[0] = 2 * v3; g.Wr[0] = 2 * V;
        g.Wb[1] = W1 + V; g.Wz[1] = 2 * v3; g.Wr[1] = 2 * V;
        g.Wb[2] = Wg[1];  g.Wz[2] = V;      g.Wr[2] = ldw;
        g.Wb[3] = Wg[0];  g.Wz[3] = V;      g.Wr[3] = ldw;
        g.Wb[4] = Wg[3];  g.Wz[4] = V;      g.Wr[4] = ldw;
        g.Wb[5] = Wg[2];  g.Wz[5] = V;      g.Wr[5] = ldw;
        g.G = Gijab_; g.t1 = t1_; g.eo = eo_; g.ev = ev_;
        g.o = o; g.v = v; g.i0 = i0; g.j = j; g.k = k;
        hipLaunchKernelGGL(triples_energy_kernel, dim3((unsigned)ncube, nb), dim3(kTThreads), 0, stream_, g,
                           partials.p);
        check_launch("triples_energy");
        hipLaunchKernelGGL(sum_to_slot, dim3(1), dim3(256), 0, stream_, partials.p, ncube * nb, acc.p, slot);
        check_launch("triples_sum");
        ++slot;
      }
  std::vector<double> h(nchunks);
  MPQC_HIP_CHECK(hipMemcpyAsync(h.data(), acc.p, nchunks * sizeof(double), hipMemcpyDeviceToHost, stream_));
  MPQC_HIP_CHECK(hipStreamSynchronize(stream_));
  return h;
}

double CCSDContext::triples(double block_bytes, double* seconds) {
  if (!have_eps_) throw std::logic_error("(T) needs the orbital energies");
  if (!prepared_) prepare();
  ensure_iabc_for_triples();
  const long V = v_;
  if (energy_cubes(V) >= (1L << 31) || V * V >= (1L << 31)) throw std::invalid_argument("v too large for (T)");
  hipEvent_t ev0, ev1;
  MPQC_HIP_CHECK(hipEventCreate(&ev0));
  MPQC_HIP_CHECK(hipEventCreate(&ev1));
  MPQC_HIP_CHECK(hipEventRecord(ev0, stream_));
  const std::vector<double> h =
      split_mode() && !summed_faster(o_, V, prec_) ? triples_orderings(block_bytes) : triples_summed(block_bytes);
  MPQC_HIP_CHECK(hipEventRecord(ev1, stream_));
  MPQC_HIP_CHECK(hipEventSynchronize(ev1));
  float ms = 0.f;
  MPQC_HIP_CHECK(hipEventElapsedTime(&ms, ev0, ev1));
  (void)hipEventDestroy(ev0);
  (void)hipEventDestroy(ev1);
  if (seconds) *seconds = ms * 1e-3;
  double e = 0.0;
  for (double x : h) e += x;
  if (!std::isfinite(e)) throw std::runtime_error("non-finite (T) energy");
  return e;
}

}  // namespace mpqc_hip
