// One output tile of an FP64 contraction on v_mfma_f64_16x16x4_f64, shared by the single,
// grouped and level launches.
//
// Operand fragments of a 16x16x4 block (lane l, r = 0..3):
//   A[m = l%16][k = l/16], B[k = l/16][n = l%16], C[m = 4*r + l/16][n = l%16]
// (the accumulator layout was established on the GPU; tests/test_gpu_gemm.py
// checks every tile position through full GEMMs).
#pragma once

#include "common.hpp"

namespace mpqc_hip {

constexpr int kBK = 16;
constexpr int kThreads = 256;

struct KParams {
  const double* A;
  const double* B;
  double* C;
  double* W;  // split-K workspace (nsplit > 1)
  long lda, ldb, ldc, sA, sB, sC;
  int M, N, K;
  int kchunk;
  int nsplit;
  int nsplit_batch;  // batch entries of a grouped problem (reduce pass)
  int batch0;  // first batch index of this launch
  int tiles_m, tiles_n;
  int per_xcd;  // tiles per XCD (workgroup w runs on XCD w % 8)
  double alpha, beta;
};

// ---------------------------------------------------------------- FP64 tile
// One 64 RB x 16 CB output tile `tile` (row-major tile index) of batch/split slice z
// (z = batch * nsplit + split, batch relative to p.batch0), by KG groups of four
// wave64s.  Bound: the matrix cores, one v_mfma_f64_16x16x4f64 per 64 cycles and SIMD
// (78.6 TFLOP/s), so everything else has to leave their issue slots alone:
//  * The four waves of a group are stacked along M (16 RB rows each, all 16 CB columns),
//    so a row of A belongs to one wave and its fragments go straight from global memory
//    to registers (whole 128-byte row pieces for A, 128-byte runs of m for A^T), one
//    K slice of 16 U values (U = 2 for small tiles) ahead of the products.  Only B, shared by the waves, is staged
//    through LDS (double buffered, one barrier per slice), in 16-byte pieces.
//  * No bounds check in the K loop: rows and columns past the edge read clamped
//    addresses, and the last, partial K slice goes through checked loads with zeros.
//  * CB (1 .. 9) follows N, so that o^2, o v, nbf ... wide outputs are not padded to 64.
//  * KG groups split K inside the workgroup (their sums are added through LDS in group
//    order), for outputs of too few tiles to give every SIMD two waves.
// Measured in TFLOP/s (before: 2 x 2 waves, both operands through LDS in checked 8-byte loads,
// 64 or 128 columns): 65536 x 1024 x 65536 58.6 -> 69.8 (the rate of a large library product here: 70 to 72), 3420^3 51.5 ->
// 63.6, 6555 x 900 x 6555 46.7 -> 62.0, 1520^3 42.5 -> 55.2, 2985984 x 144 x 144 (A^T) 35.9 ->
// 52.9, 900^3 28.3 -> 37.7; 95^3 8.9 -> 5.5 us.  Tried and dropped: exec-masked loads
// in place of clamped ones (the wait for a masked load moves up to where it merges with the
// unloaded value: 1520^3 55 -> 49), slices of 32 for the large tiles (no gain).
// A slice's k = 16 t + 4 (lane / 16) + q belongs to the q-th of its four MFMA steps (any
// assignment is exact when A and B use the same one).
typedef double double2a8 __attribute__((ext_vector_type(2), aligned(8)));  // 16-byte load at 8-byte alignment

template <int CB, int U, bool TB>
struct F64Lds {
  static constexpr int kSlice = 16 * U;
  // pitches that keep the fragment reads off each other's banks
  static constexpr int kPitch = TB ? kSlice + 2 : 16 * CB + 4;
  static constexpr int kRows = TB ? 16 * CB : kSlice;
  static constexpr int kDoubles = kRows * kPitch;
};

template <int RB, int CB, int KG, int U, bool TA, bool TB>
struct F64Shared {
  static constexpr int kStage = 2 * KG * F64Lds<CB, U, TB>::kDoubles;
  static constexpr int kReduce = KG > 1 ? 64 * RB * 16 * CB : 0;
  static constexpr int kDoubles = kStage > kReduce ? kStage : kReduce;
};

template <int RB, int CB, int KG, int U, bool TA, bool TB>
__device__ __forceinline__ void dgemm_f64_tile(const KParams& p, int tile, int z, double* __restrict__ smem) {
  constexpr int BM = 64 * RB, BN = 16 * CB, BK = 16 * U;
  constexpr int PITCH = F64Lds<CB, U, TB>::kPitch;

  const int tid = threadIdx.x & (kThreads - 1);
  const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads) : 0;
  double* const Bs = smem + grp * 2 * F64Lds<CB, U, TB>::kDoubles;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;

  const int tm = tile / p.tiles_n, tn = tile - tm * p.tiles_n;
  const int b = p.batch0 + z / p.nsplit;
  const int s = z - (z / p.nsplit) * p.nsplit;
  const int m0 = tm * BM, n0 = tn * BN;
  int k_begin = s * p.kchunk;
  int k_end = min(p.K, k_begin + p.kchunk);
  int nslices = (k_end - k_begin + BK - 1) / BK;               // of the longest group
  if (KG > 1) {
    const int per = (nslices + KG - 1) / KG;
    k_begin += grp * per * BK;
    k_end = min(k_end, k_begin + per * BK);
    nslices = per;
  }
  const int full = k_end > k_begin ? (k_end - k_begin) / BK : 0;  // whole slices of this group

  // Every load of a whole slice is unconditional (a masked one would be waited for where
  // its register merges with the unloaded value): rows and columns past the edge read the
  // last ones instead, and their products are never stored.
  // A: this lane's row of each 16-row block.
  const double* ap[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const long m = min(m0 + (wave * RB + i) * 16 + lr, p.M - 1);
    ap[i] = p.A + (long)b * p.sA + (TA ? (long)(k_begin + 4 * lk) * p.lda + m : m * p.lda + k_begin + 4 * lk);
  }
  // B: this thread's 16-byte pieces, kStep columns (rows, for B^T) apart.  With an odd N
  // the pair of the last column starts one earlier and is put right when it is stored.
  constexpr int kLine = TB ? BK / 2 : kThreads / BK;  // threads per row of the stage
  constexpr int kStep = TB ? kThreads / kLine : 2 * kLine;
  constexpr int PER = (BN + kStep - 1) / kStep;
  const int bk = TB ? 2 * (tid % kLine) : tid / kLine;   // first k of the pieces
  const int bn0 = TB ? tid / kLine : 2 * (tid % kLine);  // n of piece 0
  const double* bp = p.B + (long)b * p.sB + (TB ? (long)(k_begin + bk) : (long)(k_begin + bk) * p.ldb);
  long boff[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int n = n0 + bn0 + kStep * r;
    boff[r] = TB ? (long)min(n, p.N - 1) * p.ldb : (long)max(0, min(n, p.N - 2));
  }
  double* const bdst = Bs + (TB ? bn0 * PITCH + bk : bk * PITCH + bn0);
  const bool odd_edge = !TB && (p.N & 1) && n0 + BN >= p.N;  // some thread has half a piece
  const bool narrow = !TB && p.N < 2;                        // no whole piece in a row of B

  double an[RB][4 * U];  // next slice's fragments of A
  double2a8 bn[PER];     // next slice's pieces of B
  auto load_full = [&]() {
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      if (TA) {
#pragma unroll
        for (int q = 0; q < 4 * U; ++q) an[i][q] = ap[i][(long)(16 * (q / 4) + q % 4) * p.lda];
      } else {
#pragma unroll
        for (int q = 0; q < 4 * U; q += 2) {
          const double2a8 x = *reinterpret_cast<const double2a8*>(ap[i] + 16 * (q / 4) + q % 4);
          an[i][q] = x[0];
          an[i][q + 1] = x[1];
        }
      }
      ap[i] += TA ? (long)BK * p.lda : BK;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) bn[r] = *reinterpret_cast<const double2a8*>(bp + boff[r]);
    bp += TB ? BK : (long)BK * p.ldb;
  };
  // a slice that K ends in (or any slice of a one-column B), element by element: zeros
  // from k_end on
  auto load_checked = [&](int t) {
    const int k0 = k_begin + t * BK;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int q = 0; q < 4 * U; ++q) {
        const int dk = 16 * (q / 4) + q % 4;
        an[i][q] = k0 + 4 * lk + dk < k_end ? ap[i][TA ? (long)dk * p.lda : dk] : 0.0;
      }
      if (narrow) ap[i] += TA ? (long)BK * p.lda : BK;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = k0 + bk + (TB ? h : 0);
        bn[r][h] = k < k_end ? bp[boff[r] + (narrow ? 0 : h)] : 0.0;
      }
    if (narrow) bp += (long)BK * p.ldb;
  };
  auto load = [&](int t) {
    if (t < full && !narrow) load_full();
    else load_checked(t);
  };
  auto store_b = [&](int buf) {
    if (odd_edge) {
#pragma unroll
      for (int r = 0; r < PER; ++r)
        if (n0 + bn0 + kStep * r == p.N - 1) bn[r][0] = bn[r][1];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r)
      if (BN % kStep == 0 || bn0 + kStep * r < BN)
        *reinterpret_cast<double2*>(bdst + buf * F64Lds<CB, U, TB>::kDoubles + (TB ? kStep * r * PITCH : kStep * r)) =
            double2{bn[r][0], bn[r][1]};
  };

  double4_t acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  // Steps of one slice: one k per lane group for B rows of n, a pair for B rows of k.
  // The B fragments of a step are read one step ahead of their products, across the
  // slice's barrier too, which stands before the last step: every wave then has the
  // slice's last fragments in registers, so its stage is free, and the other stage is
  // complete.  No product waits for the LDS or, at the barrier, for a slower wave's reads.
  constexpr int PAIR = TB ? 2 : 1, STEPS = 4 * U / PAIR;
  auto read_b = [&](int buf, int step, double (&f)[CB][PAIR]) {
    const double* bs = Bs + buf * F64Lds<CB, U, TB>::kDoubles;
    if constexpr (TB) {
      bs += lr * PITCH + 4 * lk + 16 * (step / 2) + 2 * (step % 2);
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const double2 x = *reinterpret_cast<const double2*>(bs + 16 * j * PITCH);
        f[j][0] = x.x;
        f[j][PAIR - 1] = x.y;
      }
    } else {
      bs += (4 * lk + 16 * (step / 4) + step % 4) * PITCH + lr;
#pragma unroll
      for (int j = 0; j < CB; ++j) f[j][0] = bs[16 * j];
    }
  };
  // (the widest tile has no registers left for a second set: it reads a step's fragments
  // just before the products)
  constexpr bool kAhead = RB * CB < 18;
  double a[RB][4 * U], fb[kAhead ? 2 : 1][CB][PAIR];
  auto products = [&](int step) {
#pragma unroll
    for (int h = 0; h < PAIR; ++h)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][step * PAIR + h], fb[kAhead ? step & 1 : 0][j][h], acc[i][j], 0, 0, 0);
  };
  if (nslices > 0) {
    load(0);
    store_b(0);
  }
  __syncthreads();
  if (nslices > 0) {
    if (kAhead) read_b(0, 0, fb[0]);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int q = 0; q < 4 * U; ++q) a[i][q] = an[i][q];
  }
  int buf = 0;
  for (int t = 0; t < nslices; ++t) {
    const bool has_next = t + 1 < nslices;
    if (has_next) load(t + 1);
#pragma unroll
    for (int step = 0; step < STEPS - 1; ++step) {
      if constexpr (kAhead) {
        read_b(buf, step + 1, fb[(step + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the products
      } else {
        read_b(buf, step, fb[0]);
      }
      products(step);
    }
    if (!kAhead) read_b(buf, STEPS - 1, fb[0]);
    if (has_next) store_b(buf ^ 1);
    __syncthreads();
    buf ^= 1;
    if (kAhead && has_next) read_b(buf, 0, fb[0]);
    __builtin_amdgcn_sched_barrier(0);
    products(STEPS - 1);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int q = 0; q < 4 * U; ++q) a[i][q] = an[i][q];
  }
  if (KG > 1) __syncthreads();

  if (KG > 1) {  // (every wave has left the K loop: the stages are free)
#pragma unroll 1
    for (int g = 1; g < KG; ++g) {
      if (grp == g) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) smem[((i * CB + j) * 4 + r) * kThreads + tid] = acc[i][j][r];
      }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] += smem[((i * CB + j) * 4 + r) * kThreads + tid];
      }
      __syncthreads();
    }
    if (grp != 0) return;
  }

  // epilogue: C, or partial sums to workspace slice z (dense M x N)
  const bool split = p.nsplit > 1;
  double* __restrict__ out = split ? p.W + (long)z * p.M * p.N : p.C + (long)b * p.sC;
  const long ldo = split ? p.N : p.ldc;
  const double beta = split ? 0.0 : p.beta;
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gm = m0 + (wave * RB + i) * 16 + r * 4 + lk;
      if (gm >= p.M) continue;
      double* c = out + (long)gm * ldo + n0 + lr;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if (n0 + 16 * j + lr >= p.N) continue;
        const double v = p.alpha * acc[i][j][r];
        c[16 * j] = (beta == 0.0) ? v : v + beta * c[16 * j];
      }
    }
}

}  // namespace mpqc_hip
