// dpd_gemm_fr.hpp -- grouped DPD GEMM on packed panels in fragment order (gfx950).
//
// The pack kernels (dpd_gemm_pk.hip) write every operand in the order in which
// the MFMA instructions take it.  A panel (task, tile, K step of 16 k's in FP64,
// 32 in FP32 and BF16x3) is a row of 16-row groups; a group is two planes of 64
// lanes x 16 bytes, 2 KiB in every mode:
//
//   FP64    lane (r & 15) + 16 (k & 3), plane k >> 3, half (k >> 2) & 1
//   FP32    lane (r & 15) + 16 (k & 3), plane k >> 4, quarter (k >> 2) & 3
//   BF16x3  lane (r & 15) + 16 (k >> 3), element k & 7; plane 0 holds
//           hi = bf16(x), plane 1 lo = bf16(x - hi)
//
// so a wave loads the fragments of a group and K step with two fully coalesced
// 1 KiB loads, straight into the registers that the MFMAs read, and an operand
// that goes through LDS is copied and read without bank conflicts.
//
// Two forms of k_gemm_fr<mode, form, TM, TN>, four waves each:
//  * FR_ROWS: tile 64 TM x 16 TN.  Every wave owns 16 TM rows and loads
//    its A fragments itself (no two waves share them); B is staged in LDS, two
//    buffers, one barrier per K step, loads two steps ahead.  TN follows N in
//    steps of 16: an N of 145 runs 160 wide, not 192 (what three tiles of 64
//    cost), and A is then read once.
//  * FR_STEPS: tile 16 TM x 16 TN.  The waves take the K steps in turn,
//    both operands come straight into registers three steps ahead, no barrier
//    until the four partial tiles are added through LDS.  For short M x N with
//    long K, where rows of their own would leave three of four waves idle.
// The MFMAs are called with the operands exchanged (B fragment first), so that
// the 16 lanes of a result register run along m, the unit stride of C: 128-byte
// runs in FP64 instead of 16 columns x 32 bytes.
// Every FR_ROWS tile sums its products in the same order over k; FR_STEPS adds
// four interleaved sums, and split-K the sums of its parts.
// Measured (MI355X, D2h/120 orbitals, 5 vectors; the tiles before were 32 to 128
// wide with both operands through LDS): ring (8 x 3000 x 600 x 600) FP64
// 432 -> 380 us, BF16x3 107 -> 77 us; pp-ladder (8 x 2957 x 145 x 2957) FP64
// 509 -> 455, BF16x3 153 -> 119; c1_r2abci (8 x 27 x 15 x 65 000) FP64 68 -> 50.
// What bounds them: a 4096^3 product runs at 68 TFLOP/s in FP64 (rocBLAS 72, a
// bare MFMA loop 76); the ring's 38 K steps leave the start and end of each
// tile uncovered, the pp-ladder reads its 0.57 GB of integrals once at 1.3 TB/s
// beside the MFMAs and its N of 100 to 200 pads by 10 to 25 %.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "dpd_kernels.hpp"

namespace dpd {
namespace fr {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));  // one 16-byte chunk
typedef double d2_t __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
constexpr int kGroupChunks = 128;  // 16-byte chunks of a 16-row group in one K step

template <int MODE>
struct Acc {
  typedef f4_t T;
  typedef float S;
};
template <>
struct Acc<PREC_F64> {
  typedef d4_t T;
  typedef double S;
};

// FP32 sums are taken in two levels: every kFoldSteps rounds of the K loop (256
// k's; 768 of a wave's in FR_STEPS) the accumulators are added to a second set
// and start again, so the rounding error follows 256 + K / 256 additions instead
// of K: error of the FP32 sigma against FP64, C2v/100 orbitals, three vectors,
// 1.5e-7 -> 8.2e-8, D2h/120 1.6e-7 -> 7.3e-8, for 592 -> 599 us.
constexpr int kFoldSteps = 8;
template <int MODE, int TM, int TN>
struct Fold {
  __device__ __forceinline__ void step(int, typename Acc<MODE>::T (*)[TN]) {}
  __device__ __forceinline__ void end(typename Acc<MODE>::T (*)[TN]) {}
};
template <int TM, int TN>
struct Fold<PREC_F32, TM, TN> {
  f4_t sum[TM][TN];
  __device__ __forceinline__ Fold() {
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int y = 0; y < TN; y++) sum[x][y] = f4_t{0, 0, 0, 0};
  }
  // after the done-th step
  __device__ __forceinline__ void step(int done, f4_t (*acc)[TN]) {
    if (done % kFoldSteps) return;  // uniform
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int y = 0; y < TN; y++) {
        sum[x][y] += acc[x][y];
        acc[x][y] = f4_t{0, 0, 0, 0};
      }
  }
  __device__ __forceinline__ void end(f4_t (*acc)[TN]) {
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int y = 0; y < TN; y++) acc[x][y] += sum[x][y];
  }
};

// result register r of a lane: column (n) offset inside the 16x16 tile; m is lane & 15
template <int MODE>
__device__ __forceinline__ int col_of(int lane, int r) {
  return MODE == PREC_F64 ? (lane >> 4) + 4 * r : 4 * (lane >> 4) + r;
}

// the products of one K step for TM row groups a[x] against one column group b
template <int MODE, int TM>
__device__ __forceinline__ void mma(typename Acc<MODE>::T* acc, int stride, const u4_t (*a)[2], const u4_t* b) {
  if constexpr (MODE == PREC_F64) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const d2_t bv = __builtin_bit_cast(d2_t, b[h]);
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int x = 0; x < TM; x++) {
          const d2_t av = __builtin_bit_cast(d2_t, a[x][h]);
          acc[x * stride] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j], av[j], acc[x * stride], 0, 0, 0);
        }
    }
  } else if constexpr (MODE == PREC_F32) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const f4_t bv = __builtin_bit_cast(f4_t, b[h]);
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int x = 0; x < TM; x++) {
          const f4_t av = __builtin_bit_cast(f4_t, a[x][h]);
          acc[x * stride] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j], av[j], acc[x * stride], 0, 0, 0);
        }
    }
  } else {
    const bf8_t bh = __builtin_bit_cast(bf8_t, b[0]), bl = __builtin_bit_cast(bf8_t, b[1]);
#pragma unroll
    for (int x = 0; x < TM; x++)
      acc[x * stride] =
          __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, __builtin_bit_cast(bf8_t, a[x][1]), acc[x * stride], 0, 0, 0);
#pragma unroll
    for (int x = 0; x < TM; x++)
      acc[x * stride] =
          __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl, __builtin_bit_cast(bf8_t, a[x][0]), acc[x * stride], 0, 0, 0);
#pragma unroll
    for (int x = 0; x < TM; x++)
      acc[x * stride] =
          __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, __builtin_bit_cast(bf8_t, a[x][0]), acc[x * stride], 0, 0, 0);
  }
}

__device__ inline int64_t digit_off(int v, const int32_t* d, const int64_t* s) {
  const int d0 = v % d[0];
  const int t = v / d[0];
  const int d1 = t % d[1];
  const int d2 = t / d[1];
  return (int64_t)d0 * s[0] + (int64_t)d1 * s[1] + (int64_t)d2 * s[2];
}

__device__ inline int task_of(const GemmTask* tasks, int ntask, int wg) {
  int lo = 0, hi = ntask - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].wg_begin <= wg) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// XCD-aware order: consecutive workgroup ids (neighbouring tiles that share
// panels) go to one XCD's L2 (dispatch deals workgroups round-robin over 8 XCDs)
__device__ __forceinline__ int xcd_wg(int nwg) {
  const int x = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int q = nwg >> 3, r = nwg & 7;
  return x * q + (x < r ? x : r) + slot;
}

// results of one lane for NY 16x16 tiles side by side: row m, columns
// n0 + 16 y + col_of(lane, 0..3).  The old values of an accumulating result are
// loaded together before the first store (a store to C may not be passed by a
// load from it).
template <int MODE, int NY>
__device__ __forceinline__ void put(const GemmLaunch& g, const GemmTask& T, int kp, double* __restrict__ C, double beta,
                                    bool c32, int lane, int m, int64_t cm, int n0, const int64_t* cn,
                                    const double (*v)[4]) {
  if (m >= T.M) return;
  if (T.ksplit > 1) {
#pragma unroll
    for (int y = 0; y < NY; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int n = n0 + 16 * y + col_of<MODE>(lane, r);
        if (n < T.N) g.partial[T.part_off + ((int64_t)kp * T.N + n) * T.M + m] = g.alpha * v[y][r];
      }
    return;
  }
  const int64_t base = T.c_off + cm;
  double old[NY][4];
  if (beta != 0.0) {
#pragma unroll
    for (int y = 0; y < NY; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int c = 16 * y + col_of<MODE>(lane, r);
        old[y][r] = 0.0;
        if (n0 + c < T.N) old[y][r] = c32 ? (double)((const float*)C)[base + cn[c]] : C[base + cn[c]];
      }
  }
#pragma unroll
  for (int y = 0; y < NY; y++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int c = 16 * y + col_of<MODE>(lane, r);
      if (n0 + c < T.N) {
        const double x = beta == 0.0 ? g.alpha * v[y][r] : beta * old[y][r] + g.alpha * v[y][r];
        if (c32) ((float*)C)[base + cn[c]] = (float)x;  // formed in FP64, rounded once
        else C[base + cn[c]] = x;
      }
    }
}

// ---- A fragments of TM row groups, a K step at a time ------------------------
// from packed panels
template <int MODE, int TM, int GA>
struct PanelA {
  const u4_t* p;
  int lane;
  __device__ __forceinline__ PanelA(const GemmLaunch&, const GemmTask& T, const void* PA, int tm, int s0, int group,
                                    int, int lane_)
      : lane(lane_) {
    constexpr int EPC = MODE == PREC_F64 ? 2 : MODE == PREC_F32 ? 4 : 8;
    p = (const u4_t*)PA + T.pa_off / EPC + (((int64_t)tm * T.steps + s0) * GA + group) * kGroupChunks;
  }
  // fragments of step s (counted from s0)
  __device__ __forceinline__ void load(int s, u4_t (*q)[2], int&) {
    const u4_t* t = p + (int64_t)s * (GA * kGroupChunks);
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int h = 0; h < 2; h++) q[x][h] = t[x * kGroupChunks + h * 64 + lane];
  }
  static __device__ __forceinline__ void finish(u4_t (*)[2], int, int) {}
};

// from the FP64 tensor where it lies (16 rows x 4 k's a load, 8 bytes a lane):
// an operand that is read once would pay for its packing with two more passes
// over memory.  K has at most two digits here, the first at least 16 long or
// all of K; rows past M read row M - 1 (their results are not written), k's past
// K read k = 0 and are zeroed before they are multiplied.
template <int TM>
struct TensorA {
  const double* A;
  const GemmTask& T;
  const GemmSeg* segs;
  int s0, lane, m0, seg, end;
  int64_t ro[TM];
  int64_t sk0, sk1;
  int kd0, K, kt0;
  __device__ __forceinline__ TensorA(const GemmLaunch& g, const GemmTask& T_, const void*, int, int s0_, int, int m0_,
                                     int lane_)
      : A((const double*)g.A), T(T_), segs(g.segs), s0(s0_), lane(lane_), m0(m0_), seg(T_.seg_begin - 1), end(0) {}
  __device__ __forceinline__ void enter(int t) {
    do {
      seg++;
      end = segs[seg].ktile_begin + segs[seg].ktiles;
    } while (t >= end);
    const GemmSeg& S = segs[seg];
    sk0 = S.sa_k[0];
    sk1 = S.sa_k[1];
    kd0 = S.kd[0];
    K = S.K;
    kt0 = S.ktile_begin;
#pragma unroll
    for (int x = 0; x < TM; x++) {
      const int m = m0 + 16 * x + (lane & 15);
      ro[x] = S.a_off + digit_off(m < T.M ? m : T.M - 1, T.md, S.sa_m);
    }
  }
  __device__ __forceinline__ void load(int s, u4_t (*q)[2], int& left) {
    const int t = s0 + s;
    if (t >= end) enter(t);  // uniform, no load in the branch that the wave waits for later
    const int kb = (t - kt0) * 16;
    left = K - kb;
    const int k = kb + (lane >> 4);
    const int d1 = k / kd0, d0 = k - d1 * kd0;
    int64_t ko[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int dj = d0 + 4 * j;
      const bool wrap = dj >= kd0;
      const int64_t o = (int64_t)(wrap ? dj - kd0 : dj) * sk0 + (int64_t)(wrap ? d1 + 1 : d1) * sk1;
      ko[j] = k + 4 * j < K ? o : 0;
    }
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        d2_t v;
        v[0] = A[ro[x] + ko[2 * h]];
        v[1] = A[ro[x] + ko[2 * h + 1]];
        q[x][h] = __builtin_bit_cast(u4_t, v);
      }
  }
  static __device__ __forceinline__ void finish(u4_t (*q)[2], int left, int lane) {
    if (left >= 16) return;  // uniform
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (4 * j + (lane >> 4) >= left) {
#pragma unroll
        for (int x = 0; x < TM; x++) {
          d2_t v = __builtin_bit_cast(d2_t, q[x][j >> 1]);
          v[j & 1] = 0.0;
          q[x][j >> 1] = __builtin_bit_cast(u4_t, v);
        }
      }
  }
};
template <int MODE, int TM, int GA, bool DIRECT>
struct SourceA {
  typedef PanelA<MODE, TM, GA> T;
};
template <int MODE, int TM, int GA>
struct SourceA<MODE, TM, GA, true> {
  typedef TensorA<TM> T;
};

// ---- tile 64 TM x 16 TN, a wave per 16 TM rows, B through LDS --------------
template <int MODE, int TM, int TN, bool DIRECT>
__device__ __forceinline__ void rows_tile(const GemmLaunch& g, const GemmTask& T, int local, const void* __restrict__ PA,
                                          const void* __restrict__ PB, double* __restrict__ C, double beta, bool c32) {
  typedef typename Acc<MODE>::T AT;
  constexpr int EPC = MODE == PREC_F64 ? 2 : MODE == PREC_F32 ? 4 : 8;  // elements per chunk
  constexpr int GA = 4 * TM;                                           // row groups of the tile
  constexpr int NB = TN * kGroupChunks;                                // B chunks of a K step
  constexpr int CB = (NB + kThreads - 1) / kThreads;
  __shared__ u4_t Bs[2][NB];
  __shared__ int64_t cn[16 * TN];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tn = local % T.tiles_n;
  local /= T.tiles_n;
  const int tm = local % T.tiles_m;
  const int kp = local / T.tiles_m;
  const int s0 = (int)((int64_t)kp * T.steps / T.ksplit);
  const int nst = (int)((int64_t)(kp + 1) * T.steps / T.ksplit) - s0;
  const int m0 = tm * 64 * TM + wave * 16 * TM;
  typename SourceA<MODE, TM, GA, DIRECT>::T src(g, T, PA, tm, s0, wave * TM, m0, lane);
  const u4_t* pb = (const u4_t*)PB + T.pb_off / EPC + ((int64_t)tn * T.steps + s0) * NB;

  AT acc[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; x++)
#pragma unroll
    for (int y = 0; y < TN; y++) acc[x][y] = AT{0, 0, 0, 0};
  Fold<MODE, TM, TN> fold;

  u4_t ra[2][TM][2], rb[2][CB];
  int left[2] = {16, 16};
  auto load_b = [&](int step, u4_t* q) {
    const u4_t* p = pb + (int64_t)step * NB;
#pragma unroll
    for (int j = 0; j < CB; j++)
      if ((j + 1) * kThreads <= NB || j * kThreads + tid < NB) q[j] = p[j * kThreads + tid];
  };
  auto store_b = [&](const u4_t* q, u4_t* dst) {
#pragma unroll
    for (int j = 0; j < CB; j++)
      if ((j + 1) * kThreads <= NB || j * kThreads + tid < NB) dst[j * kThreads + tid] = q[j];
  };
  // one K step: B of it is in Bs[u], its A in ra[u]; rb[1 - u] holds B of the next
  auto compute = [&](int u) {
    src.finish(ra[u], left[u], lane);
    u4_t b[2][2];
    b[0][0] = Bs[u][lane];
    b[0][1] = Bs[u][64 + lane];
#pragma unroll
    for (int y = 0; y < TN; y++) {
      if (y + 1 < TN) {
        b[(y + 1) & 1][0] = Bs[u][(y + 1) * kGroupChunks + lane];
        b[(y + 1) & 1][1] = Bs[u][(y + 1) * kGroupChunks + 64 + lane];
      }
      mma<MODE, TM>(&acc[0][y], TN, ra[u], b[y & 1]);
    }
  };
  if (nst > 0) {
    load_b(0, rb[0]);
    src.load(0, ra[0], left[0]);
    if (nst > 1) {
      load_b(1, rb[1]);
      src.load(1, ra[1], left[1]);
    }
    store_b(rb[0], Bs[0]);
    __syncthreads();
    int i = 0;
    // steady state without a branch around any load: the compiler then knows how
    // many loads are in flight and waits for the oldest only.  (With the loads in
    // conditional blocks it waited for the ones just issued: 45 instead of 51
    // TFLOP/s in the FP64 ring.)
    for (; i + 3 < nst; i += 2) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        load_b(i + 2 + u, rb[u]);
        compute(u);
        src.load(i + 2 + u, ra[u], left[u]);
        store_b(rb[1 - u], Bs[1 - u]);  // the other buffer: every wave left it at the last barrier
        __syncthreads();
      }
      fold.step(i + 2, acc);
    }
    for (; i < nst; i += 2) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        if (i + u < nst) {
          if (i + u + 2 < nst) load_b(i + u + 2, rb[u]);
          compute(u);
          if (i + u + 2 < nst) src.load(i + u + 2, ra[u], left[u]);
          if (i + u + 1 < nst) store_b(rb[1 - u], Bs[1 - u]);
          __syncthreads();
        }
      }
    }
    fold.end(acc);
  }

  const int n0 = tn * 16 * TN;
  if (T.ksplit <= 1) {
    for (int i = tid; i < 16 * TN; i += kThreads) cn[i] = n0 + i < T.N ? digit_off(n0 + i, T.nd, T.sc_n) : 0;
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < TM; x++) {
    const int m = m0 + 16 * x + (lane & 15);
    const int64_t cm = m < T.M ? digit_off(m, T.md, T.sc_m) : 0;
    constexpr int NY = TN % 4 == 0 ? 4 : TN % 5 == 0 ? 5 : TN % 3 == 0 ? 3 : TN % 2 == 0 ? 2 : 1;
#pragma unroll
    for (int y = 0; y < TN; y += NY) {
      double v[NY][4];
#pragma unroll
      for (int i = 0; i < NY; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) v[i][r] = (double)acc[x][y + i][r];
      put<MODE, NY>(g, T, kp, C, beta, c32, lane, m, cm, n0 + 16 * y, cn + 16 * y, v);
    }
  }
}

// ---- tile 16 TM x 16 TN, the waves take the K steps in turn ------------------
template <int MODE, int TM, int TN, bool DIRECT>
__device__ __forceinline__ void steps_tile(const GemmLaunch& g, const GemmTask& T, int local, const void* __restrict__ PA,
                                           const void* __restrict__ PB, double* __restrict__ C, double beta, bool c32) {
  typedef typename Acc<MODE>::T AT;
  typedef typename Acc<MODE>::S ST;
  constexpr int EPC = MODE == PREC_F64 ? 2 : MODE == PREC_F32 ? 4 : 8;
  constexpr int PF = 3;
  __shared__ ST red[4][TM * TN * 256];
  __shared__ int64_t cn[16 * TN];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tn = local % T.tiles_n;
  local /= T.tiles_n;
  const int tm = local % T.tiles_m;
  const int kp = local / T.tiles_m;
  const int s0 = (int)((int64_t)kp * T.steps / T.ksplit);
  const int nst = (int)((int64_t)(kp + 1) * T.steps / T.ksplit) - s0;
  const int nw = nst > wave ? (nst - wave + 3) / 4 : 0;  // this wave's steps: wave, wave + 4, ...
  const int m0 = tm * 16 * TM, n0 = tn * 16 * TN;
  typename SourceA<MODE, TM, TM, DIRECT>::T src(g, T, PA, tm, s0, 0, m0, lane);
  const u4_t* pb = (const u4_t*)PB + T.pb_off / EPC + ((int64_t)tn * T.steps + s0 + wave) * (TN * kGroupChunks);

  AT acc[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; x++)
#pragma unroll
    for (int y = 0; y < TN; y++) acc[x][y] = AT{0, 0, 0, 0};
  Fold<MODE, TM, TN> fold;
  u4_t ra[PF][TM][2], rb[PF][TN][2];
  int left[PF];
  auto load = [&](int i, u4_t (*a)[2], u4_t (*b)[2], int& rest) {
    const u4_t* q = pb + (int64_t)i * (4 * TN * kGroupChunks);
    src.load(wave + 4 * i, a, rest);
#pragma unroll
    for (int y = 0; y < TN; y++)
#pragma unroll
      for (int h = 0; h < 2; h++) b[y][h] = q[y * kGroupChunks + h * 64 + lane];
  };
#pragma unroll
  for (int u = 0; u < PF; u++)
    if (u < nw) load(u, ra[u], rb[u], left[u]);
  int i = 0;
  for (; i + 2 * PF <= nw; i += PF) {  // steady state: no branch around the loads
#pragma unroll
    for (int u = 0; u < PF; u++) {
      src.finish(ra[u], left[u], lane);
#pragma unroll
      for (int y = 0; y < TN; y++) mma<MODE, TM>(&acc[0][y], TN, ra[u], rb[u][y]);
      load(i + PF + u, ra[u], rb[u], left[u]);
    }
    fold.step(i / PF + 1, acc);
  }
  for (; i < nw; i += PF) {
#pragma unroll
    for (int u = 0; u < PF; u++) {
      if (i + u < nw) {
        src.finish(ra[u], left[u], lane);
#pragma unroll
        for (int y = 0; y < TN; y++) mma<MODE, TM>(&acc[0][y], TN, ra[u], rb[u][y]);
        if (i + u + PF < nw) load(i + u + PF, ra[u], rb[u], left[u]);
      }
    }
  }
  fold.end(acc);
#pragma unroll
  for (int x = 0; x < TM; x++)
#pragma unroll
    for (int y = 0; y < TN; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[wave][(x * TN + y) * 256 + r * 64 + lane] = acc[x][y][r];
  if (T.ksplit <= 1)
    for (int i = tid; i < 16 * TN; i += kThreads) cn[i] = n0 + i < T.N ? digit_off(n0 + i, T.nd, T.sc_n) : 0;
  __syncthreads();
  // wave w finishes the 16x16 tiles w, w + 4, ...
  for (int t = wave; t < TM * TN; t += 4) {
    const int x = t / TN, y = t % TN;
    const int m = m0 + 16 * x + (lane & 15);
    const int64_t cm = m < T.M ? digit_off(m, T.md, T.sc_m) : 0;
    double v[1][4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int e = t * 256 + r * 64 + lane;
      v[0][r] = (double)((red[0][e] + red[1][e]) + (red[2][e] + red[3][e]));
    }
    put<MODE, 1>(g, T, kp, C, beta, c32, lane, m, cm, n0 + 16 * y, cn + 16 * y, v);
  }
}

template <int MODE, int KIND, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_gemm_fr(GemmLaunch g, const void* __restrict__ PA, const void* __restrict__ PB) {
  const int wg = xcd_wg(g.nwg);
  const GemmTask& T = g.tasks[task_of(g.tasks, g.ntask, wg)];
  if constexpr (KIND == FR_ROWS)
    rows_tile<MODE, TM, TN, false>(g, T, wg - T.wg_begin, PA, PB, g.C, g.beta, g.c_f32 != 0);
  else
    steps_tile<MODE, TM, TN, false>(g, T, wg - T.wg_begin, PA, PB, g.C, g.beta, g.c_f32 != 0);
}

template <int MODE, int KIND, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_gemm_fr_grp(GemmLaunch g, GroupTab gt) {
  const int wg = xcd_wg(g.nwg);
  const GemmTask& T = g.tasks[task_of(g.tasks, g.ntask, wg)];
  const GroupEnt& e = gt.e[T.group];
  if constexpr (KIND == FR_ROWS)
    rows_tile<MODE, TM, TN, false>(g, T, wg - T.wg_begin, e.pa, e.pb, e.c, e.beta, e.c_f32 != 0);
  else
    steps_tile<MODE, TM, TN, false>(g, T, wg - T.wg_begin, e.pa, e.pb, e.c, e.beta, e.c_f32 != 0);
}

// FP64 with A where it lies (g.A), B in panels
template <int KIND, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_gemm_fr_direct(GemmLaunch g, const void* __restrict__ PB) {
  const int wg = xcd_wg(g.nwg);
  const GemmTask& T = g.tasks[task_of(g.tasks, g.ntask, wg)];
  if constexpr (KIND == FR_ROWS)
    rows_tile<PREC_F64, TM, TN, true>(g, T, wg - T.wg_begin, nullptr, PB, g.C, g.beta, false);
  else
    steps_tile<PREC_F64, TM, TN, true>(g, T, wg - T.wg_begin, nullptr, PB, g.C, g.beta, false);
}

template <int I>
hipError_t launch_direct(const GemmLaunch& g, const void* PB, hipStream_t s) {
  if constexpr (I >= kFrShapeCount) {
    return hipErrorInvalidValue;
  } else {
    if (g.cfg != I) return launch_direct<I + 1>(g, PB, s);
    constexpr FrShape S = kFrShapes[I];
    if constexpr (S.tm * S.tn > 8) {
      return hipErrorInvalidValue;  // the planner keeps to the narrower tiles (fr_direct_shape)
    } else {
      hipLaunchKernelGGL((k_gemm_fr_direct<S.kind, S.tm, S.tn>), dim3(g.nwg), dim3(256), 0, s, g, PB);
      return hipGetLastError();
    }
  }
}

// launch of configuration I (an index of kFrShapes) and the ones after it
template <int MODE, int I>
hipError_t launch_shape(const GemmLaunch& g, const GroupTab* gt, const void* PA, const void* PB, hipStream_t s) {
  if constexpr (I >= kFrShapeCount) {
    return hipErrorInvalidValue;
  } else {
    if (g.cfg != I) return launch_shape<MODE, I + 1>(g, gt, PA, PB, s);
    constexpr FrShape S = kFrShapes[I];
    if (gt)
      hipLaunchKernelGGL((k_gemm_fr_grp<MODE, S.kind, S.tm, S.tn>), dim3(g.nwg), dim3(256), 0, s, g, *gt);
    else
      hipLaunchKernelGGL((k_gemm_fr<MODE, S.kind, S.tm, S.tn>), dim3(g.nwg), dim3(256), 0, s, g, PA, PB);
    return hipGetLastError();
  }
}

}  // namespace fr
}  // namespace dpd
