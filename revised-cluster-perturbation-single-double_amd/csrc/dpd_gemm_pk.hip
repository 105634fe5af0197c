// dpd_gemm_pk.hip -- packing of DPD operands into GEMM panels (gfx950).
//
// The DPD operands of a contraction are irrep blocks addressed through
// mixed-radix digits; gathering them inside the GEMM costs address arithmetic
// and narrow loads on every K tile.  The kernels here copy each operand into
// panels (task, tile, K step) in the order in which the MFMA instructions take
// them (dpd_gemm_fr.hpp, which multiplies them): FP64 (16 k's a step), FP32
// (32) or BF16 hi + lo planes (32; x = hi + lo, hi = bf16(x), lo = bf16(x - hi)).
// Panels pad M and N to the tile and every K segment to 16 with zeros.
// Operands that do not change between calls (integrals, intermediates) are
// packed once and kept.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "dpd_kernels.hpp"

namespace dpd {

namespace {
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));  // one 16-byte chunk
typedef int i4_t __attribute__((ext_vector_type(4)));
typedef int i2_t __attribute__((ext_vector_type(2)));

__device__ inline int64_t digit_off(int v, const int32_t* d, const int64_t* s) {
  const int d0 = v % d[0];
  const int t = v / d[0];
  const int d1 = t % d[1];
  const int d2 = t / d[1];
  return (int64_t)d0 * s[0] + (int64_t)d1 * s[1] + (int64_t)d2 * s[2];
}

// round-to-nearest-even FP32 -> BF16 (finite inputs)
__device__ inline uint16_t bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf16_float(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

constexpr int kThreads = 256;

// task of a panel of one side
__device__ inline int find_task(const GemmTask* tasks, int ntask, int panel, int side) {
  int lo = 0, hi = ntask - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if ((side == 0 ? tasks[mid].pan_a : tasks[mid].pan_b) <= panel) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
}  // namespace

// ---------------------------------------------------------------------------
// pack: one block per panel.  The block first tabulates, per K granule of the
// panel (16 k's share a segment), the offset of each of its rows and of each of
// its k's (one mixed-radix decode per row and per k instead of one per element);
// every element is then one add, or, for a fused sort, one fetch from the
// unsorted tensor with the row's and the k's indices.
// ---------------------------------------------------------------------------
template <int MODE, int MAXT>
__global__ __launch_bounds__(256) void k_pack(PackArgs p) {
  // the sort's layouts are indexed by per-lane irreps: keep them in LDS
  __shared__ MapArgs smap;
  if (p.use_map) {
    for (int i = threadIdx.x; i < (int)(sizeof(MapArgs) / 4); i += blockDim.x)
      ((int32_t*)&smap)[i] = ((const int32_t*)&p.map)[i];
  }
  constexpr int KS = MODE == PREC_F64 ? 16 : 32;
  constexpr int NG = KS / 16;    // granules per panel
  __shared__ int64_t rowoff[NG][MAXT];  // row part of the address (-1: padding row)
  __shared__ int64_t koff[KS];          // k part incl. the segment base (-1: padding k)
  __shared__ int8_t rh[NG][MAXT][4], kh[KS][4];
  __shared__ int32_t rx[NG][MAXT][4], kx[KS][4], rb[NG][MAXT];
  __shared__ int sgi[NG];
  __shared__ double tv[KS][MAXT + 1];  // the panel, [k][row]
  const int pid = blockIdx.x;
  const int ti = find_task(p.tasks, p.ntask, pid, p.side);
  const GemmTask& T = p.tasks[ti];
  const int local = pid - (p.side == 0 ? T.pan_a : T.pan_b);
  const int tile = local / T.steps, step = local % T.steps;
  const int R = p.side == 0 ? T.M : T.N;
  const int r0 = tile * p.tile;
  const int64_t pan_elems = (int64_t)p.tile * KS;
  const int64_t base = (p.side == 0 ? T.pa_off : T.pb_off) + (int64_t)local * pan_elems * (MODE == PREC_BF16X3 ? 2 : 1);
  const int32_t* rd = p.side == 0 ? T.md : T.nd;
  if (threadIdx.x < NG) {
    const int gran = step * NG + threadIdx.x;
    int sg = -1;
    if (gran < T.ktiles_total) {
      sg = T.seg_begin;
      while (gran >= p.segs[sg].ktile_begin + p.segs[sg].ktiles) sg++;
    }
    sgi[threadIdx.x] = sg;
  }
  __syncthreads();
  // rows (one thread per granule and row)
  for (int t = threadIdx.x; t < NG * p.tile; t += kThreads) {
    const int g = t / p.tile, r = t % p.tile;
    const int sg = sgi[g];
    int64_t ro = -1;
    if (sg >= 0 && r0 + r < R) {
      const GemmSeg& S = p.segs[sg];
      ro = digit_off(r0 + r, rd, p.side == 0 ? S.sa_m : S.sb_n);
      if (p.use_map) {
        // indices of the row: decode the element (row, first k of the granule)
        const int gran = step * NG + g;
        const int k0 = (gran - S.ktile_begin) * 16;
        const int64_t ad = (p.side == 0 ? S.a_off : S.b_off) + ro +
                           digit_off(k0, S.kd, p.side == 0 ? S.sa_k : S.sb_k);
        const int64_t b = ad / p.xlen;
        int h[4];
        int64_t x[4];
        decode_elem(smap.out, ad - b * p.xlen, h, x);
        for (int d = 0; d < 4; d++) {
          rh[g][r][d] = (int8_t)h[d];
          rx[g][r][d] = (int32_t)x[d];
        }
        rb[g][r] = (int32_t)b;
      }
    }
    rowoff[g][r] = ro;
  }
  // k's (one thread per k of the panel)
  if (threadIdx.x < KS) {
    const int k = threadIdx.x;
    const int g = k >> 4;
    const int sg = sgi[g];
    int64_t ko = -1;
    if (sg >= 0) {
      const GemmSeg& S = p.segs[sg];
      const int gran = step * NG + g;
      const int ks = (gran - S.ktile_begin) * 16 + (k & 15);
      if (ks < S.K) {
        ko = (p.side == 0 ? S.a_off : S.b_off) + digit_off(ks, S.kd, p.side == 0 ? S.sa_k : S.sb_k);
        if (p.use_map) {
          // indices of the k: decode the element (first row of the task, k)
          const int64_t ad = ko + digit_off(0, rd, p.side == 0 ? S.sa_m : S.sb_n);
          const int64_t b = ad / p.xlen;
          int h[4];
          int64_t x[4];
          decode_elem(smap.out, ad - b * p.xlen, h, x);
          for (int d = 0; d < 4; d++) {
            kh[k][d] = (int8_t)h[d];
            kx[k][d] = (int32_t)x[d];
          }
        }
      }
    }
    koff[k] = ko;
  }
  __syncthreads();
  // read the panel in the order in which the source is contiguous (rows or
  // k's fastest) into LDS, then write it in panel order
  for (int idx = threadIdx.x; idx < pan_elems; idx += kThreads) {
    int r, k;
    if (p.rfast) {
      r = idx % p.tile;
      k = idx / p.tile;
    } else {
      k = idx % KS;
      r = idx / KS;
    }
    const int g = k >> 4;
    double v = 0.0;
    const int64_t ro = rowoff[g][r], ko = koff[k];
    if (p.code_out) {
      // code mode (no fused sort): the source of this element
      int32_t cd = 0;
      if (ro >= 0 && ko >= 0) {
        const int64_t ad = ro + ko;
        if (p.gcode) {
          const int64_t b = ad / p.gxlen, o = ad - b * p.gxlen;
          const int32_t gc = p.gcode[o];
          if (gc != 0) {
            const int64_t a1 = b * p.gbstride + (gc > 0 ? (int64_t)gc : -(int64_t)gc);
            cd = gc > 0 ? (int32_t)a1 : -(int32_t)a1;
          }
        } else {
          cd = (int32_t)(ad + 1);
        }
      }
      p.code_out[(int64_t)pid * pan_elems + fr_pos(MODE, r, k)] = cd;
      continue;
    }
    if (ro >= 0 && ko >= 0) {
      if (!p.use_map) {
        v = p.src_f32 ? (double)((const float*)p.src)[ro + ko] : p.src[ro + ko];
      } else {
        int hi[4];
        int64_t xi[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
          const bool row = (p.rowmask >> d) & 1;
          hi[smap.term[0].perm[d]] = row ? rh[g][r][d] : kh[k][d];
          xi[smap.term[0].perm[d]] = row ? rx[g][r][d] : kx[k][d];
        }
        double sg;
        const int64_t ia = fetch_addr(smap.in, hi[0], hi[1], hi[2], hi[3], xi[0], xi[1], xi[2], xi[3], &sg);
        if (ia >= 0) v = smap.alpha * (smap.term[0].coef * sg * p.src[(int64_t)rb[g][r] * p.src_bstride + ia]);
      }
    }
    tv[k][r] = v;
  }
  if (p.code_out) return;  // uniform: every thread of the block took the code branch
  __syncthreads();
  for (int e = threadIdx.x; e < pan_elems; e += kThreads) {
    int r, k;
    fr_elem(MODE, e, &r, &k);
    const double v = tv[k][r];
    if (MODE == PREC_F64) {
      ((double*)p.dst)[base + e] = v;
    } else if (MODE == PREC_F32) {
      ((float*)p.dst)[base + e] = (float)v;
    } else {
      const float f = (float)v;
      const uint16_t h = bf16_bits(f);
      const uint16_t l = bf16_bits((float)(v - (double)bf16_float(h)));
      const int64_t at = base + ((e >> 9) << 10) + (e & 511);
      ((uint16_t*)p.dst)[at] = h;
      ((uint16_t*)p.dst)[at + 512] = l;
    }
  }
}

// panels from precomputed source codes: a thread per 16-byte chunk of the panels
// (of the hi plane in BF16x3), so the codes are read and the panels written 16
// bytes a lane; the scattered source reads of a thread (2, 4 or 8) are in flight
// together.  Codes are in panel order, panels back to back.  HBM bound (codes,
// sources and panels once each; the ring operand of D2h/120, FP64: 200 MB); an
// element a thread took 73 us there, a chunk 52.
template <int MODE, typename TIN>
__global__ __launch_bounds__(256) void k_pack_code(int64_t nchunk, const int32_t* __restrict__ code,
                                                   const TIN* __restrict__ src, u4_t* __restrict__ dst) {
  constexpr int V = MODE == PREC_F64 ? 2 : MODE == PREC_F32 ? 4 : 8;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < nchunk; c += (int64_t)gridDim.x * blockDim.x) {
    int32_t cd[V];
    if constexpr (MODE == PREC_F64) {
      const i2_t q = ((const i2_t*)code)[c];
      cd[0] = q[0];
      cd[1] = q[1];
    } else {
#pragma unroll
      for (int j = 0; j < V / 4; j++) {
        const i4_t q = ((const i4_t*)code)[c * (V / 4) + j];
#pragma unroll
        for (int i = 0; i < 4; i++) cd[4 * j + i] = q[i];
      }
    }
    double v[V];
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int32_t a = cd[i] < 0 ? -cd[i] : cd[i];
      v[i] = a ? (double)src[a - 1] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < V; i++) v[i] = cd[i] < 0 ? -v[i] : v[i];
    u4_t o;
    if constexpr (MODE == PREC_F64) {
      o = __builtin_bit_cast(u4_t, *(const double __attribute__((ext_vector_type(2)))*)v);
      dst[c] = o;
    } else if constexpr (MODE == PREC_F32) {
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = __float_as_uint((float)v[i]);
      dst[c] = o;
    } else {
      u4_t lo;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint32_t h[2], l[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const double x = v[2 * i + j];
          h[j] = bf16_bits((float)x);
          l[j] = bf16_bits((float)(x - (double)bf16_float((uint16_t)h[j])));
        }
        o[i] = h[0] | (h[1] << 16);
        lo[i] = l[0] | (l[1] << 16);
      }
      const int64_t at = ((c >> 6) << 7) + (c & 63);  // 64 chunks of hi, then 64 of lo
      dst[at] = o;
      dst[at + 64] = lo;
    }
  }
}

hipError_t launch_pack_code(int mode, int src_f32, int64_t npanel, int64_t pan_elems, const int32_t* code,
                            const void* src, void* dst, hipStream_t s) {
  // panels are whole 16-row groups: a multiple of 256 (FP64) or 512 elements
  const int64_t nchunk = npanel * pan_elems / (mode == PREC_F64 ? 2 : mode == PREC_F32 ? 4 : 8);
  if (nchunk <= 0) return hipSuccess;
  int64_t b = (nchunk + 255) / 256;
  if (b > 65536) b = 65536;
  const dim3 grid((unsigned)b), blk(256);
#define PKC(M)                                                                                               \
  if (src_f32)                                                                                               \
    hipLaunchKernelGGL((k_pack_code<M, float>), grid, blk, 0, s, nchunk, code, (const float*)src, (u4_t*)dst);  \
  else                                                                                                       \
    hipLaunchKernelGGL((k_pack_code<M, double>), grid, blk, 0, s, nchunk, code, (const double*)src, (u4_t*)dst);
  switch (mode) {
    case PREC_F64: PKC(PREC_F64) break;
    case PREC_F32: PKC(PREC_F32) break;
    case PREC_BF16X3: PKC(PREC_BF16X3) break;
    default: return hipErrorInvalidValue;
  }
#undef PKC
  return hipGetLastError();
}

template <int MODE>
static hipError_t launch_pack_mode(const PackArgs& p, hipStream_t s) {
  if (p.tile <= 32) hipLaunchKernelGGL((k_pack<MODE, 32>), dim3(p.npanel), dim3(256), 0, s, p);
  else if (p.tile <= 64) hipLaunchKernelGGL((k_pack<MODE, 64>), dim3(p.npanel), dim3(256), 0, s, p);
  else if (p.tile <= 128) hipLaunchKernelGGL((k_pack<MODE, 128>), dim3(p.npanel), dim3(256), 0, s, p);
  else if (p.tile <= 192) hipLaunchKernelGGL((k_pack<MODE, 192>), dim3(p.npanel), dim3(256), 0, s, p);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_pack(const PackArgs& p, hipStream_t s) {
  if (p.npanel == 0) return hipSuccess;
  switch (p.mode) {
    case PREC_F64:
      return launch_pack_mode<PREC_F64>(p, s);
    case PREC_F32:
      return launch_pack_mode<PREC_F32>(p, s);
    case PREC_BF16X3:
      return launch_pack_mode<PREC_BF16X3>(p, s);
    default:
      return hipErrorInvalidValue;
  }
}

static hipError_t launch_fr(const GemmLaunch& g, const GroupTab* gt, const void* PA, const void* PB, hipStream_t s) {
  switch (g.prec) {
    case PREC_F64: return launch_fr_f64(g, gt, PA, PB, s);
    case PREC_F32: return launch_fr_f32(g, gt, PA, PB, s);
    case PREC_BF16X3: return launch_fr_bf16x3(g, gt, PA, PB, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_pk_grouped(const GemmLaunch& g, const GroupTab& gt, hipStream_t s) {
  if (g.nwg == 0) return hipSuccess;
  hipError_t e = launch_fr(g, &gt, nullptr, nullptr, s);
  if (e != hipSuccess) return e;
  return launch_splitk_reduce_grouped(g, gt, s);
}

hipError_t launch_gemm_pk_only(const GemmLaunch& g, const void* PA, const void* PB, hipStream_t s) {
  if (g.nwg == 0) return hipSuccess;
  return launch_fr(g, nullptr, PA, PB, s);
}

hipError_t launch_gemm_pk(const GemmLaunch& g, const void* PA, const void* PB, hipStream_t s) {
  hipError_t e = launch_gemm_pk_only(g, PA, PB, s);
  if (e != hipSuccess || g.nwg == 0) return e;
  return launch_splitk_reduce(g, s);
}

}  // namespace dpd
