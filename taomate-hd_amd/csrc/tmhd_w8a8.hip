// Selective W8A8 projection for gfx950: per-token dynamic INT8 activation
// quantization, per-output-channel INT8 weight quantization and the scaled
// INT8 GEMM with a bf16 epilogue (reference call sites:
// src/taomate_hd/inference/w8a8.py:67-73, 117-145, 175-179).
#include <math.h>

#include <type_traits>

#include <algorithm>

#include "tmhd_internal.h"

namespace tmhd {
namespace {

// ---------------------------------------------------------------------------
// Row quantization, WPR waves (1 or 4, the whole workgroup) per row.  CH =
// 8-element chunks held per lane (one pass, row kept in registers); CH = 0
// streams the row twice.  Bound by HBM.  Four waves for long rows: one wave's
// registers (167 for 5,376 columns) let three rows a SIMD be in flight and rows
// beyond 8,192 columns not be held at all.  us with one wave / four, 331 rows:
// 5,376 columns 4.6 / 3.6, 14,336 18.3 / 5.3; 4,836 rows: 17.2 / 14.9 (5.2
// TB/s), 63.6 / 34.9; 12,252 rows: 35.5 / 32.4, 163 / 96.5.  Shorter rows lose
// more by the wait for the other waves: 4,836 rows of 2,056 columns 6.6 / 8.4, of
// 2,560 7.2 / 8.4, of 3,072 8.4 / 9.0; 12,252 rows 13.8 / 16.8, 15.8 / 16.9, 18.5
// both.  Between them the rows decide: 3,584 columns, 2,048 rows 4.9 / 5.2, 4,836
// 10.1 both, 12,252 21.4 / 20.8; 4,096 columns 5.3 / 5.5, 11.2 both, 24.0 / 23.0.
// WEIGHT selects the weight formula of _quantize_cutlass_w8a8_weight:
//   scale = max(amax / 127, 1e-12), q = clamp(rint(w / scale), -127, 127)
// otherwise the activation formula:
//   scale = amax / 127, q = sat_int8(rint(x * (127 / amax))), amax = 0 -> 0.
template <int WPR, int CH, bool WEIGHT>
__global__ void __launch_bounds__(256) row_quant_kernel(int8_t *__restrict__ q, float *__restrict__ scale,
                                                        const uint16_t *__restrict__ x, int32_t rows, int32_t cols,
                                                        int64_t xs) {
  constexpr int L = 64 * WPR;  // lanes of a row
  const int lane = threadIdx.x % L;
  const int row = blockIdx.x * (4 / WPR) + threadIdx.x / L;
  if (row >= rows) return;  // WPR 4: never (a workgroup per row)
  const int nch = cols >> 3;
  const uint16_t *xr = x + (int64_t)row * xs;
  int8_t *qr = q + (int64_t)row * cols;
  float amax = 0.0f;
  i32x4 raw[CH > 0 ? CH : 1];
  if constexpr (CH > 0) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int c = lane + L * j;
      raw[j] = c < nch ? *(const i32x4 *)(xr + c * 8) : i32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = (uint32_t)raw[j][e];
        amax = fmaxf(amax, fmaxf(fabsf(bf16_bits_to_f32(w & 0xffffu)), fabsf(bf16_bits_to_f32(w >> 16))));
      }
    }
  } else {
    for (int c = lane; c < nch; c += L) {
      const i32x4 r = *(const i32x4 *)(xr + c * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = (uint32_t)r[e];
        amax = fmaxf(amax, fmaxf(fabsf(bf16_bits_to_f32(w & 0xffffu)), fabsf(bf16_bits_to_f32(w >> 16))));
      }
    }
  }
  amax = wave_max(amax);
  if constexpr (WPR > 1) {
    __shared__ float part[WPR];
    if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = amax;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WPR; ++i) amax = fmaxf(amax, part[i]);
  }
  float sc, inv;
  if constexpr (WEIGHT) {
    sc = fmaxf(__fdiv_rn(amax, 127.0f), 1e-12f);
    inv = 0.0f;
  } else {
    sc = __fdiv_rn(amax, 127.0f);
    inv = amax > 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
  }
  if (lane == 0) scale[row] = sc;
  auto qv = [&](float v) -> uint32_t {
    int r;
    if constexpr (WEIGHT) {
      r = (int)fminf(fmaxf(__builtin_rintf(__fdiv_rn(v, sc)), -127.0f), 127.0f);
    } else {
      r = quant_rne_sat(v * inv);
    }
    return (uint32_t)r & 0xffu;
  };
  auto emit = [&](int c, i32x4 r) {
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t w0 = (uint32_t)r[e], w1 = (uint32_t)r[e + 2];
      lo |= qv(bf16_bits_to_f32(w0 & 0xffffu)) << (16 * e);
      lo |= qv(bf16_bits_to_f32(w0 >> 16)) << (16 * e + 8);
      hi |= qv(bf16_bits_to_f32(w1 & 0xffffu)) << (16 * e);
      hi |= qv(bf16_bits_to_f32(w1 >> 16)) << (16 * e + 8);
    }
    *(i32x2 *)(qr + c * 8) = i32x2{(int)lo, (int)hi};
  };
  if constexpr (CH > 0) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int c = lane + L * j;
      if (c < nch) emit(c, raw[j]);
    }
  } else {
    for (int c = lane; c < nch; c += L) emit(c, *(const i32x4 *)(xr + c * 8));
  }
}

template <bool WEIGHT>
int launch_row_quant(int8_t *q, float *scale, const void *x, int32_t rows, int32_t cols, int64_t xs, void *stream,
                     const char *what) {
  if (rows < 0 || cols <= 0 || cols % 8) return set_error(TMHD_ERR_UNSUPPORTED, "%s: cols %d must be a positive multiple of 8", what, cols);
  if (xs < cols || xs % 8) return set_error(TMHD_ERR_INVALID, "%s: row stride %lld", what, (long long)xs);
  if (!q || !scale || !x || ((uintptr_t)x % 16) || ((uintptr_t)q % 8))
    return set_error(TMHD_ERR_INVALID, "%s: null or misaligned pointer", what);
  if (rows == 0) return TMHD_OK;
  hipStream_t s = (hipStream_t)stream;
  const uint16_t *xp = (const uint16_t *)x;
  const int nch = cols / 8;
  auto go = [&](auto wpr, auto ch) {
    constexpr int WPR = decltype(wpr)::value, CH = decltype(ch)::value;
    hipLaunchKernelGGL((row_quant_kernel<WPR, CH, WEIGHT>), dim3((rows + 4 / WPR - 1) / (4 / WPR)), dim3(256), 0, s, q,
                       scale, xp, rows, cols, xs);
  };
  using std::integral_constant;
  if (nch <= 64)
    go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
  else if (nch <= 2 * 64)
    go(integral_constant<int, 1>{}, integral_constant<int, 2>{});
  else if (nch <= 4 * 64)
    go(integral_constant<int, 1>{}, integral_constant<int, 4>{});
  else if (nch <= 5 * 64)
    go(integral_constant<int, 1>{}, integral_constant<int, 5>{});
  else if (nch <= 6 * 64)
    go(integral_constant<int, 1>{}, integral_constant<int, 6>{});
  else if (nch <= 8 * 64 && rows <= 4096)
    go(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  else if (nch <= 2 * 256)
    go(integral_constant<int, 4>{}, integral_constant<int, 2>{});
  else if (nch <= 3 * 256)
    go(integral_constant<int, 4>{}, integral_constant<int, 3>{});
  else if (nch <= 4 * 256)
    go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
  else if (nch <= 8 * 256)
    go(integral_constant<int, 4>{}, integral_constant<int, 8>{});
  else
    go(integral_constant<int, 4>{}, integral_constant<int, 0>{});
  return check_launch(what);
}

// ---------------------------------------------------------------------------
// INT8 GEMM: C[m][n] = sum_k A[m][k] * B[n][k] with v_mfma_i32_32x32x32_i8.
// Workgroup tile 256 (m) x 256 (n), 8 waves as 4 (m) x 2 (n), each wave
// 64 x 128 (128 int32 accumulators per lane, two waves per SIMD).  The MFMA
// computes the transposed block D[n][m] = B-rows x A-rows, so a lane holds
// four consecutive n of one m and writes 4 bf16 (8 bytes) at a time.
// k-tiles of 64 stream through a 3-deep LDS ring filled by
// global_load_lds_dwordx4; the loop is unrolled by the ring depth so every
// LDS address is a compile-time slot.  LDS rows are 64 bytes (4 chunks);
// chunk c of row r sits at c ^ ((r >> 2) & 3), so the 16 lanes of one
// ds_read_b128 phase hit 16 distinct 16-byte bank groups.
constexpr int GBM = 256, GBN = 256, GBK = 64, GWAVES = 8, GRING = 3;
constexpr int GSTAGE = (GBM + GBN) * GBK;  // bytes per ring slot

struct GArgs {
  const int8_t *a;
  const int8_t *b;
  void *out;
  const float *as;
  const float *bs;
  const uint16_t *bias;
  int32_t m, n, k;
  int64_t lda, ldb, ldo;
  int32_t tm_count, tn_count;
  int32_t vec_ok;  // bs 16-byte and bias 8-byte aligned: vector loads of 4 columns
  int32_t st_ok;   // bf16 output rows 16-byte aligned: staged 16-byte stores
  // K split of the last, partial round (one-wave-per-SIMD kernel): tiles
  // [0, full) are whole; block t * nsplit + p of the split launch is k-range p
  // of tile full + t, whose int32 partial tile goes to ws (merged afterwards)
  // (tile kernel: parts of the tiles from `full` on, or with full < 0 its own
  // tiling of the whole matrix)
  int32_t full, nsplit;
  int32_t *ws;
};

// Tile (tm, tn) of logical tile L: 4 row tiles share each column sweep (L2
// reuse).  Measured on the 12,252-row projections: 4 beats 2, 6, 8, 16 and 48
// (about 3% against 8 on 5,120 x 13,824, 1.4% on the 5,376 x 28,672 FC1).
__device__ __forceinline__ void grouped_tile(int L, int tm_count, int tn_count, int &tm, int &tn) {
  constexpr int GROUP = 4;
  const int per_group = GROUP * tn_count;
  const int first_tm = (L / per_group) * GROUP;
  const int gsize = min(tm_count - first_tm, GROUP);
  tm = first_tm + (L % per_group) % gsize;
  tn = (L % per_group) / gsize;
}

// The dequantisation epilogue of one accumulator, the same operations in the
// same order as the GEMM's own epilogue: (float)acc * b_scale * a_scale (+ bias);
// rounded to bf16 by bf16_quad.
__device__ __forceinline__ float dequant_f32(int32_t acc, float bs, float as, bool has_bias, uint32_t bias_bits) {
#pragma clang fp contract(off)
  float t = (float)acc;
  t = t * bs;
  t = t * as;
  if (has_bias) t = t + bf16_bits_to_f32(bias_bits);
  return t;
}

// Four floats -> bf16 with gfx950's conversion (round to nearest even, two
// per instruction; the same bits as f32_to_bf16_bits for every non-NaN value).
__device__ __forceinline__ void bf16_quad(const float (&t)[4], uint16_t (&v)[4]) {
  const uint32_t p01 = pack_bf16_rne(t[0], t[1]), p23 = pack_bf16_rne(t[2], t[3]);
  v[0] = (uint16_t)p01, v[1] = (uint16_t)(p01 >> 16), v[2] = (uint16_t)p23, v[3] = (uint16_t)(p23 >> 16);
}

__device__ __forceinline__ int xcd_logical_id(int b, int G) {
  const int xcd = b & 7, pos = b >> 3, per = G >> 3, rem = G & 7;
  return xcd < rem ? xcd * (per + 1) + pos : rem * (per + 1) + (xcd - rem) * per + pos;
}

__device__ __forceinline__ void load_lds16(const void *gptr, void *lds) {
  __builtin_amdgcn_global_load_lds(gptr, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}

template <bool RAW>
__global__ void __launch_bounds__(GWAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_i8_kernel(const GArgs ga) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(1024))) char smem[GRING][GSTAGE];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 31, g = lane >> 5;
  const int wm = w >> 1, wn = w & 1;  // wave tile: a rows [wm*64, +64), b rows [wn*128, +128)
  // grouped tile order: 8 row tiles share each column sweep (L2 reuse)
  const int L = xcd_logical_id(blockIdx.x, gridDim.x);
  constexpr int GROUP = 8;
  const int per_group = GROUP * ga.tn_count;
  const int grp = L / per_group;
  const int first_tm = grp * GROUP;
  const int gsize = min(ga.tm_count - first_tm, GROUP);
  const int tm = first_tm + (L % per_group) % gsize;
  const int tn = (L % per_group) / gsize;
  const int m0 = tm * GBM, n0 = tn * GBN;

  // loads: the a tile (256 rows x 64 B) and b tile are 16 wave loads each; wave w
  // loads blocks w and w + 8 of each (16 rows of 64 B per 1 KiB block)
  const int8_t *asrc[2];
  const int8_t *bsrc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int blk = w + i * GWAVES, row = blk * 16 + (lane >> 2), ch = (lane & 3) ^ ((row >> 2) & 3);
    asrc[i] = ga.a + (int64_t)min(m0 + row, ga.m - 1) * ga.lda + ch * 16;
    bsrc[i] = ga.b + (int64_t)min(n0 + row, ga.n - 1) * ga.ldb + ch * 16;
  }
  auto issue = [&](int kt, char *slot) {
    const int k0 = kt * GBK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      load_lds16(asrc[i] + k0, slot + (w + i * GWAVES) * 1024);
      load_lds16(bsrc[i] + k0, slot + GBM * GBK + (w + i * GWAVES) * 1024);
    }
  };
  // per-lane LDS byte offsets of the MFMA operands (k-step 0; k-step 1 flips chunk bit 1)
  const int arow0 = wm * 64 + lr, brow0 = wn * 128 + lr;
  const int aoff = arow0 * 64 + ((g ^ ((arow0 >> 2) & 3)) * 16);
  const int boff = GBM * GBK + brow0 * 64 + ((g ^ ((brow0 >> 2) & 3)) * 16);

  i32x16 acc[4][2];  // [n block][m block], D[n][m]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  auto compute = [&](const char *slot) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // keep each k-step's operand reads next to its MFMAs (bounds register pressure)
      __builtin_amdgcn_sched_barrier(0);
      // chunk (2*ks + g) ^ sw == (g ^ sw) ^ (2*ks): k-step 1 toggles byte offset bit 5
      i32x4 av[2], bv[4];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int off = aoff + j * 32 * 64;
        av[j] = *(const i32x4 *)(slot + (off ^ (ks * 32)));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int off = boff + i * 32 * 64;
        bv[i] = *(const i32x4 *)(slot + (off ^ (ks * 32)));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv[i], av[j], acc[i][j], 0, 0, 0);
    }
  };

  const int nk = ga.k / GBK;
  issue(0, smem[0]);
  if (nk > 1) issue(1, smem[1]);
  // iteration kt: stage kt ready (wait), everyone past iteration kt-1 (barrier),
  // refill the slot freed by kt-1 with stage kt+2, compute stage kt
  auto step = [&](int kt, char *cur, char *fill) {
    if (kt + 1 < nk)
      __builtin_amdgcn_s_waitcnt(0x0f74);  // vmcnt(4): stage kt+1's 4 loads may stay in flight
    else
      __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 2 < nk) issue(kt + 2, fill);
    compute(cur);
    __builtin_amdgcn_sched_barrier(0);
  };
  // one exit only: the accumulators keep their registers across the unrolled steps
  int kt = 0;
  for (; kt + GRING <= nk; kt += GRING) {
    step(kt, smem[0], smem[2]);
    step(kt + 1, smem[1], smem[0]);
    step(kt + 2, smem[2], smem[1]);
  }
  if (kt < nk) step(kt, smem[0], smem[2]);
  if (kt + 1 < nk) step(kt + 1, smem[1], smem[0]);

  // epilogue: lane holds m = m-block base + lr; n = n-block base + 8u + 4g + (0..3)
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = m0 + wm * 64 + j * 32 + lr;
    if (m >= ga.m) continue;
    const float asm_ = RAW ? 0.0f : ga.as[m];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + wn * 128 + i * 32 + 8 * u + 4 * g;
        if (n >= ga.n) continue;
        if constexpr (RAW) {
          int32_t *op = (int32_t *)ga.out + (int64_t)m * ga.ldo + n;
          if (n + 3 < ga.n) {
            *(i32x4 *)op = i32x4{acc[i][j][4 * u], acc[i][j][4 * u + 1], acc[i][j][4 * u + 2], acc[i][j][4 * u + 3]};
          } else {
            for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = acc[i][j][4 * u + e];
          }
        } else {
          uint16_t *op = (uint16_t *)ga.out + (int64_t)m * ga.ldo + n;
          uint16_t vals[4];
          float tv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int nn = min(n + e, ga.n - 1);
            float t = (float)acc[i][j][4 * u + e];
            t = t * ga.bs[nn];
            t = t * asm_;
            if (ga.bias) t = t + bf16_bits_to_f32(ga.bias[nn]);
            tv[e] = t;
          }
          bf16_quad(tv, vals);
          if (n + 3 < ga.n) {
            *(i32x2 *)op = i32x2{(int)((uint32_t)vals[0] | ((uint32_t)vals[1] << 16)),
                                 (int)((uint32_t)vals[2] | ((uint32_t)vals[3] << 16))};
          } else {
            for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = vals[e];
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// INT8 GEMM, one wave per SIMD: workgroup tile 256 (m) x 256 (n), 4 waves as
// 2 (m) x 2 (n), each wave 128 x 128 (64 blocks of 16 x 16, 256 int32
// accumulators per lane in AGPRs).  A 64-byte k-step reads 8 A and 8 B
// operands (ds_read_b128) for 64 v_mfma_i32_16x16x64_i8; the next k-step's
// reads are issued under the current one's MFMAs, one read per 4 MFMAs.
// The card is power-limited under this loop, and the 16 x 16 shape moves
// half the accumulator bytes per multiply-accumulate of the 32 x 32 one: on
// random int8 operands an MFMA-only stream settles at 4,085 TOPS against
// 3,430 for v_mfma_i32_32x32x32_i8 (1.96 against 1.63 GHz), and this kernel
// runs 7% faster with it than with the 32 x 32 shape at the same tiling.
// k moves in blocks of 128 bytes (two k-steps).  A block's operands sit in
// two ring units, one per 128-row half of the tile (rows of 128 bytes: whole
// cache lines, so each 1 KiB global_load_lds_dwordx4 touches 8 lines and
// every line is fetched once -- against 16 half-used lines per load with
// 64-byte rows, which measured 9% slower on the 12,252 x 5,120 x 13,824
// projection and the 12,252 x 5,376 x 28,672 FC1, with the load path's
// address unit stalled by the L1 27% of the time).  Units cycle through a
// 5-deep ring (5 x 32 KiB, all of the CU's LDS), 96 to 224 bytes of k ahead
// of their first read; a 3-deep ring of 64-byte stages (about 128 bytes
// ahead) was as fast as the 5-deep one, so the shorter lookahead costs
// nothing.
constexpr int HBM_ = 256, HBN = 256, HKD = 128, HWAVES = 4, HRING = 5;
constexpr int HUNIT = 2 * 128 * HKD;  // bytes of one ring unit: 128 rows of A, then of B

// s_waitcnt immediate that leaves n vector-memory operations in flight (and waits for nothing else)
constexpr int vmcnt_imm(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }

__device__ __forceinline__ void hload_lds16(const void *base, uint32_t off, uint32_t lds_addr) {
  asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds_addr) : "memory");
}

// GLU: the weight rows come in blocks of 256 (128 gate rows, then the 128
// matching up rows), so tile column c < 128 and c + 128 are the gate and up of
// one output column; the epilogue writes SwiGLU(gate, up) of the bf16
// projection, out[m][n0 / 2 + c] (ldo counts its columns).
template <bool RAW, bool SPLIT, bool GLU = false>
__global__ void __launch_bounds__(HWAVES * 64) __attribute__((amdgpu_waves_per_eu(1, 1)))
gemm_i8_wave128_kernel(const GArgs ga) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(1024))) char smem[HRING * HUNIT];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;  // wave tile: a rows [wm*128, +128), b rows [wn*128, +128)
  // whole tile, or (SPLIT) k-block range [d_begin, d_end) of a tile of the split round
  const int nd_all = ga.k / HKD;
  int L, part = 0, d_begin = 0, d_end = nd_all;
  if constexpr (SPLIT) {
    const int item = blockIdx.x / ga.nsplit;
    part = blockIdx.x - item * ga.nsplit;
    L = ga.full + item;
    d_begin = nd_all * part / ga.nsplit;
    d_end = nd_all * (part + 1) / ga.nsplit;
  } else {
    L = xcd_logical_id(blockIdx.x, gridDim.x);
  }
  int tm, tn;
  grouped_tile(L, ga.tm_count, ga.tn_count, tm, tn);
  const int m0 = tm * HBM_, n0 = tn * HBN;
  const int8_t *abase = ga.a + (int64_t)d_begin * HKD, *bbase = ga.b + (int64_t)d_begin * HKD;
  const int nd = d_end - d_begin;  // >= 1

  // Unit u = (k block u / 2, row half u % 2): rows [128 h, 128 h + 128) of the
  // A and the B tile over 128 bytes of k, in ring slot u % HRING (16 KiB of A,
  // then 16 KiB of B, rows of 128 bytes).  Chunk c of row r sits at
  // c ^ ((r >> 1) & 7), which keeps the operand reads free of bank conflicts
  // (their pattern is stated with the read offsets below).
  // Loads: a unit is 16 blocks of 1 KiB (8 rows x 128 bytes: whole cache
  // lines) per operand; wave w loads blocks w, w + 4, w + 8, w + 12 of each.
  // Lane: row 8 blk + lane / 8, physical chunk lane % 8, logical chunk
  // (lane % 8) ^ ((row >> 1) & 7) -- the same for all of the wave's blocks,
  // whose parity is w's.
  const int lch = (lane & 7) ^ ((4 * (w & 1) + (lane >> 4)) & 7);
  uint32_t aoff[2][4], boff[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = h * 128 + (w + 4 * i) * 8 + (lane >> 3);
      aoff[h][i] = (uint32_t)((int64_t)min(m0 + row, ga.m - 1) * ga.lda) + lch * 16;
      boff[h][i] = (uint32_t)((int64_t)min(n0 + row, ga.n - 1) * ga.ldb) + lch * 16;
    }
  // load n (0..7) of unit u: n < 4 A block w + 4 n, else B block w + 4 (n - 4).
  // Units past the last k block repeat it (in-bounds bytes into a slot nobody reads).
  auto load_one = [&](int u, int n) {
    const int j = min(u >> 1, nd - 1), h = u & 1, i = n & 3;
    const uint32_t dst = lds0 + (uint32_t)((u % HRING) * HUNIT) + (w + 4 * i) * 1024;
    if (n < 4)
      hload_lds16(abase + (int64_t)j * HKD, aoff[h][i], dst);
    else
      hload_lds16(bbase + (int64_t)j * HKD, boff[h][i], dst + HUNIT / 2);
  };
  // operand read offsets within a unit's operand part, k-step q (0..1) of the
  // block: 16x16x64 operand lane (i, g4) = lane % 16, lane / 16 holds 16 bytes
  // of row i (+ 16 per block) at logical chunk 4 q + g4.  A 16-byte read is
  // served for 32 consecutive lanes at a time from 128 4-byte banks: rows
  // i = 0..15 at two chunks, whose physical chunks under the swizzle fill all
  // 32 16-byte bank groups of the 4 row classes (row stride 128 bytes).
  const int li = lane & 15, lg = lane >> 4;
  uint32_t rdq[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) rdq[q] = (uint32_t)(li * HKD + (((4 * q + lg) ^ ((li >> 1) & 7)) * 16));
  auto rd = [&](uint32_t off) { return *(const i32x4 *)(smem + off); };

  i32x4 acc[8][8];  // [n block][m block], D[n][m]: lane (j, g4) holds n = 16 nb + 4 g4 + (0..3), m = 16 mb + j
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  // prologue: units 0..3 in flight; units 0 and 1 (k block 0) landed
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int n = 0; n < 8; ++n) load_one(u, n);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(16));  // units 2, 3 may stay in flight
  __syncthreads();
  i32x4 cur[16], nxt[16];
  // operand r of k-step q of k block d (ring position dm = d % HRING): r < 8
  // A block r from unit 2 d + wm, else B block r - 8 from unit 2 d + wn
  auto read_op = [&](int dm, int q, int r) -> i32x4 {
    if (r < 8) return rd((uint32_t)(((2 * dm + wm) % HRING) * HUNIT) + rdq[q] + r * 16 * HKD);
    return rd((uint32_t)(((2 * dm + wn) % HRING) * HUNIT + HUNIT / 2) + rdq[q] + (r - 8) * 16 * HKD);
  };
#pragma unroll
  for (int r = 0; r < 16; ++r) cur[r] = read_op(0, 0, r);

  // Epilogue operands: the column scales and bias of n-block i (the lane's
  // columns n = n0 + wn 128 + 16 i + 4 g4 + (0..3)) and the row scales of the
  // lane's 8 m-blocks.  The staged epilogue loads n-block i + 1's while it
  // converts n-block i; a tile that lies inside the matrix in n loads n-block
  // 0's and the row scales during its last k block, so that their latency
  // hides under its MFMAs.
  const bool early = !RAW && !SPLIT && ga.vec_ok && n0 + HBN <= ga.n;
  float asv[8];
  f32x4 bsc, bsn;
  i32x2 bic, bin;
  auto load_row_scales = [&]() {
#pragma unroll
    for (int j = 0; j < 8; ++j) asv[j] = ga.as[min(m0 + wm * 128 + j * 16 + li, ga.m - 1)];
  };
  // VEC: the whole tile lies inside the matrix in n and the scales and bias
  // are aligned for vector loads (`early`)
  auto load_cols = [&](auto vec_c, int i, f32x4 &bs, i32x2 &bi) {
    constexpr bool VEC = decltype(vec_c)::value;
    const int n = n0 + wn * 128 + i * 16 + 4 * lg;
    if (VEC || (ga.vec_ok && n + 3 < ga.n)) {
      bs = *(const f32x4 *)(ga.bs + n);
      bi = ga.bias ? *(const i32x2 *)(ga.bias + n) : i32x2{0, 0};
    } else {
      uint16_t bb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int nn = min(n + e, ga.n - 1);
        bs[e] = ga.bs[nn];
        bb[e] = ga.bias ? ga.bias[nn] : 0;
      }
      bi = i32x2{(int)((uint32_t)bb[0] | ((uint32_t)bb[1] << 16)), (int)((uint32_t)bb[2] | ((uint32_t)bb[3] << 16))};
    }
  };

  // k block d at ring position dm: k-steps 0 and 1 of 64 MFMAs.  MODE 0:
  // unit 2 d + 4 is loaded under k-step 0 and unit 2 d + 5 under k-step 1, one
  // load per 8 MFMAs; one barrier, in front of k-step 1: behind it, units
  // 2 d + 2 and 2 d + 3 (block d + 1) have landed for k-step 1 to read ahead
  // from, and nobody reads block d's units any more (k-step 1's operands are
  // already in registers), so their slots take units 2 d + 5 and 2 d + 6.  The
  // last two blocks load no units (none are left): MODE 1 (next to last) waits
  // for all of its loads before the barrier; MODE 2 (last) reads nothing
  // ahead, needs no barrier, and loads the first epilogue operands.
  auto block = [&](auto dm_v, auto mode_c, int d) {
    constexpr int MODE = decltype(mode_c)::value;
    const int dm = dm_v, dn = (dm + 1) % HRING;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (q == 1 && MODE != 2) {
        if (MODE == 0)
          __builtin_amdgcn_s_waitcnt(0x0f70 | 8);  // vmcnt(8): unit 2 d + 4 may stay in flight
        else
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): block d + 1 has landed
        __syncthreads();
      }
      if constexpr (MODE == 2 && !RAW && !SPLIT)
        if (q == 0 && early) {
          load_row_scales();
          load_cols(std::true_type{}, 0, bsc, bic);
        }
#pragma unroll
      for (int idx = 0; idx < 64; ++idx) {
        if (idx % 4 == 0 && !(MODE == 2 && q == 1))
          nxt[idx / 4] = q == 0 ? read_op(dm, 1, idx / 4) : read_op(dn, 0, idx / 4);
        if (MODE == 0 && q == 0 && idx % 8 == 0) load_one(2 * d + 4, idx / 8);
        if (MODE == 0 && q == 1 && idx % 8 == 0) load_one(2 * d + 5, idx / 8);
        const int nb = idx >> 3, mb = idx & 7;
        acc[nb][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur[8 + nb], cur[mb], acc[nb][mb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!(MODE == 2 && q == 1))
#pragma unroll
        for (int r = 0; r < 16; ++r) cur[r] = nxt[r];
    }
  };
  using M0 = std::integral_constant<int, 0>;
  int d = 0;
  for (; d + HRING <= nd - 2; d += HRING) {
    block(std::integral_constant<int, 0>{}, M0{}, d);
    block(std::integral_constant<int, 1>{}, M0{}, d + 1);
    block(std::integral_constant<int, 2>{}, M0{}, d + 2);
    block(std::integral_constant<int, 3>{}, M0{}, d + 3);
    block(std::integral_constant<int, 4>{}, M0{}, d + 4);
  }
  if (d < nd - 2) block(std::integral_constant<int, 0>{}, M0{}, d);
  if (d + 1 < nd - 2) block(std::integral_constant<int, 1>{}, M0{}, d + 1);
  if (d + 2 < nd - 2) block(std::integral_constant<int, 2>{}, M0{}, d + 2);
  if (d + 3 < nd - 2) block(std::integral_constant<int, 3>{}, M0{}, d + 3);
  // the last two blocks, at ring positions known at run time only
  if (nd >= 2) block((nd - 2) % HRING, std::integral_constant<int, 1>{}, nd - 2);
  block((nd - 1) % HRING, std::integral_constant<int, 2>{}, nd - 1);
  // every wave drains its loads before the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0f70);

  if constexpr (SPLIT) {
    // k-range of a split tile: the raw 256 x 256 int32 partial, row-major
    int32_t *wp = ga.ws + ((int64_t)(L - ga.full) * ga.nsplit + part) * (HBM_ * HBN);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = wm * 128 + j * 16 + li;
#pragma unroll
      for (int i = 0; i < 8; ++i) *(i32x4 *)(wp + m * HBN + wn * 128 + i * 16 + 4 * lg) = acc[i][j];
    }
    return;
  }

  if constexpr (!RAW) {
    if (ga.st_ok) {
      // bf16 tile through LDS: each wave stages its 128 x 128 outputs in rows
      // of 256 bytes whose 16-byte chunk c sits at c ^ stg_sw(row), then
      // writes 16 bytes per lane, 256-byte row segments.  A staging write (8
      // bytes per lane) covers 16 rows x 2 chunks, a read 2 rows x 16 chunks:
      // under the swizzle both meet every bank once.
      constexpr int ROWB = 128 * 2;
      static_assert(HWAVES * 128 * ROWB <= HRING * HUNIT, "staging fits the ring");
      auto stg_sw = [](int row) { return 2 * ((row >> 1) & 7); };
      __syncthreads();  // every wave is done with the ring
      const uint32_t wt = (uint32_t)(w * 128 * ROWB);
      if (!early) {
        load_row_scales();
        load_cols(std::false_type{}, 0, bsc, bic);
      }
      // n-blocks outermost, so that one block's column scales and converted
      // bias are live at a time (the next block's are in flight), and the
      // bias test outside the element loops (per element: convert, two
      // multiplies, the bias add, half a pack)
      auto stage_tile = [&](auto has_bias, auto vec_c) {
        constexpr bool HB = decltype(has_bias)::value;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (i < 7) load_cols(vec_c, i + 1, bsn, bin);
          float bf[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t bw = (uint32_t)bic[e >> 1];
            bf[e] = HB ? bf16_bits_to_f32((e & 1) ? (bw >> 16) : (bw & 0xffffu)) : 0.0f;
          }
          const int ch = 2 * i + (lg >> 1);  // 16-byte chunk of the lane's 4 columns
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            uint16_t vals[4];
            float tv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float t = (float)acc[i][j][e];
              t = t * bsc[e];
              t = t * asv[j];
              if constexpr (HB) t = t + bf[e];
              tv[e] = t;
            }
            bf16_quad(tv, vals);
            const int row = j * 16 + li;
            *(i32x2 *)(smem + wt + row * ROWB + (ch ^ stg_sw(row)) * 16 + (lg & 1) * 8) =
                i32x2{(int)((uint32_t)vals[0] | ((uint32_t)vals[1] << 16)),
                      (int)((uint32_t)vals[2] | ((uint32_t)vals[3] << 16))};
          }
          bsc = bsn;
          bic = bin;
        }
      };
      if (early) {
        if (ga.bias)
          stage_tile(std::true_type{}, std::true_type{});
        else
          stage_tile(std::false_type{}, std::true_type{});
      } else {
        if (ga.bias)
          stage_tile(std::true_type{}, std::false_type{});
        else
          stage_tile(std::false_type{}, std::false_type{});
      }
      if constexpr (GLU) {
        // gate halves sit in the staging rows of waves (wm, 0), up halves in
        // (wm, 1); each wave writes 64 of the tile's 256 output rows
        __syncthreads();
#pragma unroll
        for (int it = 0; it < 16; ++it) {
          const int r = w * 64 + it * 4 + (lane >> 4), c = lane & 15;
          const int wr = r >> 7, rr = r & 127;
          const uint32_t so = (uint32_t)(rr * ROWB + (c ^ stg_sw(rr)) * 16);
          const i32x4 gv = *(const i32x4 *)(smem + (uint32_t)((wr * 2) * 128 * ROWB) + so);
          const i32x4 uv = *(const i32x4 *)(smem + (uint32_t)((wr * 2 + 1) * 128 * ROWB) + so);
          i32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (int)swiglu_pair((uint32_t)gv[e], (uint32_t)uv[e]);
          const int m = m0 + r, n = n0 / 2 + c * 8;
          if (m < ga.m) *(i32x4 *)((uint16_t *)ga.out + (int64_t)m * ga.ldo + n) = o;
        }
        return;
      }
#pragma unroll
      for (int it = 0; it < 32; ++it) {
        const int r = it * 4 + (lane >> 4), c = lane & 15;
        const i32x4 v = *(const i32x4 *)(smem + wt + r * ROWB + (c ^ stg_sw(r)) * 16);
        const int m = m0 + wm * 128 + r, n = n0 + wn * 128 + c * 8;
        if (m < ga.m && n < ga.n) {
          uint16_t *op = (uint16_t *)ga.out + (int64_t)m * ga.ldo + n;
          if (n + 7 < ga.n) {
            *(i32x4 *)op = v;
          } else {
            for (int e = 0; e < 8 && n + e < ga.n; ++e) op[e] = (uint16_t)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
          }
        }
      }
      return;
    }
  }
  if constexpr (GLU) return;  // the GLU launcher always takes the staged path above
  // unstaged epilogue (bf16 rows not 16-byte aligned) and the raw int32 output
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (!RAW) load_cols(std::false_type{}, i, bsc, bic);
    const int n = n0 + wn * 128 + i * 16 + 4 * lg;
    if (n >= ga.n) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = m0 + wm * 128 + j * 16 + li;
      if (m >= ga.m) continue;
      if constexpr (RAW) {
        int32_t *op = (int32_t *)ga.out + (int64_t)m * ga.ldo + n;
        if (n + 3 < ga.n) {
          *(i32x4 *)op = acc[i][j];
        } else {
          for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = acc[i][j][e];
        }
      } else {
        const float asm_ = ga.as[m];
        uint16_t *op = (uint16_t *)ga.out + (int64_t)m * ga.ldo + n;
        uint16_t vals[4];
        float tv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float t = (float)acc[i][j][e];
          t = t * bsc[e];
          t = t * asm_;
          if (ga.bias) {
            const uint32_t bw = (uint32_t)bic[e >> 1];
            t = t + bf16_bits_to_f32((e & 1) ? (bw >> 16) : (bw & 0xffffu));
          }
          tv[e] = t;
        }
        bf16_quad(tv, vals);
        if (n + 3 < ga.n) {
          *(i32x2 *)op = i32x2{(int)((uint32_t)vals[0] | ((uint32_t)vals[1] << 16)),
                               (int)((uint32_t)vals[2] | ((uint32_t)vals[3] << 16))};
        } else {
          for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = vals[e];
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// INT8 GEMM tiles smaller than 256 x 256: 2 MH rows x 2 NH columns, 4 waves as
// 2 x 2 of MH x NH (blocks of v_mfma_i32_16x16x64_i8), for calls and last
// rounds whose 256 x 256 tiles leave CUs idle or compute rows that are not
// there.  k moves in blocks of 128 bytes, two ring units each (one per half of
// the tile's rows and columns, rows of 128 bytes with chunk c of row r at
// c ^ ((r >> 1) & 7), as in the whole-tile kernel), RING units deep.  In block d,
// k-step 0 loads unit 2 d + RING - 1 into the slot of unit 2 d - 1 and reads
// k-step 1's operands; behind the wait (units 2 d + 2 and 2 d + 3 landed) and
// the barrier, k-step 1 loads unit 2 d + RING into the slot of unit 2 d and
// reads block d + 1's first operands.  Reads and loads are dealt between the
// MFMAs.  What bounds these tiles is the latency of their loads (weights come
// from HBM once): a ring of 6 to 10 units, or two workgroups per CU, keeps
// about 100 KiB per CU in flight.
// The MFMAs are inline asm with the accumulators in VGPRs: for rings that allow
// one workgroup per CU the compiler keeps the builtin's accumulators in AGPRs
// and copies them around every MFMA (12 instructions each; 192 x 128 tiles on
// 331 x 5,376 x 10,752: 43 against 32 us).
// Tile choice and times: see pick_tile.
//
// GLU: the tile's columns are NH gate columns and their NH up columns (128
// weight rows on), in the waves (wm, 0) and (wm, 1); each hands half of its
// bf16 projection to the other through LDS and writes SwiGLU of the half it
// keeps.

__device__ __forceinline__ void mfma_i8(i32x4 &acc, const i32x4 &b, const i32x4 &a) {
  asm("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(acc) : "v"(b), "v"(a));
}

template <int MH, int NH, int RING, int WPE, bool RAW, bool GLU>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
gemm_i8_tile_kernel(const GArgs ga) {
#pragma clang fp contract(off)
  constexpr int BM = 2 * MH, BN = 2 * NH, UNIT = (MH + NH) * HKD;
  constexpr int AL = MH / 32, NL = (MH + NH) / 32;  // 1 KiB loads per wave and unit: of A, in all
  constexpr int MB = MH / 16, NB = NH / 16, NR = MB + NB, NM = MB * NB;
  constexpr int RS = NM / NR > 0 ? NM / NR : 1, LS = NM / NL > 0 ? NM / NL : 1;  // MFMAs per operand read / load
  static_assert(RING >= 5 && RING * UNIT <= 160 * 1024 && (RING - 3) * NL < 64, "ring fits the LDS and vmcnt");
  static_assert(NM >= NR && NM >= NL, "reads and loads fit between a k-step's MFMAs");
  static_assert(!GLU || (128 % NH == 0 && !RAW), "gate and up columns in blocks of 128");
  __shared__ __attribute__((aligned(1024))) char smem[RING * UNIT];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;
  const int L = xcd_logical_id(blockIdx.x, gridDim.x);
  // first row; column tile (of BN columns, or BN / 2 outputs)
  constexpr int PN = HBN / BN;  // column tiles of a 256 x 256 tile
  int m0, ct;
  if (ga.full >= 0) {
    // part of 256 x 256 tile full + L / parts: consecutive ids, which run on one
    // XCD (its L2 holds their panels)
    constexpr int PARTS = (HBM_ / BM > 0 ? HBM_ / BM : 1) * PN;
    const int sub = L % PARTS;
    int tm, tn;
    grouped_tile(ga.full + L / PARTS, ga.tm_count, ga.tn_count, tm, tn);
    m0 = tm * HBM_ + sub / PN * BM;
    ct = tn * PN + sub % PN;
  } else {
    // the row tiles that share a weight panel run next to each other
    const int tmc = (ga.m + BM - 1) / BM;
    ct = L / tmc;
    m0 = (L - ct * tmc) * BM;
  }
  // weight rows of the waves' halves: n0 + h * NS ..
  constexpr int NS = GLU ? 128 : NH;
  const int n0 = GLU ? ct / PN * HBN + ct % PN * NH : ct * BN;
  if (m0 >= ga.m || n0 >= ga.n) return;  // the whole workgroup: no barrier is left waiting
  const int nd = ga.k / HKD;  // >= 1
  // Wave w loads 8-row blocks w, w + 4, ... of each operand.  Lane: row 8 blk +
  // lane / 8, physical chunk lane % 8, logical chunk (lane % 8) ^ ((row >> 1) & 7),
  // the same for all of the wave's blocks (their parity is w's).
  const int lch = (lane & 7) ^ ((4 * (w & 1) + (lane >> 4)) & 7);
  uint32_t soff[2][NL];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      if (i < AL)
        soff[h][i] = (uint32_t)((int64_t)min(m0 + h * MH + (w + 4 * i) * 8 + (lane >> 3), ga.m - 1) * ga.lda) + lch * 16;
      else
        soff[h][i] =
            (uint32_t)((int64_t)min(n0 + h * NS + (w + 4 * (i - AL)) * 8 + (lane >> 3), ga.n - 1) * ga.ldb) + lch * 16;
    }
  // load i of unit (k block j, half h) into ring slot `slot`; units past the
  // last block repeat it, into a slot nobody reads
  auto load_one = [&](int j, int h, int slot, int i) {
    const uint32_t at = i < AL ? (w + 4 * i) * 1024 : MH * HKD + (w + 4 * (i - AL)) * 1024;
    hload_lds16((i < AL ? ga.a : ga.b) + (int64_t)min(j, nd - 1) * HKD, soff[h][i], lds0 + (uint32_t)(slot * UNIT) + at);
  };
  // operand reads: 16x16x64 lane (i, g4) holds 16 bytes of row i at logical chunk 4 q + g4
  const int li = lane & 15, lg = lane >> 4;
  uint32_t rdq[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) rdq[q] = (uint32_t)(li * HKD + (((4 * q + lg) ^ ((li >> 1) & 7)) * 16));
  // operand r of k-step q of the block whose units are in slots s0 and s1: r < MB A block r, else B block r - MB
  auto read_op = [&](int s0, int s1, int q, int r) -> i32x4 {
    if (r < MB) return *(const i32x4 *)(smem + (uint32_t)((wm ? s1 : s0) * UNIT) + rdq[q] + r * 16 * HKD);
    return *(const i32x4 *)(smem + (uint32_t)((wn ? s1 : s0) * UNIT + MH * HKD) + rdq[q] + (r - MB) * 16 * HKD);
  };
  i32x4 acc[NB][MB];  // D[n][m]: lane (j, g4) holds n = 16 nb + 4 g4 + (0..3), m = 16 mb + j
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  // prologue: units 0 .. RING - 2 in flight, units 0 and 1 landed
#pragma unroll
  for (int u = 0; u < RING - 1; ++u)
#pragma unroll
    for (int i = 0; i < NL; ++i) load_one(u >> 1, u & 1, u, i);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 3) * NL));
  __syncthreads();
  i32x4 cur[NR], nxt[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) cur[r] = read_op(0, 1, 0, r);
  auto step = [](int s, int by) { return s + by >= RING ? s + by - RING : s + by; };
  int s0 = 0;  // slot of unit 2 d
  for (int d = 0; d < nd; ++d) {
    const int s1 = step(s0, 1), sp = step(s0, RING - 1), t0 = step(s0, 2), t1 = step(s0, 3);
#pragma unroll
    for (int idx = 0; idx < NM; ++idx) {
      if (idx % RS == 0 && idx / RS < NR) nxt[idx / RS] = read_op(s0, s1, 1, idx / RS);
      if (idx % LS == 0 && idx / LS < NL) load_one(d + (RING - 1) / 2, (RING - 1) & 1, sp, idx / LS);
      mfma_i8(acc[idx / MB][idx % MB], cur[MB + idx / MB], cur[idx % MB]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 4) * NL));
    __syncthreads();
    // (after the last block: a stale slot, unused)
#pragma unroll
    for (int idx = 0; idx < NM; ++idx) {
      if (idx % RS == 0 && idx / RS < NR) cur[idx / RS] = read_op(t0, t1, 0, idx / RS);
      if (idx % LS == 0 && idx / LS < NL) load_one(d + RING / 2, RING & 1, s0, idx / LS);
      mfma_i8(acc[idx / MB][idx % MB], nxt[MB + idx / MB], nxt[idx % MB]);
      __builtin_amdgcn_sched_barrier(0);
    }
    s0 = t0;
  }
  // every wave drains its loads before the workgroup ends; the accumulators'
  // wait states before VALU code reads them
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) asm volatile("" : "+v"(acc[i][j]));

  // epilogue straight from registers: 4 consecutive n of one m per lane
  float asv[MB];
  if constexpr (!RAW) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) asv[mb] = ga.as[min(m0 + wm * MH + mb * 16 + li, ga.m - 1)];
  }
  auto columns = [&](int nb, float (&bsv)[4], uint16_t (&bbv)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nn = min(n0 + wn * NS + nb * 16 + 4 * lg + e, ga.n - 1);
      bsv[e] = ga.bs[nn];
      bbv[e] = ga.bias ? ga.bias[nn] : 0;
    }
  };
  auto project = [&](const i32x4 &v, const float (&bsv)[4], const uint16_t (&bbv)[4], float as) {
    float t[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = dequant_f32(v[e], bsv[e], as, ga.bias != nullptr, bbv[e]);
    return i32x2{(int)pack_bf16_rne(t[0], t[1]), (int)pack_bf16_rne(t[2], t[3])};
  };
  if constexpr (GLU) {
    // wave (wm, 0) keeps gate blocks [0, NB / 2) and hands over the rest, wave
    // (wm, 1) keeps up blocks [NB / 2, NB); lane layouts agree
    constexpr int HALF = NB / 2;
    static_assert(4 * HALF * MB * 512 <= RING * UNIT, "the exchange fits the ring");
    __syncthreads();  // every wave is done with the ring
    i32x2 kept[HALF][MB];
    char *mine = smem + w * (HALF * MB * 512) + lane * 8;
    const char *theirs = smem + (w ^ 1) * (HALF * MB * 512) + lane * 8;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float bsv[4];
      uint16_t bbv[4];
      columns(nb, bsv, bbv);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const i32x2 v = project(acc[nb][mb], bsv, bbv, asv[mb]);
        const int i = (nb % HALF) * MB + mb;
        if ((nb >= HALF) == (wn == 1))
          kept[nb % HALF][mb] = v;
        else
          *(i32x2 *)(mine + i * 512) = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < HALF; ++nb) {
      const int n = ct * NH + (wn * HALF + nb) * 16 + 4 * lg;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const i32x2 other = *(const i32x2 *)(theirs + (nb * MB + mb) * 512);
        const i32x2 g = wn ? other : kept[nb][mb], u = wn ? kept[nb][mb] : other;
        const int m = m0 + wm * MH + mb * 16 + li;
        if (m < ga.m)
          *(i32x2 *)((uint16_t *)ga.out + (int64_t)m * ga.ldo + n) =
              i32x2{(int)swiglu_pair((uint32_t)g[0], (uint32_t)u[0]), (int)swiglu_pair((uint32_t)g[1], (uint32_t)u[1])};
      }
    }
    return;
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = n0 + wn * NH + nb * 16 + 4 * lg;
    if (n >= ga.n) continue;
    float bsv[4];
    uint16_t bbv[4];
    if constexpr (!RAW) columns(nb, bsv, bbv);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + wm * MH + mb * 16 + li;
      if (m >= ga.m) continue;
      if constexpr (RAW) {
        int32_t *op = (int32_t *)ga.out + (int64_t)m * ga.ldo + n;
        if (n + 3 < ga.n)
          *(i32x4 *)op = acc[nb][mb];
        else
          for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = acc[nb][mb][e];
      } else {
        const i32x2 v = project(acc[nb][mb], bsv, bbv, asv[mb]);
        uint16_t *op = (uint16_t *)ga.out + (int64_t)m * ga.ldo + n;
        if (n + 3 < ga.n && ga.st_ok)
          *(i32x2 *)op = v;
        else
          for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = (uint16_t)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
      }
    }
  }
}

// Merge of the K-split GLU tiles: gate columns c .. c + 3 and up columns
// 128 + c .. of one row, each the sum of its partials, dequantised and
// rounded as the GEMM's epilogue does, then SwiGLU.  Block: 8 rows of one
// tile, 4 output columns per thread.
__global__ void __launch_bounds__(256) gemm_split_merge_glu_kernel(const GArgs ga) {
  const int item = blockIdx.x / (HBM_ / 8);
  const int r = (blockIdx.x % (HBM_ / 8)) * 8 + (threadIdx.x >> 5);
  const int c = (threadIdx.x & 31) * 4;
  int tm, tn;
  grouped_tile(ga.full + item, ga.tm_count, ga.tn_count, tm, tn);
  const int m = tm * HBM_ + r, n0 = tn * HBN;
  if (m >= ga.m) return;
  const int32_t *wp = ga.ws + (int64_t)item * ga.nsplit * (HBM_ * HBN) + r * HBN + c;
  i32x4 ag = *(const i32x4 *)wp, au = *(const i32x4 *)(wp + 128);
  for (int p = 1; p < ga.nsplit; ++p) {
    ag += *(const i32x4 *)(wp + (int64_t)p * (HBM_ * HBN));
    au += *(const i32x4 *)(wp + (int64_t)p * (HBM_ * HBN) + 128);
  }
  const float asm_ = ga.as[m];
  float tg[4], tu[4];
  uint16_t vg[4], vu[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ng = n0 + c + e, nu = ng + 128;
    tg[e] = dequant_f32(ag[e], ga.bs[ng], asm_, ga.bias != nullptr, ga.bias ? ga.bias[ng] : 0u);
    tu[e] = dequant_f32(au[e], ga.bs[nu], asm_, ga.bias != nullptr, ga.bias ? ga.bias[nu] : 0u);
  }
  bf16_quad(tg, vg);
  bf16_quad(tu, vu);
  const uint32_t o0 = swiglu_pair((uint32_t)vg[0] | ((uint32_t)vg[1] << 16), (uint32_t)vu[0] | ((uint32_t)vu[1] << 16));
  const uint32_t o1 = swiglu_pair((uint32_t)vg[2] | ((uint32_t)vg[3] << 16), (uint32_t)vu[2] | ((uint32_t)vu[3] << 16));
  *(i32x2 *)((uint16_t *)ga.out + (int64_t)m * ga.ldo + n0 / 2 + c) = i32x2{(int)o0, (int)o1};
}

// Merge of the K-split tiles: the sum of each tile's nsplit int32 partials
// (exact), then the GEMM's epilogue.  Block: 4 rows of one tile, 4 columns
// per thread.
template <bool RAW>
__global__ void __launch_bounds__(256) gemm_split_merge_kernel(const GArgs ga) {
  const int item = blockIdx.x / (HBM_ / 4);
  const int r = (blockIdx.x % (HBM_ / 4)) * 4 + (threadIdx.x >> 6);
  const int c = (threadIdx.x & 63) * 4;
  int tm, tn;
  grouped_tile(ga.full + item, ga.tm_count, ga.tn_count, tm, tn);
  const int m = tm * HBM_ + r, n = tn * HBN + c;
  if (m >= ga.m || n >= ga.n) return;
  const int32_t *wp = ga.ws + (int64_t)item * ga.nsplit * (HBM_ * HBN) + r * HBN + c;
  i32x4 acc = *(const i32x4 *)wp;
  for (int p = 1; p < ga.nsplit; ++p) acc += *(const i32x4 *)(wp + (int64_t)p * (HBM_ * HBN));
  if constexpr (RAW) {
    int32_t *op = (int32_t *)ga.out + (int64_t)m * ga.ldo + n;
    if (n + 3 < ga.n)
      *(i32x4 *)op = acc;
    else
      for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = acc[e];
  } else {
    const float asm_ = ga.as[m];
    uint16_t vals[4];
    float tv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nn = min(n + e, ga.n - 1);
      tv[e] = dequant_f32(acc[e], ga.bs[nn], asm_, ga.bias != nullptr, ga.bias ? ga.bias[nn] : 0u);
    }
    bf16_quad(tv, vals);
    uint16_t *op = (uint16_t *)ga.out + (int64_t)m * ga.ldo + n;
    if (n + 3 < ga.n)
      *(i32x2 *)op = i32x2{(int)((uint32_t)vals[0] | ((uint32_t)vals[1] << 16)),
                           (int)((uint32_t)vals[2] | ((uint32_t)vals[3] << 16))};
    else
      for (int e = 0; e < 4 && n + e < ga.n; ++e) op[e] = vals[e];
  }
}

// The k split that a last, partial round of 256 x 256 tiles (all tiles when they
// fill less than half the CUs) may take: its tiles' 128-byte k blocks are dealt
// to S parts, S up to CUs / tiles and at least 2 blocks per part, so that the
// round fills the CUs (1: no split); the partials are merged by
// gemm_split_merge_kernel.
int split_parts(int64_t tail, int32_t k, int cus) {
  return 2 * tail > cus ? 1 : std::max(1, (int)std::min<int64_t>(cus / tail, (k / HKD) / 2));
}

int64_t gemm_split_bytes(int64_t tail, int parts) { return tail * parts * HBM_ * HBN * 4; }

// How the last, partial round of 256 x 256 tiles runs (all tiles, when they do
// not fill a round).
enum Tail {
  kTailWhole = TMHD_GEMM_WHOLE,
  kTailSplit = TMHD_GEMM_SPLIT_K,
  kTail64x64 = TMHD_GEMM_64X64,
  kTail64x128 = TMHD_GEMM_64X128,
  kTail128 = TMHD_GEMM_128X128,
  kTail192x128 = TMHD_GEMM_192X128,
  kTail256x128 = TMHD_GEMM_256X128,
};

// The tiles of gemm_i8_tile_kernel and, per 128-byte block of k, the
// microseconds of a round of them: `one` + `fill` * (share of the CUs in use),
// or `two` with a second workgroup on each CU.
struct TileCost {
  Tail tail;
  int bm, bn, per_cu;
  double one, fill, two;
};
constexpr TileCost kTiles[] = {
    {kTail64x64, 64, 64, 2, 0.19, 0.02, 0.37},     {kTail64x128, 64, 128, 2, 0.24, 0.09, 0.62},
    {kTail128, 128, 128, 1, 0.42, 0.14, 0.0},      {kTail192x128, 192, 128, 1, 0.58, 0.22, 0.0},
    {kTail256x128, 256, 128, 1, 0.78, 0.26, 0.0},
};
constexpr double kTileRoundUs = 5.0;  // a round of them besides its k blocks: first loads, epilogue

// Cheapest form for `tiles` 256 x 256 tiles (fewer than cus) of an m x n x k
// product; `part`: they are the last round of more.  Fitted to k = 5,120 and
// 5,376, and checked with every form forced, on weights not read shortly
// before, over 768 products of 1 to 5,000 rows, 16 to 28,672 columns and k of
// 128 to 13,824 (profiles/gemm_form_sweep.txt): within 10% of the best form in
// all but one of 658 with k up to 7,168 (that one 15%); with longer k the split
// is taken for few tiles where 64 x 64 tiles would be up to 1.6 times as fast.
// us, m x n x k:
//   16 x 13,824 x 5,120: 64 x 64 tiles 17, 64 x 128 25, k split 34, whole 51
//   331 x 13,824 x 5,120: 192 x 128 tiles 39, k split 49, whole 55, 64 x 64 58
//   331 x 10,752 x 5,376: 128 x 128 30, 192 x 128 36, 64 x 128 38, k split 45
//   512 x 5,376 x 5,376: 128 x 128 31, 64 x 64 38, k split 40, whole 59
//   1,024 x 10,752 x 5,376 (168 tiles): whole 60, 192 x 128 68, 256 x 128 84
//   1,024 x 28,672 x 640: whole 37, 64 x 128 to 256 x 128 48 (two rounds or more)
// The k split remains for long k (8 tiles of 32,768: 26 against 56 us estimated).
Tail pick_tail(int64_t tiles, bool part, int32_t m, int32_t n, int32_t k, int cus, int parts) {
  const double nd = (double)(k / HKD);
  Tail best = kTailWhole;
  double us = nd * (0.95 + 0.45 * (double)tiles / cus) + 8.0;
  if (parts > 1) {
    // 14 us of launches and merge, and per tile the write and read of its partials
    const double t = nd / parts * 1.35 + 14.0 + 0.165 * (double)tiles;
    if (t < us) us = t, best = kTailSplit;
  }
  for (const TileCost &c : kTiles) {
    if (part && HBM_ % c.bm) continue;  // parts of a 256 x 256 tile divide it
    const int64_t wgs = part ? tiles * (HBM_ / c.bm) * (HBN / c.bn)
                             : (int64_t)((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
    const int64_t slots = (int64_t)cus * c.per_cu, rest = wgs % slots;
    const double full = c.per_cu == 2 ? c.two : c.one + c.fill;
    const double last = rest == 0 ? 0.0 : rest <= cus ? c.one + c.fill * (double)rest / cus : c.two;
    const double t = kTileRoundUs * (double)((wgs + slots - 1) / slots) + nd * ((double)(wgs / slots) * full + last);
    if (t < us) us = t, best = c.tail;
  }
  return best;
}

// The last, partial round of an m x n x k product whose rounds the whole-tile
// kernel runs: its 256 x 256 tiles (0: none, every round is whole), its form
// with a workspace of ws_bytes, and for the k split the parts.
struct LastRound {
  int64_t tiles;
  Tail form;
  int parts;
};
LastRound last_round(int32_t m, int32_t n, int32_t k, int64_t ws_bytes, int cus) {
  const int64_t tiles = (int64_t)((m + HBM_ - 1) / HBM_) * ((n + HBN - 1) / HBN);
  LastRound r{cus > 0 ? tiles % cus : 0, kTailWhole, 1};
  if (r.tiles == 0) return r;
  r.parts = split_parts(r.tiles, k, cus);
  if (ws_bytes < gemm_split_bytes(r.tiles, r.parts)) r.parts = 1;
  r.form = pick_tail(r.tiles, r.tiles < tiles, m, n, k, cus, r.parts);
  return r;
}

template <int MH, int NH, int RING, int WPE, bool RAW, bool GLU>
void launch_tiles(GArgs ga, int64_t tiles, bool part, hipStream_t s) {
  const int64_t wgs = part ? tiles * (HBM_ / (2 * MH)) * (HBN / (2 * NH))
                           : (int64_t)((ga.m + 2 * MH - 1) / (2 * MH)) * ((ga.n + 2 * NH - 1) / (2 * NH));
  if (!part) ga.full = -1;
  hipLaunchKernelGGL((gemm_i8_tile_kernel<MH, NH, RING, WPE, RAW, GLU>), dim3((unsigned)wgs), dim3(256), 0, s, ga);
}

// The GEMM (checked arguments, 32-bit row offsets, whole 128-byte k blocks) in
// rounds of whole tiles and a last round as pick_tail says.  ga.full: all tiles.
template <bool RAW, bool GLU>
void launch_rounds(GArgs ga, void *ws, int64_t ws_bytes, hipStream_t s) {
  const bool ws_ok = ws && ((uintptr_t)ws % 16) == 0;
  const LastRound r = last_round(ga.m, ga.n, ga.k, ws_ok ? ws_bytes : 0, device_cus());
  const int64_t last = r.tiles;
  if (r.form != kTailWhole) ga.full -= (int32_t)last;
  const bool part = ga.full > 0;
  if (part)
    hipLaunchKernelGGL((gemm_i8_wave128_kernel<RAW, false, GLU>), dim3((unsigned)ga.full), dim3(HWAVES * 64), 0, s, ga);
  switch (r.form) {
    case kTailWhole:
      break;
    case kTailSplit:
      ga.nsplit = r.parts;
      ga.ws = (int32_t *)ws;
      hipLaunchKernelGGL((gemm_i8_wave128_kernel<false, true>), dim3((unsigned)(last * r.parts)), dim3(HWAVES * 64), 0, s, ga);
      if constexpr (GLU)
        hipLaunchKernelGGL(gemm_split_merge_glu_kernel, dim3((unsigned)(last * (HBM_ / 8))), dim3(256), 0, s, ga);
      else
        hipLaunchKernelGGL(gemm_split_merge_kernel<RAW>, dim3((unsigned)(last * (HBM_ / 4))), dim3(256), 0, s, ga);
      break;
    case kTail64x64:
      launch_tiles<32, 32, 10, 2, RAW, GLU>(ga, last, part, s);
      break;
    case kTail64x128:
      launch_tiles<32, 64, 6, 2, RAW, GLU>(ga, last, part, s);
      break;
    case kTail128:
      launch_tiles<64, 64, 9, 1, RAW, GLU>(ga, last, part, s);
      break;
    case kTail192x128:
      launch_tiles<96, 64, 7, 1, RAW, GLU>(ga, last, part, s);
      break;
    case kTail256x128:
      launch_tiles<128, 64, 6, 1, RAW, GLU>(ga, last, part, s);
  }
}

template <bool RAW>
int launch_gemm(void *out, const int8_t *a, const int8_t *b, const float *as, const float *bs, const void *bias,
                int32_t m, int32_t n, int32_t k, int64_t lda, int64_t ldb, int64_t ldo, void *ws, int64_t ws_bytes,
                void *stream) {
  const char *what = RAW ? "tmhd_gemm_i8_i32" : "tmhd_gemm_w8a8";
  if (m < 0 || n <= 0 || k <= 0) return set_error(TMHD_ERR_INVALID, "%s: m %d n %d k %d", what, m, n, k);
  if (k % GBK) return set_error(TMHD_ERR_UNSUPPORTED, "%s: k %d must be a multiple of %d", what, k, GBK);
  if (!out || !a || !b || (!RAW && (!as || !bs))) return set_error(TMHD_ERR_INVALID, "%s: null pointer", what);
  if (((uintptr_t)a % 16) || ((uintptr_t)b % 16) || lda % 16 || ldb % 16 || lda < k || ldb < k || ldo < n)
    return set_error(TMHD_ERR_INVALID, "%s: operands must be 16-byte aligned rows with stride >= k", what);
  if (m == 0) return TMHD_OK;
  const int64_t tiles = (int64_t)((m + GBM - 1) / GBM) * ((n + GBN - 1) / GBN);
  GArgs ga{a, b, out, as, bs, (const uint16_t *)bias, m, n, k, lda, ldb, ldo, (m + GBM - 1) / GBM, (n + GBN - 1) / GBN,
           (int32_t)(((uintptr_t)bs % 16) == 0 && ((uintptr_t)bias % 8) == 0),
           (int32_t)(!RAW && ((uintptr_t)out % 16) == 0 && ldo % 8 == 0), (int32_t)tiles, 1, nullptr};
  // the one-wave-per-SIMD kernel takes 32-bit row offsets and whole 128-byte
  // k blocks; other shapes (k an odd multiple of 64) run the 8-wave kernel
  const bool wide = (int64_t)(m - 1) * lda + k < ((int64_t)1 << 32) &&
                    (int64_t)(n - 1) * ldb + k < ((int64_t)1 << 32);
  if (wide && k % HKD == 0)
    launch_rounds<RAW, false>(ga, ws, ws_bytes, (hipStream_t)stream);
  else
    hipLaunchKernelGGL(gemm_i8_kernel<RAW>, dim3((unsigned)tiles), dim3(GWAVES * 64), 0, (hipStream_t)stream, ga);
  return check_launch(what);
}

// The GEMM with the SwiGLU epilogue: out[m][n / 2] from gate / up rows
// interleaved in blocks of 128 (see the GLU kernels).
int launch_gemm_glu(void *out, const int8_t *a, const int8_t *b, const float *as, const float *bs, const void *bias,
                    int32_t m, int32_t n, int32_t k, int64_t lda, int64_t ldb, int64_t ldo, void *ws,
                    int64_t ws_bytes, void *stream) {
  const char *what = "tmhd_gemm_w8a8_swiglu_ws";
  if (m < 0 || n <= 0 || k <= 0) return set_error(TMHD_ERR_INVALID, "%s: m %d n %d k %d", what, m, n, k);
  if (k % HKD || n % 256)
    return set_error(TMHD_ERR_UNSUPPORTED, "%s: k %d (a multiple of %d), n %d (gate + up, a multiple of 256)", what,
                     k, HKD, n);
  if (!out || !a || !b || !as || !bs) return set_error(TMHD_ERR_INVALID, "%s: null pointer", what);
  if (((uintptr_t)a % 16) || ((uintptr_t)b % 16) || lda % 16 || ldb % 16 || lda < k || ldb < k || ldo < n / 2 ||
      ((uintptr_t)out % 16) || ldo % 8)
    return set_error(TMHD_ERR_INVALID, "%s: operands and output must be 16-byte aligned rows", what);
  if (m == 0) return TMHD_OK;
  if (!((int64_t)(m - 1) * lda + k < ((int64_t)1 << 32) && (int64_t)(n - 1) * ldb + k < ((int64_t)1 << 32)))
    return set_error(TMHD_ERR_UNSUPPORTED, "%s: operands beyond 32-bit row offsets", what);
  const int64_t tiles = (int64_t)((m + HBM_ - 1) / HBM_) * (n / HBN);
  GArgs ga{a, b, out, as, bs, (const uint16_t *)bias, m, n, k, lda, ldb, ldo, (m + HBM_ - 1) / HBM_, n / HBN,
           (int32_t)(((uintptr_t)bs % 16) == 0 && ((uintptr_t)bias % 8) == 0), 1, (int32_t)tiles, 1, nullptr};
  launch_rounds<false, true>(ga, ws, ws_bytes, (hipStream_t)stream);
  return check_launch(what);
}

}  // namespace
}  // namespace tmhd

extern "C" int tmhd_token_quant_i8(int8_t *q, float *scale, const void *x, int32_t rows, int32_t cols,
                                   int64_t x_stride, void *stream) {
  return tmhd::launch_row_quant<false>(q, scale, x, rows, cols, x_stride, stream, "tmhd_token_quant_i8");
}

extern "C" int tmhd_weight_quant_i8(int8_t *q, float *scale, const void *w, int32_t n, int32_t k, void *stream) {
  return tmhd::launch_row_quant<true>(q, scale, w, n, k, k, stream, "tmhd_weight_quant_i8");
}

extern "C" int tmhd_gemm_w8a8(void *out, const int8_t *a, const int8_t *b, const float *a_scale,
                              const float *b_scale, const void *bias, int32_t m, int32_t n, int32_t k, int64_t lda,
                              int64_t ldb, int64_t ldo, void *stream) {
  return tmhd::launch_gemm<false>(out, a, b, a_scale, b_scale, bias, m, n, k, lda, ldb, ldo, nullptr, 0, stream);
}

extern "C" int tmhd_gemm_i8_i32(int32_t *out, const int8_t *a, const int8_t *b, int32_t m, int32_t n, int32_t k,
                                int64_t lda, int64_t ldb, int64_t ldo, void *stream) {
  return tmhd::launch_gemm<true>(out, a, b, nullptr, nullptr, nullptr, m, n, k, lda, ldb, ldo, nullptr, 0, stream);
}

extern "C" int tmhd_gemm_last_round_form(int32_t m, int32_t n, int32_t k, int64_t workspace_bytes, int32_t cus) {
  using namespace tmhd;
  if (m <= 0 || n <= 0 || k <= 0 || k % HKD) return -1;
  return last_round(m, n, k, workspace_bytes, cus > 0 ? cus : device_cus()).form;
}

extern "C" int64_t tmhd_gemm_split_workspace_bytes(int32_t m, int32_t n, int32_t k) {
  using namespace tmhd;
  if (m <= 0 || n <= 0 || k <= 0 || k % HKD) return 0;
  const LastRound r = last_round(m, n, k, INT64_MAX, device_cus());
  return r.form == kTailSplit ? gemm_split_bytes(r.tiles, r.parts) : 0;
}

extern "C" int tmhd_gemm_w8a8_ws(void *out, const int8_t *a, const int8_t *b, const float *a_scale,
                                 const float *b_scale, const void *bias, int32_t m, int32_t n, int32_t k, int64_t lda,
                                 int64_t ldb, int64_t ldo, void *workspace, int64_t workspace_bytes, void *stream) {
  return tmhd::launch_gemm<false>(out, a, b, a_scale, b_scale, bias, m, n, k, lda, ldb, ldo, workspace,
                                  workspace_bytes, stream);
}

extern "C" int tmhd_gemm_i8_i32_ws(int32_t *out, const int8_t *a, const int8_t *b, int32_t m, int32_t n, int32_t k,
                                   int64_t lda, int64_t ldb, int64_t ldo, void *workspace, int64_t workspace_bytes,
                                   void *stream) {
  return tmhd::launch_gemm<true>(out, a, b, nullptr, nullptr, nullptr, m, n, k, lda, ldb, ldo, workspace,
                                 workspace_bytes, stream);
}

extern "C" int tmhd_gemm_w8a8_swiglu_ws(void *out, const int8_t *a, const int8_t *b, const float *a_scale,
                                        const float *b_scale, const void *bias, int32_t m, int32_t n, int32_t k,
                                        int64_t lda, int64_t ldb, int64_t ldo, void *workspace,
                                        int64_t workspace_bytes, void *stream) {
  return tmhd::launch_gemm_glu(out, a, b, a_scale, b_scale, bias, m, n, k, lda, ldb, ldo, workspace, workspace_bytes,
                               stream);
}
