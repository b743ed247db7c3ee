// Slot packing (token-major K/V rows -> head-major slot) and the smooth-K
// INT8 quantization of the INT8-QK attention path.
#include <math.h>

#include <algorithm>

#include "tmhd_internal.h"
#include "tmhd_pack.h"

namespace tmhd {
namespace {

constexpr int kTile = kPackTile;

// ---------------------------------------------------------------------------
// tmhd_kv_pack: one workgroup = 64 slot positions of one head, D threads (see
// pack_block).  A launch packs up to kMaxRanges row ranges: the 64-position
// blocks from blk0 on are range i's (one launch per range instead cost 5 to
// 9 us each for ranges of 77 to 1,337 rows).  A launch of one range, the most
// usual, takes arguments of its own size (N 1): with the whole table and the
// search 4.0 us for 8 heads of 128 and 77 rows, 3.85 without, and 0.15 to 0.2
// at every size.
constexpr int kMaxRanges = 32;
struct PackRange {
  const int32_t *rows;
  int32_t row0, n, dst, zero_to;
  int32_t p_begin;  // slot position of its first block
  int32_t blk0;     // its first block in the launch
};
template <int N>
struct PackArgs {
  const uint16_t *k, *v;
  int64_t ts, hs;
  uint16_t *ks, *vts;
  int64_t khs, vhs;
  int32_t vrs, nranges;
  PackRange r[N];
};

template <int D, int N>
__global__ void __launch_bounds__(D) kv_pack_kernel(const PackArgs<N> a) {
  int ri = 0;
  while (N > 1 && ri + 1 < a.nranges && (int)blockIdx.x >= a.r[ri + 1].blk0) ++ri;
  const PackRange &R = a.r[ri];
  pack_block<D, true>(a.k, a.v, a.ts, a.hs, R.rows, R.row0, R.n, a.ks, a.vts, a.khs, a.vhs, a.vrs, R.dst, R.zero_to,
                        R.p_begin + ((int)blockIdx.x - R.blk0) * kTile, blockIdx.y, threadIdx.x);
}

// ---------------------------------------------------------------------------
// Smooth-K mean.  Keys are summed exactly as int64 fixed point (x * 2^24,
// rounded to nearest even), so the sum does not depend on the order of the
// parallel reduction; mean = bf16(fp32(sum * 2^-24 / N)).
constexpr double kMeanFix = 16777216.0;  // 2^24

__global__ void zero_i64_kernel(int64_t *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__device__ __forceinline__ int64_t to_fixed(float x) {
  float y = x * 16777216.0f;
  y = fminf(fmaxf(y, -4.0e18f), 4.0e18f);
  return (int64_t)__builtin_rintf(y);
}

// Limits of one smooth-quant launch: calls, and key segments over all of them.
constexpr int kMaxCalls = 16, kMaxBatchSeg = 24;

// Key segments whose sums a launch takes: workgroups [blk0[i], blk0[i + 1]) of
// the grid's x dimension cover segment i, 256 of its tokens each.
struct KeySegs {
  const uint16_t *k[kMaxBatchSeg];
  int64_t khs[kMaxBatchSeg];
  int64_t *part[kMaxBatchSeg];  // partial sums: block b of head h at part + h * part_hs + b * D
  int64_t part_hs[kMaxBatchSeg];
  int32_t tokens[kMaxBatchSeg];
  int32_t blk0[kMaxBatchSeg + 1];
  int32_t n;
};

__device__ __forceinline__ int key_seg(const KeySegs &a, int b) {
  int s = 0;
  while (s + 1 < a.n && b >= a.blk0[s + 1]) ++s;
  return s;
}

// Fixed-point column sums of one head's keys over 256 tokens per workgroup.
// Thread (c, r) reads 16-byte chunk c (8 channels) of rows t0 + r, t0 + r + RPI, ...
// (all its loads issued before any is used) and keeps 8 int64 partial sums;
// partials are combined in LDS and added to ws[h][d] with one 64-bit atomic per
// channel, or (ATOMIC false) stored as the workgroup's partial sums.  Values with |x| < 127 take the int32 conversion path; a chunk
// holding a larger value takes the int64 path (both give rint(x * 2^24) exactly).
template <int D, bool ATOMIC>
__global__ void __launch_bounds__(256) k_sum_kernel(const KeySegs a, int64_t *__restrict__ ws) {
  constexpr int CPR = D / 8;      // 16-byte chunks per row
  constexpr int RPI = 256 / CPR;  // rows per pass
  constexpr int NP = 256 / RPI;   // passes per workgroup
  __shared__ long long part[RPI][D];
  const int h = blockIdx.y, tid = threadIdx.x, c = tid % CPR, r = tid / CPR;
  const int sg = key_seg(a, blockIdx.x);
  const int t0 = (blockIdx.x - a.blk0[sg]) * 256;
  const int n = min(a.tokens[sg] - t0, 256);
  const uint16_t *base = a.k[sg] + (int64_t)h * a.khs[sg] + (int64_t)t0 * D + c * 8;
  // every load issued before any is used: rows past the end re-read the last
  // row (in bounds) and are zeroed afterwards
  i32x4 raw[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) raw[p] = *(const i32x4 *)(base + (int64_t)min(p * RPI + r, n - 1) * D);
#pragma unroll
  for (int p = 0; p < NP; ++p)
    if (p * RPI + r >= n) raw[p] = i32x4{};
  long long acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    float x[8];
    float mx = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[2 * e] = bf16_bits_to_f32((uint32_t)raw[p][e] & 0xffffu);
      x[2 * e + 1] = bf16_bits_to_f32((uint32_t)raw[p][e] >> 16);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
    if (mx < 127.0f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += (long long)(int)__builtin_rintf(x[e] * 16777216.0f);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += to_fixed(x[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) part[r][c * 8 + e] = acc[e];
  __syncthreads();
  if (tid < D) {
    long long sum = 0;
    for (int i = 0; i < RPI; ++i) sum += part[i][tid];
    if constexpr (ATOMIC)
      atomicAdd((unsigned long long *)(ws + h * D + tid), (unsigned long long)sum);
    else
      a.part[sg][h * a.part_hs[sg] + (int64_t)(blockIdx.x - a.blk0[sg]) * D + tid] = sum;
  }
}

// The means of a batch of calls.  Segment i's sum is `given`, or the sum of its
// nblk partial sums, which also goes to `out` if that is set (a later segment
// may have it as `given`: both are read and written by the same thread).
// Sums wrap, so their order does not matter.  One workgroup per head; group
// r of its 512 / D takes partials r, r + 512 / D, ...  (Partial sums and this
// kernel take the place of a zeroing launch, atomics, an initial sum and a
// final division, and of one such chain for each segment whose sum is kept:
// the 768p INT8-QK call with condition and padding rows spent 21 launches of 2
// to 10 us on its quantization, and now spends 3.)
struct MeanArgs {
  const int64_t *given[kMaxBatchSeg];
  const int64_t *part[kMaxBatchSeg];
  int64_t part_hs[kMaxBatchSeg];
  int64_t *out[kMaxBatchSeg];
  int32_t nblk[kMaxBatchSeg];
  int32_t call_seg0[kMaxCalls + 1];  // call c has segments [call_seg0[c], call_seg0[c + 1])
  uint16_t *mean[kMaxCalls];
  double count[kMaxCalls];           // keys of the call
  int32_t ncalls;
};
template <int D>
__global__ void __launch_bounds__(512) k_mean_kernel(const MeanArgs a) {
  constexpr int G = 512 / D;
  __shared__ unsigned long long part[G][D];
  const int h = blockIdx.x, d = threadIdx.x % D, r = threadIdx.x / D;
  for (int c = 0; c < a.ncalls; ++c) {
    unsigned long long acc = 0;
    for (int s = a.call_seg0[c]; s < a.call_seg0[c + 1]; ++s) {
      if (a.given[s]) {
        if (r == 0) acc += (unsigned long long)a.given[s][h * D + d];
        continue;
      }
      const int64_t *p = a.part[s] + h * a.part_hs[s] + d;
      unsigned long long sum = 0;
      int b = r;
      for (; b + 7 * G < a.nblk[s]; b += 8 * G) {
        int64_t x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = p[(int64_t)(b + i * G) * D];
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += (unsigned long long)x[i];
      }
      for (; b < a.nblk[s]; b += G) sum += (unsigned long long)p[(int64_t)b * D];
      __syncthreads();  // the previous segment's reads
      part[r][d] = sum;
      __syncthreads();
      if (r == 0) {
#pragma unroll
        for (int i = 1; i < G; ++i) sum += part[i][d];
        if (a.out[s]) a.out[s][h * D + d] = (int64_t)sum;
        acc += sum;
      }
    }
    if (r == 0) {
      const double m = __ddiv_rn((double)(int64_t)acc, a.count[c] * kMeanFix);
      a.mean[c][h * D + d] = f32_to_bf16_bits((float)m);
    }
  }
}

// ---------------------------------------------------------------------------
// Per-(head, 128-row block) symmetric INT8 quantization of x = src - mean:
//   amax = max |x| over the block's valid rows, scale = amax / 127,
//   q = sat_int8(rint(x * (127 / amax))) (amax = 0: scale 0, q 0).
// Rows in [nvalid, nwrite) are written as zero; every launched block writes
// its scale (0 for a block without valid rows).
template <int D, bool MEAN>
__device__ __forceinline__ void quant_block(const uint16_t *__restrict__ src, int64_t sts, int64_t shs,
                                            const int32_t *__restrict__ rows, int32_t row0,
                                            const uint16_t *__restrict__ mean, int32_t nvalid, int32_t nwrite,
                                            int8_t *__restrict__ q8, int64_t q8hs, float *__restrict__ qscale,
                                            int32_t qshs, int h, int blk) {
  constexpr int CPR = D / 8;          // 8-element chunks per row
  constexpr int RPI = 256 / CPR;      // rows per pass
  constexpr int NP = TMHD_QUANT_BLOCK / RPI;
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int ch = tid % CPR, r0 = tid / CPR;
  // All loads are issued before any is used (one memory round trip): the
  // mean as one 16-byte read, rows past nvalid re-read row nvalid - 1 (in
  // bounds; nvalid >= 1 for every launched block) and are zeroed afterwards.
  i32x4 mraw = {0, 0, 0, 0};
  if constexpr (MEAN) mraw = *(const i32x4 *)(mean + h * D + ch * 8);
  int rix[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int ic = min(blk * TMHD_QUANT_BLOCK + p * RPI + r0, nvalid - 1);
    rix[p] = rows ? rows[ic] : row0 + ic;
  }
  i32x4 raw[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) raw[p] = *(const i32x4 *)(src + (int64_t)rix[p] * sts + (int64_t)h * shs + ch * 8);
  float mf[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    mf[2 * e] = bf16_bits_to_f32((uint32_t)mraw[e] & 0xffffu);
    mf[2 * e + 1] = bf16_bits_to_f32((uint32_t)mraw[e] >> 16);
  }
  float x[NP][8];
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const bool valid = blk * TMHD_QUANT_BLOCK + p * RPI + r0 < nvalid;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = (uint32_t)raw[p][e];
      x[p][2 * e] = valid ? bf16_bits_to_f32(w & 0xffffu) - mf[2 * e] : 0.0f;
      x[p][2 * e + 1] = valid ? bf16_bits_to_f32(w >> 16) - mf[2 * e + 1] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(x[p][e]));
  }
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float inv = amax > 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
  if (tid == 0) qscale[(int64_t)h * qshs + blk] = __fdiv_rn(amax, 127.0f);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = blk * TMHD_QUANT_BLOCK + p * RPI + r0;
    if (i < nwrite) {
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo |= ((uint32_t)quant_rne_sat(x[p][e] * inv) & 0xffu) << (8 * e);
        hi |= ((uint32_t)quant_rne_sat(x[p][4 + e] * inv) & 0xffu) << (8 * e);
      }
      *(i32x2 *)(q8 + (int64_t)h * q8hs + (int64_t)i * D + ch * 8) = i32x2{(int)lo, (int)hi};
    }
  }
}

// Every key segment's and every call's query blocks of a batch in one launch:
// workgroups from blk0[i] on are entry i's.
struct QuantEntry {
  const uint16_t *src;
  int64_t sts, shs;
  const int32_t *rows;   // queries: their row list, or row0
  const uint16_t *mean;  // keys: [H][D]; queries: nullptr
  int8_t *q8;
  int64_t q8hs;
  float *qs;
  int32_t qshs, row0, nvalid, nwrite, blk0;
};
struct QuantArgs {
  int32_t n;
  QuantEntry e[kMaxBatchSeg + kMaxCalls];
};
static_assert(sizeof(QuantArgs) <= 4096, "kernel arguments");

template <int D>
__global__ void __launch_bounds__(256) block_quant_kernel(const QuantArgs a) {
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.e[i + 1].blk0) ++i;
  const QuantEntry &E = a.e[i];
  const int blk = blockIdx.x - E.blk0;
  if (E.mean)
    quant_block<D, true>(E.src, E.sts, E.shs, nullptr, 0, E.mean, E.nvalid, E.nwrite, E.q8, E.q8hs, E.qs, E.qshs,
                         blockIdx.y, blk);
  else
    quant_block<D, false>(E.src, E.sts, E.shs, E.rows, E.row0, nullptr, E.nvalid, E.nwrite, E.q8, E.q8hs, E.qs, E.qshs,
                          blockIdx.y, blk);
}

bool aligned(const void *p, int bytes) { return ((uintptr_t)p % bytes) == 0; }

// Calls [0, n) of a batch (within the launch limits): key sums, means, then
// every key and query block.  sum_out: per call kMaxSeg pointers, or nullptr.
template <int D>
int smooth_quant(const tmhd_attn_args *a, const tmhd_qk_quant *qq, int64_t *const *sum_out, int n, hipStream_t s) {
  const int H = a->heads;
  KeySegs ks{};
  MeanArgs mean{};
  QuantArgs quant{};
  int nseg = 0, qblocks = 0;
  mean.ncalls = n;
  for (int c = 0; c < n; ++c) {
    mean.call_seg0[c] = nseg;
    mean.mean[c] = qq[c].k_mean;
    for (int i = 0; i < a[c].n_segments; ++i, ++nseg) {
      const tmhd_kv_segment &sg = a[c].seg[i];
      mean.count[c] += (double)sg.tokens;
      mean.given[nseg] = qq[c].k_sum[i];
      if (!qq[c].k_sum[i]) {
        // the quantized keys' own rows hold the partial sums until they are written:
        // D int64 per 256 tokens in the cap * D bytes of a head
        int64_t *part = (int64_t *)qq[c].k_i8[i];
        const int64_t part_hs = qq[c].k_head_stride[i] / 8;
        mean.part[nseg] = ks.part[ks.n] = part;
        mean.part_hs[nseg] = ks.part_hs[ks.n] = part_hs;
        mean.nblk[nseg] = (sg.tokens + 255) / 256;
        mean.out[nseg] = sum_out ? sum_out[c * kMaxSeg + i] : nullptr;
        ks.k[ks.n] = (const uint16_t *)sg.k;
        ks.khs[ks.n] = sg.k_head_stride;
        ks.tokens[ks.n] = sg.tokens;
        ks.blk0[ks.n + 1] = ks.blk0[ks.n] + mean.nblk[nseg];
        ++ks.n;
      }
      // rows up to the 64-token tile padding are written
      QuantEntry &e = quant.e[quant.n++];
      const int nwrite = (sg.tokens + kTile - 1) / kTile * kTile;
      e = QuantEntry{(const uint16_t *)sg.k, D, sg.k_head_stride, nullptr, qq[c].k_mean, qq[c].k_i8[i],
                     qq[c].k_head_stride[i], qq[c].k_scale[i], qq[c].k_scale_head_stride[i], 0, sg.tokens, nwrite,
                     qblocks};
      qblocks += (nwrite + TMHD_QUANT_BLOCK - 1) / TMHD_QUANT_BLOCK;
    }
    // queries: rows up to the 256-row workgroup padding are written
    const int qcap = (a[c].lq + 255) / 256 * 256;
    if (qcap == 0) continue;
    quant.e[quant.n++] = QuantEntry{(const uint16_t *)a[c].q, a[c].q_token_stride, a[c].q_head_stride, a[c].q_rows,
                                    nullptr, qq[c].q_i8, qq[c].q_head_stride, qq[c].q_scale,
                                    qq[c].q_scale_head_stride, a[c].q_row0, a[c].lq, qcap, qblocks};
    qblocks += qcap / TMHD_QUANT_BLOCK;
  }
  mean.call_seg0[n] = nseg;
  if (ks.n)
    hipLaunchKernelGGL((k_sum_kernel<D, false>), dim3(ks.blk0[ks.n], H), dim3(256), 0, s, ks, (int64_t *)nullptr);
  hipLaunchKernelGGL(k_mean_kernel<D>, dim3(H), dim3(512), 0, s, mean);
  if (int st = check_launch("smooth-K mean")) return st;
  hipLaunchKernelGGL(block_quant_kernel<D>, dim3(qblocks, H), dim3(256), 0, s, quant);
  return check_launch("block_quant");
}

}  // namespace
}  // namespace tmhd

namespace tmhd {

int kv_pack_ranges(const void *k, const void *v, int64_t token_stride, int64_t head_stride,
                   const tmhd_pack_range *ranges, int32_t nranges, void *k_slot, void *vt_slot, int64_t k_head_stride,
                   int64_t vt_head_stride, int32_t vt_row_stride, int32_t heads, int32_t head_dim, void *stream,
                   bool check_only) {
  if (head_dim != 64 && head_dim != 128) return set_error(TMHD_ERR_UNSUPPORTED, "kv_pack: head_dim %d", head_dim);
  if (nranges < 0 || (nranges > 0 && !ranges)) return set_error(TMHD_ERR_INVALID, "kv_pack: %d ranges", nranges);
  bool data = false;
  for (int i = 0; i < nranges; ++i) {
    const tmhd_pack_range &r = ranges[i];
    if (r.n < 0 || r.dst < 0 || heads <= 0)
      return set_error(TMHD_ERR_INVALID, "kv_pack: n %d dst %d heads %d", r.n, r.dst, heads);
    const int64_t end = std::max((int64_t)r.dst + r.n, (int64_t)r.zero_to);
    const int64_t p_begin = r.dst / kTile * kTile;
    const int64_t p_end = (end + kTile - 1) / kTile * kTile;
    if (p_end > vt_row_stride || vt_row_stride % kTile || (int64_t)vt_row_stride * head_dim > vt_head_stride ||
        p_end * head_dim > k_head_stride)
      return set_error(TMHD_ERR_INVALID, "kv_pack: positions [%lld, %lld) exceed the slot (cap %d)",
                       (long long)p_begin, (long long)p_end, vt_row_stride);
    data = data || r.n > 0;
  }
  if ((data && (!k || !v)) || !k_slot || !vt_slot || !aligned(k_slot, 16) || !aligned(vt_slot, 16) ||
      (data && (!aligned(k, 16) || !aligned(v, 16))) || token_stride % 8 || head_stride % 8 || k_head_stride % 8 ||
      vt_head_stride % 8)
    return set_error(TMHD_ERR_INVALID, "kv_pack: pointers and strides must be 16-byte aligned");
  if (check_only) return TMHD_OK;
  PackArgs<kMaxRanges> a{(const uint16_t *)k, (const uint16_t *)v, token_stride, head_stride, (uint16_t *)k_slot,
             (uint16_t *)vt_slot, k_head_stride, vt_head_stride, vt_row_stride, 0, {}};
  for (int i = 0, blocks = 0; i < nranges; ++i) {
    const tmhd_pack_range &r = ranges[i];
    const int p_begin = r.dst / kTile * kTile, end = std::max(r.dst + r.n, r.zero_to);
    const int nblk = ((end + kTile - 1) / kTile * kTile - p_begin) / kTile;
    if (nblk > 0) {
      a.r[a.nranges++] = PackRange{r.rows, r.row0, r.n, r.dst, r.zero_to, p_begin, blocks};
      blocks += nblk;
    }
    if (blocks == 0 || (a.nranges < kMaxRanges && i + 1 < nranges)) continue;
    const dim3 grid(blocks, heads);
    hipStream_t s = (hipStream_t)stream;
    const PackArgs<1> one{a.k, a.v, a.ts, a.hs, a.ks, a.vts, a.khs, a.vhs, a.vrs, 1, {a.r[0]}};
    if (a.nranges == 1 && head_dim == 128)
      hipLaunchKernelGGL((kv_pack_kernel<128, 1>), grid, dim3(128), 0, s, one);
    else if (a.nranges == 1)
      hipLaunchKernelGGL((kv_pack_kernel<64, 1>), grid, dim3(64), 0, s, one);
    else if (head_dim == 128)
      hipLaunchKernelGGL((kv_pack_kernel<128, kMaxRanges>), grid, dim3(128), 0, s, a);
    else
      hipLaunchKernelGGL((kv_pack_kernel<64, kMaxRanges>), grid, dim3(64), 0, s, a);
    if (int st = check_launch("tmhd_kv_pack")) return st;
    a.nranges = 0;
    blocks = 0;
  }
  return TMHD_OK;
}

int kv_pack(const void *k, const void *v, int64_t token_stride, int64_t head_stride, const int32_t *rows,
            int32_t row0, int32_t n, void *k_slot, void *vt_slot, int64_t k_head_stride, int64_t vt_head_stride,
            int32_t vt_row_stride, int32_t dst, int32_t zero_to, int32_t heads, int32_t head_dim, void *stream,
            bool check_only) {
  const tmhd_pack_range r{rows, row0, n, dst, zero_to};
  return kv_pack_ranges(k, v, token_stride, head_stride, &r, 1, k_slot, vt_slot, k_head_stride, vt_head_stride,
                        vt_row_stride, heads, head_dim, stream, check_only);
}

}  // namespace tmhd

extern "C" int tmhd_kv_pack_ranges(const void *k, const void *v, int64_t token_stride, int64_t head_stride,
                                   const tmhd_pack_range *ranges, int32_t n_ranges, void *k_slot, void *vt_slot,
                                   int64_t k_head_stride, int64_t vt_head_stride, int32_t vt_row_stride,
                                   int32_t heads, int32_t head_dim, void *stream) {
  return tmhd::kv_pack_ranges(k, v, token_stride, head_stride, ranges, n_ranges, k_slot, vt_slot, k_head_stride,
                              vt_head_stride, vt_row_stride, heads, head_dim, stream, false);
}

extern "C" int tmhd_kv_pack(const void *k, const void *v, int64_t token_stride, int64_t head_stride,
                            const int32_t *rows, int32_t row0, int32_t n, void *k_slot, void *vt_slot,
                            int64_t k_head_stride, int64_t vt_head_stride, int32_t vt_row_stride, int32_t dst,
                            int32_t zero_to, int32_t heads, int32_t head_dim, void *stream) {
  return tmhd::kv_pack(k, v, token_stride, head_stride, rows, row0, n, k_slot, vt_slot, k_head_stride, vt_head_stride,
                       vt_row_stride, dst, zero_to, heads, head_dim, stream, false);
}

namespace tmhd {
namespace {

// Checks one call of the smooth quantization.
int check_smooth_quant(const tmhd_attn_args *args, const tmhd_qk_quant *quant) {
  const int D = args->head_dim;
  if (D != 64 && D != 128) return set_error(TMHD_ERR_UNSUPPORTED, "smooth_quant: head_dim %d", D);
  if (args->n_segments < 1 || args->n_segments > kMaxSeg || args->heads <= 0 || args->lq < 0)
    return set_error(TMHD_ERR_INVALID, "smooth_quant: bad segment count / heads / lq");
  if (!quant->k_mean || !quant->q_i8 || !quant->q_scale)
    return set_error(TMHD_ERR_INVALID, "smooth_quant: null output buffers");
  if (!aligned(quant->k_mean, 16)) return set_error(TMHD_ERR_INVALID, "smooth_quant: k_mean must be 16-byte aligned");
  const int qcap = (args->lq + 255) / 256 * 256;
  if (quant->q_head_stride < (int64_t)qcap * D || quant->q_scale_head_stride < qcap / TMHD_QUANT_BLOCK ||
      !aligned(quant->q_i8, 16) || quant->q_head_stride % 16)
    return set_error(TMHD_ERR_INVALID, "smooth_quant: quantized query buffer below round_up(lq, 256) rows");
  if (args->lq > 0 && (!args->q || !aligned(args->q, 16) || args->q_token_stride % 8 || args->q_head_stride % 8))
    return set_error(TMHD_ERR_INVALID, "smooth_quant: query pointer/strides must be 16-byte aligned");
  for (int i = 0; i < args->n_segments; ++i) {
    const tmhd_kv_segment &sg = args->seg[i];
    if (quant->k_sum[i] && !aligned(quant->k_sum[i], 8))
      return set_error(TMHD_ERR_INVALID, "smooth_quant: segment %d key sums must be 8-byte aligned", i);
    const int64_t cap = ((int64_t)sg.tokens + kTile - 1) / kTile * kTile;
    if (sg.tokens <= 0 || !sg.k || !aligned(sg.k, 16) || sg.k_head_stride < cap * D || sg.k_head_stride % 8)
      return set_error(TMHD_ERR_INVALID, "smooth_quant: segment %d keys are not a slot", i);
    if (!quant->k_i8[i] || !quant->k_scale[i] || !aligned(quant->k_i8[i], 16) || quant->k_head_stride[i] < cap * D ||
        quant->k_head_stride[i] % 16 ||
        quant->k_scale_head_stride[i] < (sg.tokens + TMHD_QUANT_BLOCK - 1) / TMHD_QUANT_BLOCK)
      return set_error(TMHD_ERR_INVALID, "smooth_quant: segment %d quantized key buffers too small", i);
  }
  return TMHD_OK;
}

int smooth_quant_batch(const tmhd_attn_args *args, const tmhd_qk_quant *quant, int64_t *const *sum_out, int32_t n,
                       void *stream) {
  if (n < 0 || (n > 0 && (!args || !quant))) return set_error(TMHD_ERR_INVALID, "smooth_quant: null arguments");
  // every call is checked before the first launch
  for (int i = 0; i < n; ++i) {
    if (int st = check_smooth_quant(args + i, quant + i)) return st;
    if (args[i].heads != args->heads || args[i].head_dim != args->head_dim)
      return set_error(TMHD_ERR_INVALID, "smooth_quant: the calls of a batch must share heads and head_dim");
    for (int j = 0; sum_out && j < args[i].n_segments; ++j)
      if (sum_out[i * kMaxSeg + j] && !aligned(sum_out[i * kMaxSeg + j], 8))
        return set_error(TMHD_ERR_INVALID, "smooth_quant: segment %d key sums must be 8-byte aligned", j);
  }
  hipStream_t s = (hipStream_t)stream;
  for (int i = 0; i < n;) {
    int m = 0, segs = 0;
    while (i + m < n && m < kMaxCalls && segs + args[i + m].n_segments <= kMaxBatchSeg) segs += args[i + m++].n_segments;
    int64_t *const *so = sum_out ? sum_out + i * kMaxSeg : nullptr;
    if (int st = args->head_dim == 128 ? smooth_quant<128>(args + i, quant + i, so, m, s)
                                       : smooth_quant<64>(args + i, quant + i, so, m, s))
      return st;
    i += m;
  }
  return TMHD_OK;
}

}  // namespace
}  // namespace tmhd

extern "C" int tmhd_qk_smooth_quant(const tmhd_attn_args *args, const tmhd_qk_quant *quant, void *stream) {
  if (!args || !quant) return tmhd::set_error(TMHD_ERR_INVALID, "smooth_quant: null arguments");
  return tmhd::smooth_quant_batch(args, quant, nullptr, 1, stream);
}

extern "C" int tmhd_qk_smooth_quant_batch(const tmhd_attn_args *args, const tmhd_qk_quant *quant,
                                          int64_t *const *k_sum_out, int32_t n, void *stream) {
  return tmhd::smooth_quant_batch(args, quant, k_sum_out, n, stream);
}

extern "C" int tmhd_k_fixed_sum(const void *k, int64_t k_head_stride, int32_t tokens, int32_t heads, int32_t head_dim,
                                int64_t *sum, void *stream) {
  using namespace tmhd;
  if (head_dim != 64 && head_dim != 128) return set_error(TMHD_ERR_UNSUPPORTED, "k_fixed_sum: head_dim %d", head_dim);
  if (tokens <= 0 || heads <= 0 || k_head_stride < (int64_t)tokens * head_dim || k_head_stride % 8)
    return set_error(TMHD_ERR_INVALID, "k_fixed_sum: tokens %d heads %d head stride %lld", tokens, heads,
                     (long long)k_head_stride);
  if (!k || !sum || !aligned(k, 16) || !aligned(sum, 8))
    return set_error(TMHD_ERR_INVALID, "k_fixed_sum: keys must be 16-byte and sums 8-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  KeySegs t{};
  t.n = 1;
  t.k[0] = (const uint16_t *)k;
  t.khs[0] = k_head_stride;
  t.tokens[0] = tokens;
  t.blk0[0] = 0;
  t.blk0[1] = (tokens + 255) / 256;
  hipLaunchKernelGGL(zero_i64_kernel, dim3((heads * head_dim + 255) / 256), dim3(256), 0, s, sum, heads * head_dim);
  if (head_dim == 128)
    hipLaunchKernelGGL((k_sum_kernel<128, true>), dim3(t.blk0[1], heads), dim3(256), 0, s, t, sum);
  else
    hipLaunchKernelGGL((k_sum_kernel<64, true>), dim3(t.blk0[1], heads), dim3(256), 0, s, t, sum);
  return check_launch("tmhd_k_fixed_sum");
}
