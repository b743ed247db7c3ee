// The K/V pack of one 64-position block of one head, shared by the pack kernel
// and the staged norm + RoPE kernel.
#pragma once

#include "tmhd_internal.h"

namespace tmhd {

constexpr int kPackTile = 64;

// Slot positions p0 .. p0 + 63 of head h, by D threads (tid 0 .. D - 1).
// Position p of the slot is: data row (p - dst) if dst <= p < dst + n,
// zero if dst + n <= p < zero_to, untouched otherwise.
// WITH_K false: the key rows of data positions are left to the caller (the
// staged norm + RoPE kernel writes them); zero positions are still cleared.
// Thread (dc, g) owns the 16-byte column chunk dc (columns 8 dc .. 8 dc + 7) of
// the 8 tokens stored at transposed positions 8 g .. 8 g + 7: it loads their 8
// key and value chunks, copies the keys, and transposes the 8 x 8 block of
// values in registers into 8 transposed rows of 8 positions. A wave's loads
// and stores are whole 128-byte lines; no LDS and no barrier.
template <int D, bool WITH_K>
__device__ __forceinline__ void pack_block(const uint16_t *__restrict__ k, const uint16_t *__restrict__ v, int64_t ts,
                                           int64_t hs, const int32_t *__restrict__ rows, int32_t row0, int32_t n,
                                           uint16_t *__restrict__ ks, uint16_t *__restrict__ vts, int64_t khs,
                                           int64_t vhs, int32_t vrs, int32_t dst, int32_t zero_to, int p0, int h,
                                           int tid) {
  const int dc = tid >> 3, g = tid & 7;
  int tok[8], kind[8];  // kind: 0 untouched, 1 data, 2 zero
  bool all = true, any = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    tok[e] = vt_position(g * 8 + e);
    const int p = p0 + tok[e];
    kind[e] = (p >= dst && p < dst + n) ? 1 : (p >= dst + n && p < zero_to) ? 2 : 0;
    all = all && kind[e] != 0;
    any = any || kind[e] != 0;
  }
  i32x4 kv[8], vv[8];
  if (n > 0) {
    // every load issued before any is used: indices are clamped into the
    // data rows and the values of other positions are dropped afterwards
    int64_t src[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = min(max(p0 + tok[e] - dst, 0), n - 1);
      src[e] = (int64_t)(rows ? rows[i] : row0 + i) * ts + (int64_t)h * hs + dc * 8;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (WITH_K) kv[e] = *(const i32x4 *)(k + src[e]);
      vv[e] = *(const i32x4 *)(v + src[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (n == 0 || kind[e] != 1) kv[e] = vv[e] = i32x4{0, 0, 0, 0};
  uint16_t *kout = ks + (int64_t)h * khs + dc * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (WITH_K ? kind[e] != 0 : kind[e] == 2) *(i32x4 *)(kout + (int64_t)(p0 + tok[e]) * D) = kv[e];
  if (!any) return;
  uint16_t *out = vts + (int64_t)h * vhs + (int64_t)(dc * 8) * vrs + p0 + g * 8;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    i32x4 w;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t x = (uint32_t)vv[2 * m][j >> 1], y = (uint32_t)vv[2 * m + 1][j >> 1];
      w[m] = (int)((j & 1) ? (x >> 16) | (y & 0xffff0000u) : (x & 0xffffu) | (y << 16));
    }
    if (all) {
      *(i32x4 *)(out + (int64_t)j * vrs) = w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (kind[e] != 0) out[(int64_t)j * vrs + e] = (uint16_t)((uint32_t)w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

}  // namespace tmhd
