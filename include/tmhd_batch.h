/*
 * tmhd_batch.h - batched forms of tmhd.h's attention, INT8-QK quantization and
 * K/V pack: several independent calls in one launch.  Conventions, formats and
 * status codes are tmhd.h's.
 */
#ifndef TMHD_BATCH_H
#define TMHD_BATCH_H

#include "tmhd.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * n independent attention calls (args[0 .. n)) in one launch, or as few as
 * their segments fit (16 calls and 24 segments each): the same results as n
 * calls, up to where the key ranges of a split last round are cut.  The calls
 * share heads, head_dim, scale and the query and output strides; args[0]'s
 * split workspace serves all of them; their output rows must not overlap.
 * A hook call's condition, media and padding attention, and a packed
 * sequence's documents, are such calls.  Replaces the SDPA / SageAttention
 * calls per document and part of src/taomate_hd/streaming/attention_hook.py:384-465
 * and model/layers.py:202-255.
 */
int tmhd_attn_fwd_bf16_batch(const tmhd_attn_args *args, int32_t n, void *stream);
int tmhd_attn_fwd_i8qk_batch(const tmhd_attn_args *args, const tmhd_qk_quant *quant, int32_t n,
                             void *stream);

/*
 * tmhd_qk_smooth_quant of n calls that share heads and head_dim, in three
 * launches (per 16 calls and 24 segments).  The q_i8, q_scale, k_mean, k_i8 and
 * k_scale of one call must not overlap those of another, also where two calls
 * name the same keys: k_i8 holds partial sums on the way, and each call has its
 * own mean.  k_sum_out (NULL: none) holds n *
 * TMHD_MAX_SEGMENTS pointers: entry [i * TMHD_MAX_SEGMENTS + j], where set and
 * where call i's k_sum[j] is NULL, receives segment j's exact key sums
 * (tmhd_k_fixed_sum's, 8-byte aligned); a later call of the batch may name the
 * same memory as its k_sum.
 */
int tmhd_qk_smooth_quant_batch(const tmhd_attn_args *args, const tmhd_qk_quant *quant,
                               int64_t *const *k_sum_out, int32_t n, void *stream);

/*
 * tmhd_kv_pack of several row ranges of the same K/V into one slot, in one
 * launch (of up to 32 ranges): each range as tmhd_kv_pack with its rows /
 * row0, n, dst and zero_to.  The slot positions that the ranges write must not
 * share a 64-position tile.  Replaces the per-part copies of
 * src/taomate_hd/streaming/attention_hook.py:56-97 and model/layers.py:202-255.
 */
typedef struct tmhd_pack_range {
  const int32_t *rows; /* device row list of length n, or NULL */
  int32_t row0;        /* first source row when rows is NULL */
  int32_t n;
  int32_t dst;
  int32_t zero_to;
} tmhd_pack_range;
int tmhd_kv_pack_ranges(const void *k, const void *v, int64_t token_stride, int64_t head_stride,
                        const tmhd_pack_range *ranges, int32_t n_ranges, void *k_slot, void *vt_slot,
                        int64_t k_head_stride, int64_t vt_head_stride, int32_t vt_row_stride,
                        int32_t heads, int32_t head_dim, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* TMHD_BATCH_H */
