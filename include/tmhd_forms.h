/*
 * tmhd_forms.h - which form of its kernels a call of tmhd.h takes.
 */
#ifndef TMHD_FORMS_H
#define TMHD_FORMS_H

#include "tmhd.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * The form that the last, partial round of an m x n x k product
 * (tmhd_gemm_w8a8_ws and the other GEMMs) takes with workspace_bytes of scratch
 * on a device of `cus` CUs (0: the current one): whole 256 x 256 tiles (also
 * where there is no partial round), the k split, or smaller tiles of the stated
 * rows x columns.  -1 for k not a multiple of 128, which has no such rounds.
 * Launches nothing, and needs no GPU if cus > 0.  No counterpart in the
 * reference.
 */
enum {
  TMHD_GEMM_WHOLE,
  TMHD_GEMM_SPLIT_K,
  TMHD_GEMM_64X64,
  TMHD_GEMM_64X128,
  TMHD_GEMM_128X128,
  TMHD_GEMM_192X128,
  TMHD_GEMM_256X128
};
int tmhd_gemm_last_round_form(int32_t m, int32_t n, int32_t k, int64_t workspace_bytes, int32_t cus);

/*
 * Into how many key ranges an attention call of `items` 256-row query tiles
 * (over all heads) and `key_tiles` 64-key tiles cuts the items of its last,
 * partial round, on either backend (i8qk != 0: INT8-QK), with workspace_bytes
 * of split workspace on a device of `cus` CUs (0: the current one); 1: it runs
 * them whole.  -1 for sizes or a head_dim that no call has.  Launches nothing,
 * and needs no GPU if cus > 0.  No counterpart in the reference.
 */
int tmhd_attn_last_round_ranges(int32_t items, int32_t key_tiles, int32_t head_dim, int32_t i8qk,
                                int64_t workspace_bytes, int32_t cus);

#ifdef __cplusplus
}
#endif

#endif /* TMHD_FORMS_H */
