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

#ifdef __cplusplus
}
#endif

#endif /* TMHD_FORMS_H */
