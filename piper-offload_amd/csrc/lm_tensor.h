// lm_tensor.h -- the fast per-tensor merges (lm_tensor.hip, a translation unit
// of its own).
#pragma once
#include "lm_impl.h"

// a.red: the workspace reduction slots that the prep launch cleared.  For the
// layouts of tensor_fast_ok.
__attribute__((visibility("hidden"))) int tensor_merge_run(const RowArgs& a, int kind, int nkc, bool sr, hipStream_t st);

// The row kernels' 32-bit offsets and 64-column tiles, fp32 scales, symmetric
// codes.  The amax pass's partials, one per workgroup, follow the first 64
// reduction slots: with tiles of 64 rows x 1024 columns and more they fit the
// 2 Mpad words there (short weights of very long rows do not and run
// k_blocks); the small tiles of run()'s first rule, 32 x 256, go on into the
// norm and bound regions behind, which NVFP4 alone uses (ceil(M / 32) *
// ceil(N / 256) <= ub_words).
static inline bool tensor_fast_ok(int kind, int cd, int sdt, bool asym, int nkc, int64_t M, int64_t N) {
  return sdt == LM_F32 && rows_fast_ok(kind, cd, sdt, asym, nkc, M, N) &&
         (M + 63) / 64 * ((N + 1023) / 1024) <= red_words(M) - 64;
}
