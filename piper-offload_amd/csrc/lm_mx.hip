// lm_mx.hip -- MX (TorchAO MXTensor: MXFP4 / MXFP8) entry points.
#include "lm_dequant.h"
#include "lm_mx_fast.h"
#include "lm_requant.h"

// ---------------------------------------------------------------------------
// MX
// ---------------------------------------------------------------------------
static int check_mx(int64_t M, int64_t N, int32_t elem, int32_t scaling) {
  if (M <= 0 || N <= 0) return fail(LM_EINVAL, "MX merge requires a non-empty weight");
  if (N % 32 != 0) return fail(LM_EINVAL, "MX requires columns divisible by 32, got %lld", (long long)N);
  if (elem != LM_E2M1 && elem != LM_E4M3 && elem != LM_E5M2) return fail(LM_EUNSUPPORTED, "unsupported MX element dtype");
  if (scaling < 0 || scaling > 3) return fail(LM_EINVAL, "unknown MX scaling mode %d", scaling);
  return LM_OK;
}
template <int PASS>
static int run_mx(const BlkArgs& a, int elem, int cd, int nkc, bool sr, hipStream_t st) {
  if (elem == LM_E2M1) return run_blocks<B_MXFP4, PASS>(a, cd, nkc, sr, st);
  if (elem == LM_E4M3) return run_blocks<B_MXE4M3, PASS>(a, cd, nkc, sr, st);
  return run_blocks<B_MXE5M2, PASS>(a, cd, nkc, sr, st);
}
extern "C" int lm_mx_merge(uint8_t* q, uint8_t* scale, int64_t M, int64_t N, int32_t elem_dtype, int32_t scaling,
                           int32_t swizzled, const lm_lora* lora, const lm_rounding* rounding, void* workspace,
                           size_t workspace_bytes, void* stream) {
  int rc;
  if (!q || !scale) return fail(LM_EINVAL, "MX pointers must be non-null");
  if (!lora) return fail(LM_EINVAL, "lm_mx_merge requires LoRA factors");
  if ((rc = check_mx(M, N, elem_dtype, scaling))) return rc;
  if ((rc = check_lora(lora, M, N))) return rc;
  if ((rc = check_rounding(rounding))) return rc;
  Ctx c;
  const int nkc = rpad_of(lora->rank) / 16;
  const bool fast = mx_fast_ok(lora->dtype, nkc, M, N);
  // rank 16 on the fast kernel: A^T in its macro-tile order
  if ((rc = setup(c, M, N, lora, workspace, workspace_bytes, stream, false, false,
                  fast && nkc_bucket(nkc) == 1 ? AT_NV16 : AT_PLAIN)))
    return rc;
  if (fast) {
    MxArgs ma;
    ma.q = q;
    ma.scale = scale;
    ma.at = c.at;
    ma.bp = c.bp;
    ma.M = M;
    ma.N = N;
    ma.strength = lora->strength;
    ma.swizzled = swizzled;
    ma.mode = scaling;
    ma.seed = rounding ? rounding->seed : 0;
    return mx_fast_run(ma, elem_dtype, c.nkc, is_sr(rounding), c.st);
  }
  BlkArgs a = blk_args_base(c, M, N, lora, rounding);
  a.q = q;
  a.scale = scale;
  a.q_out = q;
  a.scale_out = scale;
  a.swizzled = swizzled;
  a.mx_mode = scaling;
  return run_mx<P_FULL>(a, elem_dtype, lora->dtype, c.nkc, is_sr(rounding), c.st);
}
extern "C" int lm_mx_requant(const void* dense, int32_t dense_dtype, uint8_t* q_out, uint8_t* scale_out, int64_t M,
                             int64_t N, int32_t elem_dtype, int32_t scaling, int32_t swizzled, const lm_rounding* rounding,
                             void* workspace, size_t workspace_bytes, void* stream) {
  int rc;
  if (!dense || !q_out || !scale_out) return fail(LM_EINVAL, "MX requant pointers must be non-null");
  if ((rc = check_mx(M, N, elem_dtype, scaling))) return rc;
  if ((rc = check_rounding(rounding))) return rc;
  if ((rc = check_workspace(ws_layout(M, N, 0), workspace, workspace_bytes))) return rc;
  hipStream_t st = (hipStream_t)stream;
  RqArgs a = rq_args(dense, q_out, scale_out, nullptr, M, N, rounding);
  a.swizzled = swizzled;
  a.mx_mode = scaling;
  if (swizzled && (rc = zero_swizzle_pad(scale_out, M, N / 32, st))) return rc;
  const bool sr = is_sr(rounding);
  if (elem_dtype == LM_E2M1) return run_rq_blocks<B_MXFP4>(a, dense_dtype, sr, workspace, st);
  if (elem_dtype == LM_E4M3) return run_rq_blocks<B_MXE4M3>(a, dense_dtype, sr, workspace, st);
  return run_rq_blocks<B_MXE5M2>(a, dense_dtype, sr, workspace, st);
}
extern "C" int lm_mx_dequant(const uint8_t* q, const uint8_t* scale, int64_t M, int64_t N, int32_t elem_dtype,
                             int32_t swizzled, const lm_lora* lora, void* out, int32_t out_dtype, void* workspace,
                             size_t workspace_bytes, void* stream) {
  int rc;
  if (!q || !scale || !out) return fail(LM_EINVAL, "MX dequant pointers must be non-null");
  if ((rc = check_mx(M, N, elem_dtype, 0))) return rc;
  if ((rc = check_lora(lora, M, N))) return rc;
  if (!lora) {
    if ((rc = check_dequant(M, N, out_dtype, workspace, workspace_bytes))) return rc;
    DqArgs d{q, scale, nullptr, out, M, N, N, LM_F32, swizzled, {}};
    if (elem_dtype == LM_E2M1) return run_dequant<B_MXFP4>(d, out_dtype, (hipStream_t)stream);
    if (elem_dtype == LM_E4M3) return run_dequant<B_MXE4M3>(d, out_dtype, (hipStream_t)stream);
    return run_dequant<B_MXE5M2>(d, out_dtype, (hipStream_t)stream);
  }
  Ctx c;
  if ((rc = setup(c, M, N, lora, workspace, workspace_bytes, stream))) return rc;
  BlkArgs a = blk_args_base(c, M, N, lora, nullptr);
  a.q = q;
  a.scale = scale;
  a.swizzled = swizzled;
  a.out = out;
  a.out_dt = out_dtype;
  return run_mx<P_TODENSE>(a, elem_dtype, lora->dtype, c.nkc, false, c.st);
}

