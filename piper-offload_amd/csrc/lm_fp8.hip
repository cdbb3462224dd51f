// lm_fp8.hip -- scaled FP8 (TorchAO Float8Tensor) entry points.
#include "lm_dequant.h"
#include "lm_group.h"
#include "lm_requant.h"
#include "lm_tensor.h"

// ---------------------------------------------------------------------------
// FP8
// ---------------------------------------------------------------------------
static int check_fp8_layout(int64_t M, int64_t N, int64_t group, int32_t fmt) {
  if (M <= 0 || N <= 0) return fail(LM_EINVAL, "FP8 merge requires a non-empty weight");
  if (fmt != LM_E4M3 && fmt != LM_E5M2) return fail(LM_EUNSUPPORTED, "FP8 storage must be e4m3fn or e5m2");
  if (group != N && group != M * N && !group_size_ok(N, group))
    return fail(LM_EUNSUPPORTED,
                "FP8 supports per-row, per-tensor and per-group layouts (group 16, 32 or a multiple of 64 dividing "
                "N), got group %lld for N=%lld",
                (long long)group, (long long)N);
  return LM_OK;
}

template <int KIND, int BF>
static int fp8_merge(const uint8_t* q, const float* scale, uint8_t* q_out, float* scale_out, int64_t M, int64_t N,
                     int64_t group, const lm_lora* lora, const lm_rounding* rnd, void* ws, size_t wsb, void* stream) {
  int rc;
  const int cd = lora->dtype;
  const bool sr = is_sr(rnd);
  const bool split = group == N && rows_split_wanted(KIND, cd, LM_F32, false, sr, rpad_of(lora->rank) / 16, M, N);
  Ctx c;
  if ((rc = setup(c, M, N, lora, ws, wsb, stream, split))) return rc;
  const bool tensor = group == M * N && group != N;
  if (!tensor || tensor_fast_ok(KIND, cd, LM_F32, false, c.nkc, M, N)) {
    RowArgs a;
    memset(&a, 0, sizeof a);
    a.q = q;
    a.scale = scale;
    a.q_out = q_out;
    a.scale_out = scale_out;
    a.at = c.at;
    a.bp = c.bp;
    a.M = M;
    a.N = N;
    a.strength = lora->strength;
    a.seed = seed_of(rnd);
    a.red = split || tensor ? c.red : nullptr;
    if (tensor) return tensor_merge_run(a, KIND, c.nkc, sr, c.st);
    if (group != N) return run_groups<KIND, false>(a, group, cd, LM_F32, false, sr, c.nkc, c.st);
    return run_rows<KIND, false>(a, cd, LM_F32, false, sr, c.nkc, c.st);
  }
  BlkArgs a = blk_args_base(c, M, N, lora, rnd);
  a.q = q;
  a.scale = scale;
  a.q_out = q_out;
  a.scale_out = scale_out;
  a.scale_dt = LM_F32;
  a.group = group;
  if ((rc = run_blocks<BF, P_AMAX>(a, cd, c.nkc, false, c.st))) return rc;
  if ((rc = run_blocks<BF, P_QUANT>(a, cd, c.nkc, sr, c.st))) return rc;
  return run_finalize<BF>(a, cd, c.st) ? fail(LM_EHIP, "finalize launch failed") : LM_OK;
}
template <int KIND>
static int fp8_requant(const RqArgs& r, int64_t group, int cd, bool sr, void* ws, hipStream_t st) {
  if (group == r.M * r.N && group != r.N) return run_rq_tensor<KIND>(r, cd, false, sr, ws, st);
  const RqPlan plan = rq_plan(r, group);
  if (plan != RQ_NONE) return run_rq_rows<KIND>(r, plan, group, cd, false, sr, st);
  RowArgs a = rq_row_args(r);
  if (group != r.N) return run_groups<KIND, true>(a, group, cd, LM_F32, false, sr, 0, st);
  return run_rows<KIND, true>(a, cd, LM_F32, false, sr, 0, st);
}

extern "C" int lm_fp8_merge(const uint8_t* q, const float* scale, uint8_t* q_out, float* scale_out, int64_t M, int64_t N,
                            int64_t group, int32_t fp8_dtype, const lm_lora* lora, const lm_rounding* rounding,
                            void* workspace, size_t workspace_bytes, void* stream) {
  if (!q || !scale) return fail(LM_EINVAL, "FP8 inputs must be non-null");
  if (!lora) return fail(LM_EINVAL, "lm_fp8_merge requires LoRA factors");
  int rc;
  if ((rc = check_fp8_layout(M, N, group, fp8_dtype))) return rc;
  if ((rc = check_lora(lora, M, N))) return rc;
  if ((rc = check_rounding(rounding))) return rc;
  if (!q_out || !scale_out) return fail(LM_EINVAL, "FP8 outputs must be non-null");
  if (fp8_dtype == LM_E4M3)
    return fp8_merge<K_E4M3, B_E4M3>(q, scale, q_out, scale_out, M, N, group, lora, rounding, workspace, workspace_bytes,
                                     stream);
  return fp8_merge<K_E5M2, B_E5M2>(q, scale, q_out, scale_out, M, N, group, lora, rounding, workspace, workspace_bytes,
                                   stream);
}
extern "C" int lm_fp8_requant(const void* dense, int32_t dense_dtype, uint8_t* q_out, float* scale_out, int64_t M,
                              int64_t N, int64_t group, int32_t fp8_dtype, const lm_rounding* rounding, void* workspace,
                              size_t workspace_bytes, void* stream) {
  if (!dense) return fail(LM_EINVAL, "dense input must be non-null");
  if (dense_dtype != LM_BF16 && dense_dtype != LM_F16) return fail(LM_EUNSUPPORTED, "requant input must be bf16/fp16");
  int rc;
  if ((rc = check_fp8_layout(M, N, group, fp8_dtype))) return rc;
  if ((rc = check_rounding(rounding))) return rc;
  if (!q_out || !scale_out) return fail(LM_EINVAL, "FP8 outputs must be non-null");
  if ((rc = check_workspace(ws_layout(M, N, 0), workspace, workspace_bytes))) return rc;
  RqArgs r = rq_args(dense, q_out, scale_out, nullptr, M, N, rounding);
  r.scale_dt = LM_F32;
  if (fp8_dtype == LM_E4M3)
    return fp8_requant<K_E4M3>(r, group, dense_dtype, is_sr(rounding), workspace, (hipStream_t)stream);
  return fp8_requant<K_E5M2>(r, group, dense_dtype, is_sr(rounding), workspace, (hipStream_t)stream);
}
extern "C" int lm_fp8_dequant(const uint8_t* q, const float* scale, int64_t M, int64_t N, int64_t group, int32_t fp8_dtype,
                              const lm_lora* lora, void* out, int32_t out_dtype, void* workspace, size_t workspace_bytes,
                              void* stream) {
  int rc;
  if (!q || !scale || !out) return fail(LM_EINVAL, "FP8 dequant pointers must be non-null");
  if ((rc = check_fp8_layout(M, N, group, fp8_dtype))) return rc;
  if ((rc = check_lora(lora, M, N))) return rc;
  if (!lora) {
    if ((rc = check_dequant(M, N, out_dtype, workspace, workspace_bytes))) return rc;
    DqArgs d{q, scale, nullptr, out, M, N, group, LM_F32, 0, {}};
    if (fp8_dtype == LM_E4M3) return run_dequant<B_E4M3>(d, out_dtype, (hipStream_t)stream);
    return run_dequant<B_E5M2>(d, out_dtype, (hipStream_t)stream);
  }
  Ctx c;
  if ((rc = setup(c, M, N, lora, workspace, workspace_bytes, stream))) return rc;
  BlkArgs a = blk_args_base(c, M, N, lora, nullptr);
  a.q = q;
  a.scale = scale;
  a.scale_dt = LM_F32;
  a.group = group;
  a.out = out;
  a.out_dt = out_dtype;
  if (fp8_dtype == LM_E4M3) return run_blocks<B_E4M3, P_TODENSE>(a, lora->dtype, c.nkc, false, c.st);
  return run_blocks<B_E5M2, P_TODENSE>(a, lora->dtype, c.nkc, false, c.st);
}

