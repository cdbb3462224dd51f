// lm_tensor.hip -- per-tensor INT8 (symmetric, fp32 scale) and scaled FP8
// merges with bf16 factors and N % 64 == 0: one scale for the whole weight,
// so every merged value is needed before the first can be quantized
// (P/_triton_float8_lora.py:400-483, P/_triton_int8_lora.py:316-370; P/ = the
// reference's src/piper_offload/).
//
// Two launches over the codes, each a free tiling of the weight as in
// k_rows_split (a wave holds RB 16-row blocks that share each 64-column
// tile's A^T operands and walks TPW tiles; the workgroup's 4 waves take
// neighbouring tiles):
//   amax   merge, max |bf16(merged)|, one partial per workgroup in the
//          workspace; the first workgroup copies the input scale to red[1]
//          and the zero point, if there is one, to red[2];
//   quant  each workgroup reduces the partials (a few KB from L2), merges
//          again (the same MFMA chains and arithmetic, so the values are
//          those the amax pass reduced), quantizes and stores; the first
//          stores the scale.  It reads the input scale and zero point from
//          red[1] and red[2], since the outputs may alias them.
// The codes are read twice, the second time from the last-level cache where
// they fit.  What bounds the passes is the latency of their loads and the
// merge arithmetic.  Atomics do not pay here: the waves of one generation end
// together, all find the slot low, and their atomics on it run one by one (FP8
// [8192, 4096] rank 32: 57.9 us with one conditional atomic per wave, 30.5 with
// partials).  Per call, against the k_blocks passes that these layouts took
// before: FP8 [13800, 5120] rank 32 157 -> 62 us, [14336, 4096] rank 16
// stochastic 141 -> 47, [8192, 8192] rank 64 199 -> 73; INT8 [14336, 4096] rank
// 16 132 -> 42, with a zero point to subtract 135 -> 42.
#include "lm_tensor.h"

namespace {

constexpr int TT_NW = 4;
constexpr int TT_PART = 64;  // the partials follow the 64 slots that the prep launch clears

template <int KIND, bool SR, int NKC, int RB, int TPW, bool QUANT>
__global__ __launch_bounds__(TT_NW * 64) void k_tensor_pass(RowArgs a, int wg_per_group, int npart) {
  __shared__ float sh[TT_NW];
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15;
  const int ntiles = (int)(a.N >> 6);
  // one contiguous eighth of the weight per XCD: with 2, 4 or 8 workgroups per
  // row group each XCD would otherwise read the same columns of every row,
  // which meet on a few of its L2 channels (FP8 [8192, 4096]: 38.9 -> 36.2 us)
  const uint32_t unit = (uint32_t)xcd_unit(blockIdx.x, gridDim.x);
  const uint32_t grp = unit / (uint32_t)wg_per_group;
  const int t0 = (int)(unit - grp * (uint32_t)wg_per_group) * TT_NW * TPW + wave;
  const bool first = unit == 0 && threadIdx.x == 0;
  LM_GLOBAL uint32_t* red = (LM_GLOBAL uint32_t*)a.red;
  LM_GLOBAL float* part = (LM_GLOBAL float*)(red + TT_PART);  // one maximum per amax workgroup
  // a symmetric INT8 weight may come with a zero point (usually 0), subtracted here; the merged codes have none
  constexpr bool ZP = KIND == K_INT8;
  float s_in, z_in = 0.0f;
  RowQP qp = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (QUANT) {
    s_in = u2f(red[1]);
    if (ZP && a.zp) z_in = u2f(red[2]);
    float mx = 0.0f;
    for (int i = threadIdx.x; i < npart; i += TT_NW * 64) mx = __builtin_fmaxf(mx, part[i]);
    mx = wave_max(mx);
    if (lane == 0) sh[wave] = mx;
    __syncthreads();
    mx = __builtin_fmaxf(__builtin_fmaxf(sh[0], sh[1]), __builtin_fmaxf(sh[2], sh[3]));
    float stored;
    if constexpr (KIND == K_INT8) {
      int zp;
      qp = int8_qparams<BF16, F32, false>(-mx, mx, a.qmin, a.qmax, stored, zp);
      if (first && a.zp_out) a.zp_out[0] = 0;
    } else {
      qp = fp8_qparams<BF16, KIND>(mx, stored);
    }
    if (first) *(LM_GLOBAL float*)a.scale_out = stored;
  } else {
    s_in = *(const LM_GLOBAL float*)a.scale;
    if (first) red[1] = f2u(s_in);
    if (ZP && a.zp) {
      z_in = (float)*(const LM_GLOBAL int8_t*)a.zp;
      if (first) red[2] = f2u(z_in);
    }
  }
  // a wave without tiles has no steps; it takes part in the barriers
  const int left = (ntiles - t0 + TT_NW - 1) / TT_NW, steps = left < TPW ? left : TPW;
  const int tl = t0 < ntiles ? t0 : ntiles - 1;  // its loads stay in bounds
  FastLane L[RB];
  v4i16 bop[RB][NKC];
  bool rok[RB];
  float amax = 0.0f;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int64_t row = (int64_t)grp * (16 * RB) + 16 * rb + rl;
    rok[rb] = row < a.M;
    // rows past M work on row M-1 (valid memory, a value that counts anyway) and never store
    const int64_t rowc = rok[rb] ? row : a.M - 1;
    L[rb] = fast_lane<NKC>(a, rowc, lane);
    load_bop<NKC>(a.bp, rowc, lane, bop[rb]);
  }
  v4i16 aop[4][NKC];
  uint4 raw[RB];
  fast_load_aop<NKC>(L[0], tl, aop);  // A^T offsets depend on the lane only
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) raw[rb] = fast_load_codes(L[rb], tl);
  // Row block rb is merged while rb + 1's MFMAs run; a block's next codes are
  // requested as soon as its current ones are merged and the next A^T operands
  // once the last MFMA has read them.  (The last step requests itself again.)
  for (int i = 0; i < steps; ++i) {
    const int mt = t0 + TT_NW * i, next = i + 1 < steps ? mt + TT_NW : mt;
    float d[2][16];
    fast_tile_delta<NKC>(aop, bop[0], d[0]);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (rb + 1 < RB) fast_tile_delta<NKC>(aop, bop[rb + 1], d[(rb + 1) & 1]);
      else fast_load_aop<NKC>(L[0], next, aop);
      float m[16];
      fast_merge_vals<KIND, !QUANT, false, ZP>(a, raw[rb], d[rb & 1], s_in, m, amax, nullptr, z_in);
      raw[rb] = fast_load_codes(L[rb], next);
      if constexpr (QUANT) {
        uint32_t old[8];
#pragma unroll
        for (int j = 0; j < 16; ++j) m[j] = bf16r(m[j]);
#pragma unroll
        for (int k = 0; k < 8; ++k) old[k] = f2u(m[2 * k]);
        fast_quant_store_vals<KIND, SR>(a, L[rb], rok[rb], mt, qp, m, old);
      }
    }
  }
  if constexpr (!QUANT) {
    amax = wave_max(amax);
    if (lane == 0) sh[wave] = amax;
    __syncthreads();
    // = max |bf16(merged)|: rounding is monotone
    if (threadIdx.x == 0)
      part[unit] = bf16r(__builtin_fmaxf(__builtin_fmaxf(sh[0], sh[1]), __builtin_fmaxf(sh[2], sh[3])));
  }
}

template <int KIND, bool SR, int NKC, int RB, int TPW, bool QUANT>
int pass(const RowArgs& a, int& npart, hipStream_t st) {
  const int64_t wgs = (a.N / 64 + TT_NW * TPW - 1) / (TT_NW * TPW), n = (a.M + 16 * RB - 1) / (16 * RB) * wgs;
  if (n > 0x7fffffff) return fail(LM_EUNSUPPORTED, "weight too large for one launch");
  if (!QUANT) npart = (int)n;
  TimedLaunch timed(QUANT ? "blocks_quant" : "blocks_amax", st);
  hipLaunchKernelGGL((k_tensor_pass<KIND, SR, NKC, RB, TPW, QUANT>), dim3((unsigned)n), dim3(TT_NW * 64), 0, st, a,
                     (int)wgs, npart);
  LAUNCH_CHECK();
  return LM_OK;
}
// Wave tiles (row blocks x tiles), amax and quant pass; us per call, FP8.
// Below 2^23 elements the larger tiles leave SIMDs without a wave: 2 x 1 for
// both passes ([1024, 4096] rank 32 11.9, rank 64 16.4; with the tiles that
// follow 19.9 and 31.5; k_blocks 22.6 and 27.7; [2000, 4096] rank 64 24.0
// against 32.1), unless a row has fewer than 4 tiles, so that only row
// blocks share operands.  Above, rank <= 32: 4 x 8 and 2 x 4 ([13800, 5120]
// rank 32 57.8 with 4 x 8 and 4 x 8 57.6, 4 x 4 and 2 x 4 59.7, 2 x 4 and 2 x 4
// 63.3).  Rank 64, whose operands cost more per tile: 8 x 4 and 4 x 4, from 2^26
// elements on 8 x 8 and 4 x 8.  The lines, rank 64: the first pair and the
// second, [4096, 6144] 42.8 and 52, [4096, 11008] 62 and 67, [4096, 14336] 72.3
// and 68.2, [8192, 8192] 72.4 and 67.9, [13800, 5120] 91 and 91.
template <int KIND, bool SR, int NKC>
int run(const RowArgs& a, hipStream_t st) {
  int npart = 0, rc;
  const int64_t n = a.M * a.N;
  if (n < (INT64_C(1) << 23) && a.N >= 64 * TT_NW) {
    rc = pass<KIND, false, NKC, 2, 1, false>(a, npart, st);
    return rc ? rc : pass<KIND, SR, NKC, 2, 1, true>(a, npart, st);
  }
  if constexpr (NKC < 4) {
    rc = pass<KIND, false, NKC, 4, 8, false>(a, npart, st);
    return rc ? rc : pass<KIND, SR, NKC, 2, 4, true>(a, npart, st);
  } else if (n >= (INT64_C(1) << 26)) {
    rc = pass<KIND, false, NKC, 8, 8, false>(a, npart, st);
    return rc ? rc : pass<KIND, SR, NKC, 4, 8, true>(a, npart, st);
  } else {
    rc = pass<KIND, false, NKC, 8, 4, false>(a, npart, st);
    return rc ? rc : pass<KIND, SR, NKC, 4, 4, true>(a, npart, st);
  }
}

}  // namespace

int tensor_merge_run(const RowArgs& a, int kind, int nkc, bool sr, hipStream_t st) {
#define TT(K_)                                                          \
  if (sr) {                                                             \
    NKC_SWITCH(nkc_bucket(nkc), return (run<K_, true, NKC_>(a, st)));   \
  } else {                                                              \
    NKC_SWITCH(nkc_bucket(nkc), return (run<K_, false, NKC_>(a, st)));  \
  }
  if (kind == K_INT8) { TT(K_INT8) } else if (kind == K_E4M3) { TT(K_E4M3) } else { TT(K_E5M2) }
#undef TT
  return LM_OK;
}
