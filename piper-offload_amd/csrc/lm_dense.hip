// lm_dense.hip -- plain bf16/fp16 weight merge (addmm_) entry point.
#include "lm_impl.h"

// ---------------------------------------------------------------------------
// dense bf16 / fp16 weight: w += strength * B@A
// ---------------------------------------------------------------------------
// A wave keeps the A^T operands of one 64-column tile in registers and walks
// 16-row tiles: per tile it needs 16 rows of Bp (L2) and the weight itself, which
// it reads one tile ahead and writes back in whole cache lines (trade_rows8).
// Traffic bounds it: 4 bytes per element.  (k_blocks, which still takes rows of
// odd length or stride, re-read the A^T operands for every 16 x 64 tile, rank / 16
// bytes per weight byte, and moved half lines, four tiles in series.)
// The deltas come from the same MFMA chains, so results are the same bits.  Per
// call, against k_blocks: [4096, 14336] rank 32 71.8 -> 54.6 us, [14336, 4096]
// rank 16 59.2 -> 50.7, [8192, 8192] fp16 rank 64 120 -> 65.6 (copying such a
// weight in place: 42).
//
// In the tile lane group g = lane >> 4 holds columns 8 g .. + 7 (piece a, MFMAs
// 0 and 1) and 32 + 8 g .. + 7 (piece b, MFMAs 2 and 3) of row lane & 15.
namespace {

constexpr int DN_NW = 4;

template <bool HALF, int NKC>
__global__ __launch_bounds__(DN_NW * 64) void k_dense_merge(uint16_t* w, const uint16_t* at, const uint16_t* bp, int M,
                                                            int N, int ld, float strength, int tiles_per_wg) {
  constexpr int DT = HALF ? F16 : BF16;
  constexpr int RPAD = NKC * 16;
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15, g = lane >> 4;
  const int c0 = ((int)blockIdx.x * DN_NW + wave) * 64;  // the wave's column tile
  if (c0 >= N) return;
  // the lane's piece of both accesses: half rl >> 3 of row rl & 7 (+ 8)
  const int col = c0 + 32 * (rl >> 3) + 8 * g, r8 = rl & 7;
  const bool cok = col < N;  // N % 8 == 0: a piece is whole or outside
  v4i16 aop[4][NKC];
#pragma unroll
  for (int k4 = 0; k4 < 4; ++k4)  // At has columns up to N rounded up to 128
    load_kchunks_g<NKC>((const LM_GLOBAL uint16_t*)at +
                            (int64_t)(c0 + 32 * (k4 >> 1) + 8 * (rl >> 2) + 4 * (k4 & 1) + (rl & 3)) * RPAD + g * (NKC * 4),
                        aop[k4]);
  const int tiles = (M + 15) >> 4;
  const int tb = (int)blockIdx.y * tiles_per_wg, te = tb + tiles_per_wg < tiles ? tb + tiles_per_wg : tiles;
  const uint32_t off0 = 2u * (uint32_t)(r8 * ld + (cok ? col : 0)), off1 = off0 + 16u * (uint32_t)ld;
  const uint32_t step = 32u * (uint32_t)ld;  // bytes of a row tile
  LM_GLOBAL uint8_t* base = (LM_GLOBAL uint8_t*)w;
  lm_u32x4 w0, w1;
  v4i16 bop[NKC];
  auto load = [&](int tt) {
    // rows past M read row M - 1; Bp has rows up to M rounded up to 16
    const int last = M - 1 - 16 * tt;
    const uint32_t b0 = r8 > last ? (uint32_t)(r8 - last) : 0u, b1 = r8 + 8 > last ? (uint32_t)(r8 + 8 - last) : 0u;
    const LM_GLOBAL uint8_t* p = base + (int64_t)tt * step;
    w0 = *(const LM_GLOBAL lm_u32x4*)(p + (off0 - b0 * 2u * (uint32_t)ld));
    w1 = *(const LM_GLOBAL lm_u32x4*)(p + (off1 - b1 * 2u * (uint32_t)ld));
    load_bop_g<NKC>(bp, (int64_t)tt * 16 + rl, lane, bop);
  };
  load(tb);
  for (int tt = tb; tt < te; ++tt) {
    float d[16];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      const v4f32 acc = mfma_chain<NKC, HALF>(aop[k4], bop);
#pragma unroll
      for (int j = 0; j < 4; ++j) d[4 * k4 + j] = acc[j];
    }
    trade_rows8(w0, w1);  // pieces a and b of the lane's own row
    lm_u32x4 o0, o1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float a0 = __builtin_fmaf(d[2 * k], strength, val_dt<DT>(w0[k] & 0xffffu));
      const float a1 = __builtin_fmaf(d[2 * k + 1], strength, val_dt<DT>(w0[k] >> 16));
      const float b0 = __builtin_fmaf(d[8 + 2 * k], strength, val_dt<DT>(w1[k] & 0xffffu));
      const float b1 = __builtin_fmaf(d[9 + 2 * k], strength, val_dt<DT>(w1[k] >> 16));
      if constexpr (HALF) {
        o0[k] = (uint32_t)f16_bits(a0) | ((uint32_t)f16_bits(a1) << 16);
        o1[k] = (uint32_t)f16_bits(b0) | ((uint32_t)f16_bits(b1) << 16);
      } else {
        o0[k] = pack_bf16x2(a0, a1);
        o1[k] = pack_bf16x2(b0, b1);
      }
    }
    load(tt + 1 < te ? tt + 1 : tt);
    trade_rows8(o0, o1);
    LM_GLOBAL uint8_t* p = base + (int64_t)tt * step;
    if (cok && 16 * tt + r8 < M) *(LM_GLOBAL lm_u32x4*)(p + off0) = o0;
    if (cok && 16 * tt + r8 + 8 < M) *(LM_GLOBAL lm_u32x4*)(p + off1) = o1;
  }
}

// about this many waves: 4096 and 16384 took 56.8 and 57.1 us against 54.6 for
// [4096, 14336] rank 32, and 4096 is far too few for smaller weights
constexpr int64_t DN_WAVES = 8192;
int dense_run(uint16_t* w, const Ctx& c, int64_t M, int64_t N, int64_t ld, const lm_lora* lora) {
  const int64_t cts = (N + 63) / 64, tiles = (M + 15) / 16;
  int64_t groups = (DN_WAVES + cts - 1) / cts;
  if (groups > tiles) groups = tiles;
  const int64_t per = (tiles + groups - 1) / groups;
  groups = (tiles + per - 1) / per;
  if (groups > 65535) return fail(LM_EUNSUPPORTED, "dense weight too large for one launch");
  const dim3 grid((unsigned)((cts + DN_NW - 1) / DN_NW), (unsigned)groups), block(DN_NW * 64);
  TimedLaunch timed("blocks_full", c.st);
#define DN(H_)                                                                                                       \
  NKC_SWITCH(nkc_bucket(c.nkc), hipLaunchKernelGGL((k_dense_merge<H_, NKC_>), grid, block, 0, c.st, w, c.at, c.bp,     \
                                                   (int)M, (int)N, (int)ld, lora->strength, (int)per))
  if (lora->dtype == LM_F16) { DN(true) } else { DN(false) }
#undef DN
  LAUNCH_CHECK();
  return LM_OK;
}

}  // namespace

extern "C" int lm_dense_merge(void* w, int64_t M, int64_t N, int64_t ldw, const lm_lora* lora, void* workspace,
                              size_t workspace_bytes, void* stream) {
  int rc;
  if (!w || !lora) return fail(LM_EINVAL, "dense merge pointers must be non-null");
  if (M <= 0 || N <= 0 || ldw < N) return fail(LM_EINVAL, "dense merge shape is invalid");
  if ((rc = check_lora(lora, M, N))) return rc;
  Ctx c;
  if ((rc = setup(c, M, N, lora, workspace, workspace_bytes, stream))) return rc;
  // whole 16-byte pieces, 32-bit lane offsets of a 16-row tile
  if ((N & 7) == 0 && (ldw & 7) == 0 && ((uintptr_t)w & 15) == 0 && ldw < (INT64_C(1) << 26) && M < (INT64_C(1) << 31) - 16)
    return dense_run((uint16_t*)w, c, M, N, ldw, lora);
  BlkArgs a = blk_args_base(c, M, N, lora, nullptr);
  a.q = w;
  a.q_out = w;
  a.ld = ldw;
  return run_blocks<B_DENSE, P_FULL>(a, lora->dtype, c.nkc, false, c.st);
}
