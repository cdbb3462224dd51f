// lm_routed.hip -- routed-LoRA residual: out = y + sum_i s_i ((x A_i^T) B_i^T + bias_i)
// (P/lora.py:801-829, _routed_residual), the inference path of the reference's
// routed mode, which adds the LoRA contribution after a Linear instead of
// merging it into the weight.
//
// The reference's operation order and roundings, all in the output dtype
// (bf16 or fp16) with fp32 matmul accumulation:
//   p_i    = dt(x A_i^T)                       [T, r_i]
//   ps_i   = dt(p_i s_i)
//   part_i = dt(ps_i B_i^T)                    [T, N]
//   part_i = dt(part_i + dt(bias_i s_i))       (when a bias is present)
//   total  = part_0, then dt(total + part_i)
//   out    = dt(y + total)
//
// At most 16 tokens (decode): one kernel, k_routed_small, and no workspace.
// Otherwise two (or three):
// * k_routed_down: MFMA x A^T by 16-wave workgroups whose waves split K and meet
//   in LDS; writes ps = dt(dt(p) s) in the dtype, [T][C * 16] (C = sum of
//   ceil(r_i / 16) rank chunks), or, where few tokens leave the GPU idle, the
//   sums of one of S spans of K (down_plan), which the up kernel adds itself
//   (SPANS) or, when they are many, k_routed_finalize;
// * k_routed_up: a wave keeps the B operands of one 64-column tile in
//   registers and walks 16-token tiles: one MFMA chain per factor, the rest
//   of the rounding chain and one read and one write of y / out: the only
//   traffic that scales with T N.
// Lane layout (the merge kernels' convention): a wave owns 16 tokens; lane l
// holds token l & 15 and 16 columns of a 64-column tile (up_col).
#include "lm_impl.h"

namespace {

constexpr int RT_NW = 4;
constexpr int RT_MAX_FACTORS = 8;
constexpr int RT_MAX_CHUNKS = 16;  // sum of ceil(rank / 16) over the factors

struct RoutedArgs {
  const uint16_t* x;    // [T, K]
  const uint16_t* y;    // [T, N] (the Linear output)
  uint16_t* out;        // [T, N] (may alias y)
  uint16_t* ps;         // [T][C * 16]: dt(dt(p) s) of each factor's ranks (zero past the rank)
  float* part;          // S > 1: [S][T][C * 16], the spans' sums
  int64_t T, K, N;
  int64_t kspan;        // K columns per span of the down projection
  int S;                // spans
  int nf, nchunks;
  int tiles_per_wg;     // token tiles per up workgroup
  const uint16_t* a[RT_MAX_FACTORS];
  const uint16_t* b[RT_MAX_FACTORS];
  const uint16_t* bias[RT_MAX_FACTORS];
  float s[RT_MAX_FACTORS];
  int rank[RT_MAX_FACTORS];
  int chunk0[RT_MAX_FACTORS];  // first rank chunk of factor i
  int cfac[RT_MAX_CHUNKS];     // factor of rank chunk c
};

// 4 consecutive 16-bit values from row `row` of a [rows, cols] matrix at
// column c (zero outside the matrix); 8-byte loads when cols % 4 == 0
__device__ __forceinline__ v4i16 load4(const uint16_t* p, int64_t rows, int64_t cols, int64_t row, int64_t c) {
  v4i16 v = {0, 0, 0, 0};
  if (row >= rows) return v;
  const uint16_t* q = p + row * cols + c;
  if ((cols & 3) == 0) {
    if (c + 3 < cols) v = __builtin_bit_cast(v4i16, *(const uint2*)q);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c + i < cols) v[i] = (short)q[i];
  }
  return v;
}

typedef short rt_v8i16 __attribute__((ext_vector_type(8)));
typedef __bf16 rt_v8bf16 __attribute__((ext_vector_type(8)));
typedef _Float16 rt_v8f16 __attribute__((ext_vector_type(8)));

// 8 consecutive 16-bit values (zero outside the matrix); 16-byte loads when cols % 8 == 0
__device__ __forceinline__ rt_v8i16 load8(const uint16_t* p, int64_t rows, int64_t cols, int64_t row, int64_t c) {
  rt_v8i16 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row >= rows) return v;
  const uint16_t* q = p + row * cols + c;
  if ((cols & 7) == 0) {
    if (c + 7 < cols) v = __builtin_bit_cast(rt_v8i16, *(const uint4*)q);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (c + i < cols) v[i] = (short)q[i];
  }
  return v;
}

// D = A B + C over K = 32: lane l supplies row l & 15, k = 8 (l >> 4) .. + 7
template <bool HALF>
__device__ __forceinline__ v4f32 mfma32(const rt_v8i16& a, const rt_v8i16& b, const v4f32& acc) {
  if constexpr (HALF)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(rt_v8f16, a), __builtin_bit_cast(rt_v8f16, b),
                                                  acc, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rt_v8bf16, a), __builtin_bit_cast(rt_v8bf16, b),
                                                   acc, 0, 0, 0);
}

template <bool HALF>
__device__ __forceinline__ v4f32 mfma1(const v4i16& a, const v4i16& b, const v4f32& acc) {
  if constexpr (HALF)
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4f16, a), __builtin_bit_cast(v4f16, b), acc, 0,
                                                 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
}

// grid (token tiles x chunk blocks, S).  A workgroup takes CB rank chunks of 16
// tokens over one of S spans of K; its 16 waves split the span.  A round is
// RT_DU steps of 32 columns per wave, in pairs of 64 neighbouring columns whose
// rows load as whole cache lines (trade_rows8); all of a round's loads are
// issued before the MFMAs (4096 columns are one round).  For rank chunk c the
// MFMA computes D[r][t] = sum_k A_i[r][k] x[t][k]: lane l holds ranks 16 c' + 4
// (l >> 4) + 0..3 of token l & 15.  The CB chunks share each round's x values;
// the waves' sums meet in LDS and one thread per (chunk, rank, token) adds them
// in wave order.  With S = 1 it rounds and writes ps; otherwise it writes the
// span's partial.
constexpr int RT_DNW = 16;
constexpr int RT_DU = 8;
constexpr int RT_DSTEP = 64 * RT_DNW;  // columns of one pair per wave: spans are multiples of it
// columns k .. k + 63 (below ke) of rows row0 .. row0 + 15 as two accesses of whole lines;
// trade_pair then gives lane (rl, g) columns k + 8 g .. and k + 32 + 8 g .. of row rl
__device__ __forceinline__ void load_pair(const uint16_t* p, int64_t rows, int64_t cols, int64_t row0, int64_t k,
                                          int64_t ke, int rl, int g, rt_v8i16& v0, rt_v8i16& v1) {
  const int64_t c = k + 32 * (rl >> 3) + 8 * g;
  const rt_v8i16 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  v0 = c < ke ? load8(p, rows, cols, row0 + (rl & 7), c) : zero;
  v1 = c < ke ? load8(p, rows, cols, row0 + (rl & 7) + 8, c) : zero;
}
__device__ __forceinline__ void trade_pair(rt_v8i16& v0, rt_v8i16& v1) {
  lm_u32x4 x = __builtin_bit_cast(lm_u32x4, v0), y = __builtin_bit_cast(lm_u32x4, v1);
  trade_rows8(x, y);
  v0 = __builtin_bit_cast(rt_v8i16, x);
  v1 = __builtin_bit_cast(rt_v8i16, y);
}
template <bool HALF, int CB>
__global__ __launch_bounds__(RT_DNW * 64) void k_routed_down(RoutedArgs a, FastDiv blocks) {
  constexpr int DT = HALF ? F16 : BF16;
  __shared__ float sh[CB][RT_DNW][256];
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15, g = lane >> 4;
  const uint32_t tile = div_by(blocks, blockIdx.x);
  const int c0 = (int)(blockIdx.x - tile * blocks.d) * CB;
  const int64_t t0 = (int64_t)tile * 16;
  const int64_t kb = (int64_t)blockIdx.y * a.kspan, ke = kb + a.kspan < a.K ? kb + a.kspan : a.K;
  v4f32 acc[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c) acc[c] = (v4f32){0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t k0 = kb + 64 * wave; k0 < ke; k0 += 32 * RT_DNW * RT_DU) {
    // loads past the span or the rows read zeros
    rt_v8i16 av[RT_DU], xv[RT_DU];
#pragma unroll
    for (int u = 0; u < RT_DU; u += 2)
      load_pair(a.x, a.T, a.K, t0, k0 + (int64_t)u * 32 * RT_DNW, ke, rl, g, xv[u], xv[u + 1]);
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      if (c0 + c >= a.nchunks) break;
      const int i = a.cfac[c0 + c], cc = c0 + c - a.chunk0[i];
#pragma unroll
      for (int u = 0; u < RT_DU; u += 2)
        load_pair(a.a[i], a.rank[i], a.K, 16 * cc, k0 + (int64_t)u * 32 * RT_DNW, ke, rl, g, av[u], av[u + 1]);
#pragma unroll
      for (int u = 0; u < RT_DU; u += 2) {
        trade_pair(av[u], av[u + 1]);
        if (c == 0) trade_pair(xv[u], xv[u + 1]);
        acc[c] = mfma32<HALF>(av[u], xv[u], acc[c]);
        acc[c] = mfma32<HALF>(av[u + 1], xv[u + 1], acc[c]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CB; ++c) *(v4f32*)&sh[c][wave][4 * lane] = acc[c];
  __syncthreads();
  for (int o = threadIdx.x; o < CB * 256; o += RT_DNW * 64) {
    const int c = o >> 8, e = o & 255;  // entry e: token (e >> 2) & 15, rank 4 (e >> 6) + (e & 3)
    const int64_t t = t0 + ((e >> 2) & 15);
    if (c0 + c < a.nchunks && t < a.T) {
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < RT_DNW; ++w) sum += sh[c][w][e];
      const int64_t at = t * (a.nchunks * 16) + (c0 + c) * 16 + 4 * (e >> 6) + (e & 3);
      if (a.S > 1) a.part[(int64_t)blockIdx.y * a.T * (a.nchunks * 16) + at] = sum;
      else a.ps[at] = bits_dt<DT>(round_dt<DT>(round_dt<DT>(sum) * a.s[a.cfac[c0 + c]]));
    }
  }
}

// four ranks of ps, two words, from the S partials at p, `stride` floats apart:
// added in span order, then p_i = dt(p), ps_i = dt(p_i s_i)
template <int DT>
__device__ __forceinline__ lm_u32x2 sum_spans(const float* p, int64_t stride, int S, float s) {
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int sp = 0; sp < S; ++sp) {
    const v4f32 w = *(const LM_GLOBAL v4f32*)(p + sp * stride);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += w[i];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = round_dt<DT>(round_dt<DT>(v[i]) * s);
  return lm_u32x2{(uint32_t)bits_dt<DT>(v[0]) | ((uint32_t)bits_dt<DT>(v[1]) << 16),
                  (uint32_t)bits_dt<DT>(v[2]) | ((uint32_t)bits_dt<DT>(v[3]) << 16)};
}
// one thread per (token, chunk, 4 ranks)
template <bool HALF>
__global__ __launch_bounds__(256) void k_routed_finalize(RoutedArgs a) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x, n = a.T * a.nchunks * 4;
  if (q >= n) return;
  ((LM_GLOBAL lm_u32x2*)a.ps)[q] =
      sum_spans<HALF ? F16 : BF16>(a.part + 4 * q, 4 * n, a.S, a.s[a.cfac[(int)(q % (a.nchunks * 4)) >> 2]]);
}

// Columns of the up kernels: in a 64-column tile lane group g = lane >> 4 holds
// columns 8 g .. 8 g + 7 (half 0, MFMAs 0 and 1) and 32 + 8 g .. + 7 (half 1,
// MFMAs 2 and 3), so that one 16-byte access of the wave covers 64 contiguous
// bytes of each of its 16 rows.  (With 16 consecutive columns per lane each
// access touched every other 16 bytes: half of each sector per store.)
__device__ __forceinline__ int up_col(int pos, int k4) {  // MFMA position -> column in the tile
  return 32 * (k4 >> 1) + 8 * (pos >> 2) + 4 * (k4 & 1) + (pos & 3);
}
__device__ __forceinline__ int64_t up_col_of(int64_t mt, int g, int j) {  // the lane's value j, 0..15
  return mt * 64 + 32 * (j >> 3) + 8 * g + (j & 7);
}
// y + total of one half (8 columns from c), rounded
template <int DT>
__device__ __forceinline__ lm_u32x4 up_sum8(const uint4& y, const float* total) {
  const uint32_t yw[4] = {y.x, y.y, y.z, y.w};
  uint32_t ow[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float lo = round_dt<DT>(val_dt<DT>(yw[k] & 0xffffu) + total[2 * k]);
    const float hi = round_dt<DT>(val_dt<DT>(yw[k] >> 16) + total[2 * k + 1]);
    ow[k] = (uint32_t)bits_dt<DT>(lo) | ((uint32_t)bits_dt<DT>(hi) << 16);
  }
  return lm_u32x4{ow[0], ow[1], ow[2], ow[3]};
}
// the lane's output of token t (vec: N % 8 == 0, halves are whole or outside)
template <int DT>
__device__ __forceinline__ void up_store(const RoutedArgs& a, int64_t t, int64_t mt, int g, bool vec, const uint4& y0,
                                         const uint4& y1, const float (&total)[16]) {
  uint16_t* orow = a.out + t * a.N;
  const int64_t ca = mt * 64 + 8 * g, cb = ca + 32;
  if (vec) {
    if (ca < a.N) store_b128_guarded((LM_GLOBAL lm_u32x4*)(orow + ca), up_sum8<DT>(y0, total));
    if (cb < a.N) store_b128_guarded((LM_GLOBAL lm_u32x4*)(orow + cb), up_sum8<DT>(y1, total + 8));
  } else {
    const uint16_t* yr = a.y + t * a.N;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int64_t c = up_col_of(mt, g, j);
      if (c < a.N) orow[c] = bits_dt<DT>(round_dt<DT>(val_dt<DT>(yr[c]) + total[j]));
    }
  }
}

// grid (column-tile groups, token groups).  Every wave owns one 64-column
// tile: its B operands (all rank chunks, CMAX at most) stay in registers
// while it walks the token tiles of its token group.  Per token tile it needs
// its rows of ps (L2) and the Linear output y (HBM); both are
// requested one token tile ahead, after the current tile's own loads, so that
// waiting for the current tile never waits for the prefetch (loads complete
// in order).
template <bool HALF, int CMAX, bool SPANS>
__global__ __launch_bounds__(RT_NW * 64) void k_routed_up(RoutedArgs a) {
  constexpr int DT = HALF ? F16 : BF16;
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15, g = lane >> 4;
  const int64_t mt = (int64_t)blockIdx.x * RT_NW + wave;  // the wave's column tile
  const int64_t ntiles = (a.N + 63) / 64;
  if (mt >= ntiles) return;
  const int64_t ca = mt * 64 + 8 * g, cb = ca + 32;  // the lane's two runs of 8 output columns
  const bool vec = (a.N & 7) == 0;
  // B operands: MFMA k4, chunk c: position p = lane & 15 is column up_col(p, k4),
  // ranks 16 c' + 4 g + 0..3 of the chunk's factor
  v4i16 bo[CMAX][4];
  const int p = lane & 15;
#pragma unroll
  for (int c = 0; c < CMAX; ++c)
    if (c < a.nchunks) {
      const int i = a.cfac[c], cc = c - a.chunk0[i];
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4)
        bo[c][k4] = load4(a.b[i], a.N, a.rank[i], mt * 64 + up_col(p, k4), 16 * cc + 4 * g);
    }
  // bias * s of the lane's columns, per factor (rounded once)
  const int64_t tiles = (a.T + 15) / 16;
  const int64_t tb = (int64_t)blockIdx.y * a.tiles_per_wg;
  const int64_t te = tb + a.tiles_per_wg < tiles ? tb + a.tiles_per_wg : tiles;
  const int64_t rowstride = (int64_t)a.nchunks * 16;
  // per token tile: the ps operands (token rl, 4 ranks per chunk) and y
  v4i16 pp[CMAX];
  uint4 y0 = make_uint4(0, 0, 0, 0), y1 = y0;
  auto load_tile = [&](int64_t tt, v4i16 (&pv)[CMAX], uint4& v0, uint4& v1) {
    const int64_t t = tt * 16 + rl;
    const bool ok = tt < te && t < a.T;
#pragma unroll
    for (int c = 0; c < CMAX; ++c) {
      pv[c] = (v4i16){0, 0, 0, 0};
      if (c < a.nchunks && ok) {
        const int64_t at = t * rowstride + c * 16 + 4 * g;
        if constexpr (SPANS)
          pv[c] = __builtin_bit_cast(v4i16, sum_spans<DT>(a.part + at, a.T * rowstride, a.S, a.s[a.cfac[c]]));
        else
          pv[c] = __builtin_bit_cast(v4i16, *(const uint2*)(a.ps + at));
      }
    }
    if (ok && vec) {
      const uint16_t* yr = a.y + t * a.N;
      if (ca < a.N) v0 = *(const uint4*)(yr + ca);
      if (cb < a.N) v1 = *(const uint4*)(yr + cb);
    }
  };
  load_tile(tb, pp, y0, y1);
  for (int64_t tt = tb; tt < te; ++tt) {
    const int64_t t = tt * 16 + rl;
    const bool tok = t < a.T;
    v4i16 ps[CMAX];
#pragma unroll
    for (int c = 0; c < CMAX; ++c) ps[c] = pp[c];
    const uint4 cy0 = y0, cy1 = y1;
    load_tile(tt + 1, pp, y0, y1);  // the next token tile, behind this one's loads
    float total[16];
    v4f32 acc[4];
#pragma unroll
    for (int c = 0; c < CMAX; ++c) {
      if (c < a.nchunks) {
        const int i = a.cfac[c], cc = c - a.chunk0[i];
        if (cc == 0) {
#pragma unroll
          for (int k4 = 0; k4 < 4; ++k4) acc[k4] = (v4f32){0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) acc[k4] = mfma1<HALF>(bo[c][k4], ps[c], acc[k4]);
        if (c + 1 == a.nchunks || a.cfac[c + 1] != i) {  // the factor's last chunk: its part is complete
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            float part = round_dt<DT>(acc[j >> 2][j & 3]);
            if (a.bias[i] && up_col_of(mt, g, j) < a.N)
              part = round_dt<DT>(part + round_dt<DT>(val_dt<DT>(a.bias[i][up_col_of(mt, g, j)]) * a.s[i]));
            total[j] = i == 0 ? part : round_dt<DT>(total[j] + part);
          }
        }
      }
    }
    if (tok) up_store<DT>(a, t, mt, g, vec, cy0, cy1, total);
  }
}

// k_routed_up for one factor of rank <= 16 NC without a bias, N % 8 == 0: the
// usual call, pared down to what it needs (62 VGPRs at rank 16, 8 waves per
// SIMD).  y and out move in whole cache lines (trade_rows8), which is what bounds
// it: 4096 tokens x 14336 took 53 us with 16 half lines per access and takes 42
// now, near a copy's 41; deeper prefetch, wider workgroups and other orders of
// the tiles changed nothing while the accesses were half lines.  A wave's
// addresses are scalar bases that advance by a token tile plus constant 32-bit
// lane offsets; the loads are unconditional (rows past T and columns past N
// read valid ones), only the stores are predicated.
template <bool HALF, int NC, bool SPANS>
__global__ __launch_bounds__(RT_NW * 64) void k_routed_up1(RoutedArgs a) {
  constexpr int DT = HALF ? F16 : BF16;
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15, g = lane >> 4;
  const int64_t mt = (int64_t)blockIdx.x * RT_NW + wave;  // the wave's column tile
  if (mt * 64 >= a.N) return;
  const int N = (int)a.N, T = (int)a.T;
  // the lane's piece of both accesses (trade_rows8): half rl >> 3 of row rl & 7 (+ 8)
  const int col = (int)(mt * 64) + 32 * (rl >> 3) + 8 * g, r8 = rl & 7;
  const bool cok = col < N;
  v4i16 bo[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4)
      bo[c][k4] = load4(a.b[0], a.N, a.rank[0], mt * 64 + up_col(rl, k4), 16 * c + 4 * g);
  const int tiles = (T + 15) >> 4;
  const int tb = (int)blockIdx.y * a.tiles_per_wg, te = tb + a.tiles_per_wg < tiles ? tb + a.tiles_per_wg : tiles;
  const uint32_t off0 = 2u * (uint32_t)(r8 * N + (cok ? col : 0)), off1 = off0 + 16u * (uint32_t)N;
  const uint32_t offp = 2u * (uint32_t)(rl * (NC * 16) + 4 * g);
  const uint32_t step = 32u * (uint32_t)N;  // bytes of a token tile
  const LM_GLOBAL uint8_t* y = (const LM_GLOBAL uint8_t*)a.y;
  const LM_GLOBAL uint8_t* ps = (const LM_GLOBAL uint8_t*)a.ps;
  LM_GLOBAL uint8_t* out = (LM_GLOBAL uint8_t*)a.out;
  lm_u32x4 y0, y1;
  lm_u32x2 pv[NC];
  auto load = [&](int tt) {
    // a ragged last tile reads row T - 1 in place of the rows past it
    const int last = T - 1 - 16 * tt;
    const uint32_t b0 = r8 > last ? (uint32_t)(r8 - last) : 0u, b1 = r8 + 8 > last ? (uint32_t)(r8 + 8 - last) : 0u;
    const uint32_t bp = rl > last ? (uint32_t)(rl - last) : 0u;
    const LM_GLOBAL uint8_t* yt = y + (int64_t)tt * step;
    y0 = *(const LM_GLOBAL lm_u32x4*)(yt + (off0 - b0 * 2u * (uint32_t)N));
    y1 = *(const LM_GLOBAL lm_u32x4*)(yt + (off1 - b1 * 2u * (uint32_t)N));
    const LM_GLOBAL uint8_t* pt = ps + (int64_t)tt * (NC * 512);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (SPANS)
        pv[c] = sum_spans<DT>(a.part + ((int64_t)(16 * tt + rl) - bp) * (NC * 16) + 16 * c + 4 * g, a.T * (NC * 16), a.S, a.s[0]);
      else
        pv[c] = *(const LM_GLOBAL lm_u32x2*)(pt + (offp - bp * (NC * 32u) + 32u * c));
    }
  };
  load(tb);
  for (int tt = tb; tt < te; ++tt) {
    float total[16];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      v4f32 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < NC; ++c) acc = mfma1<HALF>(bo[c][k4], __builtin_bit_cast(v4i16, pv[c]), acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) total[4 * k4 + j] = round_dt<DT>(acc[j]);
    }
    trade_rows8(y0, y1);  // pieces a and b of the lane's own row
    lm_u32x4 o0 = up_sum8<DT>(make_uint4(y0.x, y0.y, y0.z, y0.w), total);
    lm_u32x4 o1 = up_sum8<DT>(make_uint4(y1.x, y1.y, y1.z, y1.w), total + 8);
    load(tt + 1 < te ? tt + 1 : tt);
    trade_rows8(o0, o1);
    LM_GLOBAL uint8_t* ot = out + (int64_t)tt * step;
    if (cok && 16 * tt + r8 < T) *(LM_GLOBAL lm_u32x4*)(ot + off0) = o0;
    if (cok && 16 * tt + r8 + 8 < T) *(LM_GLOBAL lm_u32x4*)(ot + off1) = o1;
  }
}

// ---- one launch for at most 16 tokens (decode) ---------------------------------
// Several launches cost more than their work when T is small.  Here every
// workgroup computes the whole down projection of the one token tile (its
// RT_SNW waves split K, one round of RT_DU loads each at K = 4096; the sums
// meet in LDS), applies the first two roundings into LDS, then each wave
// finishes one 64-column tile as k_routed_up does.  The wave's y values and
// (for at most two rank chunks) B operands are requested before the down
// projection, so their latency overlaps it.  Every workgroup recomputes the
// down projection (x and A are read from L2 after the first).
constexpr int RT_SNW = 16;

template <bool HALF, int CMAX>
__global__ __launch_bounds__(RT_SNW * 64) void k_routed_small(RoutedArgs a) {
  constexpr int DT = HALF ? F16 : BF16;
  constexpr bool PRE = CMAX <= 2;  // B operands loaded up front
  __shared__ float sh[RT_SNW][64][4];
  __shared__ uint32_t spw[16][RT_MAX_CHUNKS * 8];      // ps of token t: ranks 2j, 2j + 1 in word j
  const int lane = threadIdx.x & 63, wave = wave_index(), rl = lane & 15, g = lane >> 4;
  const int64_t mt = (int64_t)blockIdx.x * RT_SNW + wave;
  const bool tile = mt < (a.N + 63) / 64;
  const int64_t ca = mt * 64 + 8 * g, cb = ca + 32, t = rl;
  const bool tok = tile && t < a.T, vec = (a.N & 7) == 0;
  const int p = lane & 15;
  uint4 y0 = make_uint4(0, 0, 0, 0), y1 = y0;
  if (tok && vec) {
    const uint16_t* yr = a.y + t * a.N;
    if (ca < a.N) y0 = *(const uint4*)(yr + ca);
    if (cb < a.N) y1 = *(const uint4*)(yr + cb);
  }
  v4i16 bo[PRE ? CMAX : 1][4];
  if constexpr (PRE) {
#pragma unroll
    for (int c = 0; c < CMAX; ++c) {
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) bo[c][k4] = (v4i16){0, 0, 0, 0};
      if (tile && c < a.nchunks) {
        const int i = a.cfac[c], cc = c - a.chunk0[i];
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
          bo[c][k4] = load4(a.b[i], a.N, a.rank[i], mt * 64 + up_col(p, k4), 16 * cc + 4 * g);
      }
    }
  }
  for (int c = 0; c < a.nchunks; ++c) {
    const int i = a.cfac[c], cc = c - a.chunk0[i];
    v4f32 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t k0 = 32 * wave; k0 < a.K; k0 += 32 * RT_SNW * RT_DU) {
      rt_v8i16 av[RT_DU], xv[RT_DU];
#pragma unroll
      for (int u = 0; u < RT_DU; ++u) {
        const int64_t k = k0 + (int64_t)u * 32 * RT_SNW + 8 * g;
        const bool in = k < a.K;
        av[u] = in ? load8(a.a[i], a.rank[i], a.K, 16 * cc + rl, k) : (rt_v8i16){0, 0, 0, 0, 0, 0, 0, 0};
        xv[u] = in ? load8(a.x, a.T, a.K, rl, k) : (rt_v8i16){0, 0, 0, 0, 0, 0, 0, 0};
      }
#pragma unroll
      for (int u = 0; u < RT_DU; ++u) acc = mfma32<HALF>(av[u], xv[u], acc);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) sh[wave][lane][j] = acc[j];
    __syncthreads();
    if (wave == 0) {  // lane: token rl, ranks 16 cc + 4 g + 0..3
      uint32_t w2[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float sum = 0.0f;
          for (int w = 0; w < RT_SNW; ++w) sum += sh[w][lane][2 * h + e];
          v[e] = round_dt<DT>(round_dt<DT>(sum) * a.s[i]);
        }
        w2[h] = (uint32_t)bits_dt<DT>(v[0]) | ((uint32_t)bits_dt<DT>(v[1]) << 16);
      }
      spw[rl][c * 8 + 2 * g] = w2[0];
      spw[rl][c * 8 + 2 * g + 1] = w2[1];
    }
    __syncthreads();
  }
  if (!tile) return;
  float total[16];
  v4f32 acc[4];
#pragma unroll
  for (int c = 0; c < CMAX; ++c) {
    if (c < a.nchunks) {
      const int i = a.cfac[c], cc = c - a.chunk0[i];
      if (cc == 0) {
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) acc[k4] = (v4f32){0.0f, 0.0f, 0.0f, 0.0f};
      }
      const v4i16 psv = __builtin_bit_cast(v4i16, make_uint2(spw[rl][c * 8 + 2 * g], spw[rl][c * 8 + 2 * g + 1]));
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) {
        v4i16 bv;
        if constexpr (PRE)
          bv = bo[c][k4];
        else
          bv = load4(a.b[i], a.N, a.rank[i], mt * 64 + up_col(p, k4), 16 * cc + 4 * g);
        acc[k4] = mfma1<HALF>(bv, psv, acc[k4]);
      }
      if (c + 1 == a.nchunks || a.cfac[c + 1] != i) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          float part = round_dt<DT>(acc[j >> 2][j & 3]);
          if (a.bias[i] && up_col_of(mt, g, j) < a.N)
            part = round_dt<DT>(part + round_dt<DT>(val_dt<DT>(a.bias[i][up_col_of(mt, g, j)]) * a.s[i]));
          total[j] = i == 0 ? part : round_dt<DT>(total[j] + part);
        }
      }
    }
  }
  if (tok) up_store<DT>(a, t, mt, g, vec, y0, y1, total);
}

// How the down projection is shared out: CB rank chunks per workgroup, S spans
// of K.  A workgroup is bound by the latency of its rounds (about 4 us for 4096
// columns of one chunk), so up to one per CU each more takes work off the
// others: chunk blocks (a larger block shares its x) and spans (whose S partials
// of p are summed afterwards).  Long spans take the largest block that reaches
// RT_DWG workgroups with them; where that would take spans of less than 3 steps
// (3072 columns), smaller blocks come first (1024 tokens, rank 64: K 14336 CB 4
// and S 4 41.6 us, CB 1 and S 1 45.8; K 4096 27.5 and 27.0).  Per call, K -> 4096,
// one workgroup per 16 tokens -> this: 17 tokens, rank 16, K 4096 12.5 -> 7.9 us;
// four rank-64 factors, K 4096 94 -> 28, K 14336 277 -> 29; 256 tokens, rank 64,
// K 14336 71 -> 19; 1024 tokens, rank 64, K 4096 37.1 -> 27.0.  More than RT_DWG
// workgroups do not pay (2048 tokens, K 4096: rank 16 20.0 us with 128 or 256,
// 21.7 with 512; rank 64 43.6 with 256, 48.4 with 512).
constexpr int64_t RT_DWG = 256;
constexpr int64_t RT_MAX_S = 16;
// Who adds the spans: every wave of the up kernel for its own tokens (no third
// launch, whose host side costs 2.7 us of a call of 19) with at most 3 chunks,
// each a serial sum ahead of the MFMAs, and up to RT_FOLD KB of partials read in
// all.  us, K 4096: 17 tokens rank 16 up kernel 8.1, own launch 9.1, one span 12.5;
// rank 64 14.4, 11.3, 14.6; -> 14336, rank 16: 256 tokens (14336 KB) 12.2, 12.2,
// 15.3; 512 (28672 KB) 17.9, 16.6, 18.8; 1024 (57344 KB) 23.6, 21.2, 23.2.
// Otherwise their own launch, or one span where that takes a single round.
constexpr int RT_FOLD_CHUNKS = 3;
constexpr int64_t RT_FOLD = 32768;
constexpr int64_t RT_ROUND = 32 * RT_DNW * RT_DU;  // columns of a round
struct DownPlan {
  int cb, blocks;
  int64_t S, kspan;
};
DownPlan down_plan(int64_t T, int64_t K, int chunks) {
  const int64_t tiles = (T + 15) / 16, steps = (K + RT_DSTEP - 1) / RT_DSTEP;
  DownPlan d;
  d.cb = chunks > 2 ? 4 : chunks;
  for (;; d.cb /= 2) {
    d.blocks = (chunks + d.cb - 1) / d.cb;
    d.S = RT_DWG / (tiles * d.blocks);
    if (d.S <= (steps < 6 ? 1 : steps / 3) || d.cb == 1) break;
  }
  if (d.S > RT_MAX_S) d.S = RT_MAX_S;
  if (d.S < 1) d.S = 1;
  d.kspan = (steps + d.S - 1) / d.S * RT_DSTEP;
  d.S = (K + d.kspan - 1) / d.kspan;
  return d;
}

}  // namespace

extern "C" size_t lm_routed_workspace_size(int64_t T, int64_t K, const lm_routed_factor* factors, int32_t count) {
  if (T <= 16) return 0;  // the single-launch path keeps everything in LDS
  int chunks = 0;
  for (int i = 0; i < count && factors; ++i) chunks += (factors[i].rank + 15) / 16;
  if (chunks < 1 || K < 1) return 256;  // (lm_routed_residual refuses these)
  const DownPlan d = down_plan(T, K, chunks);
  const size_t tt = (size_t)T * (size_t)chunks * 16;
  return align256(tt * sizeof(uint16_t)) + (d.S > 1 ? align256((size_t)d.S * tt * sizeof(float)) : 0);
}

extern "C" int lm_routed_residual(const void* x, const void* y, void* out, int64_t T, int64_t K, int64_t N,
                                  int32_t dtype, const lm_routed_factor* factors, int32_t count, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  if (!x || !y || !out || !factors) return fail(LM_EINVAL, "routed residual pointers must be non-null");
  if (T < 0 || K <= 0 || N <= 0) return fail(LM_EINVAL, "routed residual needs K, N > 0 and T >= 0");
  if (dtype != LM_BF16 && dtype != LM_F16)
    return fail(LM_EUNSUPPORTED, "routed residual dtype must be bfloat16 or float16, got dtype id %d", dtype);
  if (count < 1 || count > RT_MAX_FACTORS)
    return fail(LM_EUNSUPPORTED, "routed residual takes 1..%d factors, got %d", RT_MAX_FACTORS, count);
  if ((K & 3) != 0) return fail(LM_EUNSUPPORTED, "routed residual needs in_features %% 4 == 0, got %lld", (long long)K);
  if ((((uintptr_t)x) & 7) != 0) return fail(LM_EINVAL, "routed residual input must be 8-byte aligned");
  RoutedArgs a;
  memset(&a, 0, sizeof a);
  int chunks = 0;
  for (int i = 0; i < count; ++i) {
    const lm_routed_factor& f = factors[i];
    if (!f.a || !f.b) return fail(LM_EINVAL, "routed factor %d has a null A or B", i);
    if (f.rank <= 0 || f.rank > 64) return fail(LM_EUNSUPPORTED, "routed factor %d rank %d outside 1..64", i, f.rank);
    if ((((uintptr_t)f.a) & 7) != 0 || (((uintptr_t)f.b) & 7) != 0)
      return fail(LM_EINVAL, "routed factor %d must be 8-byte aligned", i);
    a.a[i] = (const uint16_t*)f.a;
    a.b[i] = (const uint16_t*)f.b;
    a.bias[i] = (const uint16_t*)f.bias;
    a.s[i] = f.strength;
    a.rank[i] = f.rank;
    a.chunk0[i] = chunks;
    const int nck = (f.rank + 15) / 16;
    if (chunks + nck > RT_MAX_CHUNKS)
      return fail(LM_EUNSUPPORTED, "routed factors need more than %d rank chunks of 16", RT_MAX_CHUNKS);
    for (int c = chunks; c < chunks + nck; ++c) a.cfac[c] = i;
    chunks += nck;
  }
  if (T == 0) return LM_OK;
  const size_t need = lm_routed_workspace_size(T, K, factors, count);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return fail(LM_EWORKSPACE, "routed residual workspace too small: %zu < %zu bytes", workspace_bytes, need);
  if (((uintptr_t)workspace & 255) != 0) return fail(LM_EINVAL, "workspace must be 256-byte aligned");
  const int64_t tiles = (T + 15) / 16;
  a.x = (const uint16_t*)x;
  a.y = (const uint16_t*)y;
  a.out = (uint16_t*)out;
  DownPlan d = down_plan(T, K, chunks);
  const bool spans = d.S > 1 && chunks <= RT_FOLD_CHUNKS && (N + 63) / 64 * tiles * chunks * d.S <= RT_FOLD;
  if (d.S > 1 && !spans && K <= RT_ROUND) {
    d.S = 1;
    d.kspan = K;
  }
  a.S = (int)d.S;
  a.ps = (uint16_t*)workspace;
  a.part = (float*)((uint8_t*)workspace + align256((size_t)T * (size_t)chunks * 16 * sizeof(uint16_t)));
  a.kspan = d.kspan;
  a.T = T;
  a.K = K;
  a.N = N;
  a.nf = count;
  a.nchunks = chunks;
  // up kernel: one 64-column tile per wave, token tiles split into groups so
  // that there are about 8192 waves in all (4096 and 16384: 57.5 and 57.7
  // against 56.3 us for 4096 tokens, 4096 -> 14336, rank 16), or 4096 from rank
  // 64 on, where a wave's B operands (2 KB a chunk) are more than a token tile
  // of y and out (4 KB): 1024 tokens, 4096 -> 14336, four rank-64 factors 149
  // against 175 us, 2048 tokens 248 and 259, 2048 tokens, 4096 -> 4096 134 and
  // 180; rank 48 in three factors 4096 tokens 108 against 92
  const int64_t ntiles = (N + 63) / 64;
  const int64_t colgroups = (ntiles + RT_NW - 1) / RT_NW;
  const int64_t waves = chunks < 4 ? 8192 : 4096;
  int64_t tgroups = (waves + ntiles - 1) / ntiles;
  if (tgroups > tiles) tgroups = tiles;
  if (tgroups < 1) tgroups = 1;
  a.tiles_per_wg = (int)((tiles + tgroups - 1) / tgroups);
  tgroups = (tiles + a.tiles_per_wg - 1) / a.tiles_per_wg;
  if (tiles * d.blocks > 0x7fffffff || tgroups > 65535 || colgroups > 0x7fffffff)
    return fail(LM_EUNSUPPORTED, "routed residual grid too large");
  hipStream_t st = (hipStream_t)stream;
  TimedLaunch timed("routed", st);
  const dim3 block(RT_NW * 64);
  if (T <= 16) {  // one token tile: a single launch
    const dim3 sgrid((unsigned)((ntiles + RT_SNW - 1) / RT_SNW)), sblock(RT_SNW * 64);
#define RT_SM(H_)                                                                                 \
  if (chunks <= 1) hipLaunchKernelGGL((k_routed_small<H_, 1>), sgrid, sblock, 0, st, a);      \
  else if (chunks <= 2) hipLaunchKernelGGL((k_routed_small<H_, 2>), sgrid, sblock, 0, st, a); \
  else if (chunks <= 4) hipLaunchKernelGGL((k_routed_small<H_, 4>), sgrid, sblock, 0, st, a); \
  else hipLaunchKernelGGL((k_routed_small<H_, RT_MAX_CHUNKS>), sgrid, sblock, 0, st, a);
    if (dtype == LM_F16) { RT_SM(true) } else { RT_SM(false) }
#undef RT_SM
    LAUNCH_CHECK();
    return LM_OK;
  }
  const dim3 ugrid((unsigned)colgroups, (unsigned)tgroups);
  // (32-bit lane offsets of a token tile)
  const bool lean = count == 1 && !a.bias[0] && (N & 7) == 0 && chunks <= 4 && chunks != 3 && N < (INT64_C(1) << 26) &&
                    T < (INT64_C(1) << 31) - 16;
#define RT_UP(H_)                                                                                           \
  if (lean && chunks == 1) hipLaunchKernelGGL((k_routed_up1<H_, 1, false>), ugrid, block, 0, st, a);        \
  else if (lean && chunks == 2) hipLaunchKernelGGL((k_routed_up1<H_, 2, false>), ugrid, block, 0, st, a);   \
  else if (lean) hipLaunchKernelGGL((k_routed_up1<H_, 4, false>), ugrid, block, 0, st, a);                  \
  else if (chunks <= 1) hipLaunchKernelGGL((k_routed_up<H_, 1, false>), ugrid, block, 0, st, a);            \
  else if (chunks <= 2) hipLaunchKernelGGL((k_routed_up<H_, 2, false>), ugrid, block, 0, st, a);            \
  else if (chunks <= 4) hipLaunchKernelGGL((k_routed_up<H_, 4, false>), ugrid, block, 0, st, a);            \
  else hipLaunchKernelGGL((k_routed_up<H_, RT_MAX_CHUNKS, false>), ugrid, block, 0, st, a);
#define RT_UP_SPANS(H_)                                                                                     \
  if (lean && chunks == 1) hipLaunchKernelGGL((k_routed_up1<H_, 1, true>), ugrid, block, 0, st, a);         \
  else if (lean && chunks == 2) hipLaunchKernelGGL((k_routed_up1<H_, 2, true>), ugrid, block, 0, st, a);    \
  else if (chunks <= 1) hipLaunchKernelGGL((k_routed_up<H_, 1, true>), ugrid, block, 0, st, a);             \
  else if (chunks <= 2) hipLaunchKernelGGL((k_routed_up<H_, 2, true>), ugrid, block, 0, st, a);             \
  else hipLaunchKernelGGL((k_routed_up<H_, RT_FOLD_CHUNKS, true>), ugrid, block, 0, st, a);
  const FastDiv by_blocks = fast_div((uint32_t)d.blocks);
  const dim3 dgrid((unsigned)(tiles * d.blocks), (unsigned)d.S), dblock(RT_DNW * 64);
  const dim3 fgrid((unsigned)((T * chunks * 4 + 255) / 256));
#define RT_RUN(H_)                                                                                      \
  if (d.cb == 1) hipLaunchKernelGGL((k_routed_down<H_, 1>), dgrid, dblock, 0, st, a, by_blocks);        \
  else if (d.cb == 2) hipLaunchKernelGGL((k_routed_down<H_, 2>), dgrid, dblock, 0, st, a, by_blocks);   \
  else hipLaunchKernelGGL((k_routed_down<H_, 4>), dgrid, dblock, 0, st, a, by_blocks);                  \
  if (d.S > 1 && !spans) hipLaunchKernelGGL(k_routed_finalize<H_>, fgrid, dim3(256), 0, st, a);         \
  if (spans) { RT_UP_SPANS(H_) } else { RT_UP(H_) }
  if (dtype == LM_F16) {
    RT_RUN(true)
  } else {
    RT_RUN(false)
  }
#undef RT_RUN
#undef RT_UP
#undef RT_UP_SPANS
  LAUNCH_CHECK();
  return LM_OK;
}
