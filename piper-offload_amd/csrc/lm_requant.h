// lm_requant.h -- encode a dense bf16/fp16 weight to a packed format: the
// second half of the reference's portable merge (P/_torchao_int8.py:143-173,
// P/_torchao_float8.py:125-161, P/_torchao_nvfp4.py:145-197,
// P/_torchao_mx.py:178-207; P/ = the reference's src/piper_offload/).
//
// There is no contraction here, so nothing ties a lane to the MFMA layout: a
// lane takes 8 (block formats 16) consecutive elements of the flat weight, a
// wave's load covers contiguous memory, and one Philox call serves a lane's 8
// elements.  HBM traffic bounds all of them (2 bytes read, 0.5 to 1 written
// per element), then the requant arithmetic.
//   k_rq_rows   per-row INT8 / FP8, except long lists of short rows (rq_plan): a
//               row's values stay in registers (8 chunks per lane, all requested
//               at once) between the row maximum and the encode; the waves of a
//               row meet in LDS.
//   k_rq_groups per-group INT8 / FP8 with groups (or whole rows) of 16 .. 512
//               elements, a power of two: the group's lanes reduce with DPP.
//   k_rq_amax   per-tensor max and min: one partial per workgroup, no atomics
//               and nothing to clear beforehand; the encode's workgroups
//               reduce the partials themselves.
//   k_rq_tensor per-tensor INT8 / FP8 encode.
//   k_rq_blocks NVFP4 (one or two levels), MX and Q8_0 encode.
// The arithmetic is that of the merge kernels' requant (lm_impl.h).  Measured
// on [14336, 4096] bf16, per call, against the MFMA-tile kernels with 2-byte
// loads and a factor-prep launch that these replace: INT8 groups of 128 51.7
// -> 38.2 us, FP8 per tensor 281 -> 54.1, NVFP4 two-level 296 -> 58.3 (swizzled,
// stochastic 295 -> 68.2), MXFP4 467 -> 30.4, MXFP8 stochastic 159 -> 37.0, Q8_0
// 414 -> 35.9.
#pragma once
#include "lm_impl.h"

struct RqArgs {
  const uint16_t* dense;
  uint8_t* q_out;
  void* scale_out;
  void* aux_out;       // INT8: zero points or null; two-level NVFP4: the per-tensor scale
  float* part;         // per-tensor partials: (max, max(-min)) per workgroup of k_rq_amax
  int npart;
  int64_t M, N;
  uint64_t seed;
  int scale_dt, qmin, qmax;
  int swizzled, mx_mode;
  int aligned;         // 16-byte aligned input and output
  int waves_per_row;   // k_rq_rows
  int group_lanes;     // k_rq_groups
  FastDiv div;         // swizzled k_rq_blocks: by the scale columns
};

// 8 elements of a dense weight; count < 8: the rest are zeros
template <int CD>
DEV void rq_load8(const uint16_t* p, int count, bool aligned, float (&v)[8]) {
  if (count == 8 && aligned) {
    const lm_u32x4 w = *(const LM_GLOBAL lm_u32x4*)p;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = val_dt<CD>((j & 1) ? (w[j >> 1] >> 16) : (w[j >> 1] & 0xffffu));
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = j < count ? val_dt<CD>(((const LM_GLOBAL uint16_t*)p)[j]) : 0.0f;
  }
}
// 8 one-byte codes
DEV void rq_store8(uint8_t* p, int count, bool aligned, const uint32_t (&w)[2]) {
  if (count == 8 && aligned) {
    *(LM_GLOBAL lm_u32x2*)p = lm_u32x2{w[0], w[1]};
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < count) ((LM_GLOBAL uint8_t*)p)[j] = (uint8_t)(w[j >> 2] >> (8 * (j & 3)));
  }
}

// the codes of 8 values at flat offset idx0 (a multiple of 8), two words
template <int KIND, int SDT, bool SR>
DEV void rq_encode8(const RqArgs& a, uint64_t idx0, const RowQP& qp, const float (&m)[8], uint32_t (&w)[2]) {
  uint32_t nw[4];  // complemented Philox words
  if constexpr (SR) sr_nwords_aligned<8>(a.seed, idx0, nw);
  if constexpr (KIND == K_INT8) {
    if constexpr (SR) {
      const float lo = 1536.0f + (float)a.qmin, hi = 1536.0f + (float)a.qmax, base = 1536.0f + qp.zp;
      uint32_t pr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pr[i] = sr_i8_pair(nw[i], sr_i8_t(m[2 * i], qp.rcp, base, lo, hi), sr_i8_t(m[2 * i + 1], qp.rcp, base, lo, hi),
                           nw[i], nw[i] << 16);
      w[0] = pack_sr_i8(pr[0], pr[1]);
      w[1] = pack_sr_i8(pr[2], pr[3]);
    } else {
      const int zp = (int)qp.zp;
      uint32_t c[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int q = (int)__builtin_rintf(round_dt<SDT>(m[j] * qp.inv)) + zp;
        c[j] = (uint32_t)(q < a.qmin ? a.qmin : (q > a.qmax ? a.qmax : q));
      }
      w[0] = pack_low_bytes(c[0], c[1], c[2], c[3]);
      w[1] = pack_low_bytes(c[4], c[5], c[6], c[7]);
    }
  } else {
    constexpr float L = FmtLimit<KIND>::v;
    constexpr int F = FmtLimit<KIND>::fmt;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = __builtin_fminf(__builtin_fmaxf(div_rn(m[j], qp.s, qp.rcp), -L), L);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (SR) w[i] = sr_fp8_nword<F>(x + 4 * i, nw + 2 * i);
      else w[i] = fp8_pack4<F>(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
    }
  }
}
template <int KIND>
DEV void rq_account(const float (&m)[8], float& vmx, float& vmn) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if constexpr (KIND == K_INT8) {
      vmx = __builtin_fmaxf(vmx, m[j]);
      vmn = __builtin_fminf(vmn, m[j]);
    } else {
      vmx = __builtin_fmaxf(vmx, __builtin_fabsf(m[j]));
    }
  }
}
// qparams from a maximum and minimum, stored at qi by the writer
template <int KIND, int CD, int SDT, bool ASYM>
DEV RowQP rq_qparams(const RqArgs& a, float mx, float mn, int64_t qi, bool writer) {
  RowQP qp;
  float stored;
  if constexpr (KIND == K_INT8) {
    int zp;
    qp = int8_qparams<CD, SDT, ASYM>(mn, mx, a.qmin, a.qmax, stored, zp);
    if (writer) {
      store_scalar(a.scale_out, qi, SDT, stored);
      if (a.aux_out) ((int8_t*)a.aux_out)[qi] = (int8_t)zp;
    }
  } else {
    qp = fp8_qparams<CD, KIND>(mx, stored);
    if (writer) ((float*)a.scale_out)[qi] = stored;
  }
  return qp;
}

// ---- per row --------------------------------------------------------------------
// N % 8 == 0, 16-byte aligned rows.  A row belongs to waves_per_row waves
// (1, 2, 4, 8 or 16) of RQ_CPT chunks per lane, so that rows of up to 65536
// elements stay in registers (32 VGPRs); short rows share a workgroup.
// INT8 rows of [14336, 4096], per call: 51.0 -> 33.6 us round to
// nearest, 56.4 -> 33.7 us stochastic (5.2 TB/s; k_rows before, 16 rows per
// workgroup in the MFMA lane layout); [4096, 14336]: 60.2 -> 33.2 us.
constexpr int RQ_CPT = 8;
template <int KIND, int CD, int SDT, bool ASYM, bool SR>
__global__ __launch_bounds__(1024) void k_rq_rows(RqArgs a) {
  __shared__ float sh_mx[16], sh_mn[16];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int wpr = a.waves_per_row, rows_per_wg = (int)(blockDim.x >> 6) / wpr;
  const int64_t row = (int64_t)blockIdx.x * rows_per_wg + wave / wpr;
  const int wr = wave % wpr;  // the wave's index in its row
  const bool rok = row < a.M;  // wave-uniform
  const int nch = (int)(a.N >> 3);
  const uint16_t* src = a.dense + row * a.N;
  lm_u32x4 raw[RQ_CPT];
#pragma unroll
  for (int i = 0; i < RQ_CPT; ++i) {
    const int c = (i * wpr + wr) * 64 + lane;
    raw[i] = lm_u32x4{0u, 0u, 0u, 0u};  // zeros do not change a maximum or minimum that include 0
    if (rok && c < nch) raw[i] = ((const LM_GLOBAL lm_u32x4*)src)[c];
  }
  float vmx = 0.0f, vmn = 0.0f;
#pragma unroll
  for (int i = 0; i < RQ_CPT; ++i) {
    float m[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = val_dt<CD>((j & 1) ? (raw[i][j >> 1] >> 16) : (raw[i][j >> 1] & 0xffffu));
    rq_account<KIND>(m, vmx, vmn);
  }
  vmx = wave_max(vmx);
  if constexpr (KIND == K_INT8) vmn = -wave_max(-vmn);
  if (wpr > 1) {
    if (lane == 0) {
      sh_mx[wave] = vmx;
      sh_mn[wave] = vmn;
    }
    __syncthreads();
    for (int w = wave - wr; w < wave - wr + wpr; ++w) {
      vmx = __builtin_fmaxf(vmx, sh_mx[w]);
      vmn = __builtin_fminf(vmn, sh_mn[w]);
    }
  }
  if (!rok) return;
  const RowQP qp = rq_qparams<KIND, CD, SDT, ASYM>(a, vmx, vmn, row, wr == 0 && lane == 0);
#pragma unroll
  for (int i = 0; i < RQ_CPT; ++i) {
    const int c = (i * wpr + wr) * 64 + lane;
    if (c >= nch) break;
    float m[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = val_dt<CD>((j & 1) ? (raw[i][j >> 1] >> 16) : (raw[i][j >> 1] & 0xffffu));
    uint32_t w[2];
    rq_encode8<KIND, SDT, SR>(a, (uint64_t)(row * a.N) + 8u * (uint32_t)c, qp, m, w);
    *(LM_GLOBAL lm_u32x2*)(a.q_out + row * a.N + 8 * c) = lm_u32x2{w[0], w[1]};
  }
}

// ---- per group --------------------------------------------------------------------
// Groups of 8 group_lanes elements (2 .. 64 lanes, a power of two): flat
// chunks, the group's lanes are neighbours.  Every lane stays active for the
// reductions; lanes past the end hold zeros and store nothing.
DEV float rq_lanes_max(float x, int lanes) {  // lanes is wave-uniform
  x = __builtin_fmaxf(x, dpp_f32<0xB1>(x));
  if (lanes >= 4) x = __builtin_fmaxf(x, dpp_f32<0x4E>(x));
  if (lanes >= 8) x = __builtin_fmaxf(x, dpp_f32<0x141>(x));
  if (lanes >= 16) x = __builtin_fmaxf(x, dpp_f32<0x140>(x));
  if (lanes >= 32) x = lanes_max16(x);
  if (lanes >= 64) x = lanes_max32(x);
  return x;
}
constexpr int RQ_U = 4;  // chunks per lane of the flat kernels, requested together
template <int KIND, int CD, int SDT, bool ASYM, bool SR>
__global__ __launch_bounds__(256) void k_rq_groups(RqArgs a) {
  const int64_t nch = (a.M * a.N) >> 3;
  const int64_t c0 = (int64_t)blockIdx.x * (256 * RQ_U) + threadIdx.x;
  const int gl = a.group_lanes, lg = __builtin_ctz(gl);
  float m[RQ_U][8];
#pragma unroll
  for (int u = 0; u < RQ_U; ++u) {
    const int64_t c = c0 + 256 * u;
    rq_load8<CD>(a.dense + 8 * c, c < nch ? 8 : 0, true, m[u]);
  }
#pragma unroll
  for (int u = 0; u < RQ_U; ++u) {
    const int64_t c = c0 + 256 * u;
    float vmx = 0.0f, vmn = 0.0f;
    rq_account<KIND>(m[u], vmx, vmn);
    vmx = rq_lanes_max(vmx, gl);
    if constexpr (KIND == K_INT8) vmn = -rq_lanes_max(-vmn, gl);
    const RowQP qp = rq_qparams<KIND, CD, SDT, ASYM>(a, vmx, vmn, c >> lg, c < nch && (c & (gl - 1)) == 0);
    uint32_t w[2];
    rq_encode8<KIND, SDT, SR>(a, 8 * (uint64_t)c, qp, m[u], w);
    if (c < nch) rq_store8(a.q_out + 8 * c, 8, true, w);
  }
}

// ---- per tensor ---------------------------------------------------------------------
template <int CD>
__global__ __launch_bounds__(256) void k_rq_amax(RqArgs a) {
  __shared__ float sh[2][4];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int64_t n = a.M * a.N, nch = (n + 7) >> 3;
  float vmx = 0.0f, vmn = 0.0f;
  for (int64_t c0 = (int64_t)blockIdx.x * (256 * RQ_U) + threadIdx.x; c0 < nch; c0 += (int64_t)gridDim.x * (256 * RQ_U)) {
    float m[RQ_U][8];
#pragma unroll
    for (int u = 0; u < RQ_U; ++u) {
      const int64_t left = n - 8 * (c0 + 256 * u);
      rq_load8<CD>(a.dense + 8 * (c0 + 256 * u), left >= 8 ? 8 : (left > 0 ? (int)left : 0), a.aligned, m[u]);
    }
#pragma unroll
    for (int u = 0; u < RQ_U; ++u) rq_account<K_INT8>(m[u], vmx, vmn);
  }
  vmx = wave_max(vmx);
  vmn = wave_max(-vmn);
  if (lane == 0) {
    sh[0][wave] = vmx;
    sh[1][wave] = vmn;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int k = threadIdx.x;
    a.part[2 * blockIdx.x + k] = __builtin_fmaxf(__builtin_fmaxf(sh[k][0], sh[k][1]), __builtin_fmaxf(sh[k][2], sh[k][3]));
  }
}
// the tensor's (max, -min) from the partials, in every thread of a 256-thread workgroup
DEV void rq_tensor_range(const RqArgs& a, float& mx, float& mn) {
  __shared__ float sh[2][4];
  const int lane = threadIdx.x & 63, wave = wave_index();
  float x = 0.0f, y = 0.0f;
  for (int i = threadIdx.x; i < a.npart; i += 256) {
    x = __builtin_fmaxf(x, ((const LM_GLOBAL float*)a.part)[2 * i]);
    y = __builtin_fmaxf(y, ((const LM_GLOBAL float*)a.part)[2 * i + 1]);
  }
  x = wave_max(x);
  y = wave_max(y);
  if (lane == 0) {
    sh[0][wave] = x;
    sh[1][wave] = y;
  }
  __syncthreads();
  mx = __builtin_fmaxf(__builtin_fmaxf(sh[0][0], sh[0][1]), __builtin_fmaxf(sh[0][2], sh[0][3]));
  mn = -__builtin_fmaxf(__builtin_fmaxf(sh[1][0], sh[1][1]), __builtin_fmaxf(sh[1][2], sh[1][3]));
}
template <int KIND, int CD, int SDT, bool ASYM, bool SR>
__global__ __launch_bounds__(256) void k_rq_tensor(RqArgs a) {
  const int64_t n = a.M * a.N, nch = (n + 7) >> 3;
  float mx, mn;
  rq_tensor_range(a, mx, mn);
  if constexpr (KIND != K_INT8) mx = __builtin_fmaxf(mx, -mn);
  const RowQP qp = rq_qparams<KIND, CD, SDT, ASYM>(a, mx, mn, 0, blockIdx.x == 0 && threadIdx.x == 0);
  for (int64_t c0 = (int64_t)blockIdx.x * (256 * RQ_U) + threadIdx.x; c0 < nch; c0 += (int64_t)gridDim.x * (256 * RQ_U)) {
    float m[RQ_U][8];
    int cnt[RQ_U];
#pragma unroll
    for (int u = 0; u < RQ_U; ++u) {
      const int64_t left = n - 8 * (c0 + 256 * u);
      cnt[u] = left >= 8 ? 8 : (left > 0 ? (int)left : 0);
      rq_load8<CD>(a.dense + 8 * (c0 + 256 * u), cnt[u], a.aligned, m[u]);
    }
#pragma unroll
    for (int u = 0; u < RQ_U; ++u) {
      const int64_t c = c0 + 256 * u;
      uint32_t w[2];
      rq_encode8<KIND, SDT, SR>(a, 8 * (uint64_t)c, qp, m[u], w);
      rq_store8(a.q_out + 8 * c, cnt[u], a.aligned, w);
    }
  }
}

// the swizzled place of block b
DEV int64_t rq_swizzled(const RqArgs& a, int64_t b, int64_t s_cols) {
  const int64_t row = b < (INT64_C(1) << 32) ? (int64_t)div_by(a.div, (uint32_t)b) : b / s_cols;
  return blocked_offset(row, b - row * s_cols, s_cols, true);
}

// ---- block formats ------------------------------------------------------------------
// A lane takes 16 elements: one NVFP4 block, or half an MX / Q8_0 block, whose
// two lanes are neighbours.  Q8_0's 34-byte blocks leave through LDS: a
// workgroup's 128 blocks are 4352 contiguous, 16-byte aligned bytes.
template <int F, int CD, bool SR>
__global__ __launch_bounds__(256) void k_rq_blocks(RqArgs a) {
  constexpr bool Q8 = F == B_Q8_0;
  constexpr int Q8_BYTES = 128 * 34;
  __shared__ __attribute__((aligned(16))) uint8_t stage[Q8 ? Q8_BYTES : 16];
  const int64_t n16 = (a.M * a.N) >> 4;  // N % 16 == 0
  float g = 1.0f;
  const bool two = F == B_NVFP4 && a.aux_out != nullptr;
  if constexpr (F == B_NVFP4) {
    if (two) {
      float mx, mn;
      rq_tensor_range(a, mx, mn);
      g = __builtin_fmaxf(__builtin_fmaxf(mx, -mn) / 2688.0f, kEps);
      if (blockIdx.x == 0 && threadIdx.x == 0) *(float*)a.aux_out = g;
    }
  }
  const float inv_g = 1.0f / g;
  for (int64_t b0 = (int64_t)blockIdx.x * 256; b0 < n16; b0 += (int64_t)gridDim.x * 256) {
    const int64_t c = b0 + threadIdx.x;  // 16-element index; lanes past the end hold zeros and store nothing
    const bool ok = c < n16;
    float m[16];
    {
      float lo[8], hi[8];
      rq_load8<CD>(a.dense + 16 * c, ok ? 8 : 0, a.aligned, lo);
      rq_load8<CD>(a.dense + 16 * c + 8, ok ? 8 : 0, a.aligned, hi);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        m[j] = lo[j];
        m[8 + j] = hi[j];
      }
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) amax = __builtin_fmaxf(amax, __builtin_fabsf(m[j]));
    uint32_t nw[8];
    if constexpr (SR) sr_nwords_aligned<16>(a.seed, 16 * (uint64_t)c, nw);
    if constexpr (F == B_NVFP4) {
      const float bscale = amax / 6.0f;
      float fs = two ? bscale / g : bscale;
      fs = __builtin_fminf(__builtin_fmaxf(fs, 0.015625f), 448.0f);
      const uint32_t sc8 = fp8_encode1<E4M3>(fs);
      fs = fp8_value<E4M3>(sc8);
      const float recip = two ? inv_g / fs : 0.0f, rfs = 1.0f / fs;
      float x[16];
#pragma unroll
      for (int j = 0; j < 16; ++j)
        x[j] = __builtin_fminf(__builtin_fmaxf(two ? m[j] * recip : div_rn(m[j], fs, rfs), -6.0f), 6.0f);
      uint32_t w[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if constexpr (SR) w[k] = sr_e2m1_nword(x + 8 * k, nw + 4 * k);
        else {
          w[k] = 0u;
#pragma unroll
          for (int t = 0; t < 4; ++t) w[k] |= e2m1_pack2(x[8 * k + 2 * t], x[8 * k + 2 * t + 1]) << (8 * t);
        }
      }
      if (ok) {
        int64_t so = c;
        if (a.swizzled) {
          so = rq_swizzled(a, c, a.N >> 4);
        }
        ((LM_GLOBAL uint8_t*)a.scale_out)[so] = (uint8_t)sc8;
        rq_store8(a.q_out + 8 * c, 8, a.aligned, w);
      }
    } else if constexpr (Q8) {
      amax = __builtin_fmaxf(amax, dpp_f32<0xB1>(amax));
      const float d = amax / 127.0f, id = d != 0.0f ? 1.0f / d : 0.0f;
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (SR) {
          uint32_t pr[2];
#pragma unroll
          for (int i = 0; i < 2; ++i)
            pr[i] = sr_i8_pair(nw[2 * k + i], sr_i8_t(m[4 * k + 2 * i], id, 1536.0f, 1409.0f, 1663.0f),
                               sr_i8_t(m[4 * k + 2 * i + 1], id, 1536.0f, 1409.0f, 1663.0f), nw[2 * k + i],
                               nw[2 * k + i] << 16);
          w[k] = pack_sr_i8(pr[0], pr[1]);
        } else {
          uint32_t q[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) q[i] = (uint32_t)(int)__builtin_roundf(m[4 * k + i] * id);
          w[k] = pack_low_bytes(q[0], q[1], q[2], q[3]);
        }
      }
      // block t / 2 of the workgroup: d, then this lane's half of the codes
      uint16_t* s16 = (uint16_t*)(stage + (threadIdx.x >> 1) * 34);
      if ((threadIdx.x & 1) == 0) s16[0] = f16_bits(d);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        s16[1 + 8 * (threadIdx.x & 1) + 2 * k] = (uint16_t)w[k];
        s16[2 + 8 * (threadIdx.x & 1) + 2 * k] = (uint16_t)(w[k] >> 16);
      }
      __syncthreads();
      const int64_t left = (n16 - b0) >> 1;  // whole 32-element blocks from b0
      const int bytes = left >= 128 ? Q8_BYTES : (int)left * 34;
      uint8_t* dst = a.q_out + b0 / 2 * 34;
      if (a.aligned) {
        for (int i = threadIdx.x * 16; i + 16 <= bytes; i += 256 * 16)
          store_b128_guarded((LM_GLOBAL lm_u32x4*)(dst + i), *(const lm_u32x4*)(stage + i));
        const int done = bytes & ~15;
        if ((int)threadIdx.x < bytes - done) dst[done + threadIdx.x] = stage[done + threadIdx.x];
      } else {
        for (int i = threadIdx.x; i < bytes; i += 256) dst[i] = stage[i];
      }
      __syncthreads();  // the staged bytes are read before the next blocks overwrite them
    } else {  // MX
      constexpr int emax = F == B_MXFP4 ? 2 : (F == B_MXE4M3 ? 8 : 15);
      constexpr float maxpos = F == B_MXFP4 ? 6.0f : (F == B_MXE4M3 ? 448.0f : 57344.0f);
      constexpr int mbits = F == B_MXFP4 ? 1 : (F == B_MXE4M3 ? 3 : 2);
      amax = __builtin_fmaxf(amax, dpp_f32<0xB1>(amax));
      float inv;
      const uint32_t enc = mx_scale(amax, a.mx_mode, emax, maxpos, mbits, inv);
      float x[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = __builtin_fminf(__builtin_fmaxf(m[j] * inv, -maxpos), maxpos);
      uint32_t w[4];
      if constexpr (F == B_MXFP4) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          if constexpr (SR) w[k] = sr_e2m1_nword(x + 8 * k, nw + 4 * k);
          else {
            w[k] = 0u;
#pragma unroll
            for (int t = 0; t < 4; ++t) w[k] |= e2m1_pack2(x[8 * k + 2 * t], x[8 * k + 2 * t + 1]) << (8 * t);
          }
        }
      } else {
        constexpr int FF = F == B_MXE4M3 ? E4M3 : E5M2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (SR) w[i] = sr_fp8_nword<FF>(x + 4 * i, nw + 2 * i);
          else w[i] = fp8_pack4<FF>(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
        }
      }
      if (ok) {
        if ((c & 1) == 0) {
          int64_t so = c >> 1;
          if (a.swizzled) {
            so = rq_swizzled(a, so, a.N >> 5);
          }
          ((LM_GLOBAL uint8_t*)a.scale_out)[so] = (uint8_t)enc;
        }
        const uint32_t lo[2] = {w[0], w[1]};
        if constexpr (F == B_MXFP4) {
          rq_store8(a.q_out + 8 * c, 8, a.aligned, lo);
        } else {
          const uint32_t hi[2] = {w[2], w[3]};
          if (a.aligned) {
            store_b128_guarded((LM_GLOBAL lm_u32x4*)(a.q_out + 16 * c), lm_u32x4{w[0], w[1], w[2], w[3]});
          } else {
            rq_store8(a.q_out + 16 * c, 8, false, lo);
            rq_store8(a.q_out + 16 * c + 8, 8, false, hi);
          }
        }
      }
    }
  }
}

// ---- host -----------------------------------------------------------------------------
static inline RqArgs rq_args(const void* dense, uint8_t* q_out, void* scale_out, void* aux_out, int64_t M, int64_t N,
                             const lm_rounding* rnd) {
  RqArgs a;
  memset(&a, 0, sizeof a);
  a.dense = (const uint16_t*)dense;
  a.q_out = q_out;
  a.scale_out = scale_out;
  a.aux_out = aux_out;
  a.M = M;
  a.N = N;
  a.seed = seed_of(rnd);
  a.aligned = (((uintptr_t)dense | (uintptr_t)q_out) & 15) == 0;
  return a;
}
// the same request for k_rows / k_groups
static inline RowArgs rq_row_args(const RqArgs& r) {
  RowArgs a;
  memset(&a, 0, sizeof a);
  a.dense = r.dense;
  a.q_out = r.q_out;
  a.scale_out = r.scale_out;
  a.zp_out = (int8_t*)r.aux_out;
  a.M = r.M;
  a.N = r.N;
  a.qmin = r.qmin;
  a.qmax = r.qmax;
  a.seed = r.seed;
  return a;
}
// the per-tensor range: up to 1024 workgroups (4 per CU), as many as there are
// RQ_U chunks for and as the workspace from its reduction slots on holds
// partials of
template <int CD>
static int rq_amax_launch(RqArgs& a, void* ws, hipStream_t st) {
  const WsLayout w = ws_layout(a.M, a.N, 0);
  a.part = (float*)((uint8_t*)ws + w.red_off);
  const int64_t room = (int64_t)((w.total - w.red_off) / (2 * sizeof(float)));
  int64_t nb = ((a.M * a.N + 7) / 8 + 256 * RQ_U - 1) / (256 * RQ_U);
  if (nb > 1024) nb = 1024;
  if (nb > room) nb = room;
  a.npart = (int)nb;
  TimedLaunch timed("blocks_amax", st);
  hipLaunchKernelGGL((k_rq_amax<CD>), dim3((unsigned)nb), dim3(256), 0, st, a);
  LAUNCH_CHECK();
  return LM_OK;
}

// a call of KERNEL<KIND, CD, SDT, ASYM, SR> for runtime values (FP8: fp32 scales, no zero point)
#define RQ_DISPATCH(KIND, CALL)                                                                                    \
  do {                                                                                                             \
    if constexpr (KIND != K_INT8) {                                                                                \
      if (cd == LM_F16) { if (sr) { CALL(F16, F32, false, true); } else { CALL(F16, F32, false, false); } }        \
      else { if (sr) { CALL(BF16, F32, false, true); } else { CALL(BF16, F32, false, false); } }                   \
    } else {                                                                                                       \
      const int k_ = (cd == LM_F16 ? 8 : 0) | (a.scale_dt == LM_BF16 ? 4 : 0) | (asym ? 2 : 0) | (sr ? 1 : 0);     \
      switch (k_) {                                                                                                \
        case 0: CALL(BF16, F32, false, false); break;                                                              \
        case 1: CALL(BF16, F32, false, true); break;                                                               \
        case 2: CALL(BF16, F32, true, false); break;                                                               \
        case 3: CALL(BF16, F32, true, true); break;                                                                \
        case 4: CALL(BF16, BF16, false, false); break;                                                             \
        case 5: CALL(BF16, BF16, false, true); break;                                                              \
        case 6: CALL(BF16, BF16, true, false); break;                                                              \
        case 7: CALL(BF16, BF16, true, true); break;                                                               \
        case 8: CALL(F16, F32, false, false); break;                                                               \
        case 9: CALL(F16, F32, false, true); break;                                                                \
        case 10: CALL(F16, F32, true, false); break;                                                               \
        case 11: CALL(F16, F32, true, true); break;                                                                \
        case 12: CALL(F16, BF16, false, false); break;                                                             \
        case 13: CALL(F16, BF16, false, true); break;                                                              \
        case 14: CALL(F16, BF16, true, false); break;                                                              \
        default: CALL(F16, BF16, true, true); break;                                                               \
      }                                                                                                            \
    }                                                                                                              \
  } while (0)

// Per row (group == N) or per group: the flat kernels need whole 16-byte chunks
// per row.  k_rq_rows takes rows that fit 16 waves' registers, but rows of less
// than 1024 elements, of which its waves hold one each, only while they are few
// enough for 16 waves per CU; longer lists of such rows, and groups, go through
// k_rq_groups (2 .. 64 lanes).  The MFMA-layout kernels k_rows and k_groups take
// the rest: odd columns, misaligned storage, groups that are no power of two and
// long lists of short rows that are none.  us per call, FP8 round to nearest:
// rows of 64, 2^26 elements k_rq_groups 34.5, k_rq_rows 394, k_rows 173; of 192
// k_rq_rows 137, k_rows 70; of 768 45 and 38.6; of 1024 36.1 and 37.1; [320, 768]
// k_rq_rows 2.4, k_rows 3.3; [64, 128] k_rq_rows 2.3, k_rq_groups 3.2.
enum RqPlan { RQ_ROWS, RQ_GROUPS, RQ_NONE };
static inline RqPlan rq_plan(const RqArgs& a, int64_t group) {
  if (!a.aligned || a.N % 8 != 0) return RQ_NONE;
  if (group == a.N && a.N <= 16 * 64 * 8 * RQ_CPT && (a.N >= 1024 || a.M <= 4096)) return RQ_ROWS;
  return group >= 16 && group <= 512 && (group & (group - 1)) == 0 ? RQ_GROUPS : RQ_NONE;
}
template <int KIND>
static int run_rq_rows(RqArgs a, RqPlan plan, int64_t group, int cd, bool asym, bool sr, hipStream_t st) {
  if (plan == RQ_ROWS) {
    int wpr = 1;
    while ((int64_t)wpr * 64 * 8 * RQ_CPT < a.N) wpr *= 2;
    a.waves_per_row = wpr;
    const int waves = wpr < 4 ? 4 : wpr, rows = waves / wpr;
    const dim3 grid((unsigned)((a.M + rows - 1) / rows)), block((unsigned)(waves * 64));
    TimedLaunch timed("rows", st);
#define RQ_CALL(CD_, SDT_, AS_, SR_) hipLaunchKernelGGL((k_rq_rows<KIND, CD_, SDT_, AS_, SR_>), grid, block, 0, st, a)
    RQ_DISPATCH(KIND, RQ_CALL);
#undef RQ_CALL
  } else {
    a.group_lanes = (int)(group / 8);
    const int64_t nb = (a.M * a.N / 8 + 256 * RQ_U - 1) / (256 * RQ_U);
    if (nb > 0x7fffffff) return fail(LM_EUNSUPPORTED, "per-group weight too large for one launch");
    const dim3 grid((unsigned)nb), block(256);
    TimedLaunch timed("groups", st);
#define RQ_CALL(CD_, SDT_, AS_, SR_) hipLaunchKernelGGL((k_rq_groups<KIND, CD_, SDT_, AS_, SR_>), grid, block, 0, st, a)
    RQ_DISPATCH(KIND, RQ_CALL);
#undef RQ_CALL
  }
  LAUNCH_CHECK();
  return LM_OK;
}
template <int KIND>
static int run_rq_tensor(RqArgs a, int cd, bool asym, bool sr, void* ws, hipStream_t st) {
  int rc = cd == LM_F16 ? rq_amax_launch<F16>(a, ws, st) : rq_amax_launch<BF16>(a, ws, st);
  if (rc) return rc;
  // at most 2048 workgroups (8 per CU): each reduces the partials first
  int64_t nb = ((a.M * a.N + 7) / 8 + 256 * RQ_U - 1) / (256 * RQ_U);
  if (nb > 2048) nb = 2048;
  const dim3 grid((unsigned)nb), block(256);
  TimedLaunch timed("blocks_quant", st);
#define RQ_CALL(CD_, SDT_, AS_, SR_) hipLaunchKernelGGL((k_rq_tensor<KIND, CD_, SDT_, AS_, SR_>), grid, block, 0, st, a)
  RQ_DISPATCH(KIND, RQ_CALL);
#undef RQ_CALL
  LAUNCH_CHECK();
  return LM_OK;
}
template <int F>
static int run_rq_blocks(RqArgs a, int cd, bool sr, void* ws, hipStream_t st) {
  const bool two = F == B_NVFP4 && a.aux_out != nullptr;
  if (two) {
    const int rc = cd == LM_F16 ? rq_amax_launch<F16>(a, ws, st) : rq_amax_launch<BF16>(a, ws, st);
    if (rc) return rc;
  }
  a.div = fast_div((uint32_t)(a.N / (F == B_NVFP4 ? 16 : 32)));
  int64_t nb = (a.M * a.N / 16 + 255) / 256;
  const int64_t most = two ? 2048 : 65536;  // (two levels: each workgroup reduces the partials first)
  if (nb > most) nb = most;
  const dim3 grid((unsigned)nb), block(256);
  TimedLaunch timed(two ? "blocks_quant" : "blocks_full", st);
  if (cd == LM_F16) {
    if (sr) hipLaunchKernelGGL((k_rq_blocks<F, F16, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_rq_blocks<F, F16, false>), grid, block, 0, st, a);
  } else {
    if (sr) hipLaunchKernelGGL((k_rq_blocks<F, BF16, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_rq_blocks<F, BF16, false>), grid, block, 0, st, a);
  }
  LAUNCH_CHECK();
  return LM_OK;
}
