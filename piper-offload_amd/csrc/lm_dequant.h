// lm_dequant.h -- decode a packed weight (INT8, FP8, NVFP4, MX) to dense
// values: the first half of the reference's portable merge
// (P/_torchao_int8.py:113-141, P/_torchao_float8.py:93-123,
// P/_torchao_nvfp4.py:106-143, P/_torchao_mx.py:143-176; P/ = the reference's
// src/piper_offload/).
//
// The work is HBM traffic: 0.53 to 1 byte of codes and scales read and 2 (or
// 4) bytes written per element, against 2 to 4 VALU instructions.  Codes and
// outputs are flat runs in the same order, so the launch ignores rows: a lane
// decodes 8 consecutive elements and stores them as 16 bytes, a wave's store
// covers 1 KiB, and each thread requests the codes and scales of DQ_U chunks
// before it decodes the first.  Only the qparam index needs the row (or
// group), one multiply-high per chunk (FastDiv).  NVFP4 [14336, 4096] to
// bf16, per call: 144.8 us as a walk over 16-row tiles with 2-byte stores
// (k_blocks), 26.4 us here (5.7 TB/s; a 1 GiB copy reaches 6.16).
#pragma once
#include "lm_impl.h"

struct DqArgs {
  const uint8_t* q;
  const void* scale;
  const void* aux;   // INT8: zero points or null; NVFP4: per-tensor scale or null
  void* out;
  int64_t M, N;
  int64_t group;     // INT8 / FP8: elements per qparam
  int scale_dt;      // INT8 / FP8
  int swizzled;      // NVFP4 / MX
  FastDiv div;       // INT8 / FP8: by group; swizzled NVFP4 / MX: by N / 8
};

constexpr int DQ_THREADS = 256;
// chunks per thread: their loads are in flight together
constexpr int DQ_U = 4;

template <int F>
struct DqTraits {
  static constexpr bool FP4 = F == B_NVFP4 || F == B_MXFP4;
  static constexpr bool BLOCK = F == B_NVFP4 || F == B_MXFP4 || F == B_MXE4M3 || F == B_MXE5M2;  // block scales
  static constexpr int BS = F == B_NVFP4 ? 16 : 32;
  static constexpr int FMT = F == B_E4M3 || F == B_MXE4M3 ? E4M3 : E5M2;
};
// the compute dtype of an output dtype: fp32 outputs hold bf16 values
template <int DT>
constexpr int dq_cd() { return DT == F16 ? F16 : BF16; }

// fp16 RNE as the conversion instruction itself: left to the optimizer,
// fp16(a * b) becomes v_fma_mixlo_f16(a, b, +0), whose addend turns a -0
// product into +0
DEV uint32_t dq_f16_bits(float x) {
  uint32_t h = f2u(x);
  asm("v_cvt_f16_f32 %0, %0" : "+v"(h));  // output tied to the input
  return h & 0xffffu;
}
template <int CD>
DEV float dq_round(float x) {
  if constexpr (CD == F16) return f16_val(dq_f16_bits(x));
  else return bf16r(x);
}

// a block's decode scale from its stored byte
template <int F, int CD>
DEV float dq_block_scale(uint32_t code, bool two, float g) {
  if constexpr (F == B_NVFP4) {
    const float bs = dq_round<CD>(fp8_value<E4M3>(code));
    return two ? dq_round<CD>(bs * g) : bs;
  } else {
    return dq_round<CD>(e8m0_value(code));
  }
}
// codes (8 bytes, or 4 for fp4) to values before their last rounding
template <int F>
DEV void dq_values8(const uint32_t (&w)[2], const float (&s)[8], const float (&z)[8], float (&v)[8]) {
  if constexpr (DqTraits<F>::FP4) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const v2f32 c = e2m1_pair(w[0], j >> 1);
      v[j] = c.x * s[j];
      v[j + 1] = c.y * s[j + 1];
    }
  } else if constexpr (F == B_INT8) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = ((float)(int8_t)(w[j >> 2] >> (8 * (j & 3))) - z[j]) * s[j];
  } else {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const v2f32 c = (j & 2) ? fp8_decode_pair<DqTraits<F>::FMT, true>(w[j >> 2])
                              : fp8_decode_pair<DqTraits<F>::FMT, false>(w[j >> 2]);
      v[j] = c.x * s[j];
      v[j + 1] = c.y * s[j + 1];
    }
  }
}

template <int DT>
DEV void dq_store8(void* out, int64_t e0, const float (&v)[8]) {
  if constexpr (DT == F32) {
    LM_GLOBAL lm_u32x4* o = (LM_GLOBAL lm_u32x4*)((LM_GLOBAL float*)out + e0);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      store_b128_guarded(o + h, lm_u32x4{f2u(bf16r(v[4 * h])), f2u(bf16r(v[4 * h + 1])), f2u(bf16r(v[4 * h + 2])),
                                         f2u(bf16r(v[4 * h + 3]))});
  } else {
    lm_u32x4 w;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = DT == BF16 ? pack_bf16x2(v[2 * k], v[2 * k + 1]) : dq_f16_bits(v[2 * k]) | (dq_f16_bits(v[2 * k + 1]) << 16);
    store_b128_guarded((LM_GLOBAL lm_u32x4*)((LM_GLOBAL uint16_t*)out + e0), w);
  }
}

// one element, any shape and alignment
template <int F, int DT>
DEV void dq_one(const DqArgs& a, int64_t e) {
  constexpr int CD = dq_cd<DT>();
  float v;
  if constexpr (DqTraits<F>::BLOCK) {
    const int64_t row = e / a.N, col = e - row * a.N;
    const uint32_t sc = ((const uint8_t*)a.scale)[blocked_offset(row, col / DqTraits<F>::BS, a.N / DqTraits<F>::BS, a.swizzled)];
    const bool two = F == B_NVFP4 && a.aux != nullptr;
    const float s = dq_block_scale<F, CD>(sc, two, two ? *(const float*)a.aux : 1.0f);
    if constexpr (DqTraits<F>::FP4) v = e2m1_value((a.q[e >> 1] >> (4 * (int)(e & 1))) & 15u) * s;
    else v = fp8_value<DqTraits<F>::FMT>(a.q[e]) * s;
  } else {
    const int64_t qi = e / a.group;
    const float s = load_scalar(a.scale, qi, a.scale_dt);
    if constexpr (F == B_INT8) v = ((float)(int8_t)a.q[e] - (a.aux ? (float)((const int8_t*)a.aux)[qi] : 0.0f)) * s;
    else v = fp8_value<DqTraits<F>::FMT>(a.q[e]) * s;
  }
  if constexpr (DT == F32) ((float*)a.out)[e] = bf16r(v);
  else if constexpr (DT == BF16) ((uint16_t*)a.out)[e] = bf16_bits(v);
  else ((uint16_t*)a.out)[e] = (uint16_t)dq_f16_bits(v);
}

// M N < 2^32 and at most 2^32 swizzled scales (32-bit chunk, element and scale
// indices), 8-byte aligned codes (4 for fp4) and 16-byte aligned output (one
// load and one store per chunk), qparam groups of at least 8 elements (a chunk
// meets at most two)
template <int F, int DT>
__global__ __launch_bounds__(DQ_THREADS) void k_dequant(DqArgs a) {
  constexpr int CD = dq_cd<DT>();
  const uint32_t n = (uint32_t)(a.M * a.N), nch = n >> 3;
  const uint32_t c0 = blockIdx.x * (DQ_THREADS * DQ_U) + threadIdx.x;
  float g = 1.0f;
  const bool two = F == B_NVFP4 && a.aux != nullptr;
  if (two) g = *(const LM_GLOBAL float*)a.aux;
  uint32_t w[DQ_U][2];
  uint32_t sc[DQ_U];             // block formats: the scale byte
  float s0[DQ_U], s1[DQ_U];      // INT8 / FP8: the chunk's scale and, past `rem` elements, the next one
  float z0[DQ_U], z1[DQ_U];
  uint32_t rem[DQ_U];
#pragma unroll
  for (int u = 0; u < DQ_U; ++u) {
    const uint32_t c = c0 + u * DQ_THREADS;
    if (c >= nch) continue;
    if constexpr (DqTraits<F>::FP4) {
      w[u][0] = ((const LM_GLOBAL uint32_t*)a.q)[c];
      w[u][1] = 0u;
    } else {
      const lm_u32x2 x = ((const LM_GLOBAL lm_u32x2*)a.q)[c];
      w[u][0] = x.x;
      w[u][1] = x.y;
    }
    if constexpr (DqTraits<F>::BLOCK) {
      constexpr int CB = DqTraits<F>::BS / 8;  // chunks per block; plain scales are flat too
      uint32_t so = c / CB;
      if (a.swizzled) {
        const uint32_t row = div_by(a.div, c), scol = (c - row * a.div.d) / CB, ncb = (uint32_t)((a.N / DqTraits<F>::BS + 3) >> 2);
        so = ((row >> 7) * ncb + (scol >> 2)) * 512u + (row & 31u) * 16u + ((row >> 5) & 3u) * 4u + (scol & 3u);
      }
      sc[u] = ((const LM_GLOBAL uint8_t*)a.scale)[so];
    } else {
      const uint32_t e0 = 8u * c, qi = div_by(a.div, e0);
      rem[u] = qi * a.div.d + (a.div.d - e0);  // elements left in this qparam's group
      // (a chunk can cross into the next group only in rows of odd length)
      const uint32_t qn = rem[u] < 8u ? qi + 1 : qi;
      s0[u] = load_scalar(a.scale, qi, a.scale_dt);
      s1[u] = qn != qi ? load_scalar(a.scale, qn, a.scale_dt) : s0[u];
      z0[u] = z1[u] = 0.0f;
      if (F == B_INT8 && a.aux) {
        z0[u] = (float)((const LM_GLOBAL int8_t*)a.aux)[qi];
        z1[u] = qn != qi ? (float)((const LM_GLOBAL int8_t*)a.aux)[qn] : z0[u];
      }
    }
  }
#pragma unroll
  for (int u = 0; u < DQ_U; ++u) {
    const uint32_t c = c0 + u * DQ_THREADS;
    if (c >= nch) continue;
    float s[8], z[8], v[8];
    if constexpr (DqTraits<F>::BLOCK) {
      const float bs = dq_block_scale<F, CD>(sc[u], two, g);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        s[j] = bs;
        z[j] = 0.0f;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        s[j] = (uint32_t)j < rem[u] ? s0[u] : s1[u];
        z[j] = (uint32_t)j < rem[u] ? z0[u] : z1[u];
      }
    }
    dq_values8<F>(w[u], s, z, v);
    dq_store8<DT>(a.out, (int64_t)8 * c, v);
  }
  // the last n % 8 elements
  if (blockIdx.x == 0 && threadIdx.x < (n & 7u)) dq_one<F, DT>(a, (int64_t)(n & ~7u) + threadIdx.x);
}

// everything else: an element per thread
template <int F, int DT>
__global__ __launch_bounds__(DQ_THREADS) void k_dequant_any(DqArgs a) {
  const int64_t n = a.M * a.N, step = (int64_t)gridDim.x * DQ_THREADS;
  for (int64_t e = (int64_t)blockIdx.x * DQ_THREADS + threadIdx.x; e < n; e += step) dq_one<F, DT>(a, e);
}

template <int F, int DT>
static int launch_dequant(DqArgs a, hipStream_t st) {
  const int64_t n = a.M * a.N;
  const uintptr_t qmask = DqTraits<F>::FP4 ? 3 : 7;
  TimedLaunch timed("todense", st);
  // the swizzled layout pads rows to 128: a few very long rows have far more scale bytes than n / BS
  const int64_t scales = a.swizzled ? (a.M + 127) / 128 * ((a.N / DqTraits<F>::BS + 3) / 4) * 512 : 0;
  if (n < (INT64_C(1) << 32) - 8 && scales <= (INT64_C(1) << 32) && ((uintptr_t)a.q & qmask) == 0 &&
      ((uintptr_t)a.out & 15) == 0 && (DqTraits<F>::BLOCK || a.group >= 8)) {
    a.div = fast_div((uint32_t)(DqTraits<F>::BLOCK ? a.N / 8 : a.group));
    const int64_t nb = (n / 8 + DQ_THREADS * DQ_U - 1) / (DQ_THREADS * DQ_U);
    hipLaunchKernelGGL((k_dequant<F, DT>), dim3((unsigned)(nb > 0 ? nb : 1)), dim3(DQ_THREADS), 0, st, a);
  } else {
    const int64_t nb = (n + DQ_THREADS - 1) / DQ_THREADS;
    hipLaunchKernelGGL((k_dequant_any<F, DT>), dim3((unsigned)(nb < 65536 ? nb : 65536)), dim3(DQ_THREADS), 0, st, a);
  }
  LAUNCH_CHECK();
  return LM_OK;
}
// argument checks of a decode (the workspace is not used, but the entry points ask for one)
static inline int check_dequant(int64_t M, int64_t N, int out_dt, const void* ws, size_t wsb) {
  if (out_dt != LM_BF16 && out_dt != LM_F16 && out_dt != LM_F32)
    return fail(LM_EINVAL, "dequant output dtype must be bf16, f16 or f32");
  return check_workspace(ws_layout(M, N, 0), ws, wsb);
}
template <int F>
static int run_dequant(const DqArgs& a, int out_dt, hipStream_t st) {
  if (out_dt == LM_BF16) return launch_dequant<F, BF16>(a, st);
  if (out_dt == LM_F16) return launch_dequant<F, F16>(a, st);
  return launch_dequant<F, F32>(a, st);
}
