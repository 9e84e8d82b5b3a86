// Quantization grids: E8M0 scale choice, E2M1 / E4M3 encoders, MXFP RTN and
// dequant, affine MSE clip search with storage-rounded params, affine RTN.
// Element-parallel, HBM-bound kernels; the hot solver kernels reuse the same
// device encoders from mgq_common.h.
#include <string.h>

#include "affine_clip.h"
#include "mgq_capi.h"
#include "mgq_common.h"
#include "mx_hw.h"

namespace mgq {
namespace {

constexpr int kThreads = 256;

// NaN-propagating max / min (torch amax / amin semantics).
__device__ inline float nan_max(float m, float a) { return (a > m || a != a) ? a : m; }
__device__ inline float nan_min(float m, float a) { return (a < m || a != a) ? a : m; }

__device__ inline float affine_q(float w, float b, float s_safe, float maxq) {
  float q = rintf((w - b) / s_safe);
  if (q != q) return q;
  return fminf(fmaxf(q, 0.0f), maxq);
}

// ---------------------------------------------------------------------------
__global__ void choose_mxfp_scale_kernel(const float* __restrict__ w, int64_t n_groups,
                                         int64_t len, float fmax, uint8_t* __restrict__ bytes,
                                         float* __restrict__ scales) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n_groups;
       g += (int64_t)gridDim.x * blockDim.x) {
    const float* p = w + g * len;
    float m = fabsf(p[0]);
    for (int64_t i = 1; i < len; ++i) m = nan_max(m, fabsf(p[i]));
    const int e = e8m0_exponent(m, fmax);
    bytes[g] = static_cast<uint8_t>(e + 127);
    scales[g] = exp2_int(e);
  }
}

__global__ void quantize_mxfp_kernel(const float* __restrict__ w, const float* __restrict__ scales,
                                     int64_t n, int64_t len, int mode, uint8_t* __restrict__ q,
                                     float* __restrict__ dq) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    float d;
    q[i] = static_cast<uint8_t>(mx_quant(w[i], scales[i / len], mode, &d));
    dq[i] = d;
  }
}

__device__ inline float scale_from_byte(uint32_t b) {
  // torch.pow(2, byte - 127) in fp32: 2^128 overflows to inf.
  const int e = static_cast<int>(b) - 127;
  return e > 127 ? __uint_as_float(0x7f800000u) : exp2_int(e);
}

__global__ void dequantize_mxfp_kernel(const uint8_t* __restrict__ q,
                                       const uint8_t* __restrict__ bytes, int64_t n, int mode,
                                       float* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float s = scale_from_byte(bytes[i / kMxGroup]);
    const uint32_t c = q[i];
    const float v = (mode == kMxfp4) ? e2m1_value(c & 15u) : e4m3_value(c);
    out[i] = v * s;
  }
}

// Dequantization of whole 4-code pieces: a wave reads 256 bytes of codes and
// writes 1 KB of values per step, kDqAhead steps in flight per thread. The
// group of piece t is t >> shift (group lengths of 4, 8, 16, .. codes).
// [14336 x 4096], 4 bytes written per byte read: affine (G = 64) 164 us with a
// code and a 64-bit division per thread, now 63 us (75 us with the storage type
// branched on at run time, which keeps the loads of the steps apart); MXFP4 139
// us, MXFP8 135 us, now 57 us (5.2 TB/s).
constexpr int kDqAhead = 4;

template <int MODE, int STORAGE>
__global__ void __launch_bounds__(kThreads)
    dequantize_vec_kernel(const uint32_t* __restrict__ q, const void* __restrict__ scales,
                          const void* __restrict__ biases, int64_t n4, int shift,
                          float4* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t t0 = blockIdx.x * (int64_t)kThreads + threadIdx.x; t0 < n4;
       t0 += stride * kDqAhead) {
    uint32_t c[kDqAhead];
    float s[kDqAhead], b[kDqAhead];
#pragma unroll
    for (int u = 0; u < kDqAhead; ++u) {
      const int64_t t = t0 + u * stride;
      if (t >= n4) continue;
      c[u] = q[t];
      if constexpr (MODE == kAffine) {
        s[u] = load_storage(scales, t >> shift, STORAGE);
        b[u] = load_storage(biases, t >> shift, STORAGE);
      } else {
        s[u] = scale_from_byte(static_cast<const uint8_t*>(scales)[t >> shift]);
      }
    }
#pragma unroll
    for (int u = 0; u < kDqAhead; ++u) {
      const int64_t t = t0 + u * stride;
      if (t >= n4) continue;
      float v[4];
      if constexpr (MODE == kAffine) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = static_cast<float>((c[u] >> (8 * k)) & 0xffu) * s[u] + b[u];
      } else if constexpr (MODE == kMxfp4) {
        // one code per byte: the low nibble's value of each
        v[0] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[u], 1.0f, 0)[0] * s[u];
        v[1] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[u], 1.0f, 1)[0] * s[u];
        v[2] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[u], 1.0f, 2)[0] * s[u];
        v[3] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[u], 1.0f, 3)[0] * s[u];
      } else {
        const auto lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(c[u], 1.0f, false);
        const auto hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(c[u], 1.0f, true);
        v[0] = lo[0] * s[u], v[1] = lo[1] * s[u], v[2] = hi[0] * s[u], v[3] = hi[1] * s[u];
      }
      out[t] = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

// shift for dequantize_vec_kernel, or -1 where it does not apply
int dequant_shift(const uint8_t* q, const float* out, int64_t group_len) {
  if ((reinterpret_cast<uintptr_t>(q) & 3u) || (reinterpret_cast<uintptr_t>(out) & 15u)) return -1;
  if (group_len < 4 || (group_len & (group_len - 1))) return -1;
  int shift = 0;
  while ((int64_t{4} << shift) < group_len) ++shift;
  return shift;
}

// A workgroup takes kDqAhead steps of the grid, fewer while that leaves a CU with
// less than four workgroups (128 x 256: 2.5 us by kDqAhead steps, 2.1 us so).
constexpr int64_t kDqBlocks = 1024;
unsigned dequant_blocks(int64_t n4) {
  const int64_t one_step = ceil_div(n4, kThreads);
  if (one_step <= kDqBlocks) return static_cast<unsigned>(one_step);
  const unsigned blocks = elementwise_blocks(ceil_div(n4, kDqAhead), kThreads);
  return blocks < kDqBlocks ? static_cast<unsigned>(kDqBlocks) : blocks;
}

// One thread per 32-value group: scale choice + projection (grid.py:142-151).
__global__ void rtn_mxfp_kernel(const void* __restrict__ W, int dtype, int64_t n_groups,
                                int mode, uint8_t* __restrict__ q, uint8_t* __restrict__ bytes,
                                float* __restrict__ dq) {
  const float fmax = (mode == kMxfp4) ? 6.0f : 448.0f;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n_groups;
       g += (int64_t)gridDim.x * blockDim.x) {
    float v[kMxGroup];
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < kMxGroup; ++i) {
      v[i] = load_any(W, g * kMxGroup + i, dtype);
      m = (i == 0) ? fabsf(v[i]) : nan_max(m, fabsf(v[i]));
    }
    const int e = e8m0_exponent(m, fmax);
    const float s = exp2_int(e);
    bytes[g] = static_cast<uint8_t>(e + 127);
#pragma unroll
    for (int i = 0; i < kMxGroup; ++i) {
      float d;
      q[g * kMxGroup + i] = static_cast<uint8_t>(mx_quant(v[i], s, mode, &d));
      dq[g * kMxGroup + i] = d;
    }
  }
}

// The same for 16-byte aligned W, q and dq: one thread per group with
// 16-byte loads and stores, and the hardware MX encoders (mx_hw.h, equal to
// mx_quant for every input: w / s == w * (1/s) for power-of-two s).
template <typename TIn, bool IS_F16>
__global__ void rtn_mxfp_vec_kernel(const TIn* __restrict__ W, int64_t n_groups, int mode,
                                    uint8_t* __restrict__ q, uint8_t* __restrict__ bytes,
                                    float* __restrict__ dq) {
  const float fmax = (mode == kMxfp4) ? 6.0f : 448.0f;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n_groups;
       g += (int64_t)gridDim.x * blockDim.x) {
    float v[kMxGroup];
    if constexpr (sizeof(TIn) == 4) {
      const float4* p = reinterpret_cast<const float4*>(W + g * kMxGroup);
#pragma unroll
      for (int i = 0; i < kMxGroup / 4; ++i) {
        const float4 x = p[i];
        v[4 * i] = x.x, v[4 * i + 1] = x.y, v[4 * i + 2] = x.z, v[4 * i + 3] = x.w;
      }
    } else {
      const uint4* p = reinterpret_cast<const uint4*>(W + g * kMxGroup);
#pragma unroll
      for (int i = 0; i < kMxGroup / 8; ++i) {
        const uint4 x = p[i];
        const uint32_t d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint16_t lo = static_cast<uint16_t>(d[k] & 0xffffu), hi = static_cast<uint16_t>(d[k] >> 16);
          v[8 * i + 2 * k] = IS_F16 ? f16_to_f32(lo) : bf16_to_f32(lo);
          v[8 * i + 2 * k + 1] = IS_F16 ? f16_to_f32(hi) : bf16_to_f32(hi);
        }
      }
    }
    float m = fabsf(v[0]);
#pragma unroll
    for (int i = 1; i < kMxGroup; ++i) m = nan_max(m, fabsf(v[i]));
    const int e = e8m0_exponent(m, fmax);
    const float s = exp2_int(e), inv = exp2_int(-e);
    bytes[g] = static_cast<uint8_t>(e + 127);
    uint32_t codes[kMxGroup / 4];
    float d[kMxGroup];
#pragma unroll
    for (int i = 0; i < kMxGroup / 4; ++i) codes[i] = 0u;
#pragma unroll
    for (int i = 0; i < kMxGroup; ++i) {
      const uint32_t c = (mode == kMxfp4) ? mx4_encode_hw(v[i], inv, s, &d[i])
                                          : mx8_encode_hw(v[i], inv, s, &d[i]);
      codes[i / 4] |= c << (8 * (i % 4));
    }
    uint4* qp = reinterpret_cast<uint4*>(q + g * kMxGroup);
    qp[0] = make_uint4(codes[0], codes[1], codes[2], codes[3]);
    qp[1] = make_uint4(codes[4], codes[5], codes[6], codes[7]);
    float4* op = reinterpret_cast<float4*>(dq + g * kMxGroup);
#pragma unroll
    for (int i = 0; i < kMxGroup / 4; ++i) op[i] = make_float4(d[4 * i], d[4 * i + 1], d[4 * i + 2], d[4 * i + 3]);
  }
}

__global__ void dequantize_affine_kernel(const uint8_t* __restrict__ q, const void* scales,
                                         const void* biases, int storage, int64_t n, int64_t len,
                                         float* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = i / len;
    out[i] = static_cast<float>(q[i]) * load_storage(scales, g, storage) +
             load_storage(biases, g, storage);
  }
}

// One value as fp32: TIn float, or the bit pattern of a bf16 or f16.
template <typename TIn, bool IS_F16>
__device__ inline float widen(TIn x) {
  if constexpr (sizeof(TIn) == 4) return x;
  else return IS_F16 ? f16_to_f32(x) : bf16_to_f32(x);
}

// grid.py:167-212 for one group. Returns the chosen (s, b) in fp32 (already
// rounded to the storage dtype).
template <typename TIn, bool IS_F16>
__device__ inline void choose_qparams_group(const TIn* __restrict__ w, int64_t len, float maxq,
                                            int storage, const float2* tab, int n, float* s_out,
                                            float* b_out) {
  auto p = [&](int64_t i) { return widen<TIn, IS_F16>(w[i]); };
  maxq = __builtin_canonicalizef(maxq);  // once, or every clamp does it again
  float wmin = p(0), wmax = wmin;
  for (int64_t i = 1; i < len; ++i) {
    wmin = nan_min(wmin, p(i));
    wmax = nan_max(wmax, p(i));
  }
  const float range = wmax - wmin;
  float best_err = 0.0f, best_s = 0.0f, best_b = 0.0f;
  for (int c = 0; c < n; ++c) {
    const float s = round_to_storage(range * tab[c].x, storage);
    const float b = round_to_storage(wmin * tab[c].y, storage);
    const float s_safe = (fabsf(s) < 1e-12f) ? 1.0f : s;
    float err = 0.0f;
#pragma unroll 4  // four loads in flight
    for (int64_t i = 0; i < len; ++i) {
      const float x = p(i);
      const float q = affine_q(x, b, s_safe, maxq);
      const float d = q * s + b - x;
      err += d * d;
    }
    if (c == 0 || err < best_err) {
      best_err = err;
      best_s = s;
      best_b = b;
    }
  }
  *s_out = best_s;
  *b_out = best_b;
}

__global__ void choose_qparams_kernel(const float* __restrict__ w, int64_t n_groups, int64_t len,
                                      float maxq, int storage, Shrinks sh, void* s_store,
                                      void* b_store, float* __restrict__ s32,
                                      float* __restrict__ b32) {
  __shared__ float2 tab[kMaxShrinks];
  stage_shrinks(sh, tab);
  __syncthreads();
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n_groups;
       g += (int64_t)gridDim.x * blockDim.x) {
    float s, b;
    choose_qparams_group<float, false>(w + g * len, len, maxq, storage, tab, sh.n, &s, &b);
    store_storage(s_store, g, s, storage);
    store_storage(b_store, g, b, storage);
    s32[g] = s;
    b32[g] = b;
  }
}

__global__ void quantize_with_params_kernel(const float* __restrict__ w,
                                            const float* __restrict__ s32,
                                            const float* __restrict__ b32, int64_t n, int64_t len,
                                            float maxq, float* __restrict__ q,
                                            float* __restrict__ dq) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = i / len;
    const float s = s32[g], b = b32[g];
    const float s_safe = (fabsf(s) < 1e-12f) ? 1.0f : s;
    const float qq = affine_q(w[i], b, s_safe, maxq);
    q[i] = qq;
    dq[i] = qq * s + b;
  }
}

// choose_qparams (RTN = false: scales and biases, also in fp32) and
// rtn_quantize (RTN = true: scales, biases, codes and dequantized values) of
// groups of G = LN * NS values, LN lanes per group, each lane holding the
// 4-value pieces l, l + LN, ... (16-byte loads of f32, 8-byte of bf16 / f16,
// so W is read once and as it is). [4 x 1536 x 2048] bf16 at G = 64, 21
// candidates: 82 us for rtn_quantize + pack_q, against 1494 us with one
// thread per group reading its values again from memory for every candidate
// and a float copy of W. Bound by the search's instruction issue
// (affine_clip.h).
template <typename TIn, bool IS_F16, int LN, int NS, bool RTN>
__global__ void __launch_bounds__(kThreads)
    affine_groups_kernel(const TIn* __restrict__ W, int64_t n_groups, float maxq, int storage,
                         Shrinks sh, uint8_t* __restrict__ q, void* s_store, void* b_store,
                         float* __restrict__ dq, float* __restrict__ s32,
                         float* __restrict__ b32) {
  constexpr int G = LN * NS;
  __shared__ float2 tab[kMaxShrinks];
  stage_shrinks(sh, tab);
  __syncthreads();
  const int l = threadIdx.x & (LN - 1);
  const int64_t per = kThreads / LN;
  const bool on[NS] = {};
  // a whole workgroup takes every step (the search's lane operations need
  // its lanes on); the groups past the last one repeat it
  for (int64_t g0 = blockIdx.x * per; g0 < n_groups; g0 += gridDim.x * per) {
    const int64_t gw = g0 + threadIdx.x / LN;
    const bool live = gw < n_groups;
    const int64_t base = (live ? gw : n_groups - 1) * G + 4 * l;
    float w[NS];
#pragma unroll
    for (int t = 0; t < NS / 4; ++t) {
      if constexpr (sizeof(TIn) == 4) {
        const float4 x = *reinterpret_cast<const float4*>(W + base + 4 * LN * t);
        w[4 * t] = x.x, w[4 * t + 1] = x.y, w[4 * t + 2] = x.z, w[4 * t + 3] = x.w;
      } else {
        const uint2 x = *reinterpret_cast<const uint2*>(W + base + 4 * LN * t);
        const uint16_t h[4] = {static_cast<uint16_t>(x.x & 0xffffu), static_cast<uint16_t>(x.x >> 16),
                               static_cast<uint16_t>(x.y & 0xffffu), static_cast<uint16_t>(x.y >> 16)};
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * t + e] = IS_F16 ? f16_to_f32(h[e]) : bf16_to_f32(h[e]);
      }
    }
    float s, b;
    clip_search<LN, NS, true>(w, on, tab, sh.n, maxq, storage, s, b);
    if (live && l == 0) {
      store_storage(s_store, gw, s, storage);
      store_storage(b_store, gw, b, storage);
      if constexpr (!RTN) {
        s32[gw] = s;
        b32[gw] = b;
      }
    }
    if constexpr (RTN) {
      const float ss = safe_scale(s), ys = div_exact_recip(ss);
#pragma unroll
      for (int t = 0; t < NS / 4; ++t) {
        uint32_t code = 0;
        float d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float qq = affine_q_exact(w[4 * t + e], b, ss, ys, maxq);
          code |= (qq == qq ? static_cast<uint32_t>(qq) : 0u) << (8 * e);
          d[e] = qq * s + b;
        }
        if (live) {
          *reinterpret_cast<uint32_t*>(q + base + 4 * LN * t) = code;
          *reinterpret_cast<float4*>(dq + base + 4 * LN * t) = make_float4(d[0], d[1], d[2], d[3]);
        }
      }
    }
  }
}

// rtn_quantize (grid.py:224-246) of any group length: one thread per group,
// bound by the latency of its loads and of the chain of error sums. [1536 x
// 1920] bf16, G = 240, 21 candidates: 1029 us for an fp32 copy and a load per
// value, 1555 with the type looked at for every value, now 528.
template <typename TIn, bool IS_F16>
__global__ void rtn_affine_kernel(const TIn* __restrict__ W, int64_t n_groups, int len, float maxq,
                                  int storage, Shrinks sh, uint8_t* __restrict__ q, void* s_store,
                                  void* b_store, float* __restrict__ dq) {
  __shared__ float2 tab[kMaxShrinks];
  stage_shrinks(sh, tab);
  __syncthreads();
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n_groups;
       g += (int64_t)gridDim.x * blockDim.x) {
    const TIn* p = W + g * len;
    float s, b;
    choose_qparams_group<TIn, IS_F16>(p, len, maxq, storage, tab, sh.n, &s, &b);
    store_storage(s_store, g, s, storage);
    store_storage(b_store, g, b, storage);
    const float s_safe = (fabsf(s) < 1e-12f) ? 1.0f : s;
    for (int i = 0; i < len; ++i) {
      const float qq = affine_q(widen<TIn, IS_F16>(p[i]), b, s_safe, maxq);
      q[g * len + i] = (qq == qq) ? static_cast<uint8_t>(qq) : 0;
      dq[g * len + i] = qq * s + b;
    }
  }
}

// Whether affine_groups_kernel takes these groups: the MLX group sizes, W
// (and dq) aligned to its 4-value pieces, codes to four bytes.
bool whole_groups(int64_t group_len, const void* W, int w_dtype, const void* q, const void* dq) {
  const uintptr_t w_mask = w_dtype == kF32 ? 15u : 7u;
  return (group_len == 32 || group_len == 64 || group_len == 128) &&
         (reinterpret_cast<uintptr_t>(W) & w_mask) == 0 &&
         (reinterpret_cast<uintptr_t>(q) & 3u) == 0 && (reinterpret_cast<uintptr_t>(dq) & 15u) == 0;
}

// Groups of 32 and 64 take a quad each (the fewest lanes, so the most groups
// per instruction); a quad's 32 values per lane at 128 would need twice the
// registers, so those take a DPP row.
template <bool RTN>
int launch_groups(const void* W, int w_dtype, int64_t n_groups, int64_t group_len, float maxq,
                  int storage, const Shrinks& sh, uint8_t* q, void* s_store, void* b_store,
                  float* dq, float* s32, float* b32, hipStream_t st, const char* what) {
  const int64_t lanes = n_groups * (group_len == 128 ? 16 : 4);
  const unsigned blocks = elementwise_blocks(lanes, kThreads);
#define MGQ_GROUPS(T, F16, LN, NS)                                                             \
  affine_groups_kernel<T, F16, LN, NS, RTN><<<blocks, kThreads, 0, st>>>(                      \
      static_cast<const T*>(W), n_groups, maxq, storage, sh, q, s_store, b_store, dq, s32, b32)
#define MGQ_GROUPS_LEN(T, F16)                                    \
  do {                                                            \
    if (group_len == 32) MGQ_GROUPS(T, F16, 4, 8);                \
    else if (group_len == 64) MGQ_GROUPS(T, F16, 4, 16);          \
    else MGQ_GROUPS(T, F16, 16, 8);                               \
  } while (0)
  if constexpr (RTN) {
    if (w_dtype == kBF16) {
      MGQ_GROUPS_LEN(uint16_t, false);
      return check_launch(what);
    }
    if (w_dtype == kF16) {
      MGQ_GROUPS_LEN(uint16_t, true);
      return check_launch(what);
    }
  }
  MGQ_GROUPS_LEN(float, false);
#undef MGQ_GROUPS_LEN
#undef MGQ_GROUPS
  return check_launch(what);
}

int check_mx_mode(int mode) {
  MGQ_REQUIRE(mode == kMxfp4 || mode == kMxfp8, MGQ_ERR_VALUE,
              "not a microscaling mode: %d", mode);
  return MGQ_OK;
}

int check_dtype(int dtype, const char* what) {
  MGQ_REQUIRE(dtype == kF32 || dtype == kBF16 || dtype == kF16, MGQ_ERR_VALUE,
              "%s: unsupported dtype code %d", what, dtype);
  return MGQ_OK;
}

int check_bits(int bits) {
  MGQ_REQUIRE(bits >= 1 && bits <= 8, MGQ_ERR_VALUE, "unsupported bits: %d", bits);
  return MGQ_OK;
}


// Range audit of one stored artifact against its source weights
// (validate_artifacts.py:15-68), fused into one pass: every element is
// dequantized in-register (dequantize_artifact, grid.py:154-164), and per
// 32-column group g the kernel forms smax = max|source|, amax = max|deq|,
// limit = max(fp64(smax) * 32, 2^-126) and ratio = fp64(amax) / limit.
// Results go to `stats` (zeroed by the caller) with one atomic per block:
//   u64[0] non-finite dequantized values, u64[1] groups with amax > limit,
//   u64[2] max ratio (bits of a non-negative fp64; NaN ratios skipped),
//   u64[3] max |source| (bits of a non-negative fp32), u64[4] max |deq|.
// The grid is capped (grid-stride loop): every workgroup's atomics go to one
// cache line and are done one by one there, about 10 ns each, all at the end of
// the pass. 2048 workgroups of 256 threads: 110 us for [14336 x 4096] bf16,
// 1024: 79 us, 512: 52 us; one of 1024 threads per CU: 36 us. (A read of the
// field first, to skip a maximum that is not above it: 157 us.) Inputs that give a
// CU no more than 256 threads take workgroups of 256, whose last reduction is
// shorter (33 x 256: 4.1 us, 3.4 us so). The element-wise kernel has one load of
// each kind in flight per thread and takes two workgroups of 1024 per CU: the
// large matrix at G = 4 260 us with 2048 workgroups of 256, 388 with one of 1024
// per CU, 218 with two.
constexpr int kAuditBlocks = 256, kAuditThreads = 1024, kAuditSmall = 256;

__device__ inline float nanless_max(float a, float b) { return b > a ? b : a; }

struct AuditAcc {
  unsigned long long nonfinite = 0, exceed = 0;
  // the group with the largest ratio so far, as its two parts: two ratios are
  // compared by cross products, which are exact in fp64 (24-bit factors), so
  // only one division is done, of the largest
  double rnum = 0.0, rden = 1.0;
  float smax = 0.0f, amax = 0.0f;
  // one group's maxima, held by its leading lane
  __device__ void group(float gs, float ga) {
    const double limit = fmax(static_cast<double>(gs) * 32.0, 0x1p-126);
    const double a = static_cast<double>(ga);
    if (a > limit) ++exceed;
    // false for a NaN ratio (inf / inf) and for x / inf, as 0 > 0 would be
    const bool more = a * rden > rnum * limit;
    rnum = more ? a : rnum;
    rden = more ? limit : rden;
    smax = nanless_max(smax, gs);
    amax = nanless_max(amax, ga);
  }
  // wave, then workgroup reduction; one atomic per block and field
  template <int THREADS>
  __device__ void flush(unsigned long long* stats) {
    double rmax = rnum / rden;
    __shared__ unsigned long long s_cnt[2][THREADS / 64];
    __shared__ double s_r[THREADS / 64];
    __shared__ float s_m[2][THREADS / 64];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      nonfinite += __shfl_xor(nonfinite, o);
      exceed += __shfl_xor(exceed, o);
      rmax = fmax(rmax, __shfl_xor(rmax, o));
      smax = nanless_max(smax, __shfl_xor(smax, o));
      amax = nanless_max(amax, __shfl_xor(amax, o));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      s_cnt[0][w] = nonfinite, s_cnt[1][w] = exceed, s_r[w] = rmax;
      s_m[0][w] = smax, s_m[1][w] = amax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int k = 1; k < THREADS / 64; ++k) {
        s_cnt[0][0] += s_cnt[0][k], s_cnt[1][0] += s_cnt[1][k];
        s_r[0] = fmax(s_r[0], s_r[k]);
        s_m[0][0] = nanless_max(s_m[0][0], s_m[0][k]);
        s_m[1][0] = nanless_max(s_m[1][0], s_m[1][k]);
      }
      if (s_cnt[0][0]) atomicAdd(&stats[0], s_cnt[0][0]);
      if (s_cnt[1][0]) atomicAdd(&stats[1], s_cnt[1][0]);
      atomicMax(&stats[2], static_cast<unsigned long long>(__double_as_longlong(s_r[0])));
      atomicMax(&stats[3], static_cast<unsigned long long>(__float_as_uint(s_m[0][0])));
      atomicMax(&stats[4], static_cast<unsigned long long>(__float_as_uint(s_m[1][0])));
    }
  }
};

__device__ inline float audit_deq(uint32_t c, float sc, float bias, int mode) {
  if (mode == kAffine) return static_cast<float>(c) * sc + bias;
  return ((mode == kMxfp4) ? e2m1_value(c & 15u) : e4m3_value(c)) * sc;
}

// One element per lane (any alignment, any affine group size); the 32 lanes
// of a half-wave hold one group together (n and the stride are multiples
// of 32).
template <int THREADS>
__global__ void __launch_bounds__(THREADS)
    range_audit_kernel(const void* __restrict__ src, int src_dtype, const uint8_t* __restrict__ q,
                       const void* __restrict__ scales, const void* __restrict__ biases,
                       int storage, int mode, int64_t group_size, int64_t n,
                       unsigned long long* __restrict__ stats) {
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  AuditAcc acc;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i - (lane & 31) < n;
       i += stride) {
    const float sv = fabsf(load_any(src, i, src_dtype));
    float sc, bias = 0.0f;
    if (mode == kAffine) {
      const int64_t g = i / group_size;
      sc = load_storage(scales, g, storage);
      bias = load_storage(biases, g, storage);
    } else {
      sc = scale_from_byte(static_cast<const uint8_t*>(scales)[i / kMxGroup]);
    }
    const float v = audit_deq(q[i], sc, bias, mode);
    if (!isfinite(v)) ++acc.nonfinite;
    float gs = sv, ga = fabsf(v);
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
      gs = nanless_max(gs, __shfl_xor(gs, o));
      ga = nanless_max(ga, __shfl_xor(ga, o));
    }
    if ((lane & 31) == 0) acc.group(gs, ga);
  }
  acc.flush<THREADS>(stats);
}

// Eight elements per lane from 16-byte-aligned rows: 16 (bf16 / f16) or 32
// (f32) bytes of source and 8 code bytes per load; four lanes hold one
// 32-column group (n8 = n / 8 and the stride are multiples of 4). The
// affine group size is a multiple of 8, so a lane's eight values share one
// scale. Each lane issues the loads of kAuditUnroll grid-stride units before it
// evaluates any of them. The MX modes need no per-element dequantization: the
// values of a group share one positive power-of-two scale, so max|deq| is the
// value of the largest magnitude code (byte maxima, two codes per packed
// 16-bit maximum) times it; a lane where that is no finite number (a NaN code,
// an overflow, an infinite scale) goes value by value. max|source| is taken on the bit
// patterns with the sign cleared (monotonic in |x|; NaN patterns count as 0, as
// the float path's compare skips NaN). [14336 x 4096] bf16 source, MXFP8: 126
// us with a software decode per value and an fp64 division per group, 110 us
// without them, 36 us (5 TB/s) with the fewer workgroups of kAuditBlocks.
constexpr int kAuditUnroll = 2;
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

template <int SD>
__device__ inline float src_absmax(const uint4& a, const uint4& b) {
  if constexpr (SD == kF32) {
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t v = w[k] & 0x7fffffffu;
      m = max(m, v > 0x7f800000u ? 0u : v);
    }
    return __uint_as_float(m);
  } else {
    constexpr uint32_t kInf = (SD == kBF16) ? 0x7f80u : 0x7c00u;
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
    u16x2_t m = {0, 0};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, w[k] & 0x7fff7fffu));
    uint32_t x = max(static_cast<uint32_t>(m[0]), static_cast<uint32_t>(m[1]));
    if (x > kInf) {  // some value is a NaN: without those
      x = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t lo = w[k] & 0x7fffu, hi = (w[k] >> 16) & 0x7fffu;
        x = max(x, max(lo > kInf ? 0u : lo, hi > kInf ? 0u : hi));
      }
    }
    return (SD == kBF16) ? __uint_as_float(x << 16) : f16_to_f32(static_cast<uint16_t>(x));
  }
}

// the largest byte of (c & MASK) over eight codes
template <uint32_t MASK>
__device__ inline uint32_t max_code(uint2 c) {
  constexpr uint32_t m = MASK | (MASK << 16);
  const u16x2_t a = __builtin_bit_cast(u16x2_t, c.x & m),
                b = __builtin_bit_cast(u16x2_t, (c.x >> 8) & m),
                d = __builtin_bit_cast(u16x2_t, c.y & m),
                e = __builtin_bit_cast(u16x2_t, (c.y >> 8) & m);
  const u16x2_t x = __builtin_elementwise_max(__builtin_elementwise_max(a, b),
                                              __builtin_elementwise_max(d, e));
  return max(static_cast<uint32_t>(x[0]), static_cast<uint32_t>(x[1]));
}

template <int SD, int MODE, int THREADS>
__global__ void __launch_bounds__(THREADS)
    range_audit_vec_kernel(const void* __restrict__ src, const uint8_t* __restrict__ q,
                           const void* __restrict__ scales, const void* __restrict__ biases,
                           int storage, int64_t group_size, int64_t n8,
                           unsigned long long* __restrict__ stats) {
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  AuditAcc acc;
  for (int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t0 - (lane & 3) < n8;
       t0 += stride * kAuditUnroll) {
    uint4 ra[kAuditUnroll], rb[kAuditUnroll];
    uint2 rc[kAuditUnroll];
    float sc[kAuditUnroll], bias[kAuditUnroll];
    bool on[kAuditUnroll];
#pragma unroll
    for (int u = 0; u < kAuditUnroll; ++u) {
      const int64_t t = t0 + u * stride;
      on[u] = t - (lane & 3) < n8;  // the same in the group's four lanes
      bias[u] = 0.0f;
      if (on[u]) {
        if constexpr (SD == kF32) {
          ra[u] = reinterpret_cast<const uint4*>(src)[2 * t];
          rb[u] = reinterpret_cast<const uint4*>(src)[2 * t + 1];
        } else {
          ra[u] = reinterpret_cast<const uint4*>(src)[t];
        }
        rc[u] = reinterpret_cast<const uint2*>(q)[t];
        if constexpr (MODE == kAffine) {
          const int64_t g = (8 * t) / group_size;
          sc[u] = load_storage(scales, g, storage);
          bias[u] = load_storage(biases, g, storage);
        } else {
          sc[u] = scale_from_byte(static_cast<const uint8_t*>(scales)[t >> 2]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kAuditUnroll; ++u) {
      if (!on[u]) continue;
      float gs = src_absmax<SD>(ra[u], rb[u]);
      float ga = __uint_as_float(0x7f800000u);
      if constexpr (MODE == kMxfp4) ga = e2m1_value(max_code<0x07u>(rc[u])) * sc[u];
      // the E4M3 magnitude grows with its seven bits; 0x7f is NaN
      if constexpr (MODE == kMxfp8)
        ga = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(max_code<0x7fu>(rc[u]), 1.0f, false)[0] * sc[u];
      if (!(ga < __uint_as_float(0x7f800000u))) {
        ga = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t c = ((k < 4 ? rc[u].x : rc[u].y) >> (8 * (k & 3))) & 0xffu;
          const float v = audit_deq(c, sc[u], bias[u], MODE);
          if (!isfinite(v)) ++acc.nonfinite;
          ga = nanless_max(ga, fabsf(v));
        }
      }
      // the group's four lanes
      gs = nanless_max(gs, dpp<kQuadXor2>(gs));
      ga = nanless_max(ga, dpp<kQuadXor2>(ga));
      gs = nanless_max(gs, dpp<kQuadXor1>(gs));
      ga = nanless_max(ga, dpp<kQuadXor1>(ga));
      if ((lane & 3) == 0) acc.group(gs, ga);
    }
  }
  acc.flush<THREADS>(stats);
}

template <int MODE, int THREADS>
void launch_audit_vec(int sd, unsigned blocks, hipStream_t st, const void* src, const uint8_t* q,
                      const void* scales, const void* biases, int storage, int64_t group_size,
                      int64_t n8, unsigned long long* stats) {
  auto kernel = sd == kF32    ? range_audit_vec_kernel<kF32, MODE, THREADS>
                : sd == kBF16 ? range_audit_vec_kernel<kBF16, MODE, THREADS>
                              : range_audit_vec_kernel<kF16, MODE, THREADS>;
  kernel<<<blocks, THREADS, 0, st>>>(src, q, scales, biases, storage, group_size, n8, stats);
}

// vec: the vector kernel's n / 8 units, else the element-wise kernel's n
template <int THREADS>
void launch_audit(bool vec, int64_t max_blocks, int64_t units, int sd, hipStream_t st,
                  const void* src, const uint8_t* q, const void* scales, const void* biases,
                  int storage, int mode, int64_t group_size, unsigned long long* stats) {
  const int64_t nb = ceil_div(units, THREADS);
  const unsigned blocks = static_cast<unsigned>(nb < max_blocks ? nb : max_blocks);
  if (!vec)
    range_audit_kernel<THREADS><<<blocks, THREADS, 0, st>>>(src, sd, q, scales, biases, storage,
                                                            mode, group_size, units, stats);
  else if (mode == kMxfp4)
    launch_audit_vec<kMxfp4, THREADS>(sd, blocks, st, src, q, scales, biases, storage, group_size,
                                      units, stats);
  else if (mode == kMxfp8)
    launch_audit_vec<kMxfp8, THREADS>(sd, blocks, st, src, q, scales, biases, storage, group_size,
                                      units, stats);
  else
    launch_audit_vec<kAffine, THREADS>(sd, blocks, st, src, q, scales, biases, storage, group_size,
                                       units, stats);
}

}  // namespace
}  // namespace mgq

using namespace mgq;

extern "C" int mgq_choose_mxfp_scale(const float* w, int64_t n_groups, int64_t group_len,
                                     int mode, uint8_t* scale_bytes, float* scales,
                                     void* stream) {
  clear_error();
  if (int rc = check_mx_mode(mode)) return rc;
  MGQ_REQUIRE(n_groups >= 0 && group_len >= 1, MGQ_ERR_SHAPE, "bad shape [%lld, %lld]",
              (long long)n_groups, (long long)group_len);
  if (n_groups == 0) return MGQ_OK;
  choose_mxfp_scale_kernel<<<elementwise_blocks(n_groups, kThreads), kThreads, 0,
                             as_stream(stream)>>>(w, n_groups, group_len,
                                                  mode == kMxfp4 ? 6.0f : 448.0f, scale_bytes,
                                                  scales);
  return check_launch("choose_mxfp_scale");
}

extern "C" int mgq_quantize_mxfp_with_scale(const float* w, const float* scales,
                                            int64_t n_groups, int64_t group_len, int mode,
                                            uint8_t* q, float* dq, void* stream) {
  clear_error();
  if (int rc = check_mx_mode(mode)) return rc;
  MGQ_REQUIRE(n_groups >= 0 && group_len >= 1, MGQ_ERR_SHAPE, "bad shape");
  const int64_t n = n_groups * group_len;
  if (n == 0) return MGQ_OK;
  quantize_mxfp_kernel<<<elementwise_blocks(n, kThreads), kThreads, 0, as_stream(stream)>>>(
      w, scales, n, group_len, mode, q, dq);
  return check_launch("quantize_mxfp_with_scale");
}

extern "C" int mgq_dequantize_mxfp(const uint8_t* q, const uint8_t* scale_bytes,
                                   int64_t n_groups, int mode, float* out, void* stream) {
  clear_error();
  if (int rc = check_mx_mode(mode)) return rc;
  MGQ_REQUIRE(n_groups >= 0, MGQ_ERR_SHAPE, "bad shape");
  const int64_t n = n_groups * kMxGroup;
  if (n == 0) return MGQ_OK;
  const int shift = dequant_shift(q, out, kMxGroup);
  if (shift >= 0) {
    const unsigned blocks = dequant_blocks(n / 4);
    const uint32_t* q4 = reinterpret_cast<const uint32_t*>(q);
    float4* out4 = reinterpret_cast<float4*>(out);
    if (mode == kMxfp4)
      dequantize_vec_kernel<kMxfp4, 0><<<blocks, kThreads, 0, as_stream(stream)>>>(
          q4, scale_bytes, nullptr, n / 4, shift, out4);
    else
      dequantize_vec_kernel<kMxfp8, 0><<<blocks, kThreads, 0, as_stream(stream)>>>(
          q4, scale_bytes, nullptr, n / 4, shift, out4);
    return check_launch("dequantize_mxfp");
  }
  dequantize_mxfp_kernel<<<elementwise_blocks(n, kThreads), kThreads, 0, as_stream(stream)>>>(
      q, scale_bytes, n, mode, out);
  return check_launch("dequantize_mxfp");
}

extern "C" int mgq_rtn_quantize_mxfp(const void* W, int w_dtype, int64_t rows, int64_t cols,
                                     int mode, uint8_t* q, uint8_t* scale_bytes, float* dq,
                                     void* stream) {
  clear_error();
  if (int rc = check_mx_mode(mode)) return rc;
  if (int rc = check_dtype(w_dtype, "rtn_quantize_mxfp")) return rc;
  MGQ_REQUIRE(cols % kMxGroup == 0, MGQ_ERR_VALUE, "columns %lld not divisible by %d",
              (long long)cols, kMxGroup);
  MGQ_REQUIRE(rows >= 0 && cols >= 0, MGQ_ERR_SHAPE, "bad shape");
  const int64_t n_groups = rows * (cols / kMxGroup);
  if (n_groups == 0) return MGQ_OK;
  const bool aligned = ((reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(q) |
                         reinterpret_cast<uintptr_t>(dq)) & 15u) == 0;
  const unsigned blocks = elementwise_blocks(n_groups, kThreads);
  hipStream_t st = as_stream(stream);
  if (!aligned)
    rtn_mxfp_kernel<<<blocks, kThreads, 0, st>>>(W, w_dtype, n_groups, mode, q, scale_bytes, dq);
  else if (w_dtype == kF32)
    rtn_mxfp_vec_kernel<float, false><<<blocks, kThreads, 0, st>>>(
        static_cast<const float*>(W), n_groups, mode, q, scale_bytes, dq);
  else if (w_dtype == kBF16)
    rtn_mxfp_vec_kernel<uint16_t, false><<<blocks, kThreads, 0, st>>>(
        static_cast<const uint16_t*>(W), n_groups, mode, q, scale_bytes, dq);
  else
    rtn_mxfp_vec_kernel<uint16_t, true><<<blocks, kThreads, 0, st>>>(
        static_cast<const uint16_t*>(W), n_groups, mode, q, scale_bytes, dq);
  return check_launch("rtn_quantize_mxfp");
}

extern "C" int mgq_dequantize_affine(const uint8_t* q, const void* scales, const void* biases,
                                     int storage_dtype, int64_t n_groups, int64_t group_size,
                                     float* out, void* stream) {
  clear_error();
  if (int rc = check_dtype(storage_dtype, "dequantize_affine")) return rc;
  MGQ_REQUIRE(n_groups >= 0 && group_size >= 1, MGQ_ERR_SHAPE, "bad shape");
  const int64_t n = n_groups * group_size;
  if (n == 0) return MGQ_OK;
  const int shift = dequant_shift(q, out, group_size);
  if (shift >= 0) {
    auto kernel = storage_dtype == kF32    ? dequantize_vec_kernel<kAffine, kF32>
                  : storage_dtype == kBF16 ? dequantize_vec_kernel<kAffine, kBF16>
                                           : dequantize_vec_kernel<kAffine, kF16>;
    kernel<<<dequant_blocks(n / 4), kThreads, 0, as_stream(stream)>>>(
        reinterpret_cast<const uint32_t*>(q), scales, biases, n / 4, shift,
        reinterpret_cast<float4*>(out));
    return check_launch("dequantize_affine");
  }
  dequantize_affine_kernel<<<elementwise_blocks(n, kThreads), kThreads, 0,
                             as_stream(stream)>>>(q, scales, biases, storage_dtype, n,
                                                  group_size, out);
  return check_launch("dequantize_affine");
}

extern "C" int mgq_choose_qparams(const float* w, int64_t n_groups, int64_t group_len, int bits,
                                  int method, int storage_dtype, int grid_steps,
                                  double max_shrink, void* s_store, void* b_store, float* s32,
                                  float* b32, void* stream) {
  clear_error();
  if (int rc = check_bits(bits)) return rc;
  if (int rc = check_dtype(storage_dtype, "choose_qparams")) return rc;
  MGQ_REQUIRE(method == MGQ_CLIP_MINMAX || method == MGQ_CLIP_MSE, MGQ_ERR_VALUE,
              "unsupported clip method %d", method);
  MGQ_REQUIRE(n_groups >= 0 && group_len >= 1, MGQ_ERR_SHAPE, "bad shape");
  Shrinks sh;
  if (int rc = make_shrinks(bits, method, grid_steps, max_shrink, &sh)) return rc;
  if (n_groups == 0) return MGQ_OK;
  if (whole_groups(group_len, w, kF32, nullptr, nullptr))
    return launch_groups<false>(w, kF32, n_groups, group_len, static_cast<float>((1 << bits) - 1),
                                storage_dtype, sh, nullptr, s_store, b_store, nullptr, s32, b32,
                                as_stream(stream), "choose_qparams");
  choose_qparams_kernel<<<elementwise_blocks(n_groups, kThreads), kThreads, 0,
                          as_stream(stream)>>>(w, n_groups, group_len,
                                               static_cast<float>((1 << bits) - 1),
                                               storage_dtype, sh, s_store, b_store, s32, b32);
  return check_launch("choose_qparams");
}

extern "C" int mgq_quantize_with_params(const float* w, const float* s32, const float* b32,
                                        int64_t n_groups, int64_t group_len, int bits, float* q,
                                        float* dq, void* stream) {
  clear_error();
  if (int rc = check_bits(bits)) return rc;
  MGQ_REQUIRE(n_groups >= 0 && group_len >= 1, MGQ_ERR_SHAPE, "bad shape");
  const int64_t n = n_groups * group_len;
  if (n == 0) return MGQ_OK;
  quantize_with_params_kernel<<<elementwise_blocks(n, kThreads), kThreads, 0,
                                as_stream(stream)>>>(w, s32, b32, n, group_len,
                                                     static_cast<float>((1 << bits) - 1), q, dq);
  return check_launch("quantize_with_params");
}

extern "C" int mgq_rtn_quantize_affine(const void* W, int w_dtype, int64_t rows, int64_t cols,
                                       int bits, int group_size, int method, int storage_dtype,
                                       uint8_t* q, void* s_store, void* b_store, float* dq,
                                       void* stream) {
  clear_error();
  if (int rc = check_bits(bits)) return rc;
  if (int rc = check_dtype(w_dtype, "rtn_quantize")) return rc;
  if (int rc = check_dtype(storage_dtype, "rtn_quantize")) return rc;
  MGQ_REQUIRE(method == MGQ_CLIP_MINMAX || method == MGQ_CLIP_MSE, MGQ_ERR_VALUE,
              "unsupported clip method %d", method);
  MGQ_REQUIRE(group_size >= 1 && cols % group_size == 0, MGQ_ERR_SHAPE,
              "cols %lld not divisible by group size %d", (long long)cols, group_size);
  const int64_t n_groups = rows * (cols / group_size);
  if (n_groups == 0) return MGQ_OK;
  Shrinks sh;
  if (int rc = make_shrinks(bits, method, 20, 0.2, &sh)) return rc;
  if (whole_groups(group_size, W, w_dtype, q, dq))
    return launch_groups<true>(W, w_dtype, n_groups, group_size,
                               static_cast<float>((1 << bits) - 1), storage_dtype, sh, q, s_store,
                               b_store, dq, nullptr, nullptr, as_stream(stream), "rtn_quantize");
  const unsigned blocks = elementwise_blocks(n_groups, kThreads);
#define MGQ_RTN(T, F16)                                                                         \
  rtn_affine_kernel<T, F16><<<blocks, kThreads, 0, as_stream(stream)>>>(                        \
      static_cast<const T*>(W), n_groups, group_size, static_cast<float>((1 << bits) - 1),      \
      storage_dtype, sh, q, s_store, b_store, dq)
  if (w_dtype == kF32) MGQ_RTN(float, false);
  else if (w_dtype == kBF16) MGQ_RTN(uint16_t, false);
  else MGQ_RTN(uint16_t, true);
#undef MGQ_RTN
  return check_launch("rtn_quantize");
}

extern "C" int mgq_range_audit(const void* source, int source_dtype, const uint8_t* q,
                               const void* scales, const void* biases, int storage_dtype,
                               int mode, int64_t rows, int64_t cols, int64_t group_size,
                               unsigned long long* stats, void* stream) {
  clear_error();
  if (int rc = check_dtype(source_dtype, "range_audit")) return rc;
  MGQ_REQUIRE(mode == kAffine || mode == kMxfp4 || mode == kMxfp8, MGQ_ERR_VALUE,
              "unsupported mode %d", mode);
  MGQ_REQUIRE(rows >= 0 && cols >= 0, MGQ_ERR_SHAPE, "bad shape");
  MGQ_REQUIRE(cols % kMxGroup == 0, MGQ_ERR_SHAPE, "columns %lld not divisible by %d",
              (long long)cols, kMxGroup);
  if (mode == kAffine) {
    if (int rc = check_dtype(storage_dtype, "range_audit")) return rc;
    MGQ_REQUIRE(group_size >= 1 && cols % group_size == 0, MGQ_ERR_SHAPE,
                "columns %lld not divisible by group %lld", (long long)cols,
                (long long)group_size);
    MGQ_REQUIRE(biases != nullptr, MGQ_ERR_VALUE, "affine artifacts need biases");
  } else {
    MGQ_REQUIRE(group_size == kMxGroup, MGQ_ERR_VALUE, "mxfp requires group size %d", kMxGroup);
  }
  MGQ_REQUIRE(stats != nullptr, MGQ_ERR_VALUE, "stats required");
  const int64_t n = rows * cols;
  if (n == 0) return MGQ_OK;
  hipStream_t st = as_stream(stream);
  const bool vec = ((reinterpret_cast<uintptr_t>(source) | reinterpret_cast<uintptr_t>(q)) & 15u) == 0 &&
                   (mode != kAffine || group_size % 8 == 0);
  const int64_t units = vec ? n / 8 : n;
  const auto launch =
      units <= kAuditBlocks * kAuditSmall ? launch_audit<kAuditSmall> : launch_audit<kAuditThreads>;
  launch(vec, vec ? kAuditBlocks : 2 * kAuditBlocks, units, source_dtype, st, source, q, scales,
         biases, storage_dtype, mode, group_size, stats);
  return check_launch("range_audit");
}
