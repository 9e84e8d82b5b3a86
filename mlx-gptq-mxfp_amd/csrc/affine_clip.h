// The MSE clip search of the affine grid (grid.py:167-212) for one group of
// values held by LN consecutive lanes (LN = 4, a quad, or 16, a DPP row),
// NS values each. Shared by round-to-nearest (grid.hip) and the GPTQ column
// loop (gptq_affine.hip).
//
// Every lane operation stays in the quad or DPP row: candidates are prepared
// one per lane (scale, bias and reciprocal once per group instead of once
// per value) and broadcast by DPP (quad_perm, or row_newbcast for 16 lanes),
// and the error sums run over the values a lane holds (a tree of halves)
// and then over the lanes by DPP rotations and quad permutations. The search
// is bound by vector instruction issue: NS values and one candidate take ten
// operations each (the three of the exact division among them) and NS - 1
// additions of the error sum, the whole group another ten (LN = 4) or twelve
// (LN = 16): 55 at LN = 16, NS = 4. The fewer lanes a group takes, the more
// groups share each of those.
#pragma once

#include "mgq_capi.h"
#include "mgq_common.h"
#include "mx_hw.h"

namespace mgq {

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kRowRor8 = 0x128, kRowRor4 = 0x124, kQuadXor2 = 0x4e, kQuadXor1 = 0xb1;

// v of lane O of the lane's quad (LN = 4) or DPP row (LN = 16)
template <int LN, int O>
__device__ __forceinline__ float row_bcast(float v) {
  static_assert(LN == 4 || LN == 16, "a quad or a DPP row");
  return dpp<LN == 4 ? O * 0x55 : 0x150 + O>(v);
}

// f over the LN lanes of a row, the same result in all of them (f symmetric:
// after the rotation by 8 a lane's value depends on its lane mod 8 only, so
// the rotation by 4 reads the value of lane ^ 4)
template <int LN, typename F>
__device__ __forceinline__ float row_reduce(float v, F&& f) {
  if constexpr (LN == 16) {
    v = f(v, dpp<kRowRor8>(v));
    v = f(v, dpp<kRowRor4>(v));
  }
  v = f(v, dpp<kQuadXor2>(v));
  return f(v, dpp<kQuadXor1>(v));
}

// v[0] += the rest, pairing slot s with s + half at every level
template <int N>
__device__ __forceinline__ float tree_sum(float (&v)[N]) {
#pragma unroll
  for (int h = N / 2; h >= 1; h >>= 1)
#pragma unroll
    for (int s = 0; s < h; ++s) v[s] = v[s] + v[s + h];
  return v[0];
}

// ---- exact division by a positive divisor ----------------------------------
// a / d for d > 0 (or NaN), correctly rounded: Markstein's correction from
// y = div_exact_recip(d) (mx_hw.h); a zero numerator is returned as is (a / d
// keeps its sign for d > 0); outside the correction's range the IEEE
// division. Every divisor here is positive: the clip scale (range >= 0) and
// U's diagonal. div_fast is the correction, div_slow says when it is not
// exact (the operators are the non-short-circuit ones so that no branch is
// formed around the test).
__device__ inline float div_fast(float a, float d, float y) {
  const float q = a * y;
  const float r = fmaf(-q, d, a);
  return fmaf(r, y, q);
}
__device__ inline bool div_slow(float a, float y) {
  const uint32_t ea = f2u(a) & 0x7f800000u;
  return (a != 0.0f) & ((!(y != 0.0f)) | ((ea - (27u << 23)) > (200u << 23)));
}

__device__ inline float div_pos(float a, float d, float y) {
  float e = div_fast(a, d, y);
  const bool slow = div_slow(a, y);
  // the IEEE division only when some lane needs it: a wave-uniform branch
  // (the empty asm keeps the compiler from hoisting the division out of it)
  if (__builtin_amdgcn_ballot_w64(slow) != 0) {
    asm volatile("" ::: "memory");
    const float ref = a / d;
    e = slow ? ref : e;
  }
  return a == 0.0f ? a : e;
}

// grid.py:215-221 from a quotient (w - b) / s_safe: q = clamp(rne(quot), 0,
// maxq), NaN kept
__device__ inline float affine_round(float quot, float maxq) {
  const float q = rintf(quot);
  return q != q ? q : fminf(fmaxf(q, 0.0f), maxq);
}

// grid.py:215-221: q = clamp(rne((w - b) / s_safe), 0, maxq); ys = RN(1/s_safe)
__device__ inline float affine_q_exact(float w, float b, float s_safe, float ys, float maxq) {
  return affine_round(div_pos(w - b, s_safe, ys), maxq);
}

__device__ inline float safe_scale(float s) { return fabsf(s) < 1e-12f ? 1.0f : s; }

// The clip candidates of grid.py:189-201: candidate i scales the range by
// p_i = 1 - max_shrink * i / steps (one candidate, p = 1, for minmax).
struct Shrinks {
  int n, steps;
  double max_shrink, maxq;
};
constexpr int kMaxShrinks = 128;

// grid.py:185-192: maxq = float(2**bits - 1), one candidate for minmax
inline int make_shrinks(int bits, int method, int grid_steps, double max_shrink, Shrinks* out) {
  out->maxq = static_cast<double>((1 << bits) - 1);
  if (method == MGQ_CLIP_MINMAX) {
    out->n = out->steps = 1;
    out->max_shrink = 0.0;
    return MGQ_OK;
  }
  MGQ_REQUIRE(grid_steps >= 1 && grid_steps < kMaxShrinks, MGQ_ERR_VALUE,
              "grid_steps must be in [1, %d), got %d", kMaxShrinks, grid_steps);
  out->n = grid_steps + 1;
  out->steps = grid_steps;
  out->max_shrink = max_shrink;
  return MGQ_OK;
}

// The workgroup's table of (p_i / maxq, p_i) in LDS, formed in double as
// Python evaluates it and cast to fp32 the way torch casts a Python scalar
// operand (a barrier must follow). Formed on the device: reading a table of
// them from the kernel arguments by lane took about 2 us at every launch.
__device__ inline void stage_shrinks(const Shrinks& sh, float2* tab) {
  for (int i = threadIdx.x; i < sh.n; i += blockDim.x) {
    const double p = 1.0 - sh.max_shrink * static_cast<double>(i) / static_cast<double>(sh.steps);
    tab[i] = make_float2(static_cast<float>(p / sh.maxq), static_cast<float>(p));
  }
}

// Scale and bias (rounded to the storage dtype) of the group whose values
// this row's lanes hold in w (on[s] false: slot s holds no value; ignored
// when FULL). tab: (p / maxq, p) of the n candidates, in LDS. The first
// candidate with the smallest error wins (strict '<').
//
// The fast batch divides by Markstein's correction, which is exact when every
// numerator w - bias is zero or in [2^-100, 2^101) and the reciprocal is in
// range. That holds when all values and biases are zero or in
// [2^-76, 2^100): a nonzero difference of two such numbers is a multiple of
// 2^-99. So the range is checked once per group and candidate, not once per
// quotient; any other batch (NaN and inf included) takes the IEEE division.
//
// CS > 1: CS neighbouring rows of lanes hold the same group, and part x of
// them scores the x-th share of the candidates (all parts get the result).
template <int LN, int NS, bool FULL, int CS = 1>
__device__ __forceinline__ void clip_search(const float (&w)[NS], const bool (&on)[NS],
                                            const float2* tab, int n, float maxq, int storage,
                                            float& s_out, float& b_out) {
  constexpr uint32_t kTiny = (51u << 24) - 2u;  // 2^-76, shifted left by one, minus 2
  const int l = threadIdx.x & (LN - 1), part = (threadIdx.x / LN) & (CS - 1);
  const int per = (n + CS - 1) / CS, first = part * per;
  const int last = (first + per < n ? first + per : n) - 1;  // may precede first
  float lo = __uint_as_float(0x7f800000u), hi = __uint_as_float(0xff800000u);
  uint32_t tiny = 0xffffffffu;  // smallest nonzero magnitude (a zero wraps to the top)
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const bool a = FULL || on[s];
    lo = a ? __builtin_elementwise_minimum(lo, w[s]) : lo;
    hi = a ? __builtin_elementwise_maximum(hi, w[s]) : hi;
    tiny = min(tiny, a ? (f2u(w[s]) << 1) - 2u : 0xffffffffu);
  }
  lo = row_reduce<LN>(lo, [](float a, float b) { return __builtin_elementwise_minimum(a, b); });
  hi = row_reduce<LN>(hi, [](float a, float b) { return __builtin_elementwise_maximum(a, b); });
  const float range = hi - lo;
  const bool bad = (tiny < kTiny) | !(fabsf(lo) < 0x1p100f) | !(fabsf(hi) < 0x1p100f);
  float best = __uint_as_float(0x7f800000u), s_best = 0.0f, b_best = 0.0f;
  for (int c0 = 0; c0 < per; c0 += LN) {
    // past the part's last candidate a copy of it (an equal error takes nothing)
    const float2 t = tab[first + c0 + l < last ? first + c0 + l : last];
    const float sc = round_to_storage(range * t.x, storage);
    const float bi = round_to_storage(lo * t.y, storage);
    const float ss = safe_scale(sc), ys = div_exact_recip(ss);
    if (c0 == 0) {
      s_best = row_bcast<LN, 0>(sc);
      b_best = row_bcast<LN, 0>(bi);
    }
    const bool slow = bad | !(ys != 0.0f) | ((f2u(bi) << 1) - 2u < kTiny) | !(fabsf(bi) < 0x1p100f);
    if (__builtin_amdgcn_ballot_w64(slow) == 0) {
      // K candidates at a time, without a branch between them: their chains
      // of lane operations run side by side
      constexpr int K = NS <= 4 ? 4 : NS <= 8 ? 2 : 1;
      auto score = [&](auto ic, float& p, float& s1, float& b1) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        s1 = row_bcast<LN, i>(sc), b1 = row_bcast<LN, i>(bi);
        const float d1 = row_bcast<LN, i>(ss), y1 = row_bcast<LN, i>(ys);
        float e[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const float q = __builtin_amdgcn_fmed3f(rintf(div_fast(w[s] - b1, d1, y1)), 0.0f, maxq);
          const float d = q * s1 + b1 - w[s];
          e[s] = FULL || on[s] ? d * d : 0.0f;
        }
        p = tree_sum(e);
      };
      auto sum = [](float a, float b) { return a + b; };
      auto keep = [&](float p, float s1, float b1) __attribute__((always_inline)) {
        const bool take = p < best;
        best = take ? p : best;
        s_best = take ? s1 : s_best;
        b_best = take ? b1 : b_best;
      };
      static_for<LN / K>([&](auto tc) __attribute__((always_inline)) {
        constexpr int i0 = K * decltype(tc)::value;
        if (c0 + i0 + K <= per) {  // uniform
          float p[K], s1[K], b1[K];
          static_for<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            score(std::integral_constant<int, i0 + k>{}, p[k], s1[k], b1[k]);
          });
#pragma unroll
          for (int k = 0; k < K; ++k) p[k] = row_reduce<LN>(p[k], sum);
#pragma unroll
          for (int k = 0; k < K; ++k) keep(p[k], s1[k], b1[k]);
        } else {
          static_for<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            if (k + 1 == K || c0 + i0 + k >= per) return;
            float p, s1, b1;
            score(std::integral_constant<int, i0 + k>{}, p, s1, b1);
            keep(row_reduce<LN>(p, sum), s1, b1);
          });
        }
      });
    } else {
#pragma unroll 1
      for (int i = 0; i < LN && c0 + i < per; ++i) {
        const float s1 = __shfl(sc, i, LN), b1 = __shfl(bi, i, LN), d1 = __shfl(ss, i, LN);
        float e[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const float d = affine_round((w[s] - b1) / d1, maxq) * s1 + b1 - w[s];
          e[s] = FULL || on[s] ? d * d : 0.0f;
        }
        const float p = row_reduce<LN>(tree_sum(e), [](float a, float b) { return a + b; });
        const bool take = (first + c0 + i == 0) | (p < best);
        best = take ? p : best;
        s_best = take ? s1 : s_best;
        b_best = take ? b1 : b_best;
      }
    }
  }
  if constexpr (CS > 1) {
    // the lower part's candidate stays unless the upper part's error is smaller
#pragma unroll
    for (int x = 1; x < CS; x <<= 1) {
      const float p = __shfl_xor(best, x * LN), s1 = __shfl_xor(s_best, x * LN),
                  b1 = __shfl_xor(b_best, x * LN);
      const bool take = (part & x) == 0 ? p < best : !(best < p);
      best = take ? p : best;
      s_best = take ? s1 : s_best;
      b_best = take ? b1 : b_best;
    }
  }
  s_out = s_best;
  b_out = b_best;
}

}  // namespace mgq
