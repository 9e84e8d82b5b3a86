// The affine column loop with a wave per row, for group lengths that do not fill
// the lanes' slots of affine_block_kernel (gptq_affine.hip) while rows are few.
// Each lane holds column j + t of the group (and j + t + 64 where G > 64), so a
// group of any length up to 128 takes the same instructions, the candidates of
// the clip search run through one butterfly twelve at a time, and U's block is in
// LDS (blocks of at most kLdsBlock columns) or read where it lies: no chunk is
// waited for. The results have the bits of affine_block_kernel: every quotient is
// the correctly rounded one, and the error sums add the same pairs (columns 64
// apart, then 32, 16, 8, 4, 2, 1).
// Bound by the serial chain of one row (33 instructions per column); above two
// workgroups per CU the rows queue up and 16 lanes per row win. The lines between
// them and both sides' figures are at wave_rows in gptq_affine.hip.
#pragma once

#include "affine_clip.h"
#include "mgq_common.h"
#include "mx_hw.h"

namespace mgq {
namespace {

constexpr int kWaves = 4;
constexpr int kCand = 12;  // clip candidates scored per butterfly

// N wave sums (N a multiple of 4), each rounded like an xor butterfly with
// __shfl_xor (v <- v + partner for xor 32, 16, 8, 4, 2, 1), by recursive
// halving. The xor-32 step swaps v[i] with v[i + N/2], so lanes 0-31 keep
// sum i and lanes 32-63 sum i + N/2, both as lo + hi; the xor-16 step pairs
// those results the same way (row 2k + row 2k+1); the DPP steps then run on
// N/4 values. Because a + b == b + a bit for bit, after the 8 step a lane's
// value depends only on lane mod 8, so a rotation by 4 reads the value of
// lane ^ 4. Sum i + (N/4) r ends in u[i] of the lanes of row r (lanes 16r ..
// 16r + 15).
template <int N>
__device__ inline void wave_sum_halving(const float (&v)[N], float (&u)[N / 4]) {
  static_assert(N % 4 == 0, "N must be a multiple of 4");
  float w[N / 2];
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]),
                                                    __float_as_uint(v[i + N / 2]), false, false);
    w[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(w[i]),
                                                    __float_as_uint(w[i + N / 4]), false, false);
    u[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) u[i] += dpp<kRowRor8>(u[i]);
#pragma unroll
  for (int i = 0; i < N / 4; ++i) u[i] += dpp<kRowRor4>(u[i]);
#pragma unroll
  for (int i = 0; i < N / 4; ++i) u[i] += dpp<kQuadXor2>(u[i]);
#pragma unroll
  for (int i = 0; i < N / 4; ++i) u[i] += dpp<kQuadXor1>(u[i]);
}

// the smallest lo and the largest hi of the wave (IEEE minimum and maximum)
__device__ inline void wave_minmax(float& lo, float& hi) {
  auto mn = [](float a, float b) { return __builtin_elementwise_minimum(a, b); };
  auto mx = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };
  auto swap = [](float& v, auto&& f) __attribute__((always_inline)) {
    const uint32_t x = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const uint32_t y = __float_as_uint(f(__uint_as_float(r[0]), __uint_as_float(r[1])));
    const auto s = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    v = row_reduce<16>(f(__uint_as_float(s[0]), __uint_as_float(s[1])), f);
  };
  swap(lo, mn);
  swap(hi, mx);
}

// Row k of U restricted to the group's columns: lane t holds U[k][j + t + 64 s]
// (0 past the group). LDSU: from the block's copy Ublk[(k - i1) * n + (col -
// i1)] in LDS, else from global memory. Lanes past the group read the
// group's first column, so the load needs no branch.
template <int CPL, bool LDSU>
__device__ inline void load_urow(const float* __restrict__ Ub, const float* Ublk, int64_t C,
                                 int64_t i1, int n, int64_t k, int64_t j, int lane,
                                 const bool (&act)[CPL], float (&u)[CPL]) {
  const float* Uk = LDSU ? Ublk + (k - i1) * n + (j - i1) : Ub + k * C + j;
#pragma unroll
  for (int s = 0; s < CPL; ++s) {
    const float v = Uk[act[s] ? lane + 64 * s : 0];
    u[s] = act[s] ? v : 0.0f;
  }
}

__device__ inline float lane_read(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Grid (ceil(R / 4), B): the four waves of a workgroup take rows of one
// batch item. LDSU (blocks of at most kLdsBlock columns): the workgroup first
// copies the block's U[i1:i1+n, i1:i1+n] to LDS, so the column loop and the
// in-block updates read U rows from LDS instead of all waves fetching the
// same row from L2 at once.
constexpr int kLdsBlock = 128;

template <int CPL, bool LDSU>
__global__ void __launch_bounds__(kWaves * 64)
    affine_wave_kernel(float* __restrict__ W, const float* __restrict__ U, int64_t B, int64_t R,
                       int64_t C, int64_t i1, int n, int G, float maxq, int storage, Shrinks sh,
                       uint8_t* __restrict__ q_out, void* s_store, void* b_store,
                       float* __restrict__ Err, int64_t ld_err) {
  // the candidate table, per-wave table [kWaves][max(G, 64)] (float4: the clip
  // candidates, then the column table), errs [kWaves][n], then (LDSU) Ublk [n][n]
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float2* tab = reinterpret_cast<float2*>(smem);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tab_n = G > 64 ? G : 64;
  float* cols = smem + 2 * kMaxShrinks;
  float4* ctab = reinterpret_cast<float4*>(cols) + wave * tab_n;
  float* errs = cols + kWaves * 4 * tab_n + wave * n;
  float* Ublk = cols + kWaves * 4 * tab_n + kWaves * n;
  const int64_t b = blockIdx.y;
  const float* Ub = U + b * C * C;
  if constexpr (LDSU) {
    if ((n & 1) == 0 && (C & 1) == 0 && (i1 & 1) == 0) {
      // wave w copies rows w, w+4, ...: one 8-byte chunk per lane and row,
      // sixteen rows' loads in flight before their LDS stores
      const int half_n = n >> 1;
      const bool on = lane < half_n;
      for (int r0 = wave; r0 < n; r0 += kWaves * 16) {
        f32x2_u_t v[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int r = r0 + kWaves * t;
          v[t] = (on && r < n) ? load_f32x2(Ub + (i1 + r) * C + i1 + 2 * lane)
                               : f32x2_u_t{0.0f, 0.0f};
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int r = r0 + kWaves * t;
          if (on && r < n) *reinterpret_cast<float2*>(Ublk + r * n + 2 * lane) = float2{v[t].x, v[t].y};
        }
      }
    } else {
      for (int e = threadIdx.x; e < n * n; e += kWaves * 64) {
        const int r = e / n, c = e % n;
        Ublk[e] = Ub[(i1 + r) * C + i1 + c];
      }
    }
  }
  stage_shrinks(sh, tab);
  __syncthreads();
  const int64_t r_in = static_cast<int64_t>(blockIdx.x) * kWaves + wave;
  if (r_in >= R) return;  // whole wave exits together (no block barriers below)
  // canonicalized once, so that the clamps in affine_round do not redo it
  maxq = __builtin_canonicalizef(maxq);
  const int64_t row = b * R + r_in;
  float* Wr = W + row * C;
  const int64_t ng = C / G;
  // the clip candidates' p / maxq and p, one per lane (batches of 64)
  const int n_batches = (sh.n + 63) / 64;
  for (int64_t j = i1; j < i1 + n; j += G) {
    float acc[CPL], dg[CPL], yd[CPL];
    bool act[CPL];
#pragma unroll
    for (int s = 0; s < CPL; ++s) {
      const int col = lane + 64 * s;
      act[s] = col < G;
      acc[s] = act[s] ? Wr[j + col] : 0.0f;
      // U's diagonal of the lane's column and its reciprocal for div_pos
      const int cc = act[s] ? col : 0;
      dg[s] = act[s] ? (LDSU ? Ublk[(j - i1 + cc) * (n + 1)] : Ub[(j + cc) * (C + 1)]) : 1.0f;
      yd[s] = div_exact_recip(dg[s]);
    }
    // earlier in-block updates, in column order; sixteen rows of U in flight
    {
      const int64_t kn = j - i1;  // a multiple of G
      int64_t k = 0;
      for (; k + 16 <= kn; k += 16) {
        float u[16][CPL];
#pragma unroll
        for (int t = 0; t < 16; ++t)
          load_urow<CPL, LDSU>(Ub, Ublk, C, i1, n, i1 + k + t, j, lane, act, u[t]);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const float e = errs[k + t];
#pragma unroll
          for (int s = 0; s < CPL; ++s) acc[s] = act[s] ? acc[s] - e * u[t][s] : acc[s];
        }
      }
      for (; k < kn; ++k) {
        float u[CPL];
        load_urow<CPL, LDSU>(Ub, Ublk, C, i1, n, i1 + k, j, lane, act, u);
        const float e = errs[k];
#pragma unroll
        for (int s = 0; s < CPL; ++s) acc[s] = act[s] ? acc[s] - e * u[s] : acc[s];
      }
    }
    // clip search (grid.py:167-212) on the group's current values
    float lo = act[0] ? acc[0] : __uint_as_float(0x7f800000u);
    float hi = act[0] ? acc[0] : __uint_as_float(0xff800000u);
#pragma unroll
    for (int s = 1; s < CPL; ++s)
      if (act[s]) {
        lo = __builtin_elementwise_minimum(lo, acc[s]);
        hi = __builtin_elementwise_maximum(hi, acc[s]);
      }
    wave_minmax(lo, hi);
    const float wmin = lo, wmax = hi;
    const float range = wmax - wmin;
    float best_err = 0.0f, s32 = 0.0f, b32 = 0.0f;
    for (int bt = 0; bt < n_batches; ++bt) {
      // lane l prepares candidate 64 bt + l: scale, bias, divisor and its
      // reciprocal, into the wave's table (one LDS read per candidate)
      {
        const int cl = 64 * bt + lane < sh.n ? 64 * bt + lane : sh.n - 1;
        const float sc_l = round_to_storage(range * tab[cl].x, storage);
        const float bi_l = round_to_storage(wmin * tab[cl].y, storage);
        const float ss_l = (fabsf(sc_l) < 1e-12f) ? 1.0f : sc_l;
        ctab[lane] = float4{sc_l, bi_l, ss_l, div_exact_recip(ss_l)};
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      // candidates kCand at a time, their error sums reduced in one
      // butterfly; slots past the batch score a copy of its last candidate
      // (an equal error never replaces the earlier best under strict '<').
      // The quotients of the whole batch take the exact-division correction;
      // the numerators' magnitudes (as in the column chain) and a zero
      // reciprocal send the batch's out-of-range quotients to the IEEE
      // division.
      const int nb = sh.n - 64 * bt < 64 ? sh.n - 64 * bt : 64;
      for (int c0 = 0; c0 < nb; c0 += kCand) {
        float sc[kCand], bi[kCand], ss[kCand], ys[kCand], part[kCand];
        float num[kCand][CPL], quo[kCand][CPL];
        uint32_t mag_lo = 0xffffffffu;
        float mag_hi = 0.0f;
        bool y_zero = false;
#pragma unroll
        for (int i = 0; i < kCand; ++i) {
          const int ci = c0 + i < nb ? c0 + i : nb - 1;
          const float4 pc = ctab[ci];
          sc[i] = pc.x, bi[i] = pc.y, ss[i] = pc.z, ys[i] = pc.w;
          y_zero |= !(ys[i] != 0.0f);
#pragma unroll
          for (int s = 0; s < CPL; ++s) {
            num[i][s] = acc[s] - bi[i];
            quo[i][s] = div_fast(num[i][s], ss[i], ys[i]);
            mag_lo = min(mag_lo, (f2u(num[i][s]) << 1) - 2u);
            mag_hi = fmaxf(mag_hi, fabsf(num[i][s]));
          }
        }
        const bool slow = y_zero | (mag_lo < (27u << 24) - 2u) | !(mag_hi < 0x1p101f);
        if (__builtin_amdgcn_ballot_w64(slow) != 0) {
          asm volatile("" ::: "memory");
#pragma unroll
          for (int i = 0; i < kCand; ++i)
#pragma unroll
            for (int s = 0; s < CPL; ++s)
              if (act[s] && div_slow(num[i][s], ys[i])) quo[i][s] = num[i][s] / ss[i];
        }
#pragma unroll
        for (int i = 0; i < kCand; ++i) {
          part[i] = 0.0f;
#pragma unroll
          for (int s = 0; s < CPL; ++s) {
            // a zero numerator's quotient is that zero (see the column chain);
            // the clamp need not keep a NaN: a NaN quotient comes only from a
            // NaN acc, which makes d NaN anyway
            const float qt = copysignf(quo[i][s], num[i][s]);
            const float d = fminf(fmaxf(rintf(qt), 0.0f), maxq) * sc[i] + bi[i] - acc[s];
            part[i] = act[s] ? part[i] + d * d : part[i];
          }
        }
        float sums[kCand / 4];
        wave_sum_halving<kCand>(part, sums);
#pragma unroll
        for (int i = 0; i < kCand; ++i) {
          const float pi = lane_read(sums[i % (kCand / 4)], 16 * (i / (kCand / 4)));
          if ((bt == 0 && c0 + i == 0) || pi < best_err) {
            best_err = pi;
            s32 = sc[i];
            b32 = bi[i];
          }
        }
      }
    }
    const int64_t gi = row * ng + j / G;
    if (lane == 0) {
      store_storage(s_store, gi, s32, storage);
      store_storage(b_store, gi, b32, storage);
    }
    const float s_safe = (fabsf(s32) < 1e-12f) ? 1.0f : s32;
    const float ysafe = div_exact_recip(s_safe);
    // Sequential columns of the group. wn is the current column's value: the
    // owner lane's value after the updates of every earlier column. Before
    // column c's update the wave reads lane c+1's value (updated through
    // column c-1) and U[c, c+1], and wn = pre - e * U[c, c+1] repeats lane
    // c+1's own update (the same two roundings), so no lane read waits for
    // the column's error. Every lane past c applies w <- w - e * U[c, col]
    // (lanes past the group too: their values are never read). A column's
    // lane is not updated after its own column, so at the group's end it
    // holds the value its column was quantized from.
    //
    // The two divisions of a column take Markstein's correction without a
    // branch (EXACT = false); the operands outside its exact range are only
    // recorded. If any occurred, the group is run again from its start values
    // with the guarded division (EXACT = true), so every quotient is the
    // correctly rounded one either way.
    float acc0[CPL];
#pragma unroll
    for (int s = 0; s < CPL; ++s) acc0[s] = acc[s];
    // A divisor whose reciprocal is 0 (outside [2^-24, 2^24]) sends the
    // group to the guarded division directly.
    bool y_zero = !(ysafe != 0.0f);
#pragma unroll
    for (int s = 0; s < CPL; ++s) y_zero |= act[s] & !(yd[s] != 0.0f);
    y_zero = __builtin_amdgcn_ballot_w64(y_zero) != 0;
    // the column table: U[c][c], RN(1 / U[c][c]) and U[c][c+1] for column
    // c, read by the whole wave with one LDS read per column
#pragma unroll
    for (int s = 0; s < CPL; ++s) {
      const int col = lane + 64 * s;
      if (act[s]) {
        const int cn = col + 1 < G ? col + 1 : col;
        const float u1 = col + 1 < G ? (LDSU ? Ublk[(j - i1 + col) * n + (j - i1 + cn)]
                                             : Ub[(j + col) * C + j + cn])
                                     : 0.0f;
        ctab[col] = float4{dg[s], yd[s], u1, 0.0f};
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    auto run_columns = [&](auto exact_tag) __attribute__((always_inline)) {
      constexpr bool EXACT = decltype(exact_tag)::value;
      // The numerators' smallest nonzero magnitude (as its bit pattern
      // shifted left by one, minus 2, so that a zero wraps to the top) and
      // their largest magnitude. The correction is exact when every nonzero
      // numerator has a biased exponent in [27, 227] (div_slow).
      uint32_t mag_lo = 0xffffffffu;
      float mag_hi = 0.0f;
      float wn = lane_read(acc[0], 0);
      // column c; c1 = c + 1 (c for the last column)
      auto column = [&](int c, int c1, const float (&uc)[CPL]) __attribute__((always_inline)) {
        const int owner1 = c1 & 63, slot1 = c1 >> 6;
        float pre_v = acc[0];
#pragma unroll
        for (int s = 1; s < CPL; ++s)
          if (s == slot1) pre_v = acc[s];
        const float4 ct = ctab[c];
        const float diag = ct.x, ydg = ct.y, u1 = ct.z;
        const float pre1 = lane_read(pre_v, owner1);
        float e;
        if constexpr (EXACT) {
          const float q = affine_q_exact(wn, b32, s_safe, ysafe, maxq);
          const float dq = q * s32 + b32;
          e = div_pos(wn - dq, diag, ydg);
        } else {
          // a zero numerator's quotient is that zero: copysign turns the
          // correction's +0 into it (every other quotient has its sign)
          // NaN is not kept here: a NaN quotient means a NaN column value,
          // which reaches wn at the end of the group and sends the group to
          // the exact pass, whose rounding keeps it
          const float n1 = wn - b32;
          const float q =
              fminf(fmaxf(rintf(copysignf(div_fast(n1, s_safe, ysafe), n1)), 0.0f), maxq);
          const float dq = q * s32 + b32;
          const float n2 = wn - dq;
          e = copysignf(div_fast(n2, diag, ydg), n2);
          mag_lo = min(mag_lo, min((f2u(n1) << 1) - 2u, (f2u(n2) << 1) - 2u));
          mag_hi = fmaxf(mag_hi, fmaxf(fabsf(n1), fabsf(n2)));
        }
#pragma unroll
        for (int s = 0; s < CPL; ++s) acc[s] = lane + 64 * s > c ? acc[s] - e * uc[s] : acc[s];
        wn = pre1 - e * u1;
      };
      // Row c of the group's U block at urow + c * ust. Rows arrive eight
      // columns ahead (a slot is refilled once its column is done); the last
      // eight full columns load nothing, and the columns past the last
      // multiple of 8 load their own rows.
      const float* urow = LDSU ? Ublk + (j - i1) * n + (j - i1) : Ub + j * C + j;
      const int64_t ust = LDSU ? n : C;
      // (lanes past the group read the row's first entry: their values are
      // never read)
      auto load_row = [&](const float* p, float (&u)[CPL]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < CPL; ++s) u[s] = p[act[s] ? lane + 64 * s : 0];
      };
      const int G8 = G & ~7;
      float ring[8][CPL];
#pragma unroll
      for (int u = 0; u < 8; ++u) load_row(urow + (u < G ? u : G - 1) * ust, ring[u]);
      const float* unext = urow + 8 * ust;
      int c0 = 0;
      for (; c0 + 8 < G8; c0 += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          column(c0 + u, c0 + u + 1, ring[u]);
          load_row(unext, ring[u]);
          unext += ust;
        }
      }
      if (G8 > 0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int c = c0 + u;
          column(c, c + 1 < G ? c + 1 : c, ring[u]);
        }
      }
      for (int c = G8; c < G; ++c) {
        float uc[CPL];
        load_row(urow + c * ust, uc);
        column(c, c + 1 < G ? c + 1 : c, uc);
      }
      // nonzero numerators below 2^-100, any at or above 2^101, or a NaN
      // anywhere in the chain (it reaches the final wn through e)
      return (mag_lo < (27u << 24) - 2u) | !(mag_hi < 0x1p101f) | (wn != wn);
    };
    // every lane computed the same chain, so its verdict is wave-uniform
    if (y_zero || __builtin_amdgcn_ballot_w64(run_columns(std::false_type{})) != 0) {
#pragma unroll
      for (int s = 0; s < CPL; ++s) acc[s] = acc0[s];
      run_columns(std::true_type{});
    }
    // each lane's code, dequantized value and error, from the value its
    // column was quantized from (the same operations as the column step)
#pragma unroll
    for (int s = 0; s < CPL; ++s) {
      const float q = affine_q_exact(acc[s], b32, s_safe, ysafe, maxq);
      const float dq = q * s32 + b32;
      const float e = div_pos(acc[s] - dq, dg[s], yd[s]);
      if (!act[s]) continue;
      const int col = lane + 64 * s;
      q_out[row * C + j + col] = (q == q) ? static_cast<uint8_t>(q) : 0;
      Wr[j + col] = dq;
      errs[j + col - i1] = e;
      Err[row * ld_err + (j + col - i1)] = e;
    }
    // errs[] is read by every lane of this wave at the next group start
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace
}  // namespace mgq
