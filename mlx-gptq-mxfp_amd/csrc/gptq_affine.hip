// Affine (MLX scale/bias) GPTQ: the lazy-block column loop of
// gptq.py:229-272 with the MSE clip search of grid.py:167-212.
//
// LN consecutive lanes (a DPP row of 16, or a quad) own one (batch item,
// row), so a wave works on 4 or 16 rows at once. For each block of `bs`
// columns (a multiple of the group size G) and each G-column group in it:
//   - lane l holds columns j + l + LN s (s = 0, 1, ..); at the group start it
//     applies the earlier in-block updates
//         w <- w - err_k * U[k, col]   for k = block start .. j-1, in order,
//     which are exactly the element's updates in the reference's order;
//   - the clip search runs on those G values (affine_clip.h);
//   - the G columns are then quantized one by one; the owner lane's error
//     err = (w - dq) / U[c, c] is broadcast by DPP and every later column
//     applies w <- w - err * U[c, col].
// After the block a separate kernel applies the deferred update
//     W[:, i2:] -= Err @ U[i1:i2, i2:]
// (the reference's bmm) as an fp32 GEMM. Few rows with other group lengths than
// 32, 64 and 128 take a wave per row instead (affine_wave.h), with the same bits.
#include "affine_clip.h"
#include "affine_wave.h"
#include "mgq_capi.h"
#include "mgq_common.h"
#include "mx_hw.h"

namespace mgq {
namespace {

constexpr int kMaxBlock = 2048;  // a row's errors of one block in LDS (affine_wave.h)
constexpr int kMaxWaves = 8;
// Where the variants of affine_block_kernel start and end (us per block of
// 128 columns; rows over all items):
//   - a quad per row from quad_rows on, against a DPP row: G = 32, 32768 rows 78
//     / 91, 40000 rows 3 % behind, 49152 rows 118 / 128, 65536 rows 122 / 166,
//     66000 rows 7 % ahead, 81920 rows 173 / 204; G = 64, 32768 rows 69 / 76, 49152 rows 128 / 110,
//     65536 rows 133 / 140, 81920 rows 192 / 173, 98304 rows 198 / 205, 196608
//     rows 388 / 398. A quad's workgroup holds 128 rows, so its time goes up in
//     steps of 32768; the lines lie where a step no longer costs what it gains.
//   - four parts of the clip candidates up to kSplit4 waves of four rows, two
//     up to kSplit2, G = 64: 512 rows 14.2 / 14.7 / 17.0 (four, two, one),
//     2048 rows 21.4 / 18.3 / 19.8, 4096 rows 32.6 / 22.9 / 21.0.
//   - a wave per row where the group length leaves slots empty, up to
//     wave_rows workgroups of four rows: with U's block in LDS two of them fit a
//     CU and the 513th waits for a turn; without, more fit. The whole loop over
//     1920 columns, a wave / 16 lanes per row: G = 40, blocks of 120, 1 row 497 /
//     803, 512 rows 543 / 844, 2048 rows 662 / 886, 4096 rows (an earlier
//     build) 1336 / 922; G = 96, blocks of 96, 512 rows 520 / 699, 1536 rows 643
//     / 733; G = 48, blocks of 480, 512 rows 706 / 1398, 4096 rows 1009 / 1363,
//     8192 rows 2003 / 1449. Groups under 8 wait for a chunk of U every few
//     columns in the other form: G = 4, 4096 rows 5381 / 5811, 8192 rows 11141
//     / 6408; blocks of 512, 8192 rows 14793 / 18333, 16384 rows 28548 / 22268.
constexpr int64_t quad_rows(int G) { return G == 32 ? 49152 : 98304; }
constexpr int64_t kSplit4 = 256, kSplit2 = 768;
constexpr int64_t wave_rows(int G, int64_t n) {
  return (n <= kLdsBlock ? 512 : 1024) * (G < 8 ? 2 : 1);
}

// gptq.py:216-222 for the affine path: dead columns zeroed in W, H diag := 1.
// A workgroup looks at 256 columns' diagonals and touches `rows` rows of W only
// where one is dead (reading W to test every element's column took 264 us on 32
// experts of 1536 x 2048, now 5.5).
__global__ void __launch_bounds__(256)
    dead_fix_w_kernel(float* __restrict__ W, const float* __restrict__ H, int64_t R, int64_t C,
                      int64_t rows) {
  const int64_t b = blockIdx.z, c = blockIdx.x * int64_t{256} + threadIdx.x;
  if (c >= C || !(H[(b * C + c) * C + c] <= 0.0f)) return;
  const int64_t r0 = blockIdx.y * rows;
  const int64_t r1 = r0 + rows < R ? r0 + rows : R;
  for (int64_t r = r0; r < r1; ++r) W[(b * R + r) * C + c] = 0.0f;
}

__global__ void dead_fix_h_kernel(float* __restrict__ H, int64_t B, int64_t C) {
  const int64_t n = B * C;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / C, c = i % C;
    float* d = H + b * C * C + c * C + c;
    if (*d <= 0.0f) *d = 1.0f;
  }
}

typedef __attribute__((address_space(1))) const void global_cv;
typedef __attribute__((address_space(3))) void lds_v;

// g, opaque to the compiler: the tests of the unrolled columns against it are
// not all formed ahead of them (they would not fit the scalar registers)
__device__ __forceinline__ int opaque(int g) {
  asm volatile("" : "+s"(g));
  return g;
}

// One block [i1, i1 + n) of the column loop. Grid (row tiles, B); the waves
// of a workgroup take rows of one batch item.
//
// U comes through LDS in chunks of one group of rows by one group of columns
// (chunk (p, j): rows of group p, columns of group j, p <= j; p < j feeds the
// in-block updates of group j, p = j its column chain), fetched by LDS-direct
// loads one chunk ahead of its use (two buffers), 16 bytes a lane where U is
// aligned to that (wide).
//
// Column chain: every lane runs the column step on its own column of the
// slot being processed, and only the owner lane's error is broadcast, so no
// value is exchanged before the step (fifteen dependent operations, then one
// multiply and one subtraction per later slot). The two divisions take
// Markstein's correction without a test; the numerators of each column's
// final value are checked once at the group's end, and a group that had one
// outside the correction's range, a divisor outside [2^-24, 2^24] or a NaN is
// run again from its start values with guarded divisions: every quotient is
// the correctly rounded one either way.
//
// CS > 1: CS neighbouring DPP rows hold the same row of W, score their share
// of the clip candidates and run the same chain; the first of them stores.
//
// A wave alone on its SIMD issues one vector instruction per five cycles
// whether they depend on each other or not, so up to a few waves per SIMD
// the time is the instruction count of one wave (the column step 23, a clip
// candidate 55, at NS = 4) and rows are spread thin (CS); above that it is
// the SIMDs' issue rate, and the fewest lanes per row win (LN = 4). Measured
// for a block of 128 columns, G = 64, against the earlier form (a wave per
// row, 33 instructions per column for one row): 2048 rows 27.4 -> 18.3 us,
// 14336 rows 158 -> 43 us (G = 128: 159 -> 38), 32 x 1536 rows 544 -> 115 us.
template <int LN, int NS, bool FULL, int CS>
__global__ void __launch_bounds__(kMaxWaves * 64)
    affine_block_kernel(float* __restrict__ W, const float* __restrict__ U, int64_t R, int64_t C,
                        int64_t i1, int n, int G, float maxq, int storage, Shrinks sh,
                        bool wide, uint8_t* __restrict__ q_out, void* s_store, void* b_store,
                        float* __restrict__ Err, int64_t ld_err) {
  constexpr int GP = LN * NS;  // G rounded up to whole slots
  constexpr int RW = 64 / (LN * CS);  // rows per wave
  // rows of U read ahead of their use (an LDS read takes longer than a column)
  constexpr int kAhead = NS <= 4 ? 4 : 2;
  if constexpr (FULL) G = GP;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float2* tab = reinterpret_cast<float2*>(smem);
  float* ubuf = smem + 2 * kMaxShrinks;  // one or two chunks [G][LN][NS]
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane & (LN - 1);
  const int64_t b = blockIdx.y;
  const float* Ub = U + b * C * C + i1 * C + i1;
  const int64_t r_in = (static_cast<int64_t>(blockIdx.x) * waves + wave) * RW + lane / (LN * CS);
  const bool live = r_in < R;  // the other rows compute on zeros and store nothing
  const bool writes = live && (lane / LN) % CS == 0;
  const int64_t row = b * R + (live ? r_in : R - 1);
  float* Wr = W + row * C + i1;
  uint8_t* qr = q_out + row * C + i1;
  float* Er = Err + row * ld_err;
  const int ng = n / G;
  const int64_t g_first = row * (C / G) + i1 / G;

  auto stage = [&](int pg, int jg, int buf) {
    const float* src = Ub + static_cast<int64_t>(pg) * G * C + jg * G;
    float* dst = ubuf + buf * G * GP;
    if (wide) {  // 16 bytes a lane
      constexpr int kRows = 256 / GP > 0 ? 256 / GP : 1;  // rows of the chunk per wave and load
      const float* p = src + (wave * kRows + 4 * lane / GP) * C + 4 * lane % GP;
      for (int e0 = wave * 256; e0 < G * GP; e0 += waves * 256, p += waves * kRows * C)
        __builtin_amdgcn_global_load_lds((global_cv*)p, (lds_v*)(dst + e0), 16, 0, 0);
    } else {
      for (int e0 = wave * 64; e0 < G * GP; e0 += waves * 64) {
        const int e = e0 + lane;
        const int k = e / GP, col = e % GP;
        if (FULL || e < G * GP)
          __builtin_amdgcn_global_load_lds(
              (global_cv*)(src + static_cast<int64_t>(k) * C + (FULL || col < G ? col : 0)),
              (lds_v*)(dst + e0), 4, 0, 0);
      }
    }
  };
  // slots first .. NS - 1 of this lane in row k of a chunk
  auto load_u = [&](const float* chunk, int k, int first, float (&u)[NS])
                    __attribute__((always_inline)) {
    const float* p = chunk + k * GP + l;
#pragma unroll
    for (int t = 0; t < NS; ++t)
      if (t >= first) u[t] = p[LN * t];
  };

  stage(0, 0, 0);
  stage_shrinks(sh, tab);
  bool on[NS];
  float next[NS], errs[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    on[s] = FULL || l + LN * s < G;
    next[s] = live && on[s] ? Wr[l + LN * s] : 0.0f;
    errs[s] = 0.0f;
  }
  __syncthreads();  // the candidate table
  int buf = 0;
  for (int jg = 0; jg < ng; ++jg) {
    const int j = jg * G;
    float acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = next[s];
    if (jg + 1 < ng) {
#pragma unroll
      for (int s = 0; s < NS; ++s) next[s] = live && on[s] ? Wr[j + G + l + LN * s] : 0.0f;
    }
    // earlier in-block updates, in column order
    for (int pg = 0; pg < jg; ++pg) {
      float e[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s)
        e[s] = pg == jg - 1 ? errs[s] : (live && on[s] ? Er[pg * G + l + LN * s] : 0.0f);
      lds_handover();
      stage(pg + 1, jg, buf ^ 1);
      const float* chunk = ubuf + buf * G * GP;
      // LN columns a turn; a slot's errors come to e[0] by turns
      float ring[kAhead][NS];
#pragma unroll
      for (int d = 0; d < kAhead; ++d) load_u(chunk, d < G ? d : G - 1, 0, ring[d]);
#pragma unroll 1
      for (int k0 = 0; k0 < G; k0 += LN) {
        static_for<LN>([&](auto oc) __attribute__((always_inline)) {
          constexpr int o = decltype(oc)::value;
          if (!FULL && k0 + o >= G) return;
          const float e1 = row_bcast<LN, o>(e[0]);
          float u[NS];
#pragma unroll
          for (int t = 0; t < NS; ++t) u[t] = ring[o % kAhead][t];
          load_u(chunk, k0 + o + kAhead < G ? k0 + o + kAhead : G - 1, 0, ring[o % kAhead]);
          asm volatile("" ::: "memory");  // the row stays fetched ahead
#pragma unroll
          for (int t = 0; t < NS; ++t) acc[t] = acc[t] - e1 * u[t];
        });
#pragma unroll
        for (int s = 0; s + 1 < NS; ++s) e[s] = e[s + 1];
      }
      buf ^= 1;
    }
    // clip search (grid.py:167-212) on the group's current values
    float s32, b32;
    clip_search<LN, NS, FULL, CS>(acc, on, tab, sh.n, maxq, storage, s32, b32);
    if (writes && l == 0) {
      store_storage(s_store, g_first + jg, s32, storage);
      store_storage(b_store, g_first + jg, b32, storage);
    }
    const float ss = safe_scale(s32), ys = div_exact_recip(ss);
    lds_handover();
    if (jg + 1 < ng) stage(0, jg + 1, buf ^ 1);
    const float* chunk = ubuf + buf * G * GP;
    // U's diagonal of the lane's columns and its reciprocals
    float dg[NS], yd[NS], acc0[NS];
    bool y_zero = !(ys != 0.0f);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      dg[s] = on[s] ? chunk[(l + LN * s) * (GP + 1)] : 1.0f;
      yd[s] = div_exact_recip(dg[s]);
      y_zero |= !(yd[s] != 0.0f);
      acc0[s] = acc[s];
    }
    float ring[kAhead][NS];
#pragma unroll
    for (int d = 0; d < kAhead; ++d) load_u(chunk, d < G ? d : G - 1, 0, ring[d]);
    static_for<NS>([&](auto sc) __attribute__((always_inline)) {
      static_for<LN>([&](auto oc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value, o = decltype(oc)::value;
        constexpr int c = s * LN + o, ca = c + kAhead;
        const int g = FULL ? G : opaque(G);
        if (!FULL && c >= g) return;
        float u[NS];
#pragma unroll
        for (int t = 0; t < NS; ++t) u[t] = ring[c % kAhead][t];
        if constexpr (ca < GP) load_u(chunk, FULL || ca < g ? ca : g - 1, ca / LN, ring[c % kAhead]);
        asm volatile("" ::: "memory");  // the row stays fetched ahead
        const float q =
            __builtin_amdgcn_fmed3f(rintf(div_fast(acc[s] - b32, ss, ys)), 0.0f, maxq);
        const float dq = q * s32 + b32;
        const float e1 = row_bcast<LN, o>(div_fast(acc[s] - dq, dg[s], yd[s]));
        if constexpr (o + 1 < LN) acc[s] = l > o ? acc[s] - e1 * u[s] : acc[s];
#pragma unroll
        for (int t = s + 1; t < NS; ++t) acc[t] = acc[t] - e1 * u[t];
      });
    });
    // each lane's codes, dequantized values and errors, from the values its
    // columns were quantized from (the operations of the column step)
    uint32_t tiny = 0xffffffffu;  // smallest nonzero numerator, as in clip_search
    float big = 0.0f;
    float qv[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const float n1 = acc[s] - b32;
      qv[s] = __builtin_amdgcn_fmed3f(rintf(div_fast(n1, ss, ys)), 0.0f, maxq);
      dv[s] = qv[s] * s32 + b32;
      const float n2 = acc[s] - dv[s];
      errs[s] = div_fast(n2, dg[s], yd[s]);
      const uint32_t m = min((f2u(n1) << 1) - 2u, (f2u(n2) << 1) - 2u);
      tiny = min(tiny, on[s] ? m : 0xffffffffu);
      // NaN (kept by the IEEE maximum) and inf fail the test below
      big = on[s] ? __builtin_elementwise_maximum(
                        big, __builtin_elementwise_maximum(fabsf(n1), fabsf(n2)))
                  : big;
    }
    const bool slow = y_zero | (tiny < (27u << 24) - 2u) | !(big < 0x1p101f);
    if (__builtin_amdgcn_ballot_w64(slow) != 0) {
#pragma unroll
      for (int s = 0; s < NS; ++s) acc[s] = acc0[s];
      static_for<NS>([&](auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
#pragma unroll 1
        for (int o = 0; o < LN && s * LN + o < G; ++o) {
          float u[NS];
          load_u(chunk, s * LN + o, s, u);
          const float q = affine_q_exact(acc[s], b32, ss, ys, maxq);
          const float e1 = __shfl(div_pos(acc[s] - (q * s32 + b32), dg[s], yd[s]), o, LN);
          acc[s] = l > o ? acc[s] - e1 * u[s] : acc[s];
#pragma unroll
          for (int t = s + 1; t < NS; ++t) acc[t] = acc[t] - e1 * u[t];
        }
      });
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        qv[s] = affine_q_exact(acc[s], b32, ss, ys, maxq);
        dv[s] = qv[s] * s32 + b32;
        errs[s] = div_pos(acc[s] - dv[s], dg[s], yd[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (!writes || !on[s]) continue;
      const int c = j + l + LN * s;
      qr[c] = (qv[s] == qv[s]) ? static_cast<uint8_t>(qv[s]) : 0;
      Wr[c] = dv[s];
      Er[c] = errs[s];
    }
    buf ^= 1;
  }
}

// W[row, i2 + m] -= sum_k Err[row, k] * U[b, i1 + k, i2 + m] (the reference's
// deferred bmm): 64x64 output tiles, each wave a 32x32 block on
// v_mfma_f32_32x32x2f32 (A[l%32][k], B[k][l%32] with k = l/32 per step; result
// register r of lane l = D[8(r/4) + 4(l/32) + r%4][l%32]). K goes in chunks of
// 64: the workgroup stages the chunk's Err rows and U columns (transposed) in
// LDS with 16-byte coalesced loads, then each lane reads four consecutive k
// of its Err row and of its U column with one 16-byte LDS read each; step t
// of an 8-k group takes k = group + 4(l/32) + t for both operands (the same
// permutation of k in every build of this kernel, so the sums round the same
// way). The tile's W values are loaded before the products and updated after
// them.
constexpr int kTm = 64, kTn = 64, kLzK = 64, kLzS = kLzK + 4;  // LDS row stride (floats)
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__global__ void __launch_bounds__(256)
    lazy_update_kernel(float* __restrict__ W, const float* __restrict__ U,
                       const float* __restrict__ Err, int64_t B, int64_t R, int64_t C,
                       int64_t ld_err, int64_t i1, int n, int64_t c1) {
  __shared__ __attribute__((aligned(16))) float sE[kTm][kLzS];  // Err[r0 + i][kc + k]
  __shared__ __attribute__((aligned(16))) float sU[kTn][kLzS];  // U[i1 + kc + k][m0 + j], as [j][k]
  const int64_t i2 = i1 + n;
  const int64_t b = blockIdx.z;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int64_t R0 = static_cast<int64_t>(blockIdx.y) * kTm;
  const int64_t M0 = i2 + static_cast<int64_t>(blockIdx.x) * kTn;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int li = lane & 31, g = lane >> 5;
  const int64_t m = M0 + wc + li;
  const bool mok = m < c1;
  // this lane's 16 outputs: rows R0 + wr + 8(i/4) + 4g + i%4, column m
  float wv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t rr = R0 + wr + 8 * (i >> 2) + 4 * g + (i & 3);
    wv[i] = (rr < R && mok) ? W[(b * R + rr) * C + m] : 0.0f;
  }
  const float* Eb = Err + b * R * ld_err;
  const float* Ub = U + b * C * C;
  // (Err and U themselves need not be 16-byte aligned)
  const bool vec = (n & 3) == 0 && (ld_err & 3) == 0 && (C & 3) == 0 && (i2 & 3) == 0;
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  for (int kc = 0; kc < n; kc += kLzK) {
    // stage: thread t copies 16-byte pieces (row t / 16 + 16 p, k or column 4 (t % 16))
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int rr = tid / 16 + 16 * p, c4 = 4 * (tid % 16);
      // Err rows
      {
        const int64_t row = R0 + rr;
        const int k = kc + c4;
        float v[4];
        if (vec && row < R && k + 4 <= n) {
          const auto q = load_f32x4(Eb + row * ld_err + k);
          v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = (row < R && k + t < n) ? Eb[row * ld_err + k + t] : 0.0f;
        }
        *reinterpret_cast<float4*>(&sE[rr][c4]) = float4{v[0], v[1], v[2], v[3]};
      }
      // U row i1 + kc + rr, columns M0 + c4 .. + 3, stored transposed
      {
        const int k = kc + rr;
        const int64_t col = M0 + c4;
        float v[4];
        if (vec && k < n && col + 4 <= C) {
          const auto q = load_f32x4(Ub + (i1 + k) * C + col);
          v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = (k < n && col + t < C) ? Ub[(i1 + k) * C + col + t] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) sU[c4 + t][rr] = v[t];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k8 = 0; k8 < kLzK; k8 += 8) {
      const float4 a = *reinterpret_cast<const float4*>(&sE[wr + li][k8 + 4 * g]);
      const float4 u = *reinterpret_cast<const float4*>(&sU[wc + li][k8 + 4 * g]);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, u.x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, u.y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, u.z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, u.w, acc, 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t rr = R0 + wr + 8 * (i >> 2) + 4 * g + (i & 3);
    if (rr < R && mok) W[(b * R + rr) * C + m] = wv[i] - acc[i];
  }
}

// The same update for `blocks` consecutive blocks of n columns at once (their
// errors in columns 0 .. blocks * n - 1 of Err, their U rows from i1 on), applied
// to columns [c0, c1): where every row piece is 16-byte aligned and n a multiple
// of 8. 64 x 64 output tiles, each wave a 32 x 32 quadrant. Chunks of 32 k of
// Err rows and U rows come to LDS by direct 16-byte loads, one chunk ahead
// (two buffers; the compiler cannot tell them apart and waits for the loads
// before the reads of the present chunk, so they run beside the products of the
// CU's other workgroups), from a scalar base that moves along k plus fixed lane
// offsets. The 16-byte pieces of an Err row are permuted by the row index (the
// reads of 32 rows at one k then fall on distinct banks); U is read as it lies,
// four 4-byte reads per column and 8 k. A block's products run in
// lazy_update_kernel's order and are subtracted from W block by block, so
// the result has the bits of one launch per block, with one read and one write
// of W for all of them.
// Bound by the fp32 MFMA rate (153 TFLOP/s for a large library product here; the
// matrix pipe is 61 to 69 % busy with many columns left).
// 64 x 64 tiles keep four workgroups on a CU, so one's loads run beside the
// others' products; 128 x 128 tiles (one workgroup) were slower at every size.
// One block of 128 columns: 32 x 1536 rows, 1920 columns left 421 -> 311 us,
// 14336 rows, 3968 left 204 -> 164 us, 2048 rows, 128 left 9.8 -> 7 us against
// lazy_update_kernel. The whole column loop with a launch per block / with up
// to four blocks at once: 32 x 1536 x 2048 4.31 / 3.84 ms, 14336 x 4096 4.09 /
// 3.59 ms, 2048 x 2048 0.485 / 0.462 ms.
__global__ void __launch_bounds__(256)
    lazy_update_tiles_kernel(float* __restrict__ W, const float* __restrict__ U,
                             const float* __restrict__ Err, int64_t R, int64_t C, int64_t ld_err,
                             int64_t i1, int n, int blocks, int64_t c0, int64_t c1) {
  constexpr int T = 64, kKc = 32;
  constexpr int kPieces = kKc / 4;     // 16-byte pieces of an Err row per chunk
  constexpr int kCols = T / 4;         // 16-byte pieces of a U row of the tile
  constexpr int kPass = T * kKc / (4 * 256);  // 16-byte loads per thread, operand and chunk
  __shared__ __attribute__((aligned(16))) float sE[2][T * kKc];  // [row][piece ^ row]
  __shared__ __attribute__((aligned(16))) float sU[2][kKc * T];  // [k][column]
  const int64_t b = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t R0 = static_cast<int64_t>(blockIdx.y) * T;
  const int64_t M0 = c0 + static_cast<int64_t>(blockIdx.x) * T;
  const int wr = (wave >> 1) * (T / 2), wc = (wave & 1) * (T / 2);
  const int li = lane & 31, g = lane >> 5;

  // Byte offsets of this lane's loads from the chunk's corner of Err and U.
  // Rows past R and columns past C load the last ones (they are not stored).
  const char* Ec = reinterpret_cast<const char*>(Err + (b * R + R0) * ld_err);
  const char* Uc = reinterpret_cast<const char*>(U + (b * C + i1) * C + M0);
  const int piece_l = (lane % kPieces) ^ (lane / kPieces);
  uint32_t eoff[kPass], uoff[kPass];
#pragma unroll
  for (int p = 0; p < kPass; ++p) {
    const int rr = p * (256 / kPieces) + wave * (64 / kPieces) + lane / kPieces;
    eoff[p] = static_cast<uint32_t>(
        4 * ((R0 + rr < R ? rr : static_cast<int>(R - 1 - R0)) * ld_err + 4 * piece_l));
    const int kk = p * (256 / kCols) + wave * (64 / kCols) + lane / kCols;
    const int64_t c4 = 4 * (lane % kCols);
    uoff[p] = static_cast<uint32_t>(4 * (kk * C + (M0 + c4 + 4 <= C ? c4 : C - 4 - M0)));
  }
  auto load = [&](const char* base, uint32_t off, float* dst) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((global_cv*)(base + off), (lds_v*)dst, 16, 0, 0);
  };
  // chunk [kc, kc + 32) of the block that starts at column k0
  auto stage = [&](int k0, int kc, int buf) __attribute__((always_inline)) {
    const char* eb = Ec + static_cast<int64_t>(k0 + kc) * 4;
    const char* ub = Uc + static_cast<int64_t>(k0 + kc) * C * 4;
    // past the block's end (its last chunk of 8, 16 or 24 k) the loads repeat
    // earlier ones
    const int eback = kc + 4 * piece_l < n ? 0 : kc + 4 * piece_l - (n - 4);
#pragma unroll
    for (int p = 0; p < kPass; ++p) {
      load(eb, eoff[p] - 4 * eback, sE[buf] + 256 * (4 * p + wave));
      const int kk = kc + p * (256 / kCols) + wave * (64 / kCols) + lane / kCols;
      load(ub, uoff[p] - (kk < n ? 0u : static_cast<uint32_t>(4 * (kk - (n - 1)) * C)),
           sU[buf] + 256 * (4 * p + wave));
    }
  };
  stage(0, 0, 0);
  // this lane's outputs: rows .. + 8(i/4) + 4g + i%4, column li
  float* Wt = W + (b * R + R0) * C + M0;
  const bool inner = R0 + T <= R && M0 + T <= c1;  // uniform
  float wv[16];
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int rr = wr + 8 * (i >> 2) + 4 * g + (i & 3), m = wc + li;
    wv[i] = inner || (R0 + rr < R && M0 + m < c1) ? Wt[rr * C + m] : 0.0f;
    acc[i] = 0.0f;
  }
  const float* re[4];  // Err pieces 2j + g of this lane's row
#pragma unroll
  for (int j = 0; j < 4; ++j) re[j] = sE[0] + (wr + li) * kKc + 4 * ((2 * j + g) ^ (li % kPieces));
  const float* ru = sU[0] + 4 * g * T + wc + li;
  int k0 = 0, kc = 0;
  // one chunk; returns false after the last one
  auto step = [&](int buf) __attribute__((always_inline)) -> bool {
    lds_handover();
    __builtin_amdgcn_sched_barrier(0);
    const bool last = kc + kKc >= n;  // of its block
    const int k0n = last ? k0 + n : k0, kcn = last ? 0 : kc + kKc;
    const bool more = k0n < blocks * n;
    if (more) stage(k0n, kcn, buf ^ 1);  // every wave has left that buffer
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > 0 && kc + 8 * j >= n) break;  // uniform
      const float4 a = *reinterpret_cast<const float4*>(re[j] + buf * T * kKc);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float v = ru[buf * kKc * T + (8 * j + t) * T];
        const float at = t == 0 ? a.x : t == 1 ? a.y : t == 2 ? a.z : a.w;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(at, v, acc, 0, 0, 0);
      }
    }
    if (last) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        wv[i] = wv[i] - acc[i];
        acc[i] = 0.0f;
      }
    }
    k0 = k0n, kc = kcn;
    return more;
  };
  while (step(0) && step(1)) {
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int rr = wr + 8 * (i >> 2) + 4 * g + (i & 3), m = wc + li;
    if (inner || (R0 + rr < R && M0 + m < c1)) Wt[rr * C + m] = wv[i];
  }
}

}  // namespace
}  // namespace mgq

using namespace mgq;

extern "C" int mgq_dead_fix(float* W, int64_t B, int64_t R, int64_t C, float* H, void* stream) {
  clear_error();
  MGQ_REQUIRE(B >= 0 && R >= 0 && C >= 0, MGQ_ERR_SHAPE, "bad shape");
  if (B * C == 0) return MGQ_OK;
  hipStream_t s = as_stream(stream);
  if (W != nullptr && R > 0) {
    for (int64_t b0 = 0; b0 < B; b0 += 65535) {  // the grid's depth
      const int64_t nb = B - b0 < 65535 ? B - b0 : 65535;
      // A thread's column is one chain of stores: rows are split until every CU
      // has two workgroups. One matrix of 2048 x 2048, 1 % of the columns dead: 31
      // us with 1024 rows a workgroup, now 6.1 (all of them dead 28.6, now 7.4);
      // none dead, 14336 x 4096: 4.1 us, now 4.4 (finer splits up to 11).
      int64_t rows = 1024;
      while (rows > 16 && ceil_div(C, 256) * ceil_div(R, rows) * nb < 512) rows /= 2;
      const dim3 grid(static_cast<unsigned>(ceil_div(C, 256)),
                      static_cast<unsigned>(ceil_div(R, rows)), static_cast<unsigned>(nb));
      dead_fix_w_kernel<<<grid, 256, 0, s>>>(W + b0 * R * C, H + b0 * C * C, R, C, rows);
    }
    if (int rc = check_launch("dead fix W")) return rc;
  }
  dead_fix_h_kernel<<<elementwise_blocks(B * C, 256), 256, 0, s>>>(H, B, C);
  return check_launch("dead fix H");
}

namespace mgq {
namespace {

struct AffineArgs {
  float* W;
  const float* U;
  int64_t B, R, C;
  int group_size, bits, method, storage_dtype, grid_steps;
  double max_shrink;
  uint8_t* q_out;
  void* s_store;
  void* b_store;
};

int check_affine(const AffineArgs& a, Shrinks* sh) {
  MGQ_REQUIRE(a.bits >= 1 && a.bits <= 8, MGQ_ERR_VALUE, "unsupported bits: %d", a.bits);
  MGQ_REQUIRE(a.group_size >= 1 && a.group_size <= 128, MGQ_ERR_VALUE,
              "group size %d unsupported (1..128)", a.group_size);
  MGQ_REQUIRE(a.storage_dtype == kF32 || a.storage_dtype == kBF16 || a.storage_dtype == kF16,
              MGQ_ERR_VALUE, "bad storage dtype");
  MGQ_REQUIRE(a.method == MGQ_CLIP_MINMAX || a.method == MGQ_CLIP_MSE, MGQ_ERR_VALUE,
              "unsupported clip method %d", a.method);
  return make_shrinks(a.bits, a.method, a.grid_steps, a.max_shrink, sh);
}

int check_block(const AffineArgs& a, int64_t i1, int64_t n) {
  MGQ_REQUIRE(a.C % a.group_size == 0 && i1 % a.group_size == 0 && n % a.group_size == 0 &&
                  n >= 1 && n <= kMaxBlock && i1 + n <= a.C,
              MGQ_ERR_SHAPE, "bad block [%lld, %lld) for C=%lld, G=%d", (long long)i1,
              (long long)(i1 + n), (long long)a.C, a.group_size);
  return MGQ_OK;
}

// The same with a wave per row.
int launch_wave(const AffineArgs& a, const Shrinks& sh, int64_t i1, int64_t n, float* Err,
                int64_t ld_err, hipStream_t s) {
  const int G = a.group_size;
  const float maxq = static_cast<float>((1 << a.bits) - 1);
  const bool ldsu = n <= kLdsBlock;
  const size_t lds = sizeof(float) * (2 * kMaxShrinks + kWaves * 4 * (G > 64 ? G : 64) +
                                      kWaves * static_cast<size_t>(n) +
                                      (ldsu ? static_cast<size_t>(n) * n : 0));
  const dim3 blocks(static_cast<unsigned>(ceil_div(a.R, kWaves)), static_cast<unsigned>(a.B));
  auto kernel = G <= 64 ? (ldsu ? affine_wave_kernel<1, true> : affine_wave_kernel<1, false>)
                        : (ldsu ? affine_wave_kernel<2, true> : affine_wave_kernel<2, false>);
  kernel<<<blocks, kWaves * 64, lds, s>>>(a.W, a.U, a.B, a.R, a.C, i1, static_cast<int>(n), G, maxq,
                                          a.storage_dtype, sh, a.q_out, a.s_store, a.b_store, Err,
                                          ld_err);
  return check_launch("affine block");
}

// The column loop of block [i1, i1 + n), its errors to Err (row stride ld_err).
int launch_block(const AffineArgs& a, const Shrinks& sh, int64_t i1, int64_t n, float* Err,
                 int64_t ld_err, hipStream_t s) {
  const int64_t B = a.B, R = a.R;
  const int G = a.group_size;
  const float maxq = static_cast<float>((1 << a.bits) - 1);
  const int full = G == 32 || G == 64 || G == 128 ? G : 0;
  const bool quad = (full == 32 || full == 64) && B * R >= quad_rows(G);
  const int64_t rows4 = B * ceil_div(R, 4);
  if (!full && rows4 <= wave_rows(G, n)) return launch_wave(a, sh, i1, n, Err, ld_err, s);
  const int cs = !full || quad ? 1 : rows4 <= kSplit4 ? 4 : rows4 <= kSplit2 ? 2 : 1;
  const int rw = quad ? 16 : 4 / cs;
  const int64_t waves = B * ceil_div(R, rw);
  // few waves: small workgroups, so that every CU gets one; many: large ones,
  // so that more rows share a chunk of U
  const int wg = waves < 1024 ? 2 : waves < 2048 ? 4 : kMaxWaves;
  const int gp = G <= 16 ? 16 : G <= 32 ? 32 : G <= 64 ? 64 : 128;
  const size_t lds =
      sizeof(float) * (2 * kMaxShrinks + (n > G ? 2 : 1) * static_cast<size_t>(G) * gp);
  const bool wide = full && (reinterpret_cast<uintptr_t>(a.U) & 15u) == 0;
  const dim3 blocks(static_cast<unsigned>(ceil_div(R, static_cast<int64_t>(wg) * rw)),
                    static_cast<unsigned>(B));
#define AFFINE_LAUNCH(LN_, NS_, FULL_, CS_)                                                   \
  affine_block_kernel<LN_, NS_, FULL_, CS_><<<blocks, wg * 64, lds, s>>>(                     \
      a.W, a.U, R, a.C, i1, static_cast<int>(n), G, maxq, a.storage_dtype, sh, wide, a.q_out, \
      a.s_store, a.b_store, Err, ld_err)
#define AFFINE_SPLIT(NS_)                             \
  do {                                                \
    if (cs == 4) AFFINE_LAUNCH(16, NS_, true, 4);     \
    else if (cs == 2) AFFINE_LAUNCH(16, NS_, true, 2); \
    else AFFINE_LAUNCH(16, NS_, true, 1);             \
  } while (0)
  if (quad && full == 32) AFFINE_LAUNCH(4, 8, true, 1);
  else if (quad) AFFINE_LAUNCH(4, 16, true, 1);
  else if (full == 32) AFFINE_SPLIT(2);
  else if (full == 64) AFFINE_SPLIT(4);
  else if (full == 128) AFFINE_SPLIT(8);
  else if (G <= 16) AFFINE_LAUNCH(16, 1, false, 1);
  else if (G < 32) AFFINE_LAUNCH(16, 2, false, 1);
  else if (G < 64) AFFINE_LAUNCH(16, 4, false, 1);
  else AFFINE_LAUNCH(16, 8, false, 1);
#undef AFFINE_SPLIT
#undef AFFINE_LAUNCH
  return check_launch("affine block");
}

// Whether lazy_update_tiles_kernel takes these updates.
bool lazy_pieces(const AffineArgs& a, int64_t i1, int64_t n, const float* Err, int64_t ld_err) {
  return n % 8 == 0 && a.C % 4 == 0 && i1 % 4 == 0 && ld_err % 4 == 0 &&
         ((reinterpret_cast<uintptr_t>(a.U) | reinterpret_cast<uintptr_t>(Err)) & 15u) == 0;
}

// Columns [c0, c1) of W after `blocks` blocks of n columns from i1 on, their
// errors in Err's first columns.
int launch_lazy(const AffineArgs& a, int64_t i1, int64_t n, int64_t blocks, int64_t c0, int64_t c1,
                const float* Err, int64_t ld_err, hipStream_t s) {
  if (c0 >= c1) return MGQ_OK;
  const dim3 grid(static_cast<unsigned>(ceil_div(c1 - c0, 64)),
                  static_cast<unsigned>(ceil_div(a.R, 64)), static_cast<unsigned>(a.B));
  static_assert(kTm == 64 && kTn == 64, "one grid for both kernels");
  if (lazy_pieces(a, i1, n, Err, ld_err))
    lazy_update_tiles_kernel<<<grid, 256, 0, s>>>(a.W, a.U, Err, a.R, a.C, ld_err, i1,
                                                  static_cast<int>(n), static_cast<int>(blocks),
                                                  c0, c1);
  else  // one block, the columns right after it
    lazy_update_kernel<<<grid, 256, 0, s>>>(a.W, a.U, Err, a.B, a.R, a.C, ld_err, i1,
                                            static_cast<int>(n), c1);
  return check_launch("affine lazy update");
}

}  // namespace
}  // namespace mgq

extern "C" int mgq_gptq_affine_block(float* W, const float* U, int64_t B, int64_t R, int64_t C,
                                     int64_t i1, int64_t n, int group_size, int bits, int method,
                                     int storage_dtype, int grid_steps, double max_shrink,
                                     uint8_t* q_out, void* s_store, void* b_store, float* Err,
                                     void* stream) {
  clear_error();
  const AffineArgs a{W,      U,             B,          R,          C,     group_size, bits,
                     method, storage_dtype, grid_steps, max_shrink, q_out, s_store,    b_store};
  Shrinks sh;
  if (int rc = check_affine(a, &sh)) return rc;
  if (int rc = check_block(a, i1, n)) return rc;
  if (B * R == 0) return MGQ_OK;
  hipStream_t s = as_stream(stream);
  if (int rc = launch_block(a, sh, i1, n, Err, n, s)) return rc;
  return launch_lazy(a, i1, n, 1, i1 + n, C, Err, n, s);
}

// Every block of the column loop. Err holds the errors of err_cols / block
// blocks: those blocks update only the columns up to the last of them, one by
// one, and the columns beyond are updated once for all of them
// (lazy_update_tiles_kernel), which reads and writes W once instead of once
// per block; the bits are those of one full update per block.
extern "C" int mgq_gptq_affine(float* W, const float* U, int64_t B, int64_t R, int64_t C,
                               int64_t block, int group_size, int bits, int method,
                               int storage_dtype, int grid_steps, double max_shrink,
                               uint8_t* q_out, void* s_store, void* b_store, float* Err,
                               int64_t err_cols, void* stream) {
  clear_error();
  const AffineArgs a{W,      U,             B,          R,          C,     group_size, bits,
                     method, storage_dtype, grid_steps, max_shrink, q_out, s_store,    b_store};
  Shrinks sh;
  if (int rc = check_affine(a, &sh)) return rc;
  const int64_t bs = block < C ? block : C;
  if (int rc = check_block(a, 0, bs)) return rc;
  MGQ_REQUIRE(err_cols >= bs, MGQ_ERR_WORKSPACE, "Err holds %lld columns, a block %lld",
              (long long)err_cols, (long long)bs);
  if (B * R == 0) return MGQ_OK;
  hipStream_t s = as_stream(stream);
  // the deferred update of several blocks needs the piecewise kernel
  const int64_t span = lazy_pieces(a, bs, bs, Err, err_cols) ? err_cols / bs * bs : bs;
  for (int64_t s0 = 0; s0 < C; s0 += span) {
    const int64_t s1 = s0 + span < C ? s0 + span : C;
    for (int64_t i1 = s0; i1 < s1; i1 += bs) {
      const int64_t n = i1 + bs < C ? bs : C - i1;
      float* E = Err + (i1 - s0);
      if (int rc = launch_block(a, sh, i1, n, E, err_cols, s)) return rc;
      if (int rc = launch_lazy(a, i1, n, 1, i1 + n, s1, E, err_cols, s)) return rc;
    }
    if (int rc = launch_lazy(a, s0, bs, (s1 - s0) / bs, s1, C, Err, err_cols, s)) return rc;
  }
  return MGQ_OK;
}
