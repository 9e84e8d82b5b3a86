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
// (the reference's bmm) as an fp32 GEMM.
#include "affine_clip.h"
#include "mgq_capi.h"
#include "mgq_common.h"
#include "mx_hw.h"

namespace mgq {
namespace {

constexpr int kMaxBlock = 2048;
constexpr int kMaxWaves = 8;
// Where the variants of affine_block_kernel start and end (us per block of
// 128 columns; rows over all items):
//   - a quad per row from kQuadRows: 49152 rows 137 (G = 64) and 137 (G = 32)
//     against 116 and 147 with a DPP row, 196608 rows 380 and 300 against 450
//     and 467;
//   - four parts of the clip candidates up to kSplit4 waves of four rows, two
//     up to kSplit2, G = 64: 512 rows 14.2 / 14.7 / 17.0 (four, two, one),
//     2048 rows 21.4 / 18.3 / 19.8, 4096 rows 32.6 / 22.9 / 21.0.
constexpr int64_t kQuadRows = 98304;
constexpr int64_t kSplit4 = 256, kSplit2 = 768;

// gptq.py:216-222 for the affine path: dead columns zeroed in W, H diag := 1.
__global__ void dead_fix_w_kernel(float* __restrict__ W, float* __restrict__ H, int64_t B,
                                  int64_t R, int64_t C) {
  const int64_t n = B * R * C;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / (R * C), c = i % C;
    if (H[b * C * C + c * C + c] <= 0.0f) W[i] = 0.0f;
  }
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
// run again from its start values with guarded divisions (EXACT): every
// quotient is the correctly rounded one either way.
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
                        float* __restrict__ Err) {
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
  float* Er = Err + row * n;
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
  // this wave's loads of the next chunk have landed, and so have the others'
  auto chunk_ready = [&]() {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
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
      chunk_ready();
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
    chunk_ready();
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
                       const float* __restrict__ Err, int64_t B, int64_t R, int64_t C, int64_t i1,
                       int n) {
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
  const bool mok = m < C;
  // this lane's 16 outputs: rows R0 + wr + 8(i/4) + 4g + i%4, column m
  float wv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t rr = R0 + wr + 8 * (i >> 2) + 4 * g + (i & 3);
    wv[i] = (rr < R && mok) ? W[(b * R + rr) * C + m] : 0.0f;
  }
  const float* Eb = Err + b * R * n;
  const float* Ub = U + b * C * C;
  const bool vec = (n & 3) == 0 && (C & 3) == 0 && (i2 & 3) == 0;
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
          const float4 q = *reinterpret_cast<const float4*>(Eb + row * n + k);
          v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = (row < R && k + t < n) ? Eb[row * n + k + t] : 0.0f;
        }
        *reinterpret_cast<float4*>(&sE[rr][c4]) = float4{v[0], v[1], v[2], v[3]};
      }
      // U row i1 + kc + rr, columns M0 + c4 .. + 3, stored transposed
      {
        const int k = kc + rr;
        const int64_t col = M0 + c4;
        float v[4];
        if (vec && k < n && col + 4 <= C) {
          const float4 q = *reinterpret_cast<const float4*>(Ub + (i1 + k) * C + col);
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

int make_shrinks(int bits, int method, int grid_steps, double max_shrink, Shrinks* out) {
  out->maxq = static_cast<double>((1 << bits) - 1);
  if (method == MGQ_CLIP_MINMAX) {
    out->n = out->steps = 1;
    out->max_shrink = 0.0;
    return MGQ_OK;
  }
  MGQ_REQUIRE(grid_steps >= 1 && grid_steps < kMaxShrinks - 4, MGQ_ERR_VALUE,
              "grid_steps must be in [1, %d)", kMaxShrinks - 4);
  out->n = grid_steps + 1;
  out->steps = grid_steps;
  out->max_shrink = max_shrink;
  return MGQ_OK;
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
    dead_fix_w_kernel<<<elementwise_blocks(B * R * C, 256), 256, 0, s>>>(W, H, B, R, C);
    if (int rc = check_launch("dead fix W")) return rc;
  }
  dead_fix_h_kernel<<<elementwise_blocks(B * C, 256), 256, 0, s>>>(H, B, C);
  return check_launch("dead fix H");
}

extern "C" int mgq_gptq_affine_block(float* W, const float* U, int64_t B, int64_t R, int64_t C,
                                     int64_t i1, int64_t n, int group_size, int bits, int method,
                                     int storage_dtype, int grid_steps, double max_shrink,
                                     uint8_t* q_out, void* s_store, void* b_store, float* Err,
                                     void* stream) {
  clear_error();
  MGQ_REQUIRE(bits >= 1 && bits <= 8, MGQ_ERR_VALUE, "unsupported bits: %d", bits);
  MGQ_REQUIRE(group_size >= 1 && group_size <= 128, MGQ_ERR_VALUE,
              "group size %d unsupported (1..128)", group_size);
  MGQ_REQUIRE(storage_dtype == kF32 || storage_dtype == kBF16 || storage_dtype == kF16,
              MGQ_ERR_VALUE, "bad storage dtype");
  MGQ_REQUIRE(method == MGQ_CLIP_MINMAX || method == MGQ_CLIP_MSE, MGQ_ERR_VALUE,
              "unsupported clip method %d", method);
  MGQ_REQUIRE(C % group_size == 0 && i1 % group_size == 0 && n % group_size == 0 &&
                  n >= 1 && n <= kMaxBlock && i1 + n <= C,
              MGQ_ERR_SHAPE, "bad block [%lld, %lld) for C=%lld, G=%d", (long long)i1,
              (long long)(i1 + n), (long long)C, group_size);
  Shrinks sh;
  if (int rc = make_shrinks(bits, method, grid_steps, max_shrink, &sh)) return rc;
  if (B * R == 0) return MGQ_OK;
  hipStream_t s = as_stream(stream);
  const float maxq = static_cast<float>((1 << bits) - 1);
  const int full = group_size == 32 || group_size == 64 || group_size == 128 ? group_size : 0;
  const bool quad = (full == 32 || full == 64) && B * R >= kQuadRows;
  const int64_t rows4 = B * ceil_div(R, 4);
  const int cs = !full || quad ? 1 : rows4 <= kSplit4 ? 4 : rows4 <= kSplit2 ? 2 : 1;
  const int rw = quad ? 16 : 4 / cs;
  const int64_t waves = B * ceil_div(R, rw);
  // few waves: small workgroups, so that every CU gets one; many: large ones,
  // so that more rows share a chunk of U
  const int wg = waves < 1024 ? 2 : waves < 2048 ? 4 : kMaxWaves;
  const int gp = group_size <= 16 ? 16 : group_size <= 32 ? 32 : group_size <= 64 ? 64 : 128;
  const size_t lds = sizeof(float) * (2 * kMaxShrinks + (n > group_size ? 2 : 1) *
                                                            static_cast<size_t>(group_size) * gp);
  const bool wide = full && (reinterpret_cast<uintptr_t>(U) & 15u) == 0;
  const dim3 blocks(static_cast<unsigned>(ceil_div(R, static_cast<int64_t>(wg) * rw)),
                    static_cast<unsigned>(B));
#define AFFINE_LAUNCH(LN_, NS_, FULL_, CS_)                                                  \
  affine_block_kernel<LN_, NS_, FULL_, CS_><<<blocks, wg * 64, lds, s>>>(                    \
      W, U, R, C, i1, static_cast<int>(n), group_size, maxq, storage_dtype, sh, wide, q_out, \
      s_store, b_store, Err)
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
  else if (group_size <= 16) AFFINE_LAUNCH(16, 1, false, 1);
  else if (group_size < 32) AFFINE_LAUNCH(16, 2, false, 1);
  else if (group_size < 64) AFFINE_LAUNCH(16, 4, false, 1);
  else AFFINE_LAUNCH(16, 8, false, 1);
#undef AFFINE_SPLIT
#undef AFFINE_LAUNCH
  if (int rc = check_launch("affine block")) return rc;
  if (i1 + n < C) {
    dim3 grid(static_cast<unsigned>(ceil_div(C - i1 - n, kTn)),
              static_cast<unsigned>(ceil_div(R, kTm)), static_cast<unsigned>(B));
    lazy_update_kernel<<<grid, 256, 0, s>>>(W, U, Err, B, R, C, i1, static_cast<int>(n));
    if (int rc = check_launch("affine lazy update")) return rc;
  }
  return MGQ_OK;
}
