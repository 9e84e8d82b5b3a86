// Full-matrix damped Cholesky-inverse upper factor (gptq.py:27-66 for the
// affine solver, which factors the whole [C, C] Hessian).
//
//   U (upper) with U^T U = (H + lam I)^-1,  lam = damp * max(mean(diag H), 1e-8)
//
// As in the 32x32 kernel, Hd = V V^T is factored with V upper triangular
// ("UL" Cholesky, i.e. Cholesky in reverse index order) and U = V^-1 = W.
// The factor and its inverse are built together by recursion over 64-row
// blocks [b0, b1), split at mid (top rows T = [b0, mid), bottom rows
// S = [mid, b1)):
//   1. (V_SS, W_SS) of A_SS                          (recursion, bottom first)
//   2. P = V_TS = A_TS W_SS^T                        (GEMM)
//   3. A_TT -= P P^T                                 (GEMM, upper tiles)
//   4. Q = P W_SS                                    (GEMM)
//   5. (V_TT, W_TT) of the updated A_TT              (recursion)
//   6. W_TS = -W_TT Q                                (GEMM)
// since V V^T = [[V_TT V_TT^T + V_TS V_TS^T, V_TS V_SS^T], [., V_SS V_SS^T]]
// and V^-1 = [[W_TT, -W_TT V_TS W_SS], [0, W_SS]]. A 64x64 leaf is factored
// and inverted by one workgroup. Everything runs
// in fp64 (the factor of an fp32 matrix, rounded to fp32 once). The sums of
// 2, 4 and 6 leave out the zero part of their triangular factor (4 h^3
// operations per node of edge 2h instead of 7 h^3), so nothing below the block
// diagonal is ever read and W needs no clearing. Items whose
// pivot fails are flagged and skipped by later steps; the host escalates
// their damping and reruns them, exactly like the reference retries only the
// failed batch items.
#include <algorithm>

#include "mgq_capi.h"
#include "mgq_common.h"

namespace mgq {
namespace {

constexpr int kNb = 64;  // leaf block

typedef double f64x2_t __attribute__((ext_vector_type(2)));

// lam[b] = fp32(max(mean(diag H_b), 1e-8) * damp[b]): fp64 diagonal sum
// rounded once, then the reference's fp32 clamp and product.
__global__ void __launch_bounds__(256)
    lam_kernel(const float* __restrict__ H, int64_t C, const float* __restrict__ damp,
               const uint8_t* __restrict__ active, float* __restrict__ lam) {
  const int64_t b = blockIdx.x;
  if (!active[b]) return;
  __shared__ double part[256];
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < C; i += 256) s += static_cast<double>(H[b * C * C + i * C + i]);
  part[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float dm = static_cast<float>(part[0] / static_cast<double>(C));
    dm = dm < 1e-8f ? 1e-8f : dm;  // NaN stays NaN
    lam[b] = dm * damp[b];
  }
}

// A = fp64(H + lam I) (diagonal added in fp32, as the reference forms Hd),
// from the start of each row's diagonal 64-block on: the recursion reads no
// block below the block diagonal, of A or of W. One wave per row.
__global__ void __launch_bounds__(256)
    build_kernel(const float* __restrict__ H, int64_t C, int64_t ld, const float* __restrict__ lam,
                 const uint8_t* __restrict__ active, double* __restrict__ A) {
  const int64_t b = blockIdx.y;
  if (!active[b]) return;
  const int64_t i = blockIdx.x * int64_t{4} + (threadIdx.x >> 6);
  if (i >= C) return;
  const float l = lam[b];
  const float* Hr = H + (b * C + i) * C;
  double* Ar = A + (b * C + i) * ld;
  for (int64_t k = i / kNb * kNb + (threadIdx.x & 63); k < C; k += 64) {
    const float v = Hr[k];
    Ar[k] = static_cast<double>(k == i ? v + l : v);
  }
}

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// x of lane J of this lane's row of 16
template <int J>
__device__ inline double row_lane(double x) {
  constexpr int kRowNewbcast = 0x150;
  const int64_t v = __builtin_bit_cast(int64_t, x);
  const int64_t r = __builtin_amdgcn_update_dpp(int64_t{0}, v, kRowNewbcast + J, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}

// Orders one wave's own LDS accesses across its lanes.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Leaf: W = V^-1 for the n x n (n <= 64) diagonal block A_b = V V^T at r0
// (V upper). One workgroup of four waves per batch item. The block is taken
// with its indices reversed (i -> 63 - i), where V is a lower factor L and
// W its inverse X, and goes by 16 x 16 blocks through LDS. For block column k:
//   wave 0:     L_kk and X_kk of the updated A_kk, in registers;
//   waves 1-3:  L_ik = A_ik X_kk^T (i > k) and X_kj = -X_kk R_kj (j < k);
//   waves 1-3:  A_ij -= L_ik L_jk^T (i >= j > k), R_ij += L_ik X_kj (j <= k < i),
//               while wave 0 updates A_k+1,k+1 itself and goes on to factor it,
// the products on fp64 MFMA. In the 16 x 16 factor lane (g, i) (four rows g of
// 16 lanes) holds row i of A, the same in every g, and columns 4m + g of row i
// of the inverse, at first the identity. The sweep over j does the factor step
// and the Gauss-Jordan step of the inverse at once: with row j of both, a
// (broadcast by DPP from lane j), d = a_j and c_i = A[i][j] / d, every row i > j
// loses c_i a; at the end row i is scaled by 1 / sqrt(d_i).
// A serial chain on one CU: the 64 factor steps take 4.8 us of 14.2 us (one wave,
// some 30 instructions each), the rest is the latency of loads, products and
// barriers. 16.7 us with the whole 64 x 64 block in the registers of four waves,
// two steps per LDS exchange and barrier.
// Only the lower triangle of the block is read; rows past n are identity
// padding. A pivot <= 0 or NaN flags the item as failed.
constexpr int kLeafLd = kNb + 2;  // 16 rows x 4 columns of fp64 fall on distinct banks

struct Leaf {
  double s[kNb * kLeafLd];  // A, then L
  double x[kNb * kLeafLd];  // R, then X (lower blocks only)
  int ok;
};

// the 16 x 16 factor and inverse of block k (one wave); false if a pivot fails
__device__ inline bool leaf_factor(Leaf& w, int k) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const double* S = w.s + 16 * k * (kLeafLd + 1);
  double A[16], X[4];
#pragma unroll
  for (int c = 0; c < 16; ++c) A[c] = S[(i > c ? i : c) * kLeafLd + (i > c ? c : i)];
#pragma unroll
  for (int m = 0; m < 4; ++m) X[m] = 4 * m + g == i ? 1.0 : 0.0;
  double piv = 1.0;
  bool ok = true;
  static_for<16>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    const double d = row_lane<j>(A[j]);
    ok = ok & (d > 0.0);
    piv = i == j ? d : piv;
    const double q = A[j] * recip_f64(d);
    const double c = i > j ? q : 0.0;
#pragma unroll
    for (int n = j + 1; n < 16; ++n) A[n] = fma(-c, row_lane<j>(A[n]), A[n]);
#pragma unroll
    for (int m = 0; m <= j / 4; ++m) X[m] = fma(-c, row_lane<j>(X[m]), X[m]);
  });
  const double rs = 1.0 / sqrt(piv);
  double* out = w.x + 16 * k * (kLeafLd + 1) + i * kLeafLd + g;
#pragma unroll
  for (int m = 0; m < 4; ++m) out[4 * m] = X[m] * rs;
  return ok;
}

// acc + a * b over 16: a read by rows from `a`, b by rows (B^T stored) or
// by columns from `b`; both point at a 16 x 16 block
template <bool TRANSB>
__device__ inline f64x4_t leaf_product(const double* a, const double* b, f64x4_t acc) {
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
#pragma unroll
  for (int t = 0; t < 4; ++t)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
        a[li * kLeafLd + 4 * t + q],
        TRANSB ? b[li * kLeafLd + 4 * t + q] : b[(4 * t + q) * kLeafLd + li], acc, 0, 0, 0);
  return acc;
}

// the result layout of leaf_product: register r is row l / 16 + 4r, column l % 16
__device__ inline f64x4_t leaf_load(const double* c) {
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
  f64x4_t v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = c[(q + 4 * r) * kLeafLd + li];
  return v;
}

__device__ inline void leaf_store(double* c, f64x4_t v) {
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) c[(q + 4 * r) * kLeafLd + li] = v[r];
}

__global__ void __launch_bounds__(256)
    leaf_kernel(const double* __restrict__ A, double* __restrict__ W, int64_t C, int64_t ld,
                int64_t r0, int n,
                const uint8_t* __restrict__ active, uint8_t* __restrict__ failed) {
  const int64_t b = blockIdx.x;
  __shared__ __attribute__((aligned(16))) Leaf w;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const double* Ab = A + (b * C + r0) * ld + r0;
  const bool skip = !active[b] || failed[b];  // uniform; the loads need not wait for it
  {
    double v[kNb / 4];
#pragma unroll
    for (int p = 0; p < kNb / 4; ++p) {
      const int r = 4 * p + wave;  // rows and columns past n: identity
      v[p] = r < n && lane <= r ? Ab[r * ld + lane] : (r == lane ? 1.0 : 0.0);
    }
    if (skip) return;
#pragma unroll
    for (int p = 0; p < kNb / 4; ++p) {
      const int r = 4 * p + wave;
      if (lane <= r) w.s[(kNb - 1 - lane) * kLeafLd + kNb - 1 - r] = v[p];
    }
  }
  __syncthreads();
  auto S = [&](int i, int j) { return w.s + 16 * (i * kLeafLd + j); };
  auto X = [&](int i, int j) { return w.x + 16 * (i * kLeafLd + j); };
  const f64x4_t zero = {0.0, 0.0, 0.0, 0.0};
  // A_ij -= L_ik L_jk^T
  auto update = [&](int i, int j, int k) {
    leaf_store(S(i, j), leaf_load(S(i, j)) - leaf_product<true>(S(i, k), S(j, k), zero));
  };
  bool ok = true;
#pragma unroll 1
  for (int k = 0; k < 4; ++k) {
    if (wave == 0) {
      if (k > 0) {
        update(k, k, k - 1);
        wave_sync();
      }
      ok = leaf_factor(w, k) & ok;
    } else if (k > 0) {
      int turn = 0;  // the rest of column k - 1's updates, dealt to three waves
      for (int i = k; i < 4; ++i) {
        for (int j = k; j <= i; ++j) {
          if (j == i && j == k) continue;
          if (turn++ % 3 == wave - 1) update(i, j, k - 1);
        }
        for (int j = 0; j < k; ++j)
          if (turn++ % 3 == wave - 1)
            leaf_store(X(i, j), leaf_product<false>(S(i, k - 1), X(k - 1, j),
                                                    j == k - 1 ? zero : leaf_load(X(i, j))));
      }
    }
    __syncthreads();
    if (wave > 0 && wave <= 3 - k) {
      leaf_store(S(k + wave, k), leaf_product<true>(S(k + wave, k), X(k, k), zero));
    } else if (wave > 0) {
      const int j = wave - (3 - k) - 1;
      leaf_store(X(k, j), -leaf_product<false>(X(k, k), X(k, j), zero));
    }
    if (k == 3 && threadIdx.x == 0) w.ok = ok;
    __syncthreads();
  }
  if (!w.ok) {
    if (threadIdx.x == 0) failed[b] = 1;
    return;
  }
  double* Wb = W + (b * C + r0) * ld + r0;
#pragma unroll
  for (int p = 0; p < kNb / 4; ++p) {
    const int i = 4 * p + wave;
    if (i < n && lane < n)
      Wb[i * ld + lane] = lane >= i ? w.x[(kNb - 1 - i) * kLeafLd + kNb - 1 - lane] : 0.0;
  }
}

// One product's operands: C = alpha * A opB + beta * C, per batch item
// (row-major with leading dimensions, item strides sA, sB, sC), opB = B or B^T
// (B stored [N][K]). tri names the factor that is upper triangular: its zero
// part is left out of the sum.
enum Tri : int { kTriNone, kTriBt, kTriB, kTriA };

struct GemmArgs {
  const double* A;
  int64_t lda, sA;
  const double* B;
  int64_t ldb, sB;
  double* C;
  int64_t ldc, sC;
  int M, N, K;
  double alpha, beta;
};

typedef __attribute__((address_space(1))) const void global_cv;
typedef __attribute__((address_space(3))) void lds_v;

// A T x T output tile (T = 64 or 32) on fp64 MFMA (v_mfma_f64_16x16x4f64,
// whose operand layout is A[l%16][k], B[k][l%16] with k = l/16 per k-step, and
// result register r of lane l = D[l/16 + 4r][l%16]); each of the four waves
// has a T/2 x T/2 quadrant over the whole K range, so there is no reduction,
// and every tile size sums in the same order (a result does not depend on the
// tile chosen). Chunks of K of both operands come to LDS by LDS-direct loads,
// one chunk ahead. A rows (and rows of B when TRANSB) lie [row][k], their
// 16-byte pieces permuted by the row so that 16 rows read at one k fall on
// distinct banks; a B stored [K][N] lies [k][n] and is read by column as it
// is. Lane l of k-step t takes k = 16-group + 4(l/16) + t for both.
//
// On this GPU fp64 MFMA and vector instructions take turns on a SIMD, whichever
// wave they come from: an earlier loop with 105 vector instructions beside a
// chunk's 16 MFMAs kept the matrix pipe 62 % busy, with or without loads and
// barriers (this one 81 to 85 % in those three launches). So the chunk loop computes no addresses: global addresses are a
// scalar base that moves along K plus a fixed 32-bit lane offset, the two
// buffers are unrolled so that LDS addresses are fixed registers plus
// immediates, and K's ragged end has a chunk step of its own.
// 32 x 2048: the three launches of the top node 1534, 2920 and 1328 us (whole
// sums, 45 TFLOP/s) -> 618, 1240 and 611 us (trimmed sums, 60 TFLOP/s; a
// library fp64 product reaches 72 here).
template <int T>
struct Tile {
  static constexpr int kBk = T == 64 ? 16 : 32;
  static constexpr int kPr = kBk / 2;             // 16-byte pieces of a row of A
  static constexpr int kPc = T / 2;               // 16-byte pieces of a row of [k][n] B
  static constexpr int kPass = T * kPr / 256;     // 16-byte loads per thread and operand
  double a[2][T * kBk];
  double b[2][T * kBk];
  static __device__ int swz_row(int r) { return kPr == 16 ? r % 16 : (r >> 1) % 8; }
  static __device__ int swz_col(int k) { return 8 * ((k >> 2) & 3) % kPc; }
};

template <int T, bool TRANSB>
__device__ inline void dgemm_tile(const GemmArgs& g, Tri tri, int m0, int n0, int64_t item,
                                  Tile<T>& s) {
  constexpr int NB = T / 32;  // 16x16 blocks per wave and edge
  constexpr int kBk = Tile<T>::kBk, kPr = Tile<T>::kPr, kPc = Tile<T>::kPc;
  constexpr int kPass = Tile<T>::kPass, kH = kBk / 16;
  const int M = g.M, N = g.N, K = g.K;
  // upper triangular factor: opB[k][n] = B[n][k] is zero for k < n, B[k][n]
  // for k > n, A[m][k] for k < m
  const int kb = tri == kTriBt ? n0 : tri == kTriA ? m0 : 0;
  const int ke = tri == kTriB && n0 + T < K ? n0 + T : K;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = (wave >> 1) * (T / 2), wc = (wave & 1) * (T / 2);
  const int li = lane & 15, gq = lane >> 4;

  // Byte offsets of this lane's loads from the chunk's corner of A and B.
  // Rows and columns past M and N load the last one (they are not stored).
  const char* Ac = reinterpret_cast<const char*>(g.A + item * g.sA + m0 * g.lda);
  const char* Bc = reinterpret_cast<const char*>(g.B + item * g.sB + (TRANSB ? n0 * g.ldb : n0));
  const int r_l = wave * (64 / kPr) + lane / kPr;  // this lane's row of a pass
  const int piece_l = (lane % kPr) ^ Tile<T>::swz_row(r_l);
  uint32_t aoff[kPass], boff[kPass];
  int kk_l[kPass];  // [k][n] B: this lane's k of the chunk
#pragma unroll
  for (int p = 0; p < kPass; ++p) {
    const int r = r_l + p * (256 / kPr);
    const int ra = m0 + r < M ? r : M - 1 - m0;
    aoff[p] = static_cast<uint32_t>(ra * g.lda * 8 + 16 * piece_l);
    if constexpr (TRANSB) {
      const int rb = n0 + r < N ? r : N - 1 - n0;
      boff[p] = static_cast<uint32_t>(rb * g.ldb * 8 + 16 * piece_l);
      kk_l[p] = 0;
    } else {
      const int kk = wave * (64 / kPc) + lane / kPc + p * (256 / kPc);
      const int n = 2 * ((lane % kPc) ^ Tile<T>::swz_col(kk));
      kk_l[p] = kk;
      boff[p] = static_cast<uint32_t>(kk * g.ldb * 8 + 8 * (n0 + n < N ? n : (N - 1 - n0) & ~1));
    }
  }
  auto load = [&](const char* base, uint32_t off, double* dst) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((global_cv*)(base + off), (lds_v*)dst, 16, 0, 0);
  };
  auto stage = [&](int kc, int buf) __attribute__((always_inline)) {
    const char* ab = Ac + static_cast<int64_t>(kc) * 8;
    const char* bb = Bc + static_cast<int64_t>(kc) * (TRANSB ? 8 : g.ldb * 8);
    if (kc + kBk <= K) {
#pragma unroll
      for (int p = 0; p < kPass; ++p) load(ab, aoff[p], s.a[buf] + 128 * (4 * p + wave));
#pragma unroll
      for (int p = 0; p < kPass; ++p) load(bb, boff[p], s.b[buf] + 128 * (4 * p + wave));
    } else {  // the ragged end: k past K loads the last one (zeroed below)
      const int back = kc + 2 * piece_l < K ? 0 : kc + 2 * piece_l - ((K - 1) & ~1);
#pragma unroll
      for (int p = 0; p < kPass; ++p) {
        load(ab, aoff[p] - 8 * back, s.a[buf] + 128 * (4 * p + wave));
        const int kback = kc + kk_l[p] < K ? 0 : kc + kk_l[p] - (K - 1);
        load(bb, boff[p] - static_cast<uint32_t>(TRANSB ? 8 * back : kback * g.ldb * 8),
             s.b[buf] + 128 * (4 * p + wave));
      }
    }
  };
  // where this lane reads: four consecutive k of a row (two 16-byte pieces per
  // 16-group h), and the columns of a [k][n] B
  const double* ra[kH][2];
  const double* rb[TRANSB ? kH : NB][2];
#pragma unroll
  for (int h = 0; h < kH; ++h)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int at = li * kBk + 2 * ((8 * h + 2 * gq + q) ^ Tile<T>::swz_row(li));
      ra[h][q] = s.a[0] + wr * kBk + at;
      if constexpr (TRANSB) rb[h][q] = s.b[0] + wc * kBk + at;
    }
  if constexpr (!TRANSB)
#pragma unroll
    for (int y = 0; y < NB; ++y)
      rb[y][0] = s.b[0] + 4 * gq * T + ((wc + 16 * y + li) ^ (16 * gq % T));

  f64x4_t acc[NB][NB];
#pragma unroll
  for (int x = 0; x < NB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y) acc[x][y] = f64x4_t{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](int buf, int kc, bool ragged) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < kH; ++h) {
      double a[NB][4], b[NB][4];
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const f64x2_t v = *reinterpret_cast<const f64x2_t*>(ra[h][q] + buf * T * kBk + 16 * x * kBk);
          a[x][2 * q] = v.x, a[x][2 * q + 1] = v.y;
          if constexpr (TRANSB) {
            const f64x2_t u =
                *reinterpret_cast<const f64x2_t*>(rb[h][q] + buf * T * kBk + 16 * x * kBk);
            b[x][2 * q] = u.x, b[x][2 * q + 1] = u.y;
          }
        }
      if constexpr (!TRANSB)
#pragma unroll
        for (int y = 0; y < NB; ++y)
#pragma unroll
          for (int t = 0; t < 4; ++t) b[y][t] = rb[y][0][buf * T * kBk + (16 * h + t) * T];
      if (ragged) {
#pragma unroll
        for (int x = 0; x < NB; ++x)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const bool in = kc + 16 * h + 4 * gq + t < ke;
            a[x][t] = in ? a[x][t] : 0.0;
            b[x][t] = in ? b[x][t] : 0.0;
          }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int x = 0; x < NB; ++x)
#pragma unroll
          for (int y = 0; y < NB; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x][t], b[y][t], acc[x][y], 0, 0, 0);
    }
  };
  auto step = [&](int kc, int buf) __attribute__((always_inline)) {
    lds_handover();
    __builtin_amdgcn_sched_barrier(0);
    if (kc + kBk < ke) stage(kc + kBk, buf ^ 1);  // every wave has left that buffer
    multiply(buf, kc, false);
  };
  // whole chunks, then at most one ragged one
  const int kfull = kb + (ke - kb) / kBk * kBk;
  stage(kb, 0);
  int kc = kb;
  while (kc < kfull) {
    step(kc, 0);
    kc += kBk;
    if (kc >= kfull) break;
    step(kc, 1);
    kc += kBk;
  }
  if (kc < ke) {
    lds_handover();
    __builtin_amdgcn_sched_barrier(0);
    multiply(((kc - kb) / kBk) & 1, kc, true);
  }
  // the outputs' old values (beta != 0) are read together, ahead of the stores
  double* Cb = g.C + item * g.sC;
  auto out = [&](int x, int y, int r) {
    const int m = m0 + wr + 16 * x + gq + 4 * r, n = n0 + wc + 16 * y + li;
    return Cb + (m < M ? m : M - 1) * g.ldc + (n < N ? n : N - 1);
  };
  double old[NB][NB][4];
  if (g.beta != 0.0) {
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int y = 0; y < NB; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) old[x][y][r] = *out(x, y, r);
  }
#pragma unroll
  for (int x = 0; x < NB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wr + 16 * x + gq + 4 * r, n = n0 + wc + 16 * y + li;
        const double v = g.alpha * acc[x][y][r];
        if (m < M && n < N) *out(x, y, r) = g.beta == 0.0 ? v : v + g.beta * old[x][y][r];
      }
}

// Work item of a workgroup, of items * tiles. The hardware deals workgroups to
// the 8 XCDs in turn, and an XCD's to its 32 CUs. With more than kDealItems items,
// XCD x takes the x-th contiguous part of the (item, tile) list, so the tiles
// that share an item's operands share an L2. With fewer, a contiguous part
// would be the longest sums of an item for one XCD and the shortest for
// another: the list is dealt out in its order, longest first, every second
// round of 256 in reverse so that a CU's long and short tiles even out, and an
// XCD keeps every eighth tile of the edge that the numbering runs along.
// Measured, contiguous -> dealt out: the top node's three launches of one 4096
// matrix 260, 491 and 259 us -> 155, 342 and 161 us (its products at 52
// TFLOP/s), all of it 3307 -> 2891 us. The whole pass, in us: 4096 columns, 4
// items 6277 -> 5347, 5 7096 -> 6328, 6 7629 -> 7188, 7 8118 -> 7961, 8 8219 ->
// 8850; 2048, 4 1547 -> 1463, 5 1718 -> 1674, 6 1806 -> 1802, 7 1864 -> 1910, 8
// 1795 -> 2019; 1024 and less, even up to 5, 6 598 -> 616, 8 562 -> 631. (Eight and
// sixteen items, whole ones per XCD, are where the parts gain; with ten and
// twelve of 2048 or 4096 they are 1 to 5 % behind.)
constexpr int64_t kDealItems = 5;
__device__ inline int64_t xcd_work(int tiles) {
  constexpr int kXcds = 8, kCus = 32, kRound = kXcds * kCus;
  const int64_t n = gridDim.x, x = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  if (n <= kDealItems * tiles) {
    const int64_t round = slot / kCus, cu = slot % kCus;
    const bool whole = (round + 1) * kRound <= n;
    return round * kRound + (whole && (round & 1) ? kCus - 1 - cu : cu) * kXcds + x;
  }
  const int64_t per = n / kXcds, extra = n % kXcds;
  return x * per + (x < extra ? x : extra) + slot;
}

// P = A_TS W_SS^T (TRANSB, tri = kTriBt) and W_TS = -W_TT Q (tri = kTriA). An
// item's tiles are numbered from the longest sums to the shortest.
template <int T, bool TRANSB>
__global__ void __launch_bounds__(256)
    dgemm_kernel(GemmArgs g, Tri tri, int mt, int nt, const uint8_t* __restrict__ active,
                 const uint8_t* __restrict__ failed) {
  const int64_t work = xcd_work(mt * nt);
  const int64_t item = work / (mt * nt);
  if (!active[item] || failed[item]) return;
  __shared__ __attribute__((aligned(16))) Tile<T> s;
  const int t = static_cast<int>(work % (mt * nt));
  const int m = TRANSB ? t % mt : t / nt, n = TRANSB ? t / mt : t % nt;
  dgemm_tile<T, TRANSB>(g, tri, m * T, n * T, item, s);
}

// The two products of a recursion node that both follow P, in one launch:
// A_TT -= P P^T (its 64-blocks on and above the diagonal: a leaf reads the
// lower triangle of its 64-block; tiles [0, tiles0)) and Q = P W_SS (the
// rest). They read P and write disjoint memory.
template <int T>
__global__ void __launch_bounds__(256)
    dgemm_pair_kernel(GemmArgs g0, int nb0, int tiles0, GemmArgs g1, int nt1, int tiles1,
                      const uint8_t* __restrict__ active, const uint8_t* __restrict__ failed) {
  const int64_t work = xcd_work(tiles0 + tiles1);
  const int64_t item = work / (tiles0 + tiles1);
  if (!active[item] || failed[item]) return;
  __shared__ __attribute__((aligned(16))) Tile<T> s;
  int t = static_cast<int>(work % (tiles0 + tiles1));
  if (t < tiles0) {
    constexpr int kSub = 64 / T;  // tiles per edge of a 64-block
    const int sub = t % (kSub * kSub);
    int q = t / (kSub * kSub), m = 0;
    while (q >= nb0 - m) q -= nb0 - m++;
    dgemm_tile<T, true>(g0, kTriNone, 64 * m + T * (sub / kSub),
                        64 * (m + q) + T * (sub % kSub), item, s);
  } else {
    t -= tiles0;
    const int mt1 = tiles1 / nt1;
    dgemm_tile<T, false>(g1, kTriB, (t % mt1) * T, (nt1 - 1 - t / mt1) * T, item, s);
  }
}

// U = fp32(W) (upper), zero below the diagonal, for items that succeeded.
// One wave per row.
__global__ void __launch_bounds__(256)
    emit_u_kernel(const double* __restrict__ W, int64_t C, int64_t ld, const uint8_t* __restrict__ active,
                  const uint8_t* __restrict__ failed, float* __restrict__ U) {
  const int64_t b = blockIdx.y;
  if (!active[b] || failed[b]) return;
  const int64_t i = blockIdx.x * int64_t{4} + (threadIdx.x >> 6);
  if (i >= C) return;
  const double* Wr = W + (b * C + i) * ld;
  float* Ur = U + (b * C + i) * C;
  for (int64_t k = threadIdx.x & 63; k < C; k += 64)
    Ur[k] = k >= i ? static_cast<float>(Wr[k]) : 0.0f;
}

// Workspace plan: A, W (B x C x C fp64 each), lam (B floats), P (largest
// top x bottom block product) and one Q slot per recursion depth.
// Leading dimension of a workspace matrix of n columns: even, so that every
// row is 16-byte aligned.
int64_t pitch(int64_t n) { return (n + 1) / 2 * 2; }

struct Layout {
  int64_t lam_off, p_off, q_off[32], total;
  int64_t p_elems, q_elems[32];
};

void plan_sizes(int64_t b0, int64_t b1, int64_t C, int depth, Layout* L) {
  if (b1 - b0 <= 1) return;
  const int64_t mid = b0 + (b1 - b0) / 2;
  const int64_t r0 = b0 * kNb, rm = mid * kNb, r1 = std::min(b1 * kNb, C);
  const int64_t hs = (rm - r0) * pitch(r1 - rm);
  L->p_elems = std::max(L->p_elems, hs);
  L->q_elems[depth] = std::max(L->q_elems[depth], hs);
  plan_sizes(mid, b1, C, depth + 1, L);
  plan_sizes(b0, mid, C, depth + 1, L);
}

Layout make_layout(int64_t B, int64_t C) {
  Layout L{};
  const int64_t nblk = ceil_div(C, kNb);
  plan_sizes(0, nblk, C, 0, &L);
  int64_t off = 2 * B * C * pitch(C) * 8;
  L.lam_off = off;
  off += ceil_div(B * 4, 256) * 256;
  L.p_off = off;
  off += B * L.p_elems * 8;
  for (int d = 0; d < 32; ++d) {
    L.q_off[d] = off;
    off += B * L.q_elems[d] * 8;
  }
  L.total = off + 256;
  return L;
}

struct Ctx {
  double* A;
  double* W;
  double* P;
  double* Q[32];
  int64_t B, C;
  const uint8_t* active;
  uint8_t* failed;
  hipStream_t s;
};

GemmArgs gemm_args(const double* A, int64_t lda, int64_t sA, const double* Bm, int64_t ldb,
                   int64_t sB, double* Cm, int64_t ldc, int64_t sC, int64_t M, int64_t N,
                   int64_t K, double alpha, double beta) {
  return GemmArgs{A,  lda, sA, Bm, ldb, sB, Cm, ldc, sC, static_cast<int>(M), static_cast<int>(N),
                  static_cast<int>(K), alpha, beta};
}

// 64 x 64 tiles once they give every CU two workgroups: they read half the
// bytes per product of 32 x 32 tiles, which below that spread the work (and
// the unequal lengths of the triangular sums) over four times as many. The
// 1024-edge products of one 2048 matrix (256 or fewer 64-tiles) took 66, 102
// and 57 us on 64-tiles over whole sums and take 25, 50 and 27 us so.
constexpr int64_t kBigTiles = 512;
int64_t tiles_of(const GemmArgs& g, int t) { return ceil_div(g.M, t) * ceil_div(g.N, t); }

template <bool TRANSB>
int gemm(const Ctx& x, const GemmArgs& g, Tri tri) {
  const int t = x.B * tiles_of(g, 64) >= kBigTiles ? 64 : 32;
  const int mt = static_cast<int>(ceil_div(g.M, t)), nt = static_cast<int>(ceil_div(g.N, t));
  const unsigned grid = static_cast<unsigned>(x.B * mt * nt);
  if (t == 64)
    dgemm_kernel<64, TRANSB><<<grid, 256, 0, x.s>>>(g, tri, mt, nt, x.active, x.failed);
  else
    dgemm_kernel<32, TRANSB><<<grid, 256, 0, x.s>>>(g, tri, mt, nt, x.active, x.failed);
  return check_launch("hinv gemm");
}

// g0 = the symmetric update (its M = N a multiple of 64), g1 = Q
int gemm_pair(const Ctx& x, const GemmArgs& g0, const GemmArgs& g1) {
  const int nb0 = g0.M / kNb, upper = nb0 * (nb0 + 1) / 2;
  const int t = x.B * (upper + tiles_of(g1, 64)) >= kBigTiles ? 64 : 32;
  const int tiles0 = upper * (64 / t) * (64 / t);
  const int nt1 = static_cast<int>(ceil_div(g1.N, t));
  const int tiles1 = static_cast<int>(tiles_of(g1, t));
  const unsigned grid = static_cast<unsigned>(x.B * (tiles0 + tiles1));
  if (t == 64)
    dgemm_pair_kernel<64><<<grid, 256, 0, x.s>>>(g0, nb0, tiles0, g1, nt1, tiles1, x.active,
                                                 x.failed);
  else
    dgemm_pair_kernel<32><<<grid, 256, 0, x.s>>>(g0, nb0, tiles0, g1, nt1, tiles1, x.active,
                                                 x.failed);
  return check_launch("hinv gemm pair");
}

int factor_rec(const Ctx& x, int64_t b0, int64_t b1, int depth) {
  const int64_t C = x.C, ld = pitch(C), CC = C * ld;
  const int64_t r0 = b0 * kNb, r1 = std::min(b1 * kNb, C);
  if (b1 - b0 == 1) {
    leaf_kernel<<<static_cast<unsigned>(x.B), 256, 0, x.s>>>(x.A, x.W, C, ld, r0,
                                                            static_cast<int>(r1 - r0), x.active,
                                                            x.failed);
    return check_launch("hinv leaf");
  }
  const int64_t mid = b0 + (b1 - b0) / 2;
  const int64_t rm = mid * kNb, h = rm - r0, s2 = r1 - rm, lp = pitch(s2);
  if (int rc = factor_rec(x, mid, b1, depth + 1)) return rc;
  const double* Wss = x.W + rm * ld + rm;
  // P = A_TS W_SS^T
  if (int rc = gemm<true>(x, gemm_args(x.A + r0 * ld + rm, ld, CC, Wss, ld, CC, x.P, lp, h * lp,
                                       h, s2, s2, 1.0, 0.0), kTriBt))
    return rc;
  // A_TT -= P P^T (upper tiles) and Q = P W_SS
  double* Q = x.Q[depth];
  if (int rc = gemm_pair(x,
                         gemm_args(x.P, lp, h * lp, x.P, lp, h * lp, x.A + r0 * ld + r0, ld, CC, h,
                                   h, s2, -1.0, 1.0),
                         gemm_args(x.P, lp, h * lp, Wss, ld, CC, Q, lp, h * lp, h, s2, s2, 1.0,
                                   0.0)))
    return rc;
  if (int rc = factor_rec(x, b0, mid, depth + 1)) return rc;
  // W_TS = -W_TT Q
  return gemm<false>(x, gemm_args(x.W + r0 * ld + r0, ld, CC, Q, lp, h * lp, x.W + r0 * ld + rm, ld,
                                  CC, h, s2, h, -1.0, 0.0), kTriA);
}

}  // namespace
}  // namespace mgq

using namespace mgq;

extern "C" int64_t mgq_hinv_full_workspace_size(int64_t B, int64_t C) {
  if (B < 0 || C < 1) return 0;
  return make_layout(B, C).total;
}

// One factorisation pass for the items with active[b] != 0, using per-item
// damp[b]; failed[b] (device, cleared by the caller) reports pivot failure.
extern "C" int mgq_hinv_full_pass(const float* H, int64_t B, int64_t C, const float* damp,
                                  const uint8_t* active, uint8_t* failed, float* U,
                                  void* workspace, int64_t workspace_bytes, void* stream) {
  clear_error();
  MGQ_REQUIRE(B >= 0 && C >= 1, MGQ_ERR_SHAPE, "bad shape");
  const Layout L = make_layout(B, C);
  MGQ_REQUIRE(workspace != nullptr && workspace_bytes >= L.total, MGQ_ERR_WORKSPACE,
              "hinv workspace too small");
  if (B == 0) return MGQ_OK;
  hipStream_t s = as_stream(stream);
  // aligned to 16 bytes inside the layout's slack
  char* ws = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t{15});
  Ctx x;
  x.A = reinterpret_cast<double*>(ws);
  x.W = x.A + B * C * pitch(C);
  x.P = reinterpret_cast<double*>(ws + L.p_off);
  for (int d = 0; d < 32; ++d) x.Q[d] = reinterpret_cast<double*>(ws + L.q_off[d]);
  x.B = B;
  x.C = C;
  x.active = active;
  x.failed = failed;
  x.s = s;
  float* lam = reinterpret_cast<float*>(ws + L.lam_off);
  const unsigned gb = static_cast<unsigned>(B);
  lam_kernel<<<gb, 256, 0, s>>>(H, C, damp, active, lam);
  if (int rc = check_launch("hinv lam")) return rc;
  const dim3 rows(static_cast<unsigned>(ceil_div(C, 4)), gb);
  build_kernel<<<rows, 256, 0, s>>>(H, C, pitch(C), lam, active, x.A);
  if (int rc = check_launch("hinv build")) return rc;
  if (int rc = factor_rec(x, 0, ceil_div(C, kNb), 0)) return rc;
  emit_u_kernel<<<rows, 256, 0, s>>>(x.W, C, pitch(C), active, failed, U);
  return check_launch("hinv emit");
}
