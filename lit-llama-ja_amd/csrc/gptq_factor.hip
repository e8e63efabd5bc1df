// Matrix work of the GPTQ producer around the column loop (gptq.hip): the calibration Hessian, the inverse factor that the
// loop reads, and the update of the columns behind a block (reference lit_llama/quantization.py:516-530, 549-566, 596).
//
// All three are C -= or += A^T B (gptq_tiles.h).
// Bound: the fp32 matrix rate (157 TFLOP/s dense). A wave's 16 k of a 64 x 64 tile are 16 MFMAs of 32 cycles for 16 reads of
// 4 bytes a lane, so neither LDS nor the loads (the next tile's in registers while this one is multiplied) are near their limits.
#include "common.h"
#include "gptq_tiles.h"

namespace llj {

constexpr int kFactor = 128;  // columns per elimination step

// H = keep H + (alpha X)^T (alpha X): the tiles on and below the diagonal, each written to its place and mirrored. The sums are those
// of the library's product bit for bit (to 4,096 columns), at half its work: 2048 x 4096 358 us (96 TFLOP/s of the half; 386 with one tile
// ahead, read behind branches) for 580 with the two passes over H.
template <int BT, typename S, bool VEC>
__global__ __launch_bounds__(256) void gptq_gram_kernel(const S* __restrict__ x, int T, int K, float keep, float alpha, float* __restrict__ H) {
  typedef AtB<BT, BT, S, VEC, true> G;
  __shared__ __align__(16) float lds[G::kLds];
  const int nt = (K + BT - 1) / BT, t = xcd_run(blockIdx.x, nt * (nt + 1) / 2);
  if (t < 0) return;
  int ti, tj;
  triangle(t, ti, tj);
  const int m0 = ti * BT, n0 = tj * BT;
  f32x4 acc[G::MI][G::NI], old[G::MI][G::NI];
  // (a lane's four sums of an MFMA tile are neighbours in the mirrored place: whole vectors there, of H's own symmetric other half too. VEC says
  // nothing of where H begins.)
  const bool whole = VEC && ((uintptr_t)H & 15) == 0 && m0 + BT <= K && n0 + BT <= K;
  G::run(x + m0, K, K - m0, x + n0, K, K - n0, T, alpha, lds, acc, [&] {
    if (!whole) return;
    G::tiles([&](int a, int b, int i, int j) { old[a][b] = *reinterpret_cast<const f32x4*>(H + (size_t)(n0 + j) * K + m0 + i); });
  });
  if (whole) {
    G::tiles([&](int a, int b, int i, int j) {
      f32x4 h;
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = old[a][b][r] * keep + acc[a][b][r];
      *reinterpret_cast<f32x4*>(H + (size_t)(n0 + j) * K + m0 + i) = h;
      if (ti != tj)
#pragma unroll
        for (int r = 0; r < 4; ++r) H[(size_t)(m0 + i + r) * K + n0 + j] = h[r];
    });
    return;
  }
  G::load(old, [&](int i, int j) { return H[(size_t)min(m0 + i, K - 1) * K + min(n0 + j, K - 1)]; });
  G::both(acc, old, [&](int i, int j, float v, float h) {
    const int m = m0 + i, n = n0 + j;
    if (m >= K || n >= K) return;
    h = h * keep + v;
    H[(size_t)m * K + n] = h;
    if (ti != tj) H[(size_t)n * K + m] = h;
  });
}

// Wt[i2 + m][n] -= sum_b hinv[i1 + b][i2 + m] err[b][n]. Bound: Wt in and out beside the products; what is subtracted from is read
// after them, all of it before the first use. 3968 x 4096: 56 us for 73 as a product and a subtraction, the same bits.
template <int BM, int BN, bool VEC>
__global__ __launch_bounds__(256) void gptq_update_kernel(const float* __restrict__ hinv, int K, int i1, int blk, const float* __restrict__ err,
                                                          int N, float* __restrict__ wt) {
  typedef AtB<BM, BN, float, VEC, false> G;
  __shared__ __align__(16) float lds[G::kLds];
  const int i2 = i1 + blk, M = K - i2, mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN, t = xcd_run(blockIdx.x, mt * nt);
  if (t < 0) return;
  const int m0 = t / nt * BM, n0 = t % nt * BN;
  f32x4 acc[G::MI][G::NI], old[G::MI][G::NI];
  G::run(hinv + (size_t)i1 * K + i2 + m0, K, M - m0, err + n0, N, N - n0, blk, 1.f, lds, acc, [&] {
    G::load(old, [&](int i, int j) { return wt[(size_t)(i2 + min(m0 + i, M - 1)) * N + min(n0 + j, N - 1)]; });
  });
  G::both(acc, old, [&](int i, int j, float v, float w) {
    const int m = m0 + i, n = n0 + j;
    if (m < M && n < N) wt[(size_t)(i2 + m) * N + n] = w - v;
  });
}

// ---------------------------------------------------------------- the inverse factor
// U upper triangular with U^T U = H^-1 (torch.linalg.cholesky(cholesky_inverse(cholesky(H)), upper=True)): with the order of the
// columns reversed, H = L L^T gives U as L^-1 reversed -- one elimination instead of two factorizations and a product. Blocks of 128
// columns; step k turns row block k of [H | I] into P_k = L_kk^-1 [X_k | H_k] (gptq_panel_kernel) and takes P_k[:, i]^T P_k off every
// later row block i (gptq_step_kernel): in H's upper triangle the next matrix to factor, in the lower one the growing L^-1.
// The next diagonal block is factored by one workgroup of that launch while the others work on the rest: its chain (1.4 us
// for its loads, 4 for its product, four times 2.9 for 32 pivots, 1.7 between them, 2 for the stores) bounds a step, the products (2 K^3 / 3 in
// all, 0.3 ms at K = 4096) run beside it and bound it from 6,144 columns on. K = 4096: 1.27 ms (39.6 us a step; 1.49 with the block's whole product, the other waves' updates before
// the elimination and 4-byte stores) for 29.2 with the library's three calls, K = 512: 0.14 (35 a step; 0.17) for 3.1; error against float64 2.5e-7 for 1.1e-6 (8,192 rows).
constexpr int kFs = kFactor + 16;  // LDS row stride of the diagonal block

__device__ __forceinline__ float lane_value(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }

// S (LDS, 128 x 128, upper triangle, zeros below) -> L^-1 in the lower triangle with zeros above, S = L L^T. 32 columns at a time: one wave eliminates
// the 32 x 32 block in registers (lane c a column of the block, lane 32 + c of the identity, which lies in the rows' padding), the matrix cores do
// the rest: the other waves' products of one turn run beside the next turn's elimination, whose block that wave brings up to date itself.
// Returns false (in every thread) if a pivot was not a positive normal number.
__device__ __forceinline__ bool factor_block(float* S, int* bad) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, c16 = lane & 15;
  if (tid == 0) *bad = 0;
  for (int i = tid; i < 64 * 16; i += 256) S[(i >> 4) * kFs + kFactor + (i & 15)] = (i >> 4 & 31) == (i >> 9) * 16 + (i & 15) ? 1.f : 0.f;
  auto update = [&](int s, int ib, int jb) {  // block (ib, jb) less its product of row block s
    const float* p = S + 32 * s * kFs;
    float* o = S + 32 * ib * kFs + 32 * jb;
    f32x4 d[2][2] = {}, old[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) old[i][j][r] = o[(16 * i + 4 * q + r) * kFs + 16 * j + c16];
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          d[i][j] = mma4(p[(4 * k + q) * kFs + 32 * ib + 16 * i + c16], p[(4 * k + q) * kFs + 32 * jb + 16 * j + c16], d[i][j]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * i + 4 * q + r, col = 16 * j + c16;
          o[row * kFs + col] = ib == jb && row > col ? 0.f : old[i][j][r] - d[i][j][r];
        }
  };
  for (int s = 0; s < 4; ++s) {
    __syncthreads();
    if (wave == 0) {
      if (s) update(s - 1, s, s);
      const int c = lane & 31;
      float* d = S + 32 * s * kFs + 32 * s;
      const float* from = lane < 32 ? d + c : S + (c >> 4) * 32 * kFs + kFactor + (c & 15);
      float v[32];
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] = from[i * kFs];
      bool ok = true;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const float p = lane_value(v[j], j);
        ok = ok && p >= 0x1p-126f && p < INFINITY;  // (the root's estimate takes normal numbers)
        float r = __builtin_amdgcn_rsqf(p);
        r = __builtin_fmaf(0.5f * r, __builtin_fmaf(-p * r, r, 1.f), r);  // one Newton step
        v[j] *= r;
#pragma unroll
        for (int g = (j + 1) & ~7; g < 32; g += 8) {
#pragma unroll
          for (int i = g > j ? g : j + 1; i < g + 8; ++i) v[i] = __builtin_fmaf(-lane_value(v[j], i), v[j], v[i]);
          // updated here, not where it is read next: the lane values would pile up and spill
          asm volatile("" : "+v"(v[g]), "+v"(v[g + 1]), "+v"(v[g + 2]), "+v"(v[g + 3]), "+v"(v[g + 4]), "+v"(v[g + 5]), "+v"(v[g + 6]), "+v"(v[g + 7]));
        }
      }
      if (lane >= 32) {
#pragma unroll
        for (int i = 0; i < 32; ++i) d[i * kFs + c] = v[i];
      }
      if (!ok && lane == 0) *bad = 1;
    } else if (s) {
      int n = 0;
      for (int ib = s; ib < 4; ++ib)
        for (int jb = 0; jb < 4; ++jb) {
          if ((jb >= s && jb < ib) || (ib == s && jb == s)) continue;
          if (n++ % 3 == wave - 1) update(s - 1, ib, jb);
        }
    }
    __syncthreads();
    if (wave != s) {  // the other 32-column blocks of these rows, times the block's inverse
      float* b = S + 32 * s * kFs + 32 * wave;
      const float* a = S + 32 * s * kFs + 32 * s;
      f32x4 o[2][2] = {};
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[i][j] = mma4(a[(16 * i + c16) * kFs + 4 * k + q], b[(4 * k + q) * kFs + 16 * j + c16], o[i][j]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) b[(16 * i + 4 * q + r) * kFs + 16 * j + c16] = o[i][j][r];
    }
  }
  __syncthreads();
  return *bad == 0;
}

// the factored block: its rows of P (zeros above the diagonal) and transposed for the panel product, in whole vectors (4-byte stores: 7.8 us)
__device__ __forceinline__ void put_block(const float* S, int k, int K, float* __restrict__ P, float* __restrict__ xt, bool ok, int* info) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int b = 0; b < kFactor / 8; ++b) {
    const int i = 8 * b + (tid >> 5), j = 4 * (tid & 31);
    f32x4 v = *reinterpret_cast<const f32x4*>(S + i * kFs + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = j + e <= i ? v[e] : 0.f;
    *reinterpret_cast<f32x4*>(P + ((size_t)k * kFactor + i) * K + (size_t)k * kFactor + j) = v;
  }
#pragma unroll
  for (int b = 0; b < kFactor / 8; ++b) {  // 16 columns of 16 rows a wave
    const int i = 16 * (b >> 1) + (tid & 15), j = 64 * (b & 1) + 4 * (tid >> 4);
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = i <= j + e ? S[(j + e) * kFs + i] : 0.f;
    *reinterpret_cast<f32x4*>(xt + i * kFactor + j) = v;
  }
  if (!ok && tid == 0) *info = 1;
}

// S (LDS) = the upper triangle of M's diagonal block at r0 less X^T X, X: P's 128 x 128 block there, zeros below. Wave W: rows W and 7 - W of the
// MFMA tiles, 9 of the triangle's 36.
template <int W>
__device__ __forceinline__ void diagonal_block(const float* __restrict__ M, const float* __restrict__ p, int r0, int K, float* S) {
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c = lane & 15;
  f32x4 x[16], acc[9], old[9];
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = *reinterpret_cast<const f32x4*>(p + (size_t)(8 * i + (tid >> 5)) * K + r0 + 4 * (tid & 31));
  auto each = [&](auto f) {
#pragma unroll
    for (int t = 0; t < 9; ++t) f(t, t < 8 - W ? W : 7 - W, t < 8 - W ? W + t : t - 1);
  };
  each([&](int t, int m, int n) {
    acc[t] = f32x4{};
#pragma unroll
    for (int r = 0; r < 4; ++r) old[t][r] = M[(size_t)(r0 + 16 * m + 4 * q + r) * K + r0 + 16 * n + c];
  });
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4*>(S + (8 * i + (tid >> 5)) * kFs + 4 * (tid & 31)) = x[i];
  __syncthreads();
  float v[2][8];  // tile columns W .. 7 of four k: both operands' values
  auto read = [&](int s) {
#pragma unroll
    for (int j = W; j < 8; ++j) v[s & 1][j] = S[(4 * s + q) * kFs + 16 * j + c];
  };
  read(0);
#pragma unroll
  for (int s = 0; s < kFactor / 4; ++s) {
    if (s + 1 < kFactor / 4) read(s + 1);
    __builtin_amdgcn_sched_barrier(0);
    each([&](int t, int m, int n) { acc[t] = mma4(v[s & 1][m], v[s & 1][n], acc[t]); });
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4*>(S + (8 * i + (tid >> 5)) * kFs + 4 * (tid & 31)) = f32x4{};
  __syncthreads();
  each([&](int t, int m, int n) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * m + 4 * q + r, j = 16 * n + c;
      if (j >= i) S[i * kFs + j] = old[t][r] - acc[t][r];
    }
  });
}

// M (upper triangle) = H in the reversed order of perm (null: 0, 1, ..) with damp on the diagonal, a row to a workgroup. ROW: through LDS, where the
// gather costs least (4,096 columns: 74 us from memory).
template <bool ROW>
__global__ __launch_bounds__(256) void gptq_order_kernel(const float* __restrict__ H, const int64_t* __restrict__ perm, const float* __restrict__ damp,
                                                         int K, float* __restrict__ M) {
  extern __shared__ __align__(16) float row[];
  const int a = blockIdx.x, ra = K - 1 - a;
  const size_t i = perm ? (size_t)perm[ra] : ra;
  const float* h = H + i * K;
  const float d = *damp;
  if (ROW) {
    for (int b = threadIdx.x; b < K; b += 256) row[b] = h[b];
    __syncthreads();
  }
#pragma unroll 4
  for (int b = a + threadIdx.x; b < K; b += 256) {
    const size_t j = perm ? (size_t)perm[K - 1 - b] : K - 1 - b;
    const float v = ROW ? row[j] : h[j];
    M[(size_t)a * K + b] = a == b ? v + d : v;
  }
}

__global__ __launch_bounds__(256) void gptq_first_kernel(const float* __restrict__ M, int K, float* __restrict__ P, float* __restrict__ xt, int* info) {
  __shared__ __align__(16) float S[kFactor * kFs];
  __shared__ int bad;
  float m[kFactor * kFactor / 256];  // every load in flight before the first is used (the lower triangle is not set)
#pragma unroll
  for (int r = 0; r < kFactor * kFactor / 256; ++r) m[r] = M[(size_t)(2 * r + (threadIdx.x >> 7)) * K + (threadIdx.x & 127)];
#pragma unroll
  for (int r = 0; r < kFactor * kFactor / 256; ++r) {
    const int i = 2 * r + (threadIdx.x >> 7), j = threadIdx.x & 127;
    S[i * kFs + j] = j >= i ? m[r] : 0.f;
  }
  const bool ok = factor_block(S, &bad);
  put_block(S, 0, K, P, xt, ok, info);
}

// P's row block k outside the diagonal block: xt^T M's row block. Workgroup: 64 rows x 64 columns.
__global__ __launch_bounds__(256) void gptq_panel_kernel(const float* __restrict__ M, const float* __restrict__ xt, int k, int K, float* __restrict__ P) {
  typedef AtB<64, 64, float, true, false> G;
  __shared__ __align__(16) float lds[G::kLds];
  const int m0 = (blockIdx.x & 1) * 64, n0 = (blockIdx.x >> 1) * 64;
  if (n0 / kFactor == k) return;
  f32x4 acc[G::MI][G::NI];
  const size_t row = (size_t)k * kFactor;
  G::run(xt + m0, kFactor, kFactor - m0, M + row * K + n0, K, K - n0, kFactor, 1.f, lds, acc, [] {});
  G::each(acc, [&](int i, int j, float v) { P[(row + m0 + i) * K + n0 + j] = v; });
}

constexpr int kStepLds = kFactor * kFs, kStepAlone = 21000;  // floats: the diagonal block's, and more than half a CU's LDS
// Tiles of a step up to which workgroup 0 has its CU to itself (ALONE), so that its chain is not held up: up to some 8 tiles a CU the chain is the longer. Past that
// the products are, and one workgroup of theirs a CU, which ALONE makes of them too, is too few. ms of a factor, all steps alone -> by this rule
// (two a CU in all): 4,096 columns 1.28 -> 1.28 (1.39), 5,120 2.01 -> 1.80 (1.86), 6,144 3.08 -> 2.62 (2.65), 8,192 6.52 -> 5.31 (5.33),
// 11,008 15.3 -> 12.3 (12.3), 13,824 29.5 -> 24.1 (24.1); with 1,536 tiles 4,096 columns take 1.35, with 2,048 1.31 (their first
// steps have up to 2,077), with 3,072 5,120 take 1.95.
constexpr long kAloneTiles = 2100;

// Workgroup 0: the next diagonal block, updated and factored. The others: 64 x 64 tiles of the rows below, the lower triangle's columns
// up to block k (first sums in block k's own) and the upper triangle's.
template <bool ALONE>
__global__ __launch_bounds__(256) void gptq_step_kernel(float* __restrict__ M, float* __restrict__ P, int k, int K, float* __restrict__ xt, int* info) {
  typedef AtB<64, 64, float, true, false> G;
  __shared__ __align__(16) float lds[ALONE ? kStepAlone : kStepLds];
  __shared__ int bad;
  const float* p = P + (size_t)k * kFactor * K;
  const int r0 = (k + 1) * kFactor;
  if (blockIdx.x == 0) {
    __builtin_amdgcn_s_setprio(3);  // the longest chain of the launch (not ALONE: beside another workgroup's products)
    switch (uniform(threadIdx.x >> 6)) {  // (the same barriers on every way)
      case 0: diagonal_block<0>(M, p, r0, K, lds); break;
      case 1: diagonal_block<1>(M, p, r0, K, lds); break;
      case 2: diagonal_block<2>(M, p, r0, K, lds); break;
      default: diagonal_block<3>(M, p, r0, K, lds);
    }
    const bool ok = factor_block(lds, &bad);
    put_block(lds, k + 1, K, P, xt, ok, info);
    return;
  }
  const int R = (K - r0) / 64, C = r0 / 64, upper = R * (R + 1) / 2;
  const int t = xcd_run(blockIdx.x - 1, R * C + upper);
  if (t < 0) return;
  int m0, n0;
  if (t < R * C) {
    m0 = r0 + t / C * 64;
    n0 = t % C * 64;
  } else {
    int i, j;
    triangle(t - R * C, i, j);
    if (i < 2) return;  // workgroup 0's
    m0 = r0 + j * 64;
    n0 = r0 + i * 64;
  }
  f32x4 acc[G::MI][G::NI], old[G::MI][G::NI];
  G::run(p + m0, K, 64, p + n0, K, 64, kFactor, 1.f, lds, acc,
         [&] { G::load(old, [&](int i, int j) { return M[(size_t)(m0 + i) * K + n0 + j]; }); });
  const bool first = n0 / kFactor == k;
  G::both(acc, old, [&](int i, int j, float v, float m) { M[(size_t)(m0 + i) * K + n0 + j] = (first ? 0.f : m) - v; });
}

// Wt[place[k]][n] = W[n][k] (null: k), zero where dead[k]: 64 x 64 through LDS, whole rows of Wt moved to their places
__global__ __launch_bounds__(256) void gptq_weight_kernel(const float* __restrict__ W, const int64_t* __restrict__ place, const bool* __restrict__ dead,
                                                          int N, int K, float* __restrict__ Wt) {
  __shared__ float t[64][65];
  const int n0 = blockIdx.x * 64, k0 = blockIdx.y * 64, c = threadIdx.x & 63, r = threadIdx.x >> 6;
  const int k = min(k0 + c, K - 1);
  const bool zero = dead[k];
  float v[16];
  size_t to[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    v[i] = W[(size_t)min(n0 + r + 4 * i, N - 1) * K + k];
    const int row = min(k0 + r + 4 * i, K - 1);
    to[i] = place ? (size_t)place[row] : row;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) t[r + 4 * i][c] = zero ? 0.f : v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (n0 + c < N && k0 + r + 4 * i < K) Wt[to[i] * N + n0 + c] = t[c][r + 4 * i];
}

// U = P's lower triangle in reversed order, zeros below the diagonal
__global__ __launch_bounds__(256) void gptq_reverse_kernel(const float* __restrict__ P, int K, float* __restrict__ U) {
  const int a = blockIdx.y, b = blockIdx.x * 256 + threadIdx.x;
  if (b < K) U[(size_t)a * K + b] = b >= a ? P[(size_t)(K - 1 - a) * K + K - 1 - b] : 0.f;
}

}  // namespace llj

using namespace llj;

extern "C" {

int llj_gptq_gram(const void* x, int dt, int T, int K, float keep, float alpha, float* H, void* stream) {
  LLJ_REQUIRE(x && H && T > 0 && K > 0 && (dt == 0 || dt == 1));
  // 64 x 64 tiles, 32 x 32 while those leave CUs idle (1467 x 512: 49 us and 20, 357 x 1152: 17 and 12)
  const long n64 = (K + 63) / 64, n32 = (K + 31) / 32;
  const bool small = n64 * (n64 + 1) / 2 < 256;
  const long tiles = small ? n32 * (n32 + 1) / 2 : n64 * (n64 + 1) / 2, grid = (tiles + 7) / 8 * 8;
  const bool vec = K % 4 == 0 && ((uintptr_t)x & (dt ? 15 : 7)) == 0;
  LLJ_REQUIRE(grid < (1l << 31));
  const hipStream_t s = (hipStream_t)stream;
#define LLJ_GRAM_T(B, S, V) \
  hipLaunchKernelGGL((gptq_gram_kernel<B, S, V>), dim3((unsigned)grid), dim3(256), 0, s, (const S*)x, T, K, keep, alpha, H)
#define LLJ_GRAM(S, V)                 \
  do {                                 \
    if (small) LLJ_GRAM_T(32, S, V);   \
    else LLJ_GRAM_T(64, S, V);         \
  } while (0)
  if (dt) {
    if (vec) LLJ_GRAM(float, true);
    else LLJ_GRAM(float, false);
  } else {
    if (vec) LLJ_GRAM(bf16_t, true);
    else LLJ_GRAM(bf16_t, false);
  }
#undef LLJ_GRAM
#undef LLJ_GRAM_T
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_gptq_update(const float* hinv, int K, int i1, int blocksize, const float* err, int N, float* wt, void* stream) {
  LLJ_REQUIRE(hinv && err && wt && K > 0 && N > 0 && i1 >= 0 && blocksize > 0 && i1 + blocksize <= K);
  const int M = K - i1 - blocksize;
  if (M == 0) return 0;
  const bool vec = K % 4 == 0 && N % 4 == 0 && (i1 + blocksize) % 4 == 0 && (((uintptr_t)hinv | (uintptr_t)err) & 15) == 0;
  const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64), grid = (tiles + 7) / 8 * 8;
  LLJ_REQUIRE(grid < (1l << 31));
  if (vec)
    hipLaunchKernelGGL((gptq_update_kernel<64, 64, true>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, hinv, K, i1, blocksize, err, N, wt);
  else
    hipLaunchKernelGGL((gptq_update_kernel<64, 64, false>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, hinv, K, i1, blocksize, err, N, wt);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_gptq_weight(const float* W, const int64_t* place, const void* dead, int N, int K, float* Wt, void* stream) {
  LLJ_REQUIRE(W && dead && Wt && N > 0 && K > 0 && (K + 63) / 64 <= 65535);
  hipLaunchKernelGGL(gptq_weight_kernel, dim3((N + 63) / 64, (K + 63) / 64), dim3(256), 0, (hipStream_t)stream, W, place, (const bool*)dead, N, K, Wt);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_gptq_factor(const float* H, const int64_t* perm, const float* damp, int K, float* M, float* P, float* xt, int* info, void* stream) {
  LLJ_REQUIRE(H && damp && M && P && xt && info && K >= kFactor && K % kFactor == 0 && K <= 65535);
  LLJ_REQUIRE((((uintptr_t)M | (uintptr_t)P | (uintptr_t)xt) & 15) == 0);
  const hipStream_t s = (hipStream_t)stream;
  const int nb = K / kFactor;
  if (K <= 16384) hipLaunchKernelGGL(gptq_order_kernel<true>, dim3(K), dim3(256), (size_t)K * 4, s, H, perm, damp, K, M);
  else hipLaunchKernelGGL(gptq_order_kernel<false>, dim3(K), dim3(256), 0, s, H, perm, damp, K, M);
  hipLaunchKernelGGL(gptq_first_kernel, dim3(1), dim3(256), 0, s, M, K, P, xt, info);
  for (int k = 0; k < nb; ++k) {
    hipLaunchKernelGGL(gptq_panel_kernel, dim3(K / 64 * 2), dim3(256), 0, s, M, xt, k, K, P);
    if (k + 1 == nb) break;
    const long R = (K - (k + 1) * kFactor) / 64, C = (k + 1) * kFactor / 64, tiles = R * C + R * (R + 1) / 2;
    const dim3 grid((unsigned)(1 + (tiles + 7) / 8 * 8));
    if (tiles <= kAloneTiles) hipLaunchKernelGGL(gptq_step_kernel<true>, grid, dim3(256), 0, s, M, P, k, K, xt, info);
    else hipLaunchKernelGGL(gptq_step_kernel<false>, grid, dim3(256), 0, s, M, P, k, K, xt, info);
  }
  hipLaunchKernelGGL(gptq_reverse_kernel, dim3((K + 255) / 256, K), dim3(256), 0, s, P, K, M);
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
