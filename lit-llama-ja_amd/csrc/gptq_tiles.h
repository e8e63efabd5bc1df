// Products C = A^T B of the GPTQ producer in fp32 (gptq_factor.hip, gptq.hip): both operands stored along their output index
// ("k-major": X of the Hessian is tokens x columns, a block of the factor and the block's errors are 128 x columns), which
// v_mfma_f32_16x16x4_f32 takes from LDS without a transposition: lane l reads element (k + l / 16, m + l % 16), rows 16 banks
// apart. One accumulator per output, ascending k. Two tiles of K are on their way to registers while a third is multiplied from LDS (2048 rows, half the
// product: 4,096 columns 386 -> 358 us, 11,008 with 1,500 rows 1,782 -> 1,660).
#pragma once
#include "common.h"

namespace llj {

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// four consecutive elements; not VEC: none past the last-th
template <bool VEC>
__device__ __forceinline__ f32x4 ld4(const float* p, int last) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4*>(p);
  return f32x4{p[0], p[min(1, last)], p[min(2, last)], p[min(3, last)]};
}
template <bool VEC>
__device__ __forceinline__ f32x4 ld4(const bf16_t* p, int last) {
  if constexpr (VEC) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    return f32x4{bflo(w.x), bfhi(w.x), bflo(w.y), bfhi(w.y)};
  }
  return f32x4{bf2f(p[0]), bf2f(p[min(1, last)]), bf2f(p[min(2, last)]), bf2f(p[min(3, last)])};
}

// acc = A^T B of one BM x BN tile by 256 threads (2 x 2 waves): A: kd x ma, B: kd x nb, k-major, pointers at the tile's first column,
// ma / nb columns left from there (VEC: multiples of 4, rows aligned to four elements). SCALE: elements times alpha, rounded. also(): loads of
// the caller's to be in flight over the products, behind the first tiles'.
template <int BM, int BN, typename S, bool VEC, bool SCALE>
struct AtB {
  static constexpr int KD = 32, SA = BM + 16, SB = BN + 16, MI = BM / 32, NI = BN / 32;
  static constexpr int kLds = 2 * KD * (SA + SB);  // floats
  static constexpr int TA = BM / 4, RA = 256 / TA, PA = KD / RA, TB = BN / 4, RB = 256 / TB, PB = KD / RB;

  template <typename F>
  static __device__ __forceinline__ void run(const S* A, size_t lda, int ma, const S* B, size_t ldb, int nb, int kd, float alpha,
                                             float* lds, f32x4 (&acc)[MI][NI], F also) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ra = tid / TA, ca = (tid % TA) * 4, rb = tid / TB, cb = (tid % TB) * 4;
    // No load is behind a branch, so that the count of those in flight is known where one is waited for: columns past the last give outputs
    // that nobody takes, rows past the last are zeroed on their way to LDS.
    const int va = min(ca, (ma - 1) & ~3), vb = min(cb, (nb - 1) & ~3);
    f32x4 fa[2][PA], fb[2][PB];
    auto fetch = [&](int s, int k) {
#pragma unroll
      for (int p = 0; p < PA; ++p) fa[s][p] = ld4<VEC>(A + (size_t)min(k + ra + p * RA, kd - 1) * lda + va, ma - 1 - va);
#pragma unroll
      for (int p = 0; p < PB; ++p) fb[s][p] = ld4<VEC>(B + (size_t)min(k + rb + p * RB, kd - 1) * ldb + vb, nb - 1 - vb);
    };
    auto stage = [&](int s, int k) {
      float* a = lds + ((k / KD) & 1) * KD * (SA + SB);
      float* b = a + KD * SA;
#pragma unroll
      for (int p = 0; p < PA; ++p)
        *reinterpret_cast<f32x4*>(a + (ra + p * RA) * SA + ca) = k + ra + p * RA >= kd ? f32x4{} : SCALE ? fa[s][p] * alpha : fa[s][p];
#pragma unroll
      for (int p = 0; p < PB; ++p)
        *reinterpret_cast<f32x4*>(b + (rb + p * RB) * SB + cb) = k + rb + p * RB >= kd ? f32x4{} : SCALE ? fb[s][p] * alpha : fb[s][p];
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{};
    const int oa = (lane >> 4) * SA + (wave & 1) * (BM / 2) + (lane & 15), ob = (lane >> 4) * SB + (wave >> 1) * (BN / 2) + (lane & 15);
    auto step = [&](int s, int k) {  // tile k / KD is in LDS; the one after it in registers or on its way
      __syncthreads();  // it is staged, and every wave is done with the other buffer
      fetch(s, k + 2 * KD);
      const float* a = lds + ((k / KD) & 1) * KD * (SA + SB) + oa;
      const float* b = lds + ((k / KD) & 1) * KD * (SA + SB) + KD * SA + ob;
      float xa[2][MI], xb[2][NI];
      auto read = [&](int q) {
#pragma unroll
        for (int i = 0; i < MI; ++i) xa[q & 1][i] = a[4 * q * SA + 16 * i];
#pragma unroll
        for (int j = 0; j < NI; ++j) xb[q & 1][j] = b[4 * q * SB + 16 * j];
      };
      read(0);
#pragma unroll
      for (int q = 0; q < KD / 4; ++q) {  // (the next operands are read over the products, not at their use)
        if (q + 1 < KD / 4) read(q + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = mma4(xa[q & 1][i], xb[q & 1][j], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    fetch(0, 0);
    fetch(1, KD);
    also();
    stage(0, 0);
    for (int k = 0; k < kd; k += 2 * KD) {  // (an odd number of tiles: zeros behind the last; behind a branch its loads would move to their use)
      step(0, k);
      stage(1, k + KD);
      step(1, k + KD);
      stage(0, k + 2 * KD);
    }
  }
  // acc = f(row, column) of every output of the tile: all loads before the first use
  template <typename F>
  static __device__ __forceinline__ void load(f32x4 (&acc)[MI][NI], F f) {
    each(acc, [&](int i, int j, float& v) { v = f(i, j); });
  }
  // f(i, j, row, column) of every MFMA tile of the lane: acc[i][j] holds rows row .. row + 3 of a column
  template <typename F>
  static __device__ __forceinline__ void tiles(F f) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) f(i, j, (wave & 1) * (BM / 2) + 16 * i + 4 * (lane >> 4), (wave >> 1) * (BN / 2) + 16 * j + (lane & 15));
  }
  // f(row, column, sum) of every output of the tile
  template <typename F>
  static __device__ __forceinline__ void each(f32x4 (&acc)[MI][NI], F f) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[i][j][r];
          f((wave & 1) * (BM / 2) + 16 * i + 4 * (lane >> 4) + r, (wave >> 1) * (BN / 2) + 16 * j + (lane & 15), v);
          acc[i][j][r] = v;
        }
  }
  template <typename F>
  static __device__ __forceinline__ void both(f32x4 (&acc)[MI][NI], f32x4 (&old)[MI][NI], F f) {
    int at = 0;
    each(acc, [&](int i, int j, float v) {
      f(i, j, v, old[at / (4 * NI)][at / 4 % NI][at % 4]);
      ++at;
    });
  }
};

// block b of a grid padded to a multiple of 8 -> its place in a list of n tiles that gives each XCD (b % 8) one run of neighbours
__device__ __forceinline__ int xcd_run(int b, int n) {
  const int per = (n + 7) / 8, t = (b & 7) * per + (b >> 3);
  return (b >> 3) < per && t < n ? t : -1;
}
// t -> (i, j <= i) of a triangle's tiles, row by row
__device__ __forceinline__ void triangle(int t, int& i, int& j) {
  i = (int)((__builtin_sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
  while (i * (i + 1) / 2 > t) --i;
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  j = t - i * (i + 1) / 2;
}

}  // namespace llj
