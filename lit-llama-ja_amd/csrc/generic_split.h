// fp32 products of more than GL_ROWS rows on the bf16 matrix cores: y = x . W^T for any M, N, K and strides.
//
// An fp32 value is the sum of three bf16 values (each the rest's nearest: 8 + 8 + 8 bits), and a product of two such sums needs six of the
// nine partial products: the three left out are together below 2^-24 of the product, 2^-27.5 in the root mean square over random
// mantissas, and of either sign. The bf16 rate is 16 times the fp32 one, so six products leave 2.7 times its ceiling (157 TFLOP/s dense).
//
// A workgroup computes 16 MI rows x 128 columns, wave w all rows of columns 32 w .. +31. The weights go from memory to the wave's registers
// (each wave has its own columns, so LDS would move them twice) and are split there, one tile of 32 values of K ahead; the rows of x are split
// on their way into LDS, three planes of 64 bytes a row, and are read by all four waves. Lane group g of an MFMA holds the values 4 g .. 4 g + 3
// and 16 + 4 g .. of a tile, so that 16 lanes' loads are 16 runs of 64 bytes; the 16-byte chunk g of row r is at place g ^ (r / 4 % 4), which
// spreads 16 rows over all banks. Two to four workgroups a CU: one's splitting (5.5 instructions a value) runs beside another's products.
//
// Sums: the six products of a tile make one chain from zero, the small ones first; tiles are added in fp32, eight at a time. The matrix cores round
// a sum of products towards minus infinity, which would add up over K (a mean error of 0.6 of its deviation at K = 4096, 0.73 at 11008), so
// every other tile is formed with -x and subtracted. Error against float64 in the 2-norm, random operands (fp32 MFMA before): 7.7e-8 at K = 780
// (9.1e-8), 1.03e-7 at 4096 in one piece and 8.8e-8 in four (1.40e-7, 1.32e-7 in three), 1.01e-7 at 11008 in four (1.36e-7 in eight).
// Both operands are multiplied by 2^24 before they are split and the sums by 2^-48 at the end: the lowest part of any fp32 value, the smallest
// denormal's included, is then a normal bf16 number, and no part of a product falls below fp32's range (unscaled, rows of 1e-35 were 2.7e-6 from
// float64, rows of 1e-37 2.6e-4; scaled 1.03e-7 as at any size). Sums past 2^79 and values past 2^103 leave the range at the other end and are
// formed again as below. It costs an instruction a value: 301 rows 4096 -> 12288 212 us and 215, 4096 -> 4096 70 and 72,
// 11008 -> 4096 165 and 180, 780 -> 2048 the same.
//
// Up to kGgFineK without K ranges the sums of K's halves are kept apart from 8 tiles on (the second half starts at the same sign).
//
// A value that is not finite, or rounds to infinity, spoils its outputs' other parts: outputs that are not finite are formed again on the
// fp32 matrix cores at the end, a row of tiles at a time, in chains of 4 values, their pairs up to two tiles, and fours (K = 4096 in one piece 1.10e-7 against
// 1.15e-6 in one chain, 1.40e-7 in the fp32 products before; K = 780 8.9e-8, 5.0e-7 and 9.1e-8).
//
// Bound: the bf16 rate at the clock that it sustains (about 1.3 PFLOP/s, 217 TFLOP/s in sixths); below some 40 rows the weights' bytes. us before
// (v_mfma_f32_32x32x2_f32) and now, weights from memory: 301 rows 4096 -> 12288 270, 215 (141 TFLOP/s), 4096 -> 4096 103, 72, 11008 -> 4096 267, 180,
// 4096 -> 32000 695, 512 (154), 2048 rows 4096 -> 4096 534, 432 (159), 16 rows 4096 -> 12288 69, 48 (4.2 TB/s), 1000 rows 780 -> 2304 76, 43, 70 rows
// 780 -> 2304 23, 14.
#pragma once
#include "common.h"
#include "generic_gemm.h"

namespace llj {

constexpr int kGsBN = 128, kGsKT = 32, kGsMostMI = 6;
constexpr float kGsUp = 0x1p24f, kGsDown = 0x1p-48f;  // of both operands before they are split, of the sums

// two fp32 values as three pairs of bf16
__device__ __forceinline__ void gs_split(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  p0 = cvt_pk(f32x2{a, b});
  a -= bflo(p0);
  b -= bfhi(p0);
  p1 = cvt_pk(f32x2{a, b});
  a -= bflo(p1);
  b -= bfhi(p1);
  p2 = cvt_pk(f32x2{a, b});
}

// elements k .. k + 3 of a row, k in the tile (or half of one) that ends before `end`. LD: 2 aligned, K a multiple of 32; 1 aligned, K a multiple of 4; 0
// neither: 16 bytes from any element on, single elements where the tile passes K (single ones everywhere: 3101 -> 3000, 64 rows 44 us for 23).
// Past K: zeros, or (FILL false) other elements of the row.
typedef f32x4 __attribute__((aligned(4))) gs_any4;
template <int LD, bool FILL>
__device__ __forceinline__ f32x4 gs_ld(const float* row, int k, int end, int K) {
  f32x4 v;
  if constexpr (LD == 0) {
    if (end <= K) return *reinterpret_cast<const gs_any4*>(row + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = row[min(k + i, K - 1)];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = !FILL || k + i < K ? v[i] : 0.f;
  } else {
    v = *reinterpret_cast<const f32x4*>(row + (LD == 2 ? k : min(k, K - 4)));
    if (LD == 1 && FILL) v = k < K ? v : f32x4{};
  }
  return v;
}

// part: as gg_kernel's. Blocks: gg_kernel's from eight column tiles on; below, where a column tile to an XCD would leave XCDs without work, tile by tile.
// Past K the weights are other elements of their row, times the zeros of x (one that is not finite: formed again as below).
template <int MI, int LD>
__global__ __launch_bounds__(256, 2) void gs_kernel(const float* __restrict__ x, int ldx, int M, int K, const float* __restrict__ W, int N,
                                                    float* __restrict__ y, int ldy, const float* resid, int ldr, float* __restrict__ part,
                                                    int split_tiles) {
  constexpr int BM = 16 * MI, JX = (BM * 8 + 255) / 256, PL = BM * 64;  // JX: 16-byte loads of x per thread, PL: bytes of a plane
  __shared__ __align__(16) char lds[2][3 * PL];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), g = lane >> 4, r = lane & 15;
  const int mt = (M + BM - 1) / BM, cols = (N + kGsBN - 1) / kGsBN, local = blockIdx.x >> 3;
  int nt = (int)(blockIdx.x & 7) + 8 * (local / mt), mb = local % mt;
  if (cols < 8) {  // (gs_launch: tile by tile, or all on one XCD)
    const int b = (int)gridDim.x == cols * mt ? (int)blockIdx.x : blockIdx.x & 7 ? cols * mt : local;
    nt = b / mt;
    mb = b % mt;
  }
  if (nt >= cols) return;
  const int m0 = mb * BM, n0 = nt * kGsBN + wave * 32;
  const int t0 = blockIdx.y * split_tiles, t1 = min((K + kGsKT - 1) / kGsKT, t0 + split_tiles);

  const float *xr[JX], *wr[2];
  int xo[JX];
#pragma unroll
  for (int j = 0; j < JX; ++j) {
    const int row = (tid + 256 * j) >> 3, c = tid & 7;  // c: 16 bytes of the tile's 128
    xr[j] = x + (size_t)min(m0 + row, M - 1) * ldx;
    xo[j] = row * 64 + (((c & 3) ^ (row >> 2 & 3)) << 4) + (c >> 2) * 8;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) wr[j] = W + (size_t)min(n0 + 16 * j + r, N - 1) * K;
  // an odd MI leaves half a load per thread: waves 0 and 1 take it
  auto mine = [&](int j) { return MI % 2 == 0 || j + 1 < JX || wave < 2; };
  f32x4 xv[JX], wv[2][2];
  auto fetch_x = [&](int t) {
#pragma unroll
    for (int j = 0; j < JX; ++j)
      if (mine(j)) xv[j] = gs_ld<LD, true>(xr[j], t * kGsKT + 4 * (tid & 7), t * kGsKT + kGsKT, K);
  };
  auto fetch_w = [&](int t) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) wv[j][h] = gs_ld<LD, false>(wr[j], t * kGsKT + 16 * h + 4 * g, t * kGsKT + kGsKT, K);
  };
  auto stage_x = [&](int t, bool negative) {
    char* b = lds[(t - t0) & 1];
#pragma unroll
    for (int j = 0; j < JX; ++j)
      if (mine(j)) {
        uint2 p0, p1, p2;
        const f32x4 v = xv[j] * (negative ? -kGsUp : kGsUp);
        gs_split(v[0], v[1], p0.x, p1.x, p2.x);
        gs_split(v[2], v[3], p0.y, p1.y, p2.y);
        *reinterpret_cast<uint2*>(b + xo[j]) = p0;
        *reinterpret_cast<uint2*>(b + PL + xo[j]) = p1;
        *reinterpret_cast<uint2*>(b + 2 * PL + xo[j]) = p2;
      }
  };

  f32x4 mid[MI][2] = {}, tot[MI][2] = {};
  const int ra = r * 64 + ((g ^ (r >> 2)) << 4);
  // past the last tile: its own elements again, not used; not at all where they may be single elements, each as many requests as 16 bytes
  auto wanted = [&](int t) { return LD != 0 || t < t1; };
  fetch_x(t0);
  fetch_w(t0);  // (before x is waited for)
  stage_x(t0, false);
  if (wanted(t0 + 1)) fetch_x(min(t0 + 1, t1 - 1));
  auto step = [&](int t, bool negative, bool next) {  // the signs of tile t and the next one (constants at every call)
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");  // tile t is staged, and every wave is done with the other buffer
    uint4 w[2][3];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      wv[j][0] *= kGsUp;
      wv[j][1] *= kGsUp;
      gs_split(wv[j][0][0], wv[j][0][1], w[j][0].x, w[j][1].x, w[j][2].x);
      gs_split(wv[j][0][2], wv[j][0][3], w[j][0].y, w[j][1].y, w[j][2].y);
      gs_split(wv[j][1][0], wv[j][1][1], w[j][0].z, w[j][1].z, w[j][2].z);
      gs_split(wv[j][1][2], wv[j][1][3], w[j][0].w, w[j][1].w, w[j][2].w);
    }
    if (wanted(t + 1)) fetch_w(min(t + 1, t1 - 1));
    if (t + 1 < t1) stage_x(t + 1, next);
    if (wanted(t + 2)) fetch_x(min(t + 2, t1 - 1));
    const char* b = lds[(t - t0) & 1] + ra;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      bf16x8 a[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8*>(b + p * PL + i * 1024);
      f32x4 s[2] = {};
      constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kW[6] = {0, 2, 1, 0, 1, 0};  // the parts' products, the smallest first
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          s[j] = mfma_bf16(a[kA[q]], __builtin_bit_cast(bf16x8, w[j][kW[q]]), s[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) mid[i][j] = negative ? mid[i][j] - s[j] : mid[i][j] + s[j];
    }
    __builtin_amdgcn_s_setprio(0);
  };
  auto flush = [&] {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        tot[i][j] += mid[i][j];
        mid[i][j] = f32x4{};
      }
  };
  const int th = K <= kGgFineK && gridDim.y == 1 && t1 - t0 >= 8 ? t0 + (t1 - t0 + 1) / 2 : t1;  // the second half's first tile
  for (int lo = t0, hi = th; lo < t1; lo = hi, hi = t1) {
    int t = lo;
    for (; t + 1 < hi; t += 2) {
      step(t, false, true);
      step(t + 1, true, false);
      if (((t - lo) & 6) == 6) flush();
    }
    if (t < hi) step(t, false, false);
    if (hi < t1) flush();
  }

  flush();
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    uint32_t bad = 0;  // a bit an output
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      bad |= fabsf(tot[i][u >> 2][u & 3]) < INFINITY ? 0u : 1u << u;
      tot[i][u >> 2][u & 3] *= kGsDown;
    }
    if (!__any(bad != 0)) continue;
    // 4 values a chain, pairs of those to two tiles, four of these, and the rest: no further from float64 than the fp32 sums of gg_kernel
    const float* row = x + (size_t)min(m0 + 16 * i + r, M - 1) * ldx;
    const int k0 = t0 * kGsKT, k1 = min(t1 * kGsKT, K);
    f32x4 held[2] = {}, part8[2] = {}, sum[2] = {};
    for (int k = k0; k < k1; k += 32) {
      f32x4 tile[2] = {};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kh = k + 16 * h;
        const f32x4 a = gs_ld<LD, true>(row, kh + 4 * g, kh + 16, K);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const f32x4 w = gs_ld<LD, true>(wr[j], kh + 4 * g, kh + 16, K);
          f32x4 s[4] = {};
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], w[e], s[e], 0, 0, 0);
          tile[j] += (s[0] + s[1]) + (s[2] + s[3]);
        }
      }
      const bool second = (k - k0) & 32, last = k + 32 >= k1;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (second) part8[j] += held[j] + tile[j];
        else if (last) part8[j] += tile[j];
        held[j] = tile[j];
        if (((k - k0) & 224) == 224 || last) {
          sum[j] += part8[j];
          part8[j] = f32x4{};
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) tot[i][u >> 2][u & 3] = bad >> u & 1 ? sum[u >> 2][u & 3] : tot[i][u >> 2][u & 3];
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + 16 * j + r;
      if (n >= N) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + 16 * i + 4 * g + e;
        if (m >= M) continue;
        const float v = tot[i][j][e];
        if (part) part[((size_t)blockIdx.y * M + m) * N + n] = v;
        else y[(size_t)m * ldy + n] = resid ? resid[(size_t)m * ldr + n] + v : v;
      }
    }
}

// Rows of a workgroup and K ranges. Microseconds: a workgroup's tile step alone on a CU (the loads' latency and the splitting: 0.88, 1.09, 1.25
// at 2, 4, 5) and its share of a CU that has several (0.75, 0.96, 1.04 at 4, 5, 6; below, the weights' bytes), partials written and
// read at 4.9 TB/s, 3 for the second launch.
struct GsPlan {
  int mi, splits;
};
inline GsPlan gs_plan(int M, int N, int K, bool split) {
  static const double kAlone[kGsMostMI] = {0.77, 0.88, 0.98, 1.09, 1.25, 1.35}, kShare[kGsMostMI] = {0.3, 0.42, 0.58, 0.75, 0.96, 1.04};
  const int all = (K + kGsKT - 1) / kGsKT;
  GsPlan best = {1, 1};
  double least = 0;
  for (int mi = 1; mi <= kGsMostMI; ++mi) {
    if (mi > 1 && 16 * (mi - 1) >= M) break;
    const long mt = (M + 16 * mi - 1) / (16 * mi), nt = (N + kGsBN - 1) / kGsBN;
    for (int s = 1; s <= (split ? kGgMaxSplit : 1) && s <= all; ++s) {
      const int per = (all + s - 1) / s;
      if ((all + per - 1) / per != s) continue;
      const double share = (double)(nt < 8 ? (nt * mt * s + 255) / 256 : ((nt + 7) / 8 * mt * s + 31) / 32) * kShare[mi - 1];
      const double us = per * (share > kAlone[mi - 1] ? share : kAlone[mi - 1]) + (s > 1 ? 3.0 + s * (double)M * N * 8 / 4.9e6 : 0.0);
      if (least == 0 || us < least) best = {mi, s}, least = us;
    }
  }
  return best;
}

inline bool gs_takes(int wkind, int dt) { return wkind == 1 && dt == 1; }

inline int gs_launch(GsPlan p, const float* x, int ldx, int M, int K, const float* W, int N, float* y, int ldy, const float* resid, int ldr, float* part,
                     hipStream_t s) {
  const int mt = (M + 16 * p.mi - 1) / (16 * p.mi), nt = (N + kGsBN - 1) / kGsBN, all = (K + kGsKT - 1) / kGsKT, per = (all + p.splits - 1) / p.splits;
  // below eight column tiles: tile by tile over the XCDs; an output of one workgroup of gg_reduce_kernel, where the parts' workgroups find a CU
  // each on that one's XCD, there: its L2 then holds the parts (both launches: 29 rows 512 -> 1, 16 ranges 8.2 us tile by tile and 5.8; with more
  // workgroups than CUs, 232 rows 2304 -> 1, 10.7 and 16.7)
  const bool one = nt < 8 && p.splits > 1 && (long)M * N <= 256 && (long)nt * mt * p.splits <= 32;
  const long blocks = one ? 8L * nt * mt : nt < 8 ? (long)nt * mt : (long)((nt + 7) / 8) * 8 * mt;
  LLJ_REQUIRE(blocks < (1L << 31));
  const dim3 grid((unsigned)blocks, p.splits);
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && (((uintptr_t)x | (uintptr_t)W) & 15) == 0;
  if (p.splits == 1) part = nullptr;
#define LLJ_GS_LD(MI, LD) \
  hipLaunchKernelGGL((gs_kernel<MI, LD>), grid, dim3(256), 0, s, x, ldx, M, K, W, N, y, ldy, resid, ldr, part, per)
#define LLJ_GS(MI)                                     \
  case MI:                                             \
    if (vec && K % kGsKT == 0) LLJ_GS_LD(MI, 2);       \
    else if (vec) LLJ_GS_LD(MI, 1);                    \
    else LLJ_GS_LD(MI, 0);                             \
    break
  switch (p.mi) {
    LLJ_GS(1);
    LLJ_GS(2);
    LLJ_GS(3);
    LLJ_GS(4);
    LLJ_GS(5);
    LLJ_GS(6);
  }
#undef LLJ_GS
#undef LLJ_GS_LD
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // namespace llj
