// Tiled matrix products of the any-shape path (generic.hip's llj_g_linear / _ws for more than GL_ROWS rows): y = x . W^T for
// any M, N, K and strides, on the matrix cores: bf16 rows, and rows of either type on codes (dense fp32: generic_split.h).
//
// A workgroup computes 64 rows x 128 columns: fp32 four waves of two 32x32 accumulators, bf16 and short fp32 chains eight of one (four of
// two: 136 us for 120 at 2048 x 4096 x 4096 bf16, more steps between barriers that one wave cannot fill). Both operands go through
// LDS as rows of 128 bytes of K (32 fp32 / 64 bf16 values), the 16-byte chunk c of row r at place c ^ (r / 2 % 8): 16 lanes
// reading one chunk of 16 consecutive rows then fall on 16 different groups of four banks (padded rows, as free of
// conflicts, left room for two workgroups per CU instead of three). One read of 16 bytes per lane (lanes 0-31 the even
// chunks, 32-63 the odd ones) is four fp32 or one bf16 MFMA step -- the products' order over K is free as long as both
// operands agree. Two LDS buffers, the next tile's loads in registers while the current one is multiplied, one barrier
// per tile.
//
// Bound: the MFMA rate (fp32 operands: v_mfma_f32_32x32x2_f32, 157 TFLOP/s dense; they need 32 of LDS's 128 bytes per clock), so
// no larger tile is needed to feed it; 64 rows waste little on prompts of some hundred rows. bf16, 100 rows, 780 -> 2304: 11 us (87 with
// one output column per wave, which reads x through the cache 8 times per weight element).
//
// fp32 sums (codes): from K = kGgFineK down an accumulator runs over 8 values of K, four of those are added pairwise, four of
// these sums in a second and the rest in a third accumulator, and from 8 tiles on each half of K by itself; above it 32 values,
// eight of those, and the rest (2-norm error against float64, random operands: 9.0e-8 at K = 780, 1.3e-7 to 1.7e-7 at 4096 and above).
#pragma once
#include "common.h"
#include "elem.h"

namespace llj {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kGgBM = 64, kGgBN = 128;
constexpr int kGgRow = 128;  // bytes of one operand row in LDS
constexpr int kGgMaxSplit = 16;
constexpr int kGgFineK = 3071;
constexpr size_t kGgForced = (size_t)128 << 20;  // most scratch of two ranges that are not there for speed

__device__ __forceinline__ f32x16 gg_mma(f32x4 a, f32x4 b, f32x16 c, float) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ f32x16 gg_mma(f32x4 a, f32x4 b, f32x16 c, bf16_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ int gg_at(int row, int chunk) { return row * kGgRow + ((chunk ^ (row >> 1 & 7)) << 4); }

// 16 bytes of one operand row in the compute type CT, from a row-major matrix of S (S = CT, or bf16 widened to fp32). VE:
// elements per load, a divisor of K and of the row stride with the rows aligned to it; zeros past K.
template <typename S, typename CT, int VE>
struct GgDense {
  static constexpr int E = 16 / (int)sizeof(CT);
  typedef S vec __attribute__((ext_vector_type(VE)));
  union {
    vec v[E / VE];
    S e[E];
  };
  __device__ __forceinline__ void load(const S* row, int k, int K) {
#pragma unroll
    for (int i = 0; i < E / VE; ++i) {
      const int kk = k + i * VE;
      v[i] = kk < K ? *reinterpret_cast<const vec*>(row + kk) : vec(0);
    }
  }
  __device__ __forceinline__ void store(void* lds) const {
    if constexpr (sizeof(S) == sizeof(CT)) {
      *reinterpret_cast<f32x4*>(lds) = __builtin_bit_cast(f32x4, *this);
    } else {
      f32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = ldv(e, i);
      *reinterpret_cast<f32x4*>(lds) = o;
    }
  }
};

// The weight tile's share of one of NT threads. Dense: 16-byte chunks of rows NT / 8 apart.
template <typename CT, int VE, int NT>
struct GgWeightDense {
  static constexpr int C = kGgBN * 8 / NT;
  GgDense<CT, CT, VE> c[C];
  __device__ __forceinline__ void load(const void* W, const float*, const float*, int, int, int n0, int N, int k0, int K, int tid) {
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int n = n0 + (tid >> 3) + NT / 8 * i;
      c[i].load(reinterpret_cast<const CT*>(W) + (size_t)(n < N ? n : N - 1) * K, k0 + (tid & 7) * (16 / (int)sizeof(CT)), K);
    }
  }
  __device__ __forceinline__ void store(char* lds, int, int, int, int, int tid) const {
#pragma unroll
    for (int i = 0; i < C; ++i) c[i].store(lds + gg_at((tid >> 3) + NT / 8 * i, tid & 7));
  }
};

// ColBlockQuantizedLinear's codes: thread t takes column t % 128 (neighbouring bytes, the storage is column-major) and
// KN of the tile's 32 values of K; the element is (q - zero) * scale in fp32.
template <int BITS, int NT>
struct GgWeightCodes {
  static constexpr int KN = 32 * kGgBN / NT, EPB = 8 / BITS, NB = KN / EPB;
  unsigned char q[NB];
  const float *sc, *zr;
  float s0, z0;
  __device__ __forceinline__ void load(const void* W, const float* scales, const float* zeros, int, int G, int n0, int N, int k0,
                                       int K, int tid) {
    const int n = n0 + (tid & 127), nn = n < N ? n : N - 1, j0 = (k0 + KN * (tid >> 7)) / EPB;
    sc = scales + (size_t)nn * G;
    zr = zeros + (size_t)nn * G;
    s0 = sc[0];
    z0 = zr[0];
#pragma unroll
    for (int i = 0; i < NB; ++i) q[i] = j0 + i < K / EPB ? reinterpret_cast<const unsigned char*>(W)[(size_t)(j0 + i) * N + nn] : 0;
  }
  __device__ __forceinline__ void store(char* lds, int group, int G, int k0, int K, int tid) const {
    const int kt = k0 + KN * (tid >> 7);
    float s = s0, z = z0;
    int g = 0;
#pragma unroll
    for (int i = 0; i < KN / 4; ++i) {
      f32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 4 * i + j, k = kt + r;
        if (G > 1 && k < K && k / group != g) {
          g = k / group;
          s = sc[g];
          z = zr[g];
        }
        o[j] = k < K ? ((float)((q[r / EPB] >> (r % EPB * BITS)) & ((1 << BITS) - 1)) - z) * s : 0.f;
      }
      *reinterpret_cast<f32x4*>(lds + gg_at(tid & 127, (tid >> 7) * (KN / 4) + i)) = o;
    }
  }
};

// WL: the weight tile's loader; T: activations and output, CT: compute type, VEX: elements per load of x, J: accumulators per wave.
// part (splits > 1): this split's fp32 sums at [split][M][N], summed by gg_reduce_kernel. FINE: short chains of sums (above), HALVES:
// those of each half of K by themselves.
// Blocks: (8 * ceil(column tiles / 8) * row tiles, splits); block b runs on XCD b % 8, whose L2 keeps a column tile's weights
// for its row tiles.
// (At least two waves per SIMD: registers stay below 256, where the compiler keeps the accumulators in plain registers and the sums
// need no copies out of the accumulation registers.)
template <typename WL, typename T, typename CT, int VEX, int J, bool FINE, bool HALVES>
__global__ __launch_bounds__(512 / J, 2) void gg_kernel(const T* __restrict__ x, int ldx, int M, int K, const void* __restrict__ W,
                                                     const float* __restrict__ sc, const float* __restrict__ zr, int group,
                                                     int N, T* __restrict__ y, int ldy, const T* resid, int ldr,
                                                     float* __restrict__ part, int split_tiles) {
  __shared__ __align__(16) char lds[2][(kGgBM + kGgBN) * kGgRow];
  constexpr int KT = kGgRow / (int)sizeof(CT), EX = 16 / (int)sizeof(CT), RT = 64 / J;  // RT: rows that the threads cover
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int mt = (M + kGgBM - 1) / kGgBM, local = blockIdx.x >> 3;
  const int nt = (int)(blockIdx.x & 7) + 8 * (local / mt);
  if (nt * kGgBN >= N) return;
  const int m0 = (local % mt) * kGgBM, n0 = nt * kGgBN, G = (K + group - 1) / group;
  const int t0 = blockIdx.y * split_tiles, all = (K + KT - 1) / KT, t1 = min(all, t0 + split_tiles);

  const T* xr[J];
#pragma unroll
  for (int j = 0; j < J; ++j) xr[j] = x + (size_t)min(m0 + (tid >> 3) + RT * j, M - 1) * ldx;
  GgDense<T, CT, VEX> a[J];
  WL w;
  auto fetch = [&](int t) {
#pragma unroll
    for (int j = 0; j < J; ++j) a[j].load(xr[j], t * KT + (tid & 7) * EX, K);
    w.load(W, sc, zr, group, G, n0, N, t * KT, K, tid);
  };
  auto stage = [&](int t) {
    char* b = lds[t & 1];
#pragma unroll
    for (int j = 0; j < J; ++j) a[j].store(b + gg_at((tid >> 3) + RT * j, tid & 7));
    w.store(b + kGgBM * kGgRow, group, G, t * KT, K, tid);
  };

  f32x16 acc[J] = {}, mid[J] = {}, tot[J] = {}, front[J] = {};
  const int th = HALVES ? t0 + (t1 - t0 + 1) / 2 : t1;  // the second half's first tile
  const int nw = (wave >> 1) * 32 * J;  // the wave's first column
  const int ra = gg_at((wave & 1) * 32 + (lane & 31), lane >> 5), rb = gg_at(kGgBM + nw + (lane & 31), lane >> 5);
  fetch(t0);
  stage(t0);
  for (int t = t0; t < t1; ++t) {
    if (HALVES && t == th) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        front[j] = tot[j] + mid[j];
        tot[j] = mid[j] = f32x16{};
      }
    }
    __syncthreads();  // tile t is staged, and every wave is done with the other buffer
    if (t + 1 < t1) fetch(t + 1);
    const char* b = lds[t & 1];
    f32x4 fa[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) fa[g] = *reinterpret_cast<const f32x4*>(b + (ra ^ g << 5));  // chunks 2 g and 2 g + 1 of the rows
    auto fb = [&](int g, int j) { return *reinterpret_cast<const f32x4*>(b + (rb ^ g << 5) + 32 * j * kGgRow); };
    if constexpr (FINE) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        f32x16 p[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) p[g] = gg_mma(fa[g], fb(g, j), f32x16{}, CT());
        mid[j] += (p[0] + p[1]) + (p[2] + p[3]);
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[j] = gg_mma(fa[g], fb(g, j), acc[j], CT());
      if constexpr (sizeof(CT) == 4) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
          mid[j] += acc[j];
          acc[j] = f32x16{};
        }
      }
    }
    if (sizeof(CT) == 4 && ((t - (HALVES && t >= th ? th : t0)) & (FINE ? 3 : 7)) == (FINE ? 3 : 7)) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        tot[j] += mid[j];
        mid[j] = f32x16{};
      }
    }
    if (t + 1 < t1) stage(t + 1);
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if constexpr (sizeof(CT) == 4) tot[j] += mid[j];
    else tot[j] = acc[j];
    if constexpr (HALVES) tot[j] = front[j] + tot[j];
    const int n = n0 + nw + 32 * j + (lane & 31);
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + (wave & 1) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
      if (m >= M) continue;
      if (part) {
        part[((size_t)blockIdx.y * M + m) * N + n] = tot[j][i];
      } else {
        float v = rnd<T>(tot[j][i]);
        if (resid) v = ldv(resid, (size_t)m * ldr + n) + v;
        stv(y, (size_t)m * ldy + n, v);
      }
    }
  }
}

// y = the splits' sums, added pairwise (and the residual), as gg_kernel's own epilogue
template <typename T>
__global__ __launch_bounds__(256) void gg_reduce_kernel(const float* __restrict__ part, int splits, int M, int N, T* __restrict__ y,
                                                        int ldy, const T* resid, int ldr) {
  const size_t n = (size_t)M * N;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    float v4[4] = {0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < splits; p += 4)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (p + j < splits) v4[j] += part[(p + j) * n + i];
    const float s = (v4[0] + v4[1]) + (v4[2] + v4[3]);
    const size_t m = i / N, c = i - m * N;
    float v = rnd<T>(s);
    if (resid) v = ldv(resid, m * ldr + c) + v;
    stv(y, m * ldy + c, v);
  }
}

template <typename T>
inline int gg_reduce(const float* part, int splits, int M, int N, T* y, int ldy, const T* resid, int ldr, hipStream_t s) {
  const size_t blocks = ((size_t)M * N + 255) / 256;
  hipLaunchKernelGGL(gg_reduce_kernel<T>, dim3(blocks < 4096 ? (unsigned)blocks : 4096u), dim3(256), 0, s, part, splits, M, N, y, ldy, resid, ldr);
  LLJ_CHECK_LAUNCH();
  return 0;
}

// K ranges of a product: what makes the last round of workgroups over the 256 CUs cheapest, against the partial sums'
// traffic and launch. Microseconds: a tile step at the MFMA rate of one CU (0.9 fp32, 0.2 bf16), partials
// written and read at 4.9 TB/s, 3 for the second launch. fine (fp32 operands, K <= kGgFineK): at least two ranges while their scratch
// is small, for the shorter sums; larger outputs keep the halves apart inside one workgroup (HALVES).
inline int gg_splits(int M, int N, int K, bool f32, bool fine) {
  const int KT = kGgRow / (f32 ? 4 : 2), all = (K + KT - 1) / KT;
  const long tiles = (long)((M + kGgBM - 1) / kGgBM) * ((N + kGgBN - 1) / kGgBN);
  const double step = f32 ? 0.9 : 0.2;
  int best = 1;
  double least = 0;
  for (int s = fine && all >= 8 && (size_t)M * N * 8 <= kGgForced ? 2 : 1; s <= kGgMaxSplit && s <= all; ++s) {
    const int per = (all + s - 1) / s;
    if ((all + per - 1) / per != s) continue;
    const double us = (double)((tiles * s + 255) / 256) * per * step + (s > 1 ? 3.0 + s * (double)M * N * 8 / 4.9e6 : 0.0);
    if (least == 0 || us < least) best = s, least = us;
  }
  return best;
}

}  // namespace llj
