// Decode products of hybrid models with bf16 weights (N, K): few activation rows (M <= 16), each weight read once.
//
// One row runs on rowdot.h, also as the residual streams (llj_streams_linear); 2 to 8 rows run on rows_gemv_kernel. 9 to 16 rows, rows
// of values that do not fit its registers, any rows with LLJ_ACT_TILES and the row that is the residual after a sublayer
// (llj_post_linear) run on post_gemv_kernel, 2 to 8 such rows (llj_post_rows) on post_rows_kernel. Output bf16, plus a bias, optionally max(., 0)^2 or the clamped gated unit of
// interleaved columns (elem.h).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "elem.h"
#include "lit_llama_amd.h"
#include "rowdot.h"

namespace llj {

struct PostGemvParams {
  const bf16_t* A;  // plain: rows, stride lda
  int lda, ldt, ldx;  // post: row strides of t, of x and x'
  const bf16_t* t;  // post: sublayer output (C), norm weight (C), residual in / out (C)
  const bf16_t* w;
  const float* x;
  float* xo;
  float eps;
  int C;
  const bf16_t* W;  // (N, K)
  bf16_t* out;
  int ldo, M, N, K;
  const float* bias;  // (N) or NULL
  float limit, alpha;  // clamped gated unit
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// the 4x4 MFMA, 16 blocks: lane 4 b + j holds 4 values of row / column j of block b; result r of the lane: row r, column j
__device__ __forceinline__ f32x4 mfma4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, u32x2{a0, a1}), __builtin_bit_cast(s16x4, u32x2{b0, b1}), c, 0, 0, 0);
}
// x summed over the two halves of the wave (WIDE) or of each 32 lanes in the lower half's lanes, y likewise in the upper half's
template <bool WIDE>
__device__ __forceinline__ float lane_split(float x, float y) {
  if constexpr (WIDE) asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
  else asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
  return x + y;
}
// with the value 4 (8) lanes further on within 16 lanes
template <int N>
__device__ __forceinline__ float quad_add(float v) { return v + dpp_f32<0x120 + N>(v); }  // row_ror

// 2 to 8 rows. Bound: the weights' bytes, and at these sizes (tens of MB) the first bytes' latency. Each of a workgroup's NW waves
// keeps the rows' values of its own share of K (up to S chunks of 128) in registers, as operands of the 4x4 MFMA whose 16 blocks
// take 16 neighbouring pieces of K: a load is 256 consecutive bytes of each of 4 columns, and the sums of a group of 4 columns
// leave the blocks once per wave, by lane swaps that halve the rows a lane holds. G groups' loads are in flight per wave, each
// chunk's register loaded anew as soon as its products are done. The 16x16 form (below) reads its rows again from L2 for every 16
// columns and, at 8 rows, multiplies as many zeros. us in a graph (TB/s), 8 rows, 16x16 form -> this:
//   2048 -> 8448   12.5 (2.8) -> 9.3 (3.7)      8448 -> 2048   13.4 (2.6) -> 10.9 (3.2)    2048 -> 6272   9.3 (2.8) -> 7.6 (3.4)
//   2048 -> 2048    6.7 (1.3) -> 5.1 (1.7)      2048 -> 32000  31.8 (4.1) -> 23.1 (5.7)    4096 -> 4096  10.6 (3.2) -> 9.0 (3.7)
//   4096 -> 26112  54.1 (4.0) -> 35.0 (6.1)    16512 -> 4096   37.6 (3.6) -> 33.4 (4.1)   13056 -> 4096  28.5 (3.8) -> 22.1 (4.8)
//   2 rows: 2048 -> 8448 11.1 -> 7.9, 4096 -> 26112 47.3 -> 35.8, 16512 -> 4096 34.8 -> 28.4
template <int NW, int S, int G, int MG, int ACT>
__global__ __launch_bounds__(NW * 64) void rows_gemv_kernel(PostGemvParams p) {
  extern __shared__ __align__(16) float part[];  // [column][NW][RW]
  constexpr int RW = 4 * MG;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), b = lane >> 2, j = lane & 3;
  const int K = p.K, KC = K >> 7, groups = p.N >> 2;
  const int g0 = (int)((long)blockIdx.x * groups / gridDim.x), g1 = (int)((long)(blockIdx.x + 1) * groups / gridDim.x);
  const int k0 = KC * wave / NW, n = KC * (wave + 1) / NW - k0;  // this wave's chunks, at most S
  u32x4 a[S][MG], wr[G][S];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int g = 0; g < MG; ++g) {
      const int m = 4 * g + j, c = k0 + s < KC ? k0 + s : KC - 1;
      a[s][g] = *reinterpret_cast<const u32x4*>(p.A + (size_t)(m < p.M ? m : 0) * p.lda + 128 * c + 8 * b);
    }
  // This workgroup's columns as a buffer: a load past this wave's chunks or past the columns fetches nothing, so that the count of
  // loads in flight is the same everywhere.
  const __amdgpu_buffer_rsrc_t weights =
      __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + (size_t)4 * g0 * K), 0, (g1 - g0) * 8 * K, 0x00020000);
  const int lane_at = 2 * (j * K + 128 * k0 + 8 * b);
  auto load = [&](int g, int s, int grp) {
    const int at = s < n && grp < g1 ? lane_at + 8 * (grp - g0) * K + 256 * s : 0x7ffffff0;  // (all of it in the checked offset)
    wr[g][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(weights, at, 0, 2));  // non-temporal
  };
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int s = 0; s < S; ++s) load(g, s, g0 + g);
  auto round = [&](int grp, auto more) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4 acc[MG];
#pragma unroll
      for (int i = 0; i < MG; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const u32x4 w = wr[g][s];
        if (s < n) {  // (uniform)
#pragma unroll
          for (int i = 0; i < MG; ++i) {
            acc[i] = mfma4(a[s][i][0], a[s][i][1], w[0], w[1], acc[i]);
            acc[i] = mfma4(a[s][i][2], a[s][i][3], w[2], w[3], acc[i]);
          }
        }
        if constexpr (decltype(more)::value) load(g, s, grp + G + g);
      }
      if (grp + g >= g1) continue;
      // acc[i][r]: row 4 i + r, column j, block b's share. Lanes 0-31 / 32-63, then the 16-lane rows, keep half of the rows each.
      // (The first additions are the compiler's, which waits for the products; the swaps' asm does not.)
#pragma unroll
      for (int i = 0; i < MG; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = quad_add<4>(acc[i][r]);
      float* dst = part + ((size_t)(4 * (grp + g - g0) + j) * NW + wave) * RW + (RW / 2) * (lane >> 5) + (RW / 4) * ((lane >> 4) & 1);
      if constexpr (MG == 2) {
        f32x4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = lane_split<true>(acc[0][r], acc[1][r]);
        const float y0 = quad_add<8>(lane_split<false>(h[0], h[2])), y1 = quad_add<8>(lane_split<false>(h[1], h[3]));
        if ((lane & 15) < 4) *reinterpret_cast<float2*>(dst) = make_float2(y0, y1);
      } else {
        const float y = quad_add<8>(lane_split<false>(lane_split<true>(acc[0][0], acc[0][2]), lane_split<true>(acc[0][1], acc[0][3])));
        if ((lane & 15) < 4) *dst = y;
      }
    }
  };
  int grp = g0;
  for (; grp + G < g1; grp += G) round(grp, std::true_type{});
  round(grp, std::false_type{});
  __syncthreads();
  auto column = [&](int m, int c) {
    float y = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) y += part[((size_t)c * NW + w) * RW + m];
    if (ACT != 1) y += p.bias ? p.bias[4 * g0 + c] : 0.f;
    return y;
  };
  const int cols = (4 * (g1 - g0)) >> (ACT == 2 ? 1 : 0), o0 = (4 * g0) >> (ACT == 2 ? 1 : 0);
  for (int i = tid; i < cols * RW; i += NW * 64) {
    const int m = i % RW, c = i / RW;
    if (m >= p.M) continue;
    float y;
    if constexpr (ACT == 2) {
      y = clamped_glu(column(m, 2 * c), column(m, 2 * c + 1), p.limit, p.alpha);
    } else {
      y = column(m, c);
      if (ACT == 1) y = fmaxf(y, 0.f) * fmaxf(y, 0.f);
    }
    p.out[(size_t)m * p.ldo + o0 + c] = f2bf(y);
  }
}

constexpr int kRowsMaxK = 8 * 17 * 128;

template <int NW, int S, int G, int MG, int ACT>
static int rows_gemv_go(const PostGemvParams& p, hipStream_t s) {
  // one, two, four .. workgroups per CU, 8 waves per CU at most, at least 8 column groups each: the rows' loads are the same in
  // every workgroup (2048 -> 8448, 8 rows: 512 workgroups 10.7 us, 256 9.3; 2048 -> 2048: 512 7.7, 256 5.1). Very wide outputs: the
  // sums of a share stay within 48 KiB.
  const int groups = p.N / 4, most = 48 * 1024 / (4 * NW * 4 * MG * 4) - 1;
  int grid = 2048 / NW;
  while (grid > 256 && groups < 8 * grid) grid /= 2;
  grid = std::max(std::min(grid, groups), (groups + most - 1) / most);
  const size_t lds = (size_t)((groups + grid - 1) / grid) * 4 * NW * 4 * MG * 4;
  hipLaunchKernelGGL((rows_gemv_kernel<NW, S, G, MG, ACT>), dim3(grid), dim3(NW * 64), lds, s, p);
  LLJ_CHECK_LAUNCH();
  return 0;
}

template <int MG, int ACT>
static int rows_gemv_k(const PostGemvParams& p, hipStream_t s) {
  const int KC = p.K / 128;  // chunks; S: the least built that covers them (8 rows against the 16x16 form inside the steps: 3072 -> 3072
                             // 10.7 -> 7.3 us, 5120 -> 5120 22.4 -> 12.9, 17408 -> 512 20.7 -> 13.6)
  if (KC <= 8) return rows_gemv_go<2, 4, 4, MG, ACT>(p, s);
  if (KC <= 16) return rows_gemv_go<4, 4, 4, MG, ACT>(p, s);
  if (KC <= 32) return rows_gemv_go<8, 4, 4, MG, ACT>(p, s);
  if (KC <= 56) return rows_gemv_go<8, 7, 2, MG, ACT>(p, s);
  if (KC <= 72) return rows_gemv_go<8, 9, 2, MG, ACT>(p, s);
  if (KC <= 104) return rows_gemv_go<8, 13, 1, MG, ACT>(p, s);
  return rows_gemv_go<8, 17, 1, MG, ACT>(p, s);
}

template <int ACT>
static int rows_gemv_launch(const PostGemvParams& p, hipStream_t s) {
  return p.M <= 4 ? rows_gemv_k<1, ACT>(p, s) : rows_gemv_k<2, ACT>(p, s);
}

// A workgroup owns 16 output columns; its NW waves take the 128-deep K chunks round robin, D chunks in
// flight per wave, and their partial tiles are summed through LDS. A load is 256 contiguous bytes of each of 4 columns;
// the MFMA's operand (one column per lane and 16 bytes of four pieces of it) is made from four of them in a 4 KB
// patch of LDS that is the wave's own. Loads in the operand's own order touch 64 bytes of each of 16 columns. us in a graph
// (TB/s), that form -> this, the same sums:
//   8 rows: 2048 -> 8448 13.3 (2.6) -> 10.3 (3.4)   8448 -> 2048 14.8 (2.3) -> 10.3 (3.4)   2048 -> 6272 9.6 (2.7) -> 8.1 (3.2)
//           2048 -> 2048 6.7 (1.3) -> 4.2 (2.0)     2048 -> 32000 34.6 (3.8) -> 26.2 (5.0)  4096 -> 12544 32.4 (3.2) -> 22.4 (4.6)
//           4096 -> 16512 40.5 (3.3) -> 27.6 (4.9)  16512 -> 4096 40.9 (3.3) -> 32.9 (4.1)
//   post:   2048 -> 8448 11.7 -> 9.7, 4096 -> 16512 34.4 -> 28.5, 2048 -> 2048 4.9 -> 4.0
// Activation rows:
//   plain   read as MFMA fragments from memory (L2) next to the weights: no staging, no barrier before
//           the stream; lanes of rows past M read row 0 and their results are dropped;
//   post    one row (M = 1) that is the fp32 residual after a sublayer: x' = x + t / rms(t) * (1 + w) is formed
//           by every workgroup in its prologue (its operands are loaded ahead of the weight stream, which
//           then covers the reduction), rounded to bf16 as the product's input, and written once to x'.
// Few columns (N / 16 workgroups would leave CUs idle): HALF forms take 8 columns per workgroup and up to 8 rows
// and put the two halves of K side by side in the MFMA tile -- operand rows 0-7 / columns 0-7 the first
// half, rows 8-15 / columns 8-15 the second; the two diagonal quarters of the result are added.
// A row's sums are the same however many of the up to 8 rows there are. NV: post, 8-column vectors per thread that cover C (0: plain).
template <int NW, int D, int NV, int ACT, bool HALF>
__global__ __launch_bounds__(NW * 64) void post_gemv_kernel(PostGemvParams p) {
  constexpr bool POST = NV > 0;  // the row comes from LDS
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* red = reinterpret_cast<float*>(smem);            // [NW][64][4]
  float* rs = red + NW * 256;                             // [2][NW]
  constexpr int kOwn = (NW * 256 + 16) * 4;               // a chunk of weights per wave
  bf16_t* As = reinterpret_cast<bf16_t*>(smem + kOwn + NW * 4096);  // post: the row (K)
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int row = lane & 15, g = lane >> 4;
  constexpr int CW = HALF ? 8 : 16;
  const int K = p.K, KC = HALF ? K >> 8 : K >> 7, n0 = blockIdx.x * CW;
  const int rc = HALF ? row & 7 : row, koff = HALF && row >= 8 ? K >> 1 : 0;  // column / row of the lane, its K half
  // load s of a chunk: operand column 4 s + g, 16 bytes each of its 16 lanes -> LDS, 16-byte piece q of column v at place q ^ v -> as
  // the MFMA reads them
  unsigned char* mine = smem + kOwn + wave * 4096;
  const u32x4* wp[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int v = 4 * s + g;
    wp[s] = reinterpret_cast<const u32x4*>(p.W + (size_t)(n0 + (HALF ? v & 7 : v)) * K + (HALF && v >= 8 ? K >> 1 : 0)) + row;
  }
  const u32x4* ap = POST ? nullptr : reinterpret_cast<const u32x4*>(p.A + (size_t)(rc < p.M ? rc : 0) * p.lda + koff + 8 * g);
  u32x4 wr[D][4], ar[POST ? 1 : D][4];
  auto load = [&](int d, int i) {
    int c = wave + NW * i;
    c = c < KC ? c : KC - 1;  // past the end: a valid chunk, not used
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (!POST) ar[d][s] = ap[(size_t)c * 16 + 4 * s];
      wr[d][s] = __builtin_nontemporal_load(wp[s] + (size_t)c * 16);
    }
  };
  const int n = KC > wave ? (KC - wave + NW - 1) / NW : 0;
  if constexpr (POST) {
    u32x4 tv[NV], gv[NV];
    float xv[NV][8];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int k = 8 * (tid + NW * 64 * v), kk = k < p.C ? k : 0;
      tv[v] = *reinterpret_cast<const u32x4*>(p.t + kk);
      gv[v] = *reinterpret_cast<const u32x4*>(p.w + kk);
      ld8(p.x + kk, xv[v]);
    }
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d);
    float ss = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (8 * (tid + NW * 64 * v) < p.C) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += bflo(tv[v][e]) * bflo(tv[v][e]) + bfhi(tv[v][e]) * bfhi(tv[v][e]);
      }
    }
    ss = wave_sum(ss);
    if (lane == 0) rs[wave] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) tot += rs[i];
    const float r = 1.f / sqrtf(tot / (float)p.C + p.eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int k = 8 * (tid + NW * 64 * v);
      if (k < K) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float tt = (e & 1) ? bfhi(tv[v][e >> 1]) : bflo(tv[v][e >> 1]);
          const float gg = (e & 1) ? bfhi(gv[v][e >> 1]) : bflo(gv[v][e >> 1]);
          xv[v][e] = k < p.C ? xv[v][e] + tt * r * (1.f + gg) : 0.f;
        }
        st8(As + k, xv[v]);
        if (k < p.C && (unsigned)(k >> 3) % gridDim.x == blockIdx.x) st8(p.xo + k, xv[v]);
      }
    }
    for (int k = 8 * (tid + NW * 64 * NV); k < K; k += 8 * NW * 64)  // K's padding past the vectors
      *reinterpret_cast<uint4*>(As + k) = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d);
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < n; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int i = i0 + d;
      if (i < n) {  // (uniform)
#pragma unroll
        for (int s = 0; s < 4; ++s) *reinterpret_cast<u32x4*>(mine + 256 * (4 * s + g) + 16 * (row ^ (4 * s + g))) = wr[d][s];
        u32x4 wt[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) wt[s] = *reinterpret_cast<const u32x4*>(mine + 256 * row + 16 * ((4 * s + g) ^ row));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          u32x4 a;
          if constexpr (POST) a = *reinterpret_cast<const u32x4*>(As + koff + 128 * (wave + NW * i) + 32 * s + 8 * g);
          else a = ar[d][s];
          acc = mfma_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, wt[s]), acc);
        }
        if (i + D < n) load(d, i + D);
      }
    }
  }
  // lane: rows 4 g + r, column n0 + row
  *reinterpret_cast<f32x4*>(red + (wave * 64 + lane) * 4) = acc;
  __syncthreads();
  auto column = [&](int m, int c) {
    float y = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      y += red[(w * 64 + (m >> 2) * 16 + c) * 4 + (m & 3)];
      if (HALF) y += red[(w * 64 + ((m + 8) >> 2) * 16 + c + 8) * 4 + (m & 3)];
    }
    if (ACT != 1) y += p.bias ? p.bias[n0 + c] : 0.f;
    return y;
  };
  constexpr int OW = ACT == 2 ? CW / 2 : CW;  // output columns
  for (int i = tid; i < p.M * OW; i += NW * 64) {
    const int m = i / OW, c = i % OW;
    float y;
    if constexpr (ACT == 2) {
      y = clamped_glu(column(m, 2 * c), column(m, 2 * c + 1), p.limit, p.alpha);
    } else {
      y = column(m, c);
      if (ACT == 1) y = fmaxf(y, 0.f) * fmaxf(y, 0.f);
    }
    p.out[(size_t)m * p.ldo + (ACT == 2 ? n0 / 2 : n0) + c] = f2bf(y);
  }
}

template <int NW, int D, int NV, bool HALF>
static int post_gemv_go(const PostGemvParams& p, int act, hipStream_t s) {
  const size_t lds = (size_t)(NW * 256 + 16) * 4 + NW * 4096 + (NV > 0 ? (size_t)p.K * 2 : 0);
  const dim3 grid(p.N / (HALF ? 8 : 16)), nt(NW * 64);
  auto go = [&](auto kern) -> int {
    if (lds > 64 * 1024) {
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kern, grid, nt, lds, s, p);
    LLJ_CHECK_LAUNCH();
    return 0;
  };
  if (act == 2) return go(post_gemv_kernel<NW, D, NV, 2, HALF>);
  if (act) return go(post_gemv_kernel<NW, D, NV, 1, HALF>);
  return go(post_gemv_kernel<NW, D, NV, 0, HALF>);
}

constexpr int kHalfRows = 8;  // most rows of the half-K forms
static int post_threads(int K) { return K > 4096 ? 512 : 256; }

template <int NV>
static int post_gemv_launch(const PostGemvParams& p, int act, hipStream_t s) {
  const bool half = p.M <= kHalfRows && p.N / 16 < 256 && p.K % 256 == 0 && p.K >= 1024;
  if constexpr (NV > 0) {  // (the thread count is post_threads')
    if (post_threads(p.K) == 512) return half ? post_gemv_go<8, 4, NV, true>(p, act, s) : post_gemv_go<8, 4, NV, false>(p, act, s);
    return half ? post_gemv_go<4, 3, NV, true>(p, act, s) : post_gemv_go<4, 4, NV, false>(p, act, s);
  } else {
    // waves: 8 for long K, so that a wave's chunks stay within a few rounds of the D in flight. D: few enough that two workgroups
    // share a CU and one streams while the other starts and ends (8 rows, us at D = 2 / 3 / 4: 4096 -> 12544 22.4 / 25.6 / 26.3,
    // 2048 -> 8448 10.9 / 10.3 / 10.6; halves, 16512 -> 4096 34.1 / 32.9 / 34.8, 2048 -> 2048, whose waves have two chunks, 4.2 / 4.9 / 5.4)
    if (half) return p.K > 4096 ? post_gemv_go<8, 3, 0, true>(p, act, s) : post_gemv_go<4, 2, 0, true>(p, act, s);
    return p.K > 2048 ? post_gemv_go<8, 2, 0, false>(p, act, s) : post_gemv_go<4, 3, 0, false>(p, act, s);
  }
}

// 2 to 8 rows that are the fp32 residual after a sublayer (as above for one), to the bits of postnorm.hip's launch and the plain form: row by row the
// same sums over the same threads, the product's chunks on the same waves in the same order.
// Bound: the weights' bytes. A launch of its own for the norm costs 2 to 2.7 us; here every workgroup forms the rows under its first weights in
// flight, so that a CU's share of the columns is one workgroup: TW tiles side by side, NW waves and all their chunks (n = D, or D ahead) each, and past
// 256 workgroups one such group after another. us in a graph, norm + product -> this (the product alone):
//   2 rows: 2048 -> 8448 11.3 -> 9.5 (9.1)   2048 -> 6272 9.7 -> 7.2 (7.1)   4096 -> 16512 26.0 -> 23.3 (22.8)   4096 -> 12544 21.7 -> 18.9 (19.9)
//   8 rows: 2048 -> 8448 11.8 -> 11.9 (9.6)  2048 -> 6272 9.8 -> 9.6 (7.5)   4096 -> 16512 27.6 -> 26.8 (25.0)   4096 -> 12544 23.3 -> 22.5 (20.4)
// and of a program of 32 steps, whose rows come from other XCDs: 1B, 2 / 3 / 5 / 8 sequences 38.5 / 39.3 / 38.4 / 40.7 -> 35.1 / 37.0 / 37.3 / 39.4 ms, 7B,
// 2 / 3 / 8 107.4 / 108.6 / 113.0 -> 101.5 / 105.0 / 110.9. (2048 -> 8448, 8 rows, with two tiles: 264 workgroups, 15.9; at 128 registers 19.6.)
template <int NW, int TW, int D, int NV, int MR, int ACT, bool MORE>
__global__ __launch_bounds__(NW * TW * 64) void post_rows_kernel(PostGemvParams p, int rounds) {
  constexpr int NT = NW * TW * 64, RH = (MR + NT / 256 - 1) / (NT / 256);  // rows to 256 threads
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int K = p.K, KC = K >> 7, AS = K + 8;  // (rows 4 banks apart)
  unsigned char* patch = smem;                                                      // [waves][4096] a chunk of weights each
  float* rs = reinterpret_cast<float*>(smem + NW * TW * 4096);                      // [MR][4]
  bf16_t* As = reinterpret_cast<bf16_t*>(smem + NW * TW * 4096 + MR * 16);          // [MR][AS]
  float* red = reinterpret_cast<float*>(As + (size_t)MR * AS);                      // [rounds > 1 ? 2 : 1][waves][64][4]
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), team = wave / NW, w = wave % NW;
  const int row = lane & 15, g = lane >> 4, tiles = p.N >> 4, step = gridDim.x * TW, first = blockIdx.x * TW + team;
  unsigned char* mine = patch + wave * 4096;
  u32x4 wr[D][4];
  // (a load past the last tile fetches nothing, so that the count of loads in flight is the same everywhere)
  const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc((void*)p.W, 0, 2 * p.N * K, 0x00020000);
  const int lane_at = 2 * (g * K + 8 * row);
  auto load = [&](int d, int tile, int c) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int at = tile < tiles ? lane_at + 2 * (tile * 16 + 4 * s) * K + 256 * c : 0x7ffffff0;
      wr[d][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(weights, at, 0, 2));  // non-temporal
    }
  };
  // ---- the rows
  const int part = tid >> 8, lt = tid & 255;
  {
    u32x4 tv[RH][NV], gv[NV];
    float xv[RH][NV][8];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int k = 8 * (lt + 256 * v), kk = k < p.C ? k : 0;
      gv[v] = *reinterpret_cast<const u32x4*>(p.w + kk);
#pragma unroll
      for (int r = 0; r < RH; ++r) {
        const int m = part * RH + r < p.M ? part * RH + r : 0;
        tv[r][v] = *reinterpret_cast<const u32x4*>(p.t + (size_t)m * p.ldt + kk);
        ld8(p.x + (size_t)m * p.ldx + kk, xv[r][v]);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, first, w + NW * d);
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const bool in = 8 * (lt + 256 * v) < p.C;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float tt = (e & 1) ? bfhi(tv[r][v][e >> 1]) : bflo(tv[r][v][e >> 1]);
          ss += in ? tt * tt : 0.f;
        }
      }
      ss = wave_sum(ss);
      if (lane == 0 && part * RH + r < MR) rs[(part * RH + r) * 4 + (wave & 3)] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      const int m = part * RH + r;
      if (m >= MR) break;  // (uniform)
      const f32x4 q = *reinterpret_cast<const f32x4*>(rs + 4 * m);
      const float f = 1.f / sqrtf((q[0] + q[1] + q[2] + q[3]) / (float)p.C + p.eps);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int k = 8 * (lt + 256 * v);
        if (k >= K) continue;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float tt = (e & 1) ? bfhi(tv[r][v][e >> 1]) : bflo(tv[r][v][e >> 1]);
          const float gg = (e & 1) ? bfhi(gv[v][e >> 1]) : bflo(gv[v][e >> 1]);
          o[e] = k < p.C ? xv[r][v][e] + tt * f * (1.f + gg) : 0.f;
        }
        st8(As + (size_t)m * AS + k, o);
        if (k < p.C && m < p.M && (unsigned)(k >> 3) % gridDim.x == blockIdx.x) st8(p.xo + (size_t)m * p.ldx + k, o);
      }
    }
    __syncthreads();
  }
  // ---- the products
  const bf16_t* a0 = As + (size_t)(row & (MR - 1)) * AS + 8 * g;
  const int n = KC / NW;  // a multiple of D
  for (int t = 0; t < rounds; ++t) {
    const int tile = first + t * step;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < n; i0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int c = w + NW * (i0 + d);
#pragma unroll
        for (int s = 0; s < 4; ++s) *reinterpret_cast<u32x4*>(mine + 256 * (4 * s + g) + 16 * (row ^ (4 * s + g))) = wr[d][s];
        const bool next = i0 + D >= n;  // (uniform) this chunk's registers take the next tile's
        if (MORE) load(d, !next ? tile : t + 1 < rounds ? tile + step : tiles, next ? w + NW * d : c + NW * D);
        u32x4 wt[4], a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          wt[s] = *reinterpret_cast<const u32x4*>(mine + 256 * row + 16 * ((4 * s + g) ^ row));
          a[s] = *reinterpret_cast<const u32x4*>(a0 + 128 * c + 32 * s);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = mfma_bf16(__builtin_bit_cast(bf16x8, a[s]), __builtin_bit_cast(bf16x8, wt[s]), acc);
      }
    }
    float* sums = red + (t & 1) * NW * TW * 256;
    *reinterpret_cast<f32x4*>(sums + (wave * 64 + lane) * 4) = acc;
    __syncthreads();
    for (int i = tid; i < TW * p.M * 16; i += NT) {
      const int c = i & 15, m = (i >> 4) % p.M, tm = (i >> 4) / p.M, at = blockIdx.x * TW + tm + t * step;
      float y = 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q) y += sums[((tm * NW + q) * 64 + (m >> 2) * 16 + c) * 4 + (m & 3)];
      if (ACT == 1) y = fmaxf(y, 0.f) * fmaxf(y, 0.f);
      if (at < tiles) p.out[(size_t)m * p.ldo + 16 * at + c] = f2bf(y);
    }
  }
}

template <int NW, int TW, int D, int NV, int MR>
static int post_rows_go(const PostGemvParams& p, int act, hipStream_t s) {
  const int units = (p.N / 16 + TW - 1) / TW, rounds = (units + 255) / 256, grid = (units + rounds - 1) / rounds;
  const size_t lds = NW * TW * 4096 + MR * 16 + (size_t)MR * (p.K + 8) * 2 + (size_t)(rounds > 1 ? 2 : 1) * NW * TW * 1024;
  auto go = [&](auto kern) -> int {
    if (lds > 64 * 1024) {
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * TW * 64), lds, s, p, rounds);
    LLJ_CHECK_LAUNCH();
    return 0;
  };
  const bool more = rounds > 1 || p.K / 128 / NW > D;
  if (act) return more ? go(post_rows_kernel<NW, TW, D, NV, MR, 1, true>) : go(post_rows_kernel<NW, TW, D, NV, MR, 1, false>);
  return more ? go(post_rows_kernel<NW, TW, D, NV, MR, 0, true>) : go(post_rows_kernel<NW, TW, D, NV, MR, 0, false>);
}
template <int NW, int TW, int D, int NV>
static int post_rows_m(const PostGemvParams& p, int act, hipStream_t s) {
  if (p.M <= 2) return post_rows_go<NW, TW, D, NV, 2>(p, act, s);
  return p.M <= 4 ? post_rows_go<NW, TW, D, NV, 4>(p, act, s) : post_rows_go<NW, TW, NW == 8 ? 2 : D, NV, 8>(p, act, s);  // (8 rows of 4096: registers)
}

constexpr int kPostMaxK = 28544;  // widest weight rows of the post form, whose row lies in LDS (96 KB with the waves' patches); llj_streams_linear keeps the same limit

template <int PRO>
static int rowdot_act(const RowDotParams& r, int act, hipStream_t s) {
  if (act == 2) {
    return rowdot_launch<PRO, RD_GLU>(r, s);
  } else if (act == 1) {
    if constexpr (PRO != RD_STREAMS) return rowdot_launch<PRO, RD_RELU2>(r, s);
  } else {
    return rowdot_launch<PRO, RD_STORE>(r, s);
  }
  return LLJ_EINVAL;
}

}  // namespace llj

using namespace llj;

extern "C" {
LLJ_TRACE_EXPORT(post_gemv)

int llj_rows_linear(int act, const void* A, int lda, const void* W, const float* bias, void* out, int ldo, int M, int N, int K,
                    float limit, float alpha, void* stream) {
  const bool tiles = act & LLJ_ACT_TILES;
  act &= ~LLJ_ACT_TILES;
  LLJ_REQUIRE(act >= 0 && act <= 2 && (act != 1 || !bias) && A && W && out && M >= 1 && M <= 16 && N > 0 && N % 16 == 0 &&
              K > 0 && K % 128 == 0 && lda >= K && (lda & 7) == 0 && ldo >= (act == 2 ? N / 2 : N) &&
              (((uintptr_t)A | (uintptr_t)W) & 15) == 0);
  if (!tiles && M == 1 && K <= kRdMaxC) {
    RowDotParams r{};
    r.A = (const bf16_t*)A; r.W = (const bf16_t*)W; r.out = (bf16_t*)out; r.N = N; r.K = r.C = K; r.bias = bias;
    r.limit = limit; r.alpha = alpha;
    return rowdot_act<RD_PLAIN>(r, act, (hipStream_t)stream);
  }
  PostGemvParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.W = (const bf16_t*)W; p.out = (bf16_t*)out; p.ldo = ldo; p.M = M; p.N = N; p.K = K;
  p.bias = bias; p.limit = limit; p.alpha = alpha;
  hipStream_t s = (hipStream_t)stream;
  if (!tiles && M <= 8 && K <= kRowsMaxK) return act == 2 ? rows_gemv_launch<2>(p, s) : act ? rows_gemv_launch<1>(p, s) : rows_gemv_launch<0>(p, s);
  return post_gemv_launch<0>(p, act, s);
}

int llj_post_linear(int act, const void* t, const void* norm_w, float eps, const float* x, float* x_out, int C,
                    const void* W, void* out, int N, int K, void* stream) {
  LLJ_REQUIRE((act == 0 || act == 1) && t && norm_w && x && x_out && x != x_out && W && out && C > 0 && C % 8 == 0 &&
              C <= K && C <= 8192 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && K <= kPostMaxK &&
              (((uintptr_t)t | (uintptr_t)norm_w | (uintptr_t)x | (uintptr_t)x_out | (uintptr_t)W) & 15) == 0);
  PostGemvParams p{};
  p.t = (const bf16_t*)t; p.w = (const bf16_t*)norm_w; p.x = x; p.xo = x_out; p.eps = eps; p.C = C;
  p.W = (const bf16_t*)W; p.out = (bf16_t*)out; p.ldo = N; p.M = 1; p.N = N; p.K = K;
  hipStream_t s = (hipStream_t)stream;
  const int nt = post_threads(K), nv = (C / 8 + nt - 1) / nt;
  if (nv <= 1) return post_gemv_launch<1>(p, act, s);
  return post_gemv_launch<2>(p, act, s);  // C <= 8192 over 512 threads, C <= 4096 over 256
}

// K: the hybrid models' two widths, the two that were measured; every wave has whole rounds of its D chunks there. N: below 4096 columns the rows by
// themselves take the half-K form, which adds in another order.
static bool post_rows_takes(int M, int N, int K, int C) {
  return M >= 2 && M <= 8 && C > 0 && C % 8 == 0 && C <= K && (K == 2048 || K == 4096) && N >= 4096 && N % 16 == 0 && N < (1 << 29) / K;
}

// Where it is the faster. Up to 4 rows: everywhere (within 0.9 us where it is not). 5 to 8 rows cost every workgroup 1.3 us more, which pays where the product alone leaves
// most of a round of 256 workgroups empty. us with the product before it, norm and product -> this, 5 / 8 rows:
//   4096 ->  4352 21.4 / 22.5 -> 21.7 / 22.6   8448 25.3 / 27.5 -> 25.2 / 26.3   12544 30.6 / 31.4 -> 30.4 / 31.3   16512 34.2 / 36.8 -> 34.6 / 35.9, but
//            4096 18.5 / 18.7 -> 20.1 / 21.2   7168 22.7 / 23.6 -> 24.0 / 24.6    8192 22.9 / 24.6 -> 24.6 / 25.8   12288 28.1 / 29.2 -> 29.8 / 31.0
//   2048 ->  4352 13.5 / 14.0 -> 12.9 / 13.9   6272 13.8 / 15.4 -> 13.5 / 14.5    8448 15.6 / 17.1 -> 16.2 / 16.7, but
//            4096 12.3 / 12.4 -> 12.8 / 13.5  12288 17.1 / 18.4 -> 18.2 / 18.7   12544 18.7 / 18.8 -> 20.1 / 20.6   26112 26.2 / 28.3 -> 26.9 / 27.5
int llj_post_rows_ok(int M, int N, int K, int C) {
  return post_rows_takes(M, N, K, C) && (M <= 4 || (K == 2048 ? N > 4096 && N < 12288 : (N / 16 - 1) % 256 < 64));
}

int llj_post_rows(int act, const void* t, int ldt, const void* norm_w, float eps, const float* x, float* x_out, int ldx, int C, const void* W,
                  void* out, int ldo, int M, int N, int K, void* stream) {
  LLJ_REQUIRE((act == 0 || act == 1) && t && norm_w && x && x_out && x != x_out && W && out && post_rows_takes(M, N, K, C) && ldt >= C && ldx >= C &&
              ldo >= N && (ldt & 7) == 0 && (ldx & 3) == 0 &&
              (((uintptr_t)t | (uintptr_t)norm_w | (uintptr_t)x | (uintptr_t)x_out | (uintptr_t)W) & 15) == 0);
  PostGemvParams p{};
  p.t = (const bf16_t*)t; p.ldt = ldt; p.w = (const bf16_t*)norm_w; p.x = x; p.xo = x_out; p.ldx = ldx; p.eps = eps; p.C = C;
  p.W = (const bf16_t*)W; p.out = (bf16_t*)out; p.ldo = ldo; p.M = M; p.N = N; p.K = K;
  hipStream_t s = (hipStream_t)stream;
  if (K == 2048) return N <= 8192 ? post_rows_m<4, 2, 4, 1>(p, act, s) : post_rows_m<4, 3, 4, 1>(p, act, s);
  return post_rows_m<8, 1, 4, 2>(p, act, s);
}

int llj_streams_linear_ok(int streams, int C) { return streams >= 1 && streams <= kRdStreams && C % 8 == 0 && C > 0 && C <= 8192; }

int llj_streams_linear(int act, const void* y, const float* out_w, const float* mix, const float* x, float* x_out, int ldx,
                       int streams, const float* in, const void* norm_w, float eps, int C, const void* W, const float* bias,
                       void* out, int N, int K, float limit, float alpha, void* stream) {
  LLJ_REQUIRE((act == 0 || act == 2) && y && out_w && mix && x && x_out && x != x_out && in && norm_w && W && out &&
              llj_streams_linear_ok(streams, C) && C <= K && ldx >= C && ldx % 4 == 0 && N > 0 && N % 16 == 0 && K > 0 &&
              K % 128 == 0 && K <= kPostMaxK && (((uintptr_t)y | (uintptr_t)norm_w | (uintptr_t)x | (uintptr_t)x_out | (uintptr_t)W) & 15) == 0);
  RowDotParams r{};
  r.t = (const bf16_t*)y; r.w = (const bf16_t*)norm_w; r.x = x; r.xo = x_out; r.ldx = ldx; r.eps = eps; r.C = C;
  r.so = out_w; r.sm = mix; r.si = in; r.S = streams;
  r.W = (const bf16_t*)W; r.out = (bf16_t*)out; r.N = N; r.K = K; r.bias = bias; r.limit = limit; r.alpha = alpha;
  return rowdot_act<RD_STREAMS>(r, act, (hipStream_t)stream);
}

}  // extern "C"
