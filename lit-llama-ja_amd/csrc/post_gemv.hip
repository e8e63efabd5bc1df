// Decode products of hybrid models with bf16 weights (N, K): few activation rows (M <= 16), each
// weight read once and fed straight from its registers to the MFMA units.
//
// One row runs on rowdot.h, also as the residual after a sublayer (llj_post_linear) and as the residual streams
// (llj_streams_linear). From two rows on (and for a row of more than kRdMaxC values):
// a workgroup owns 16 output columns; its NW waves take the 128-deep K chunks round robin, D chunks in
// flight per wave (a chunk of a column is 256 contiguous bytes, 16 B per lane and MFMA step), and their
// partial tiles are summed through LDS. Activation rows are read as MFMA fragments from memory (L2) next to the weights:
// no staging, no barrier before the stream; lanes of rows past M read row 0 and their results are dropped.
// Few columns (N / 16 workgroups would leave CUs idle): HALF forms take 8 columns per workgroup and up to 8 rows
// and put the two halves of K side by side in the MFMA tile -- operand rows 0-7 / columns 0-7 the first
// half, rows 8-15 / columns 8-15 the second; the two diagonal quarters of the result are added.
// Output bf16, plus a bias, optionally max(., 0)^2 or the clamped gated unit of interleaved columns (elem.h).
#include "common.h"
#include "elem.h"
#include "lit_llama_amd.h"
#include "rowdot.h"

namespace llj {

struct PostGemvParams {
  const bf16_t* A;  // rows, stride lda
  int lda;
  const bf16_t* W;  // (N, K)
  bf16_t* out;
  int ldo, M, N, K;
  const float* bias;  // (N) or NULL
  float limit, alpha;  // clamped gated unit
};

template <int NW, int D, int ACT, bool HALF>
__global__ __launch_bounds__(NW * 64) void post_gemv_kernel(PostGemvParams p) {
  __shared__ __align__(16) float red[NW * 256];  // [NW][64][4]
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int row = lane & 15, g = lane >> 4;
  constexpr int CW = HALF ? 8 : 16;
  const int K = p.K, KC = HALF ? K >> 8 : K >> 7, n0 = blockIdx.x * CW;
  const int rc = HALF ? row & 7 : row, koff = HALF && row >= 8 ? K >> 1 : 0;  // column / row of the lane, its K half
  const u32x4* wp = reinterpret_cast<const u32x4*>(p.W + (size_t)(n0 + rc) * K + koff + 8 * g);
  const u32x4* ap = reinterpret_cast<const u32x4*>(p.A + (size_t)(rc < p.M ? rc : 0) * p.lda + koff + 8 * g);
  u32x4 wr[D][4], ar[D][4];
  auto load = [&](int d, int i) {
    int c = wave + NW * i;
    c = c < KC ? c : KC - 1;  // past the end: a valid chunk, not used
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ar[d][s] = ap[(size_t)c * 16 + 4 * s];
      wr[d][s] = __builtin_nontemporal_load(wp + (size_t)c * 16 + 4 * s);
    }
  };
  const int n = KC > wave ? (KC - wave + NW - 1) / NW : 0;
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < n; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int i = i0 + d;
      if (i < n) {  // (uniform)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          acc = mfma_bf16(__builtin_bit_cast(bf16x8, ar[d][s]), __builtin_bit_cast(bf16x8, wr[d][s]), acc);
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

template <int NW, int D, bool HALF>
static int post_gemv_go(const PostGemvParams& p, int act, hipStream_t s) {
  const dim3 grid(p.N / (HALF ? 8 : 16)), nt(NW * 64);
  if (act == 2) hipLaunchKernelGGL((post_gemv_kernel<NW, D, 2, HALF>), grid, nt, 0, s, p);
  else if (act) hipLaunchKernelGGL((post_gemv_kernel<NW, D, 1, HALF>), grid, nt, 0, s, p);
  else hipLaunchKernelGGL((post_gemv_kernel<NW, D, 0, HALF>), grid, nt, 0, s, p);
  LLJ_CHECK_LAUNCH();
  return 0;
}

#ifndef LLJ_PG_HALF_M
#define LLJ_PG_HALF_M 8  // largest row count that takes the half-K form where it applies (A/B; 0: never)
#endif
static int post_gemv_launch(const PostGemvParams& p, int act, hipStream_t s) {
  // waves: 8 for long K, so that a wave's chunks stay within a few rounds of the D in flight
  if (p.M <= LLJ_PG_HALF_M && p.N / 16 < 256 && p.K % 256 == 0 && p.K >= 1024)
    return p.K > 4096 ? post_gemv_go<8, 5, true>(p, act, s) : post_gemv_go<4, 4, true>(p, act, s);
  return p.K > 2048 ? post_gemv_go<8, 4, false>(p, act, s) : post_gemv_go<4, 4, false>(p, act, s);
}

constexpr int kPostMaxK = 28544;  // widest weight rows of the post and streams forms

template <int PRO>
static int rowdot_act(const RowDotParams& r, int act, hipStream_t s) {
  if (act == 2) {
    if constexpr (PRO != RD_POST) return rowdot_launch<PRO, RD_GLU>(r, s);
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
  LLJ_REQUIRE(act >= 0 && act <= 2 && (act != 1 || !bias) && A && W && out && M >= 1 && M <= 16 && N > 0 && N % 16 == 0 &&
              K > 0 && K % 128 == 0 && lda >= K && (lda & 7) == 0 && ldo >= (act == 2 ? N / 2 : N) &&
              (((uintptr_t)A | (uintptr_t)W) & 15) == 0);
  if (M == 1 && K <= kRdMaxC) {
    RowDotParams r{};
    r.A = (const bf16_t*)A; r.W = (const bf16_t*)W; r.out = (bf16_t*)out; r.N = N; r.K = r.C = K; r.bias = bias;
    r.limit = limit; r.alpha = alpha;
    return rowdot_act<RD_PLAIN>(r, act, (hipStream_t)stream);
  }
  PostGemvParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.W = (const bf16_t*)W; p.out = (bf16_t*)out; p.ldo = ldo; p.M = M; p.N = N; p.K = K;
  p.bias = bias; p.limit = limit; p.alpha = alpha;
  return post_gemv_launch(p, act, (hipStream_t)stream);
}

int llj_post_linear(int act, const void* t, const void* norm_w, float eps, const float* x, float* x_out, int C,
                    const void* W, void* out, int N, int K, void* stream) {
  LLJ_REQUIRE((act == 0 || act == 1) && t && norm_w && x && x_out && x != x_out && W && out && C > 0 && C % 8 == 0 &&
              C <= K && C <= 8192 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && K <= kPostMaxK &&
              (((uintptr_t)t | (uintptr_t)norm_w | (uintptr_t)x | (uintptr_t)x_out | (uintptr_t)W) & 15) == 0);
  RowDotParams r{};
  r.t = (const bf16_t*)t; r.w = (const bf16_t*)norm_w; r.x = x; r.xo = x_out; r.eps = eps; r.C = C;
  r.W = (const bf16_t*)W; r.out = (bf16_t*)out; r.N = N; r.K = K;
  return rowdot_act<RD_POST>(r, act, (hipStream_t)stream);
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
