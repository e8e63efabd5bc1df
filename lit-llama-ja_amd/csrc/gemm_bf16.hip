// Instantiations of the prefill GEMMs (gemm_impl.h) for bf16 (N, K) weights, and the plain products of
// models whose residual is not bf16: activation epilogues and a split-K form without a residual.
#include "gemm_impl.h"

namespace llj {

// Products of small models' prompts: so few of the other kernels' tiles that a launch is one chain of K / 64 chunk loads on a few CUs. A workgroup takes
// 16 columns and 32 rows, its 8 waves a share of K each: all of a share's operands (S steps of 32), straight from memory as the MFMA wants them, are in
// flight at once, and the shares meet in LDS in wave order. Bound: one memory trip and, past a workgroup a CU, the caches' 16 lines a load. us in a graph
// with the weights in the last-level cache, the tiles -> this, 17 / 32 / 64 / 100 / 160 / 250 rows (64 rows to a workgroup: 640 -> 1920, 64 and 160 rows 6.4, 9.1):
//   512 -> 1536  8.2 -> 3.3, 3.8, 3.8, 5.2, 5.3, 6.8   1536 -> 512  8.5 .. 10.5 -> 5.9, 7.2, 7.1, 6.7, 7.0, 7.0   640 -> 1920  9.3 .. 9.6 -> 4.0, 4.7, 4.6, 7.1, 9.3 (250: 10.0, 11.3)
//   640 -> 640   9.2 .. 9.8 -> 3.8, 4.5, 4.5, 4.3, 4.4, 6.5   1792 -> 640  8.6 .. 10.1 -> 6.4, 8.1, 7.8, 7.4, 7.8 (250: 11.4, 12.5)   1024 -> 3072  8.8 .. 11.4 -> 4.5, 5.5, 8.5, 11.3
template <int EP, int S>
__global__ __launch_bounds__(512) void gemm_few_kernel(GemmParams p) {
  constexpr int NW = 8, MT = 2;  // waves; blocks of 16 rows
  __shared__ __align__(16) float red[NW][MT][64][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), row = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT, K = p.K, KS = K >> 5, k0 = KS * wave / NW, k1 = KS * (wave + 1) / NW;
  // the epilogue's operands, ahead of the product's: an element to a thread
  const int r = tid >> 4, m = m0 + r, n = n0 + (tid & 15), Cd = p.n_head * p.head_size, mm = m < p.M ? m : p.M - 1;
  const QkvRow qr = EP == GEP_QKV ? qkv_row(p, mm) : QkvRow{};
  const QkvCol qc = EP == GEP_QKV ? qkv_col(p, n0, n, Cd) : QkvCol{};
  const float2 op = gemm_operand<EP>(p, mm, n, qr, qc);
  const bf16_t* w = reinterpret_cast<const bf16_t*>(p.W) + (size_t)(n0 + row) * K + 8 * g;
  const bf16_t* a[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a[i] = p.A + (size_t)min(m0 + 16 * i + row, p.M - 1) * p.lda + 8 * g;
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wv[S], av[S][MT];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = 32 * min(k0 + s, k1 - 1);  // (past the share: its last step again, not used)
    wv[s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + k));
#pragma unroll
    for (int i = 0; i < MT; ++i) av[s][i] = *reinterpret_cast<const u32x4*>(a[i] + k);
  }
  __builtin_amdgcn_sched_barrier(0);  // (else each step's loads move to its products)
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (k0 + s >= k1) break;  // (uniform)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = mfma_bf16(__builtin_bit_cast(bf16x8, av[s][i]), __builtin_bit_cast(bf16x8, wv[s]), acc[i]);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4*>(red[wave][i][lane]) = acc[i];
  __syncthreads();
  float y = 0.f;
#pragma unroll
  for (int q = 0; q < NW; ++q) y += red[q][r >> 4][((r & 15) >> 2) * 16 + (tid & 15)][r & 3];
  gemm_store_elem<EP>(p, y, m, n, m < p.M, tid & 15, Cd, op, qr, qc);
}

template <int EP>
static int gemm_few_go(const GemmParams& p, hipStream_t s) {
  const dim3 grid(p.N / 16, (p.M + 31) / 32);
  const int steps = (p.K / 32 + 7) / 8;  // of the largest share
#define LLJ_FEW(S) hipLaunchKernelGGL((gemm_few_kernel<EP, S>), grid, dim3(512), 0, s, p)
  if (steps <= 2) LLJ_FEW(2);  // (a step more than the share has costs what a step of it does)
  else if (steps == 3) LLJ_FEW(3);
  else if (steps == 4) LLJ_FEW(4);
  else if (steps <= 6) LLJ_FEW(6);
  else LLJ_FEW(7);
#undef LLJ_FEW
  LLJ_CHECK_LAUNCH();
  return 0;
}

// Up to 256 workgroups, of short sums 512 or 400,000 steps of K (the times above: 640 -> 1920 at 600 9.3 for the tiles' 9.6, at 960 11.3 for 10.0; 1024 -> 1024 at 512 8.1 for 10.7), but no more
// than three a CU (256 -> 4608 at 864 7.8 for 6.7, 256 -> 4096 at 768 6.4 for 6.6 and at 1,024 7.8 for 6.6; 384 -> 8192 at 1,024 8.7 for 7.6, 384 -> 4096 at 768 6.9 for 7.6).
// Only for the LLaMA entries: other models' logits move with the order of a product's sums. -1: not taken.
int gemm_few_run(int ep, const GemmParams& p, hipStream_t s) {
  const long groups = (long)(p.N / 16) * ((p.M + 31) / 32);
  if (p.M < 1 || p.K % 32 || p.K < 256 || p.K > 1792 || p.N % 16 || groups > (p.K > 1024 ? 256 : std::min(768, std::max(512, 400000 / p.K))) || (((uintptr_t)p.A | (uintptr_t)p.W) & 15) || (p.lda & 7)) return -1;
  switch (ep) {
    case GEP_STORE: return gemm_few_go<GEP_STORE>(p, s);
    case GEP_RESID: return gemm_few_go<GEP_RESID>(p, s);
    case GEP_QKV: return gemm_few_go<GEP_QKV>(p, s);
    case GEP_SILU_MUL: return gemm_few_go<GEP_SILU_MUL>(p, s);
  }
  return -1;
}

template <int EP>
static int bf16_run(const GemmParams& p, size_t ws_bytes, hipStream_t s) {
  if (p.M >= 256 && glds_enabled(GWF_BF16)) return gemm_glds_run<GWF_BF16, EP>(p, s);
  if (LLJ_GEMM_BM256 && p.M >= 256) return gemm_launch<GWF_BF16, EP, 256>(p, s);
  return gemm_split_launch<GWF_BF16, EP>(p, ws_bytes, s);
}

int gemm_bf16_run(int ep, const GemmParams& p, size_t ws_bytes, hipStream_t s) {
  switch (ep) {
    case GEP_STORE: return bf16_run<GEP_STORE>(p, ws_bytes, s);
    case GEP_RESID: return bf16_run<GEP_RESID>(p, ws_bytes, s);
    case GEP_QKV: return bf16_run<GEP_QKV>(p, ws_bytes, s);
    case GEP_SILU_MUL: return bf16_run<GEP_SILU_MUL>(p, ws_bytes, s);
    case GEP_RELU2: return bf16_run<GEP_RELU2>(p, ws_bytes, s);
    case GEP_BIAS: return bf16_run<GEP_BIAS>(p, ws_bytes, s);
    case GEP_GLU: return bf16_run<GEP_GLU>(p, ws_bytes, s);
    case GEP_PARTIAL: return gemm_glds_launch<GWF_BF16, GEP_PARTIAL, 128>(p, s);
  }
  return LLJ_EINVAL;
}

// C = bf16(sum over the slices of their fp32 partials + bias), slices in order
__global__ __launch_bounds__(256) void gemm_splitk_store_kernel(const float* __restrict__ ws, int nsplit, int M, int N,
                                                                const float* __restrict__ bias, bf16_t* __restrict__ C, int ldc) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= (size_t)M * N) return;
  const int m = (int)(i / N), n = (int)(i % N);
  float4 y = *reinterpret_cast<const float4*>(ws + i);
  for (int sp = 1; sp < nsplit; ++sp) {
    const float4 v = *reinterpret_cast<const float4*>(ws + (size_t)sp * M * N + i);
    y.x += v.x; y.y += v.y; y.z += v.z; y.w += v.w;
  }
  if (bias) {
    const float4 b = *reinterpret_cast<const float4*>(bias + n);
    y.x += b.x; y.y += b.y; y.z += b.z; y.w += b.w;
  }
  *reinterpret_cast<uint2*>(C + (size_t)m * ldc + n) = make_uint2(pack2bf(y.x, y.y), pack2bf(y.z, y.w));
}

}  // namespace llj

using namespace llj;

extern "C" {
LLJ_TRACE_EXPORT(gemm_bf16)

size_t llj_gemm_bf16_ws_bytes(int M, int N, int K) {
  int kcs = 0;
  const int ns = splitk_plan(GWF_BF16, M, N, K, &kcs);
  return ns ? (size_t)ns * M * N * sizeof(float) : gemm_split_bytes(GWF_BF16, M, N, K);
}

int llj_gemm_bf16(int act, const void* A, int lda, const void* W, const float* bias, void* C, int ldc, int M, int N, int K,
                  float limit, float alpha, void* ws, size_t ws_bytes, void* stream) {
  LLJ_REQUIRE(act >= 0 && act <= 2 && (act != 1 || !bias) && A && W && C && M > 0 && N % kGBN == 0 && K % 128 == 0 && N > 0 &&
              K > 0 && lda >= K && ldc >= (act == 2 ? N / 2 : N) && (lda & 7) == 0 && (ldc & 3) == 0 &&
              ((uintptr_t)bias & 15) == 0);
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.C = (bf16_t*)C; p.ldc = ldc;
  p.bias = bias; p.limit = limit; p.alpha = alpha;
  hipStream_t s = (hipStream_t)stream;
  int kcs = 0;
  const int ns = act == 0 && ws ? splitk_plan(GWF_BF16, M, N, K, &kcs) : 0;
  if (!ns) {
    p.ws = (float*)ws;
    return gemm_bf16_run(act == 2 ? GEP_GLU : act ? GEP_RELU2 : bias ? GEP_BIAS : GEP_STORE, p, ws_bytes, s);
  }
  LLJ_REQUIRE(ws_bytes >= (size_t)ns * M * N * sizeof(float));
  p.ws = (float*)ws; p.nsplit = ns; p.kcs = kcs;
  if (const int rc = gemm_bf16_run(GEP_PARTIAL, p, ws_bytes, s)) return rc;
  const size_t n4 = (size_t)M * N / 4;
  hipLaunchKernelGGL(gemm_splitk_store_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, (const float*)ws, ns, M,
                     N, bias, (bf16_t*)C, ldc);
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
