// C-ABI entry points of the prefill GEMMs and their instantiations for the quantized weight formats
// (device code: gemm_impl.h; bf16 weights: gemm_bf16.hip).
#include <algorithm>

#include "gemm_impl.h"

namespace llj {

// split-K residual GEMM (few row tiles: a prompt of 256..1024 rows leaves the 4096-column GEMMs at
// 64..128 workgroups): x = bf16(x + bf16(sum over the slices of their fp32 partials)), slices in order
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ ws, int nsplit, int M, int N,
                                                                 bf16_t* __restrict__ x, int ldx) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;  // 4 consecutive columns (N % 4 == 0)
  if (i >= (size_t)M * N) return;
  const int m = (int)(i / N), n = (int)(i % N);
  float4 y = *reinterpret_cast<const float4*>(ws + i);
  for (int sp = 1; sp < nsplit; ++sp) {
    const float4 v = *reinterpret_cast<const float4*>(ws + (size_t)sp * M * N + i);
    y.x += v.x; y.y += v.y; y.z += v.z; y.w += v.w;
  }
  uint2* xp = reinterpret_cast<uint2*>(x + (size_t)m * ldx + n);
  const uint2 xv = *xp;
  const uint32_t lo = pack2bf(round_bf(bflo(xv.x) + round_bf(y.x)), round_bf(bfhi(xv.x) + round_bf(y.y)));
  const uint32_t hi = pack2bf(round_bf(bflo(xv.y) + round_bf(y.z)), round_bf(bfhi(xv.y) + round_bf(y.w)));
  *xp = make_uint2(lo, hi);
}

template <int EP>
static int gemm_run(int wfmt, GemmParams& p, void* ws, size_t ws_bytes, void* stream) {
  p.ws = (float*)ws;  // K slices of fewer than 256 rows (llj_gemm_ws_bytes)
  const bool zint = (wfmt & LLJ_WF_ZINT) != 0;  // int4 only: every zero is an integer
  wfmt &= ~LLJ_WF_ZINT;
  if (zint && wfmt != GWF_W4) return LLJ_EINVAL;
  if (p.M < 1 || p.N % kGBN || p.K % kGBK || p.K < kGBK || (p.lda & 7)) return LLJ_EINVAL;
  if (EP != GEP_QKV && (!p.C || (p.ldc & 1))) return LLJ_EINVAL;
  // the int4 / bf16 kernels assume an even count of 64-deep chunks (gemm_body's __builtin_assume)
  if ((wfmt == GWF_W4 || wfmt == GWF_BF16) && p.K % 128) return LLJ_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  if (wfmt == GWF_W4) {
    if (!p.sz) return LLJ_EINVAL;
    if (zint && p.M >= 256 && w4z_enabled()) return gemm_glds_launch<GWF_W4Z, EP, 128>(p, s);
    // 129 to 255 rows: one convert-once tile of 256 against two of 128, us at 160 / 255 rows: 4096 -> 12288 50 / 50 -> 41 / 44,
    // 11008 -> 4096 45 / 50 -> 36 / 39, 4096 -> 4096 29 / 32 -> 30 / 32. Up to 128 rows one tile of 128 is the cheaper (64 rows 35, 32,
    // 23 -> 37, 32, 24), and for short sums, whose pipeline fills and drains more often (2048 -> 5632, 255 rows 28 -> 30).
    if (zint && p.M > kGBM && p.M < 256 && p.K >= 4096 && w4z_enabled()) return gemm_split_launch<GWF_W4Z, EP>(p, ws_bytes, s);
    if (p.M >= 256 && p.K % 128 == 0 && glds_enabled(GWF_W4)) return gemm_glds_run<GWF_W4, EP>(p, s);
    if (LLJ_GEMM_BM256_W4 && p.M >= 256) return gemm_launch<GWF_W4, EP, 256>(p, s);
    return gemm_split_launch<GWF_W4, EP>(p, ws_bytes, s);
  }
  if (wfmt == GWF_W8) return p.sz ? gemm_split_launch<GWF_W8, EP>(p, ws_bytes, s) : LLJ_EINVAL;
  if ((wfmt & 0xff) == GWF_W4G) {  // grouped int4: group size (128-deep chunks) in the bits above
    p.gch = wfmt >> 8;
    return (p.sz && p.gch >= 1 && p.K % 128 == 0) ? gemm_split_launch<GWF_W4G, EP>(p, ws_bytes, s) : LLJ_EINVAL;
  }
  if (wfmt == GWF_BF16) {
    const int rc = gemm_few_run(EP, p, s);
    return rc < 0 ? gemm_bf16_run(EP, p, ws_bytes, s) : rc;
  }
  if (wfmt == GWF_I8) {
    if (!p.sz || !p.i8ws || p.K % 128) return LLJ_EINVAL;
    if (!p.ao16 != !p.w16 || (p.ao16 && (p.kpad < 64 || p.kpad % 64))) return LLJ_EINVAL;
    if (LLJ_GEMM_BM256_I8 && p.M >= 256) return gemm_launch<GWF_I8, EP, 256>(p, s);
    return gemm_split_launch<GWF_I8, EP>(p, ws_bytes, s);
  }
  return LLJ_EINVAL;
}

}  // namespace llj

using namespace llj;

extern "C" {

int llj_gemm_linear_ws(int wfmt, const void* A, int lda, const void* W, const void* sz, void* C, int ldc, int M, int N,
                    int K, void* ws,
    size_t ws_bytes, void* stream) {
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.sz = (const float2*)sz;
  p.C = (bf16_t*)C; p.ldc = ldc;
  return gemm_run<GEP_STORE>(wfmt, p, ws, ws_bytes, stream);
}

int llj_gemm_linear(int wfmt, const void* A, int lda, const void* W, const void* sz, void* C, int ldc, int M, int N,
                    int K, void* stream) {
  return llj_gemm_linear_ws(wfmt, A, lda, W, sz, C, ldc, M, N, K, nullptr, 0, stream);
}

int llj_gemm_resid(int wfmt, const void* A, int lda, const void* W, const void* sz, void* x, int ldx, int M, int N,
                   int K, void* stream) {
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.sz = (const float2*)sz;
  p.C = (bf16_t*)x; p.ldc = ldx;
  return gemm_run<GEP_RESID>(wfmt, p, nullptr, 0, stream);
}

int llj_gemm_silu_mul_ws(int wfmt, const void* A, int lda, const void* W, const void* sz, void* h, int ldh, int M, int N,
                      int K, void* ws,
    size_t ws_bytes, void* stream) {
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.sz = (const float2*)sz;
  p.C = (bf16_t*)h; p.ldc = ldh;
  return gemm_run<GEP_SILU_MUL>(wfmt, p, ws, ws_bytes, stream);
}

int llj_gemm_silu_mul(int wfmt, const void* A, int lda, const void* W, const void* sz, void* h, int ldh, int M, int N,
                      int K, void* stream) {
  return llj_gemm_silu_mul_ws(wfmt, A, lda, W, sz, h, ldh, M, N, K, nullptr, 0, stream);
}

// Workspace bytes llj_gemm_resid_ws needs for this residual GEMM of 256 rows or more (0: it would not split K).
size_t llj_gemm_resid_ws_bytes(int wfmt, int M, int N, int K) {
  int kcs = 0;
  const int ns = splitk_plan(wfmt, M, N, K, &kcs);
  return ns ? (size_t)ns * M * N * sizeof(float) : 0;
}

// Scratch of the _ws forms below 256 rows (0: they would not split K).
size_t llj_gemm_ws_bytes(int wfmt, int M, int N, int K) {
  const size_t n = gemm_split_bytes(wfmt & 0xff, M, N, K);
  return (wfmt & 0xff) == GWF_W4 ? std::max(n, gemm_split_bytes(GWF_W4Z, M, N, K)) : n;  // (enough for either form of int4)
}

// llj_gemm_resid with the K range split over workgroups (few row tiles): fp32 partials into ws
// (llj_gemm_resid_ws_bytes), then one reduce launch adds them in slice order and the residual.
int llj_gemm_resid_ws(int wfmt, const void* A, int lda, const void* W, const void* sz, void* x, int ldx, int M, int N,
                      int K, void* ws, size_t ws_bytes, void* stream) {
  int kcs = 0;
  const int ns = splitk_plan(wfmt, M, N, K, &kcs);
  if (!ns) {
    GemmParams p{};
    p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.sz = (const float2*)sz;
    p.C = (bf16_t*)x; p.ldc = ldx;
    return gemm_run<GEP_RESID>(wfmt, p, ws, ws_bytes, stream);
  }
  if (!ws || ws_bytes < (size_t)ns * M * N * sizeof(float) || (lda & 7) || (ldx & 3) || !A || !W || !x) return LLJ_EINVAL;
  if ((wfmt & ~LLJ_WF_ZINT) == GWF_W4 && !sz) return LLJ_EINVAL;
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = W; p.sz = (const float2*)sz;
  p.ws = (float*)ws; p.nsplit = ns; p.kcs = kcs;
  hipStream_t s = (hipStream_t)stream;
  const int rc = wfmt == GWF_BF16 ? gemm_bf16_run(GEP_PARTIAL, p, ws_bytes, s)
                                  : gemm_glds_launch<GWF_W4Z, GEP_PARTIAL, 128>(p, s);
  if (rc) return rc;
  const size_t n4 = (size_t)M * N / 4;
  hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, (const float*)ws, ns,
                     M, N, (bf16_t*)x, ldx);
  LLJ_CHECK_LAUNCH();
  return 0;
}

// the dual SwiGLU pass's tail: h[m, n] = bf16(silu(bf16(a))) * bf16(b), a / b the c_fc1 / c_fc2 partials of the
// slices summed in slice order (4 consecutive columns per thread, N % 4 == 0)
__global__ __launch_bounds__(256) void gemm_swiglu_reduce_kernel(const float* __restrict__ ws, int nsplit, int M, int N,
                                                                 bf16_t* __restrict__ h, int ldh) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const size_t MN = (size_t)M * N;
  if (i >= MN) return;
  const int m = (int)(i / N), n = (int)(i % N);
  float4 a = *reinterpret_cast<const float4*>(ws + i), b = *reinterpret_cast<const float4*>(ws + MN + i);
  for (int sp = 1; sp < nsplit; ++sp) {
    const float4 u = *reinterpret_cast<const float4*>(ws + 2 * sp * MN + i);
    const float4 v = *reinterpret_cast<const float4*>(ws + (2 * sp + 1) * MN + i);
    a.x += u.x; a.y += u.y; a.z += u.z; a.w += u.w;
    b.x += v.x; b.y += v.y; b.z += v.z; b.w += v.w;
  }
  const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
  float o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float a1 = round_bf(av[q]);
    const float sl = round_bf(a1 / (1.f + __expf(-a1)));  // F.silu in bf16
    o[q] = sl * round_bf(bv[q]);
  }
  *reinterpret_cast<uint2*>(h + (size_t)m * ldh + n) = make_uint2(pack2bf(o[0], o[1]), pack2bf(o[2], o[3]));
}

#ifndef LLJ_GEMM_SWIGLU_TAIL
#define LLJ_GEMM_SWIGLU_TAIL 1  // the dual SwiGLU pass's partial last wave of tiles as split-K halves
#endif
// The dual SwiGLU pass over (row tiles) x (H / 64 column tiles): when the tiles leave a partial last wave
// over the CUs, its column tiles (tc of them, at the right end) run as two K halves -- twice the
// workgroups at half the length, fitting one wave -- and the full-K launch keeps only whole waves.
// Returns the tail's column tiles (0: no split), kcs = its 64-deep chunks per half.
static int swiglu_tail_plan(int M, int H, int K, int* kcs_out) {
  if (!LLJ_GEMM_SWIGLU_TAIL || M < 256 || H % 64 || K % 128 || K / 64 < 16) return 0;
  int cus = 256;
  {
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (cus <= 0) cus = 256;
  }
  const long mt = (M + 255) / 256, ntn = H / 64, tiles = mt * ntn;
  const long full = tiles / cus * cus;
  if (full == tiles || full == 0) return 0;
  const long tc = ntn - full / mt;  // the full-K launch keeps (ntn - tc) column tiles: at most the whole waves
  if (tc <= 0 || tc >= ntn || 2 * mt * tc > cus) return 0;
  int kcs = (K / 64 + 1) / 2;
  kcs += kcs & 1;
  if (kcs_out) *kcs_out = kcs;
  return (int)tc;
}

// h[M, H] = bf16(silu(bf16(A . W1^T))) * bf16(A . W2^T) in one pass: int4 W4P with integral zeros
// (wfmt 0 | LLJ_WF_ZINT), M >= 256, H % 64 == 0 (the convert-once kernel with both weights' codes per chunk)
int llj_gemm_swiglu(int wfmt, const void* A, int lda, const void* W1, const void* sz1, const void* W2, const void* sz2,
                    void* h, int ldh, int M, int H, int K, void* stream) {
  if (wfmt != (GWF_W4 | LLJ_WF_ZINT) || M < 256 || H % 64 || K % 128 || K < 128 || (lda & 7) || (ldh & 1) || !A ||
      !W1 || !W2 || !sz1 || !sz2 || !h)
    return LLJ_EINVAL;
  GemmParams p{};
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = H; p.K = K; p.W = W1; p.sz = (const float2*)sz1;
  p.W2 = W2; p.sz2 = (const float2*)sz2; p.C = (bf16_t*)h; p.ldc = ldh;
  return gemm_glds_launch<GWF_W4Z, GEP_SWIGLU, 128>(p, (hipStream_t)stream);
}

// Workspace bytes llj_gemm_swiglu_ws needs (0: no partial last wave to split -- call llj_gemm_swiglu).
size_t llj_gemm_swiglu_ws_bytes(int wfmt, int M, int H, int K) {
  if (wfmt != (GWF_W4 | LLJ_WF_ZINT) || !w4z_enabled()) return 0;
  int kcs = 0;
  const int tc = swiglu_tail_plan(M, H, K, &kcs);
  return tc ? (size_t)2 * 2 * M * (64 * tc) * sizeof(float) : 0;
}

// llj_gemm_swiglu with the partial last wave of column tiles split into two K halves (fp32 partials of both
// weights into ws, llj_gemm_swiglu_ws_bytes), one reduce launch finishing those columns of h
int llj_gemm_swiglu_ws(int wfmt, const void* A, int lda, const void* W1, const void* sz1, const void* W2, const void* sz2,
                       void* h, int ldh, int M, int H, int K, void* ws, size_t ws_bytes, void* stream) {
  int kcs = 0;
  const int tc = (wfmt == (GWF_W4 | LLJ_WF_ZINT) && w4z_enabled()) ? swiglu_tail_plan(M, H, K, &kcs) : 0;
  if (!tc) return llj_gemm_swiglu(wfmt, A, lda, W1, sz1, W2, sz2, h, ldh, M, H, K, stream);
  const int Ht = 64 * tc, Hc = H - Ht;
  if ((lda & 7) || (ldh & 3) || !A || !W1 || !W2 || !sz1 || !sz2 || !h || !ws ||
      ws_bytes < (size_t)2 * 2 * M * Ht * sizeof(float))
    return LLJ_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  int rc = llj_gemm_swiglu(wfmt, A, lda, W1, sz1, W2, sz2, h, ldh, M, Hc, K, stream);  // whole waves, full K
  if (rc) return rc;
  GemmParams p{};  // the tail's columns Hc .. H - 1: W4P column tiles are K-contiguous, so pointer offsets
  const size_t woff = (size_t)Hc * K / 2;
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = Ht; p.K = K;
  p.W = (const char*)W1 + woff; p.sz = (const float2*)sz1 + Hc;
  p.W2 = (const char*)W2 + woff; p.sz2 = (const float2*)sz2 + Hc;
  p.ws = (float*)ws; p.nsplit = 2; p.kcs = kcs;
  rc = gemm_glds_launch<GWF_W4Z, GEP_SWIGLU_PART, 128>(p, s);
  if (rc) return rc;
  const size_t n4 = (size_t)M * Ht / 4;
  hipLaunchKernelGGL(gemm_swiglu_reduce_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, (const float*)ws, 2, M,
                     Ht, (bf16_t*)h + Hc, ldh);
  LLJ_CHECK_LAUNCH();
  return 0;
}

// LLM.int8() forms (wfmt 2): W = CB in the I8P tiling, sz = SCB (fp32), i8ws = llj_i8_stats of A
int llj_gemm_i8_linear_ws(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                       const void* w16, int kpad, void* C, int ldc, int M, int N, int K, void* ws,
    size_t ws_bytes, void* stream) {
  GemmParams p{};
  p.ao16 = (const _Float16*)ao16; p.w16 = (const _Float16*)w16; p.kpad = kpad;
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = CB; p.sz = (const float2*)SCB;
  p.C = (bf16_t*)C; p.ldc = ldc; p.i8ws = (const char*)i8ws;
  return gemm_run<GEP_STORE>(GWF_I8, p, ws, ws_bytes, stream);
}

int llj_gemm_i8_linear(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                       const void* w16, int kpad, void* C, int ldc, int M, int N, int K, void* stream) {
  return llj_gemm_i8_linear_ws(A, lda, CB, SCB, i8ws, ao16, w16, kpad, C, ldc, M, N, K, nullptr, 0, stream);
}

int llj_gemm_i8_resid_ws(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                      const void* w16, int kpad, void* x, int ldx, int M, int N, int K, void* ws,
    size_t ws_bytes, void* stream) {
  GemmParams p{};
  p.ao16 = (const _Float16*)ao16; p.w16 = (const _Float16*)w16; p.kpad = kpad;
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = CB; p.sz = (const float2*)SCB;
  p.C = (bf16_t*)x; p.ldc = ldx; p.i8ws = (const char*)i8ws;
  return gemm_run<GEP_RESID>(GWF_I8, p, ws, ws_bytes, stream);
}

int llj_gemm_i8_resid(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                      const void* w16, int kpad, void* x, int ldx, int M, int N, int K, void* stream) {
  return llj_gemm_i8_resid_ws(A, lda, CB, SCB, i8ws, ao16, w16, kpad, x, ldx, M, N, K, nullptr, 0, stream);
}

int llj_gemm_i8_silu_mul_ws(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                         const void* w16, int kpad, void* h, int ldh, int M, int N, int K, void* ws,
    size_t ws_bytes, void* stream) {
  GemmParams p{};
  p.ao16 = (const _Float16*)ao16; p.w16 = (const _Float16*)w16; p.kpad = kpad;
  p.A = (const bf16_t*)A; p.lda = lda; p.M = M; p.N = N; p.K = K; p.W = CB; p.sz = (const float2*)SCB;
  p.C = (bf16_t*)h; p.ldc = ldh; p.i8ws = (const char*)i8ws;
  return gemm_run<GEP_SILU_MUL>(GWF_I8, p, ws, ws_bytes, stream);
}

int llj_gemm_i8_silu_mul(const void* A, int lda, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                         const void* w16, int kpad, void* h, int ldh, int M, int N, int K, void* stream) {
  return llj_gemm_i8_silu_mul_ws(A, lda, CB, SCB, i8ws, ao16, w16, kpad, h, ldh, M, N, K, nullptr, 0, stream);
}

int llj_gemm_i8_qkv_rope_ws(const void* x, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                         const void* w16, int kpad, void* q_out, void* kcache, void* vcache, const float* rope,
                         const int* pos, int B, int T, int C, int n_head, int S, void* ws,
    size_t ws_bytes, void* stream) {
  if (B < 1 || T < 1 || n_head < 1 || C % n_head || S < 1 || !pos || !rope) return LLJ_EINVAL;
  GemmParams p{};
  p.ao16 = (const _Float16*)ao16; p.w16 = (const _Float16*)w16; p.kpad = kpad;
  p.A = (const bf16_t*)x; p.lda = C; p.M = B * T; p.N = 3 * C; p.K = C; p.W = CB; p.sz = (const float2*)SCB;
  p.q_out = (bf16_t*)q_out; p.kcache = (bf16_t*)kcache; p.vcache = (bf16_t*)vcache; p.rope = rope; p.pos = pos;
  p.n_head = n_head; p.head_size = C / n_head; p.S = S; p.T = T; p.i8ws = (const char*)i8ws;
  if (p.head_size & 1 || C % 16) return LLJ_EINVAL;
  return gemm_run<GEP_QKV>(GWF_I8, p, ws, ws_bytes, stream);
}

int llj_gemm_i8_qkv_rope(const void* x, const void* CB, const void* SCB, const void* i8ws, const void* ao16,
                         const void* w16, int kpad, void* q_out, void* kcache, void* vcache, const float* rope,
                         const int* pos, int B, int T, int C, int n_head, int S, void* stream) {
  return llj_gemm_i8_qkv_rope_ws(x, CB, SCB, i8ws, ao16, w16, kpad, q_out, kcache, vcache, rope, pos, B, T, C, n_head, S, nullptr, 0, stream);
}

int llj_gemm_qkv_rope_ws(int wfmt, const void* x, const void* W, const void* sz, void* q_out, void* kcache, void* vcache,
                      const float* rope, const int* pos, int B, int T, int C, int n_head, int S, void* ws,
    size_t ws_bytes, void* stream) {
  if (B < 1 || T < 1 || n_head < 1 || C % n_head || S < 1 || !pos || !rope) return LLJ_EINVAL;
  GemmParams p{};
  p.A = (const bf16_t*)x; p.lda = C; p.M = B * T; p.N = 3 * C; p.K = C; p.W = W; p.sz = (const float2*)sz;
  p.q_out = (bf16_t*)q_out; p.kcache = (bf16_t*)kcache; p.vcache = (bf16_t*)vcache; p.rope = rope; p.pos = pos;
  p.n_head = n_head; p.head_size = C / n_head; p.S = S; p.T = T;
  if (p.head_size & 1 || C % 16) return LLJ_EINVAL;
  return gemm_run<GEP_QKV>(wfmt, p, ws, ws_bytes, stream);
}

int llj_gemm_qkv_rope(int wfmt, const void* x, const void* W, const void* sz, void* q_out, void* kcache, void* vcache,
                      const float* rope, const int* pos, int B, int T, int C, int n_head, int S, void* stream) {
  return llj_gemm_qkv_rope_ws(wfmt, x, W, sz, q_out, kcache, vcache, rope, pos, B, T, C, n_head, S, nullptr, 0, stream);
}

}  // extern "C"
