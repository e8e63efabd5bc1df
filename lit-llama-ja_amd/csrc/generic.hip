// The any-shape path: LLaMA configurations the streaming kernels do not tile -- n_embd % 128 != 0
// or a head size other than 64 / 128. The JA fork's own 125M config (n_embd 780, head 78; reference
// lit_llama/model.py:48-51) and the reference test's n_embd 32 / head 2 (tests/test_model.py:108-112)
// run here: tiled matrix products from 9 rows on (generic_gemm.h), below that one output column per
// wave (generic_rows.h), fp32 accumulation, the reference's bf16 rounding points (the same ones the fast kernels keep).
// Every kernel also runs in fp32 (dt = 1: activations, dense weights, KV cache and logits fp32, no
// bf16 rounding -- the reference's float32 model, e.g. evaluate/full.py's default dtype and the
// CPU config of generate.py:121): LLaMA.forward routes an fp32 model here whatever its shape.
#include "common.h"
#include "elem.h"
#include "generic_attention.h"
#include "generic_gemm.h"
#include "generic_rows.h"
#include "generic_split.h"
#include "lit_llama_amd.h"

namespace llj {

// ---- embedding (model.py:110), any C, optionally bumping the device-side decode position
template <typename T>
__global__ __launch_bounds__(256) void g_embedding_kernel(const int* __restrict__ idx, const T* __restrict__ wte,
                                                          T* __restrict__ out, int C, int* pos_inc) {
  const int m = blockIdx.x;
  const size_t r = (size_t)idx[m];
  for (int v = threadIdx.x; v < C; v += blockDim.x) out[(size_t)m * C + v] = wte[r * C + v];
  if (pos_inc && m == 0 && threadIdx.x == 0) *pos_inc += 1;
}

// ---- RMSNorm (model.py:276-283; on bf16 tensors every op rounds): one block per row, any C
template <typename T>
__global__ __launch_bounds__(256) void g_rmsnorm_kernel(const T* __restrict__ x, int ldx, const T* __restrict__ w,
                                                        float eps, T* __restrict__ y, int ldy, int C) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  const T* xr = x + (size_t)m * ldx;
  float ss = 0.f;
  for (int k = tid; k < C; k += 256) {
    const float v = ldv(xr, k);
    ss += rnd<T>(v * v);  // x * x (model.py:281)
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float r = rnd<T>(rsqrtf(rnd<T>(rnd<T>(tot / (float)C) + eps)));
  T* yr = y + (size_t)m * ldy;
  for (int k = tid; k < C; k += 256) stv(yr, k, ldv(w, k) * rnd<T>(ldv(xr, k) * r));
}

// ---- y[m, n] = bf16(sum_k x[m, k] W[n, k]) or, with resid, bf16(resid[m, n] + that) (the residual
// adds of model.py:172-173) of up to 8 rows on the reference's ColBlockQuantizedLinear buffers untouched -- codes in
// quant_weight's column-major storage (byte (n, j) at j N + n, 8 / bits codes per byte, code of k = j epb + r at bits
// r * bits), per-group fp32 scales / zeros (N, G), group = tile_cols (K for -1); the weight element is the Triton path's
// (q - zero) * scale in fp32 (quantization.py:250-267, 390-409). One wave per output column, lanes
// over k. T: activation type.
template <typename T>
__global__ __launch_bounds__(256) void g_code_rows_kernel(const T* __restrict__ x, int ldx, int M, int K,
                                                          const unsigned char* __restrict__ W, const float* __restrict__ sc,
                                                          const float* __restrict__ zr, int bits, int group, int N,
                                                          T* __restrict__ y, int ldy, const T* resid, int ldr) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int G = (K + group - 1) / group;
  const int epb = 8 / bits;
  const uint32_t mask = (1u << bits) - 1u;
  float acc[GL_ROWS];
#pragma unroll
  for (int r = 0; r < GL_ROWS; ++r) acc[r] = 0.f;
  for (int k = lane; k < K; k += 64) {
    const int j = k / epb, sh = (k - j * epb) * bits;
    const uint32_t q = ((uint32_t)W[(size_t)j * N + n] >> sh) & mask;
    const int g = k / group;
    const float wv = ((float)q - zr[(size_t)n * G + g]) * sc[(size_t)n * G + g];
#pragma unroll
    for (int r = 0; r < GL_ROWS; ++r)
      if (r < M) acc[r] += ldv(x, (size_t)r * ldx + k) * wv;
  }
#pragma unroll
  for (int r = 0; r < GL_ROWS; ++r) {
    const float s = wave_sum(acc[r]);
    if (lane == r && r < M) {
      float v = rnd<T>(s);
      if (resid) v = ldv(resid, (size_t)r * ldr + n) + v;
      stv(y, (size_t)r * ldy + n, v);
    }
  }
}

// ---- a biased Linear's second pass: y += bias in place (act 0), or the clamped gated unit of its interleaved
// columns (gate 2 j, up 2 j + 1, bias added to both) into out[j] (act 2)
template <typename T>
__global__ __launch_bounds__(256) void g_bias_act_kernel(int act, T* y, int ldy, const float* __restrict__ bias, T* out, int ldo,
                                                         int M, int N, float limit, float alpha) {
  const int cols = act ? N / 2 : N;
  const size_t n = (size_t)M * cols;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const size_t m = i / cols;
    const int c = (int)(i - m * cols);
    if (act) {
      const float g = ldv(y, m * ldy + 2 * c) + (bias ? bias[2 * c] : 0.f);
      const float u = ldv(y, m * ldy + 2 * c + 1) + (bias ? bias[2 * c + 1] : 0.f);
      stv(out, m * ldo + c, clamped_glu(g, u, limit, alpha));
    } else {
      stv(y, m * ldy + c, ldv(y, m * ldy + c) + bias[c]);
    }
  }
}

// ---- q / k / v split of c_attn's output (model.py:204), apply_rope on q and k in fp32
// (model.py:312-329), k / v of the token at position p into cache slot p % S. Block (row, head).
template <typename TT>
__global__ __launch_bounds__(64) void g_rope_kv_kernel(const TT* __restrict__ qkv, TT* __restrict__ q_out,
                                                       TT* __restrict__ kc, TT* __restrict__ vc,
                                                       const float* __restrict__ rope, const int* __restrict__ pos,
                                                       int T, int C, int nh, int S) {
  const int m = blockIdx.x, h = blockIdx.y;
  const int hs = C / nh, b = m / T, t = m - b * T;
  const int p = pos[t], slot = p % S;
  const TT* row = qkv + (size_t)m * 3 * C + h * hs;
  const size_t cbase = (((size_t)b * nh + h) * S + slot) * hs;
  for (int i = threadIdx.x; i < hs / 2; i += 64) {
    const float c = rope[((size_t)p * (hs / 2) + i) * 2], s = rope[((size_t)p * (hs / 2) + i) * 2 + 1];
    const float q0 = ldv(row, 2 * i), q1 = ldv(row, 2 * i + 1);
    const float k0 = ldv(row, C + 2 * i), k1 = ldv(row, C + 2 * i + 1);
    const float2 q = gr_rotate(q0, q1, c, s), k = gr_rotate(k0, k1, c, s);
    stv(q_out, (size_t)m * C + h * hs + 2 * i, q.x);
    stv(q_out, (size_t)m * C + h * hs + 2 * i + 1, q.y);
    stv(kc, cbase + 2 * i, k.x);
    stv(kc, cbase + 2 * i + 1, k.y);
    vc[cbase + 2 * i] = row[2 * C + 2 * i];
    vc[cbase + 2 * i + 1] = row[2 * C + 2 * i + 1];
  }
}

// ---- causal attention (model.py:237, the tril mask rows): row m at position p attends cache
// slots [0, p] (all S slots once p >= S: the ring holds the last S positions). Scores in LDS,
// fp32 softmax, y = P V / sum (rounded to bf16 on the bf16 path). Block (row, head); LDS: S + hs floats.
template <typename TT>
__global__ __launch_bounds__(256) void g_attention_kernel(const TT* __restrict__ q, const TT* __restrict__ kc,
                                                          const TT* __restrict__ vc, TT* __restrict__ y,
                                                          const int* __restrict__ pos, int T, int C, int nh, int S) {
  extern __shared__ float g_att_lds[];
  __shared__ float red[4];
  const int m = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int hs = C / nh, b = m / T, t = m - b * T;
  const int p = pos[t];
  const int nvis = p < S ? p + 1 : S;
  float* sc = g_att_lds;       // [S]
  float* sq = g_att_lds + S;   // [hs]
  const float scale = 1.f / sqrtf((float)hs);
  for (int d = tid; d < hs; d += 256) sq[d] = ldv(q, (size_t)m * C + h * hs + d) * scale;
  __syncthreads();
  const size_t kb = ((size_t)b * nh + h) * S * hs;
  float mx = -INFINITY;
  for (int j = tid; j < nvis; j += 256) {
    const TT* kr = kc + kb + (size_t)j * hs;
    float s = 0.f;
    for (int d = 0; d < hs; ++d) s += sq[d] * ldv(kr, d);
    sc[j] = s;
    mx = fmaxf(mx, s);
  }
  // block max
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float l = 0.f;
  for (int j = tid; j < nvis; j += 256) {
    const float e = __expf(sc[j] - mx);
    sc[j] = e;
    l += e;
  }
  l = wave_sum(l);
  if ((tid & 63) == 0) red[tid >> 6] = l;
  __syncthreads();
  l = red[0] + red[1] + red[2] + red[3];
  const float inv = 1.f / l;
  for (int d = tid; d < hs; d += 256) {
    float o = 0.f;
    for (int j = 0; j < nvis; ++j) o += sc[j] * ldv(vc, kb + (size_t)j * hs + d);
    stv(y, (size_t)m * C + h * hs + d, o * inv);
  }
}

// ---- h = silu(a1) * a2 (model.py:258-259; bf16: bf16(bf16(silu(a1)) * a2))
template <typename T>
__global__ __launch_bounds__(256) void g_silu_mul_kernel(const T* __restrict__ a1, const T* __restrict__ a2,
                                                         T* __restrict__ h, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float a = ldv(a1, i);
    stv(h, i, rnd<T>(a / (1.f + expf(-a))) * ldv(a2, i));
  }
}

}  // namespace llj

using namespace llj;

// ---- LLM.int8() for any K (Linear8bitLt outside the streaming tiling, e.g. the 125M's K = 780):
// the restated bnb MatMul8bitLt (oracle/llama_np.py int8_linear, reference quantization.py:36-75):
// A16 = f16(A); outlier columns = {k : any row |A16[m, k]| >= thr}; SCA[m] = max |A16[m, k]| < thr; CA = rint(A16 * (127 / SCA)); y = f16(f16(sum_k CA CB (int32) * SCA SCB / 127^2)
// + sum_{outliers} A16 f16(CB SCB / 127)), cast to bf16. ws: K flag bytes, then M fp32 SCA.
// T: the activation type. bitsandbytes' MatMul8bitLt casts its input to fp16 (A16) whatever it is
// and casts the fp16 result back to the input dtype, so a float32 model's Linear8bitLt computes on
// f16(x) and returns fp32 holding fp16 values (no bf16 rounding, fp32 residual add).
template <typename T>
__global__ __launch_bounds__(256) void g_i8_flags_kernel(const T* __restrict__ x, int ldx, int M, int K, float thr,
                                                         unsigned char* __restrict__ flags) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= K) return;
  bool o = false;
  for (int m = 0; m < M; ++m) o |= fabsf((float)(_Float16)ldv(x, (size_t)m * ldx + k)) >= thr;
  flags[k] = o ? 1 : 0;
}
// SCA[m]: max |A16| over the row's elements below the threshold (element-wise, as double_quant's row
// statistics; an element under it in an outlier column still counts, its code is then dropped)
template <typename T>
__global__ __launch_bounds__(256) void g_i8_sca_kernel(const T* __restrict__ x, int ldx, int K, float thr,
                                                       float* __restrict__ sca) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  float mx = 0.f;
  for (int k = tid; k < K; k += 256) {
    const float a = fabsf((float)(_Float16)ldv(x, (size_t)m * ldx + k));
    if (a < thr) mx = fmaxf(mx, a);
  }
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  if (tid == 0) sca[m] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
template <typename T>
__global__ __launch_bounds__(256) void g_i8_linear_kernel(const T* __restrict__ x, int ldx, int M, int K,
                                                          const int8_t* __restrict__ CB, const float* __restrict__ SCB,
                                                          const unsigned char* __restrict__ flags,
                                                          const float* __restrict__ sca, int N, T* __restrict__ y,
                                                          int ldy, const T* resid, int ldr) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int m0 = blockIdx.y * GL_ROWS;
  const int mr = M - m0 < GL_ROWS ? M - m0 : GL_ROWS;
  const float scb = SCB[n];
  float qs[GL_ROWS];
#pragma unroll
  for (int r = 0; r < GL_ROWS; ++r) {
    const float sa = r < mr ? sca[m0 + r] : 1.f;
    qs[r] = 127.f / (sa == 0.f ? 1.f : sa);
  }
  int acc[GL_ROWS];
  float side[GL_ROWS];
#pragma unroll
  for (int r = 0; r < GL_ROWS; ++r) {
    acc[r] = 0;
    side[r] = 0.f;
  }
  for (int k = lane; k < K; k += 64) {
    const int cb = CB[(size_t)n * K + k];
    const bool o = flags[k] != 0;
    const float w16 = (float)(_Float16)((float)cb * (scb / 127.f));
#pragma unroll
    for (int r = 0; r < GL_ROWS; ++r) {
      if (r < mr) {
        const float a16 = (float)(_Float16)ldv(x, (size_t)(m0 + r) * ldx + k);
        if (o) side[r] += a16 * w16;
        else acc[r] += (int)rintf(fminf(fmaxf(a16 * qs[r], -127.f), 127.f)) * cb;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < GL_ROWS; ++r) {
    int a = acc[r];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
    const float sd = wave_sum(side[r]);
    if (lane == r && r < mr) {
      const size_t m = (size_t)(m0 + r);
      const float sa = sca[m];
      float v = (float)a * (sa * scb * (1.f / (127.f * 127.f)));
      v = (float)(_Float16)((float)(_Float16)v + sd);
      v = rnd<T>(v);
      if (resid) v = ldv(resid, m * ldr + n) + v;
      stv(y, m * ldy + n, v);
    }
  }
}

// Elements per load: 16 bytes, 8 or single elements, as x, its rows and the weights' rows are aligned. Columns per wave: four from
// 8192 on (every CU then still has 8 waves), one below.
// Pieces per round for K of n: as many as there are up to 4; then 3 or 4, whichever leaves fewer past K; single elements from 20 on 8
// (one column), where what counts is how much is in flight, and so one row of vectors to 8 in the plain form (bf16, 2080 -> 780 3.0 us, in
// rounds of 3 3.2), the last 4 behind branches. Time against 4 a round in every case (one column of the plain form 8, the last
// 4 in branches), mean over sizes, bf16 / fp32: one column, n = 1 0.86 / 0.92, 2 0.90 / 0.94, 3 0.98 / 0.97, 9 0.91 / 0.94, 40 0.79 /
// 0.88; four columns of one row, 1 0.76 / 0.71.
// 2 to 8 rows of four columns (4 weights a piece, and in the plain form as many of x as there are rows, from the caches; formed rows lie
// in LDS): fewer a round the wider the pieces. Time of 1, 2, 3, 4 a round in hundredths of what 8 behind branches took; plain, single
// elements, fp32 6 pieces 114 103 95 99, 8 126 112 107 99; of 4, bf16 6 109 92 89 101, 8 128 100 99 98; of 8, 6 98 89 94 102, 40 119 89
// 112 97; formed, single elements, fp32 6 99 88 86 89, 10 - 83 83 81; of 4, fp32 4 68 68 76 75, 12 - 89 88 87; of 8, 8 85 89 90 110, 24 92
// 94 98 132.
static int gr_pieces(int n, int ve, int nc, int M, bool plain) {
  if (nc > 1 && M > 1) {
    if (plain) return ve == 8 ? (n > 1 ? 2 : 1) : n <= 3 ? n : n == 4 ? (ve == 4 ? 2 : 4) : n <= 6 || n == 9 ? 3 : 4;
    if (ve == 1) return n == 1 ? 1 : n <= 6 ? 2 : 4;
    return n <= ve ? 1 : ve == 8 || n <= 10 ? 2 : 4;
  }
  if (n <= 4) return n;
  if (nc == 1 && (ve == 1 ? n >= 20 : n <= 8 && M == 1 && plain)) return 8;
  return (n + 2) / 3 * 3 < (n + 3) / 4 * 4 ? 3 : 4;
}

template <typename T>
static int gr_launch(int mode, const void* x, int ldx, const void* nw, float eps, int M, int K, const void* W, const void* W2,
                     int N, void* y, int ldy, const void* resid, int ldr, hipStream_t s) {
  const int el = (int)sizeof(T), nc = N >= 8192 && mode != GR_SWIGLU ? 4 : 1;
  auto fits = [&](int n) {
    return K % n == 0 && (uintptr_t)W % (n * el) == 0 && (uintptr_t)W2 % (n * el) == 0 &&
           (mode != GR_PLAIN || ((uintptr_t)x % (n * el) == 0 && (ldx % n == 0 || M == 1)));
  };
  const size_t lds = mode == GR_PLAIN ? 0 : (size_t)M * K * el;
  const dim3 grid((N + 4 * nc - 1) / (4 * nc));
#define LLJ_GR_U(VE, MB, NC, MODE, U, APART)                                                                                             \
  hipLaunchKernelGGL((g_rows_kernel<T, VE, MB, NC, MODE, U, APART>), grid, dim3(256), lds, s, (const T*)x, ldx, (const T*)nw, eps, M, K, \
                     (const T*)W, (const T*)W2, N, (T*)y, ldy, (const T*)resid, ldr)
#define LLJ_GR(VE, MB, NC, MODE)                                                                          \
  do {                                                                                                    \
    constexpr bool loop = MB > 1 && NC == 1 && MODE != GR_SWIGLU;                                         \
    constexpr bool many = MB > 1 && NC > 1, few = many && VE == 8, none3 = few || (many && MODE == GR_NORM); \
    const int n = (K + 64 * (VE) - 1) / (64 * (VE)), u = gr_pieces(n, VE, NC, M, MODE == GR_PLAIN);       \
    if (u == 1) LLJ_GR_U(VE, MB, NC, MODE, 1, !loop);                                                     \
    else if (u == 2) LLJ_GR_U(VE, MB, NC, MODE, 2, !loop);                                                \
    else if (u == 3 && loop && n == 3) LLJ_GR_U(VE, MB, NC, MODE, 3, !loop);                              \
    else if (u == 3 && !none3) LLJ_GR_U(VE, MB, NC, MODE, (none3 ? 2 : 3), true);                         \
    else if (u == 4 && loop && n == 4) LLJ_GR_U(VE, MB, NC, MODE, 4, !loop);                              \
    else if (u == 8) LLJ_GR_U(VE, MB, NC, MODE, (NC == 1 && (VE == 1 || (MB == 1 && MODE == GR_PLAIN)) ? 8 : 4), true); \
    else LLJ_GR_U(VE, MB, NC, MODE, (few ? 2 : 4), true);                                                 \
  } while (0)
#define LLJ_GR_MODE(VE, MB)                                  \
  do {                                                       \
    if (mode == GR_SWIGLU) LLJ_GR(VE, MB, 1, GR_SWIGLU);     \
    else if (mode == GR_NORM && nc == 4) LLJ_GR(VE, MB, 4, GR_NORM); \
    else if (mode == GR_NORM) LLJ_GR(VE, MB, 1, GR_NORM);    \
    else if (nc == 4) LLJ_GR(VE, MB, 4, GR_PLAIN);           \
    else LLJ_GR(VE, MB, 1, GR_PLAIN);                        \
  } while (0)
#define LLJ_GR_ROWS(VE)            \
  do {                             \
    if (M == 1) LLJ_GR_MODE(VE, 1); \
    else LLJ_GR_MODE(VE, GL_ROWS); \
  } while (0)
  if (sizeof(T) == 2 && fits(8)) LLJ_GR_ROWS((sizeof(T) == 2 ? 8 : 4));
  else if (fits(4)) LLJ_GR_ROWS(4);
  else LLJ_GR_ROWS(1);
#undef LLJ_GR_ROWS
#undef LLJ_GR_MODE
#undef LLJ_GR
#undef LLJ_GR_U
  LLJ_CHECK_LAUNCH();
  return 0;
}

extern "C" {
LLJ_TRACE_EXPORT(generic)

int llj_g_norm_ok(int M, int K, int dt) {
  return M > 0 && M <= GL_ROWS && K > 0 && (dt == 0 || dt == 1) && (size_t)M * K * (dt ? 4 : 2) <= (size_t)kGrNormLds;
}

int llj_g_norm_linear(const void* x, int ldx, const void* nw, float eps, int M, int K, const void* W, int N, void* y, int ldy,
                      int dt, void* stream) {
  LLJ_REQUIRE(x && nw && W && y && llj_g_norm_ok(M, K, dt) && N > 0 && ldx >= K && ldy >= N);
  hipStream_t s = (hipStream_t)stream;
  return dt == 0 ? gr_launch<bf16_t>(GR_NORM, x, ldx, nw, eps, M, K, W, nullptr, N, y, ldy, nullptr, 0, s)
                 : gr_launch<float>(GR_NORM, x, ldx, nw, eps, M, K, W, nullptr, N, y, ldy, nullptr, 0, s);
}

int llj_g_norm_swiglu(const void* x, int ldx, const void* nw, float eps, int M, int K, const void* W1, const void* W2, int N,
                      void* y, int ldy, int dt, void* stream) {
  LLJ_REQUIRE(x && nw && W1 && W2 && y && llj_g_norm_ok(M, K, dt) && N > 0 && ldx >= K && ldy >= N);
  hipStream_t s = (hipStream_t)stream;
  return dt == 0 ? gr_launch<bf16_t>(GR_SWIGLU, x, ldx, nw, eps, M, K, W1, W2, N, y, ldy, nullptr, 0, s)
                 : gr_launch<float>(GR_SWIGLU, x, ldx, nw, eps, M, K, W1, W2, N, y, ldy, nullptr, 0, s);
}

static size_t gr_attention_lds(int S, int hs) { return ((size_t)S + (size_t)hs * (3 + gr_groups(hs / 2))) * 4; }

int llj_g_rope_attention_ok(int S, int hs) { return S > 0 && hs > 0 && hs % 2 == 0 && gr_attention_lds(S, hs) <= 64 * 1024; }

int llj_g_rope_attention(const void* qkv, void* kcache, void* vcache, const float* rope, const int* pos, void* y, int B, int C,
                         int n_head, int S, int dt, void* stream) {
  LLJ_REQUIRE(qkv && kcache && vcache && rope && pos && y && B > 0 && n_head > 0 && C % n_head == 0 && (dt == 0 || dt == 1) &&
              llj_g_rope_attention_ok(S, C / n_head) && ((uintptr_t)kcache | (uintptr_t)vcache) % (dt ? 8 : 4) == 0);
  const size_t lds = gr_attention_lds(S, C / n_head);
  hipStream_t s = (hipStream_t)stream;
  // fp32 with more than a workgroup per CU: nothing is loaded that is not seen (12 rows of 32 heads, us without and with: heads of 80, 16 slots 8.9 and 7.2,
  // of 128 21.5 and 18.9). Heads of more than 64 there, and of more than 128, stay on the kernel with its scores in LDS, which has the registers for
  // more waves (12 rows of 32 heads of 80, 1,700 keys 88 and 81, 26 rows of 10 heads of 78 12.8 and 11.3; bf16 is ahead in registers at every size)
  const bool mask = dt == 1 && (long)B * n_head > 256;
#define LLJ_GRA(T, NQ, MASK) \
  hipLaunchKernelGGL((g_rope_attention16_kernel<T, NQ, 4, MASK>), dim3(B, n_head), dim3(kGrThreads), 0, s, (const T*)qkv, (T*)kcache, (T*)vcache, rope, pos, (T*)y, C, n_head, S)
#define LLJ_GRA_NQ(NQ)                        \
  do {                                        \
    if (dt == 0) LLJ_GRA(bf16_t, NQ, false);  \
    else if (mask) LLJ_GRA(float, (NQ > 2 ? 2 : NQ), true);  \
    else LLJ_GRA(float, NQ, false);           \
  } while (0)
  const int hs = C / n_head;
  if (hs > (mask ? 64 : 128)) {
#define LLJ_GRS(T, MASK) \
  hipLaunchKernelGGL((g_rope_attention_kernel<T, MASK>), dim3(B, n_head), dim3(kGrThreads), lds, s, (const T*)qkv, (T*)kcache, (T*)vcache, rope, pos, (T*)y, C, n_head, S)
    if (dt == 0) LLJ_GRS(bf16_t, false);
    else if (mask) LLJ_GRS(float, true);
    else LLJ_GRS(float, false);
#undef LLJ_GRS
  } else if (hs <= 32) LLJ_GRA_NQ(1);
  else if (hs <= 64) LLJ_GRA_NQ(2);
  else if (hs <= 96) LLJ_GRA_NQ(3);
  else LLJ_GRA_NQ(4);
#undef LLJ_GRA_NQ
#undef LLJ_GRA
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_embedding(const int* idx, const void* wte, void* out, int M, int C, int* pos_inc, int dt, void* stream) {
  LLJ_REQUIRE(idx && wte && out && M > 0 && C > 0 && (dt == 0 || dt == 1));
  hipStream_t s = (hipStream_t)stream;
  LLJ_DT(dt, hipLaunchKernelGGL(g_embedding_kernel<bf16_t>, dim3(M), dim3(256), 0, s, idx, (const bf16_t*)wte, (bf16_t*)out, C, pos_inc),
         hipLaunchKernelGGL(g_embedding_kernel<float>, dim3(M), dim3(256), 0, s, idx, (const float*)wte, (float*)out, C, pos_inc));
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_rmsnorm(const void* x, int ldx, const void* w, float eps, void* y, int ldy, int M, int C, int dt, void* stream) {
  LLJ_REQUIRE(x && w && y && M > 0 && C > 0 && ldx >= C && ldy >= C && (dt == 0 || dt == 1));
  hipStream_t s = (hipStream_t)stream;
  LLJ_DT(dt, hipLaunchKernelGGL(g_rmsnorm_kernel<bf16_t>, dim3(M), dim3(256), 0, s, (const bf16_t*)x, ldx, (const bf16_t*)w, eps, (bf16_t*)y, ldy, C),
         hipLaunchKernelGGL(g_rmsnorm_kernel<float>, dim3(M), dim3(256), 0, s, (const float*)x, ldx, (const float*)w, eps, (float*)y, ldy, C));
  LLJ_CHECK_LAUNCH();
  return 0;
}

size_t llj_g_linear_ws_bytes(int wkind, int M, int N, int K, int dt) {
  if (M <= GL_ROWS || N <= 0 || K <= 0) return 0;
  const int s = gs_takes(wkind, dt) ? gs_plan(M, N, K, true).splits : gg_splits(M, N, K, dt == 1 || wkind == 0, dt == 1 && K <= kGgFineK);
  return s > 1 ? (size_t)s * M * N * 4 : 0;
}

int llj_g_linear_ws(int wkind, const void* x, int ldx, int M, int K, const void* W, const float* scales, const float* zeros,
                    int bits, int group, int N, void* y, int ldy, const void* resid, int ldr, int dt, void* ws, size_t ws_bytes,
                    void* stream) {
  LLJ_REQUIRE(x && W && y && M > 0 && K > 0 && N > 0 && ldx >= K && ldy >= N && (!resid || ldr >= N) && (dt == 0 || dt == 1));
  LLJ_REQUIRE(wkind == 1 || (wkind == 0 && scales && zeros && (bits == 2 || bits == 4 || bits == 8) && group > 0 &&
                             K % (8 / bits) == 0));
  hipStream_t s = (hipStream_t)stream;
  if (M <= GL_ROWS && wkind == 1)
    return dt == 0 ? gr_launch<bf16_t>(GR_PLAIN, x, ldx, nullptr, 0.f, M, K, W, nullptr, N, y, ldy, resid, ldr, s)
                   : gr_launch<float>(GR_PLAIN, x, ldx, nullptr, 0.f, M, K, W, nullptr, N, y, ldy, resid, ldr, s);
  if (M <= GL_ROWS) {
#define LLJ_GL(T) \
  hipLaunchKernelGGL(g_code_rows_kernel<T>, dim3((N + 3) / 4), dim3(256), 0, s, (const T*)x, ldx, M, K, (const unsigned char*)W, \
                     scales, zeros, bits, group, N, (T*)y, ldy, (const T*)resid, ldr)
    LLJ_DT(dt, LLJ_GL(bf16_t), LLJ_GL(float));
#undef LLJ_GL
    LLJ_CHECK_LAUNCH();
    return 0;
  }
  if (gs_takes(wkind, dt)) {
    GsPlan p = gs_plan(M, N, K, ws != nullptr);
    if (p.splits > 1 && ws_bytes < (size_t)p.splits * M * N * 4) p = gs_plan(M, N, K, false);
    const int e = gs_launch(p, (const float*)x, ldx, M, K, (const float*)W, N, (float*)y, ldy, (const float*)resid, ldr, (float*)ws, s);
    if (e) return e;
    return p.splits > 1 ? gg_reduce((const float*)ws, p.splits, M, N, (float*)y, ldy, (const float*)resid, ldr, s) : 0;
  }
  const bool f32 = dt == 1 || wkind == 0;  // bf16 rows on codes: the weight element (q - zero) * scale is fp32
  const bool fine = dt == 1 && K <= kGgFineK;  // fp32 operands: short chains of sums
  int splits = ws ? gg_splits(M, N, K, f32, fine) : 1;
  if (splits > 1 && ws_bytes < (size_t)splits * M * N * 4) splits = 1;
  const int kt = kGgRow / (f32 ? 4 : 2), all = (K + kt - 1) / kt, per = (all + splits - 1) / splits;
  const int mt = (M + kGgBM - 1) / kGgBM, nt = (N + kGgBN - 1) / kGgBN;
  LLJ_REQUIRE((long)((nt + 7) / 8) * 8 * mt < (1L << 31));
  const dim3 grid((nt + 7) / 8 * 8 * mt, splits);
  float* part = splits > 1 ? (float*)ws : nullptr;
  // elements per load: 16, 8 (bf16) or single elements, as the rows of x and of a dense W are aligned
  const int el = dt == 1 ? 4 : 2;
  auto fits = [&](const void* p, int ld, int n) { return (uintptr_t)p % (n * el) == 0 && ld % n == 0 && K % n == 0; };
  // WL: loader of J accumulators per wave (512 / J threads)
#define LLJ_GG_GO(T, CT, VEX, J, FINE, HALVES, ...)                                                                           \
  do {                                                                                                                        \
    typedef __VA_ARGS__ wl;                                                                                                   \
    hipLaunchKernelGGL((gg_kernel<wl, T, CT, VEX, J, FINE, HALVES>), grid, dim3(512 / J), 0, s, (const T*)x, ldx, M, K, W, scales,    \
                       zeros, wkind == 1 ? K : group, N, (T*)y, ldy, (const T*)resid, ldr, part, per);                        \
  } while (0)
#define LLJ_GG_RUN(T, CT, VEX, J, FINE, ...)                                                      \
  do {                                                                                            \
    if (FINE && splits == 1 && all >= 8) LLJ_GG_GO(T, CT, VEX, J, FINE, FINE, __VA_ARGS__);       \
    else LLJ_GG_GO(T, CT, VEX, J, FINE, false, __VA_ARGS__);                                      \
  } while (0)
#define LLJ_GG_BF16(VE) LLJ_GG_RUN(bf16_t, bf16_t, VE, 1, false, GgWeightDense<bf16_t, VE, 512>)
#define LLJ_GG_BITS(B, VE)                                                                 \
  do {                                                                                     \
    if (dt == 0) LLJ_GG_RUN(bf16_t, float, VE, 2, false, GgWeightCodes<B, 256>);           \
    else if (fine) LLJ_GG_RUN(float, float, VE, 1, true, GgWeightCodes<B, 512>);           \
    else LLJ_GG_RUN(float, float, VE, 2, false, GgWeightCodes<B, 256>);                    \
  } while (0)
#define LLJ_GG_CODES(VE)                  \
  do {                                    \
    if (bits == 4) LLJ_GG_BITS(4, VE);    \
    else if (bits == 8) LLJ_GG_BITS(8, VE); \
    else LLJ_GG_BITS(2, VE);              \
  } while (0)
  if (wkind == 0) {
    if (fits(x, ldx, 4)) LLJ_GG_CODES(4);
    else LLJ_GG_CODES(1);
  } else {
    if (fits(x, ldx, 8) && fits(W, K, 8)) LLJ_GG_BF16(8);
    else if (fits(x, ldx, 4) && fits(W, K, 4)) LLJ_GG_BF16(4);
    else LLJ_GG_BF16(1);
  }
#undef LLJ_GG_CODES
#undef LLJ_GG_BITS
#undef LLJ_GG_BF16
#undef LLJ_GG_RUN
#undef LLJ_GG_GO
  LLJ_CHECK_LAUNCH();
  if (!part) return 0;
  return dt == 0 ? gg_reduce(part, splits, M, N, (bf16_t*)y, ldy, (const bf16_t*)resid, ldr, s)
                 : gg_reduce(part, splits, M, N, (float*)y, ldy, (const float*)resid, ldr, s);
}

int llj_g_linear(int wkind, const void* x, int ldx, int M, int K, const void* W, const float* scales, const float* zeros,
                 int bits, int group, int N, void* y, int ldy, const void* resid, int ldr, int dt, void* stream) {
  return llj_g_linear_ws(wkind, x, ldx, M, K, W, scales, zeros, bits, group, N, y, ldy, resid, ldr, dt, nullptr, 0, stream);
}

int llj_g_rope_kv(const void* qkv, void* q_out, void* kcache, void* vcache, const float* rope, const int* pos, int B, int T,
                  int C, int n_head, int S, int dt, void* stream) {
  LLJ_REQUIRE(qkv && q_out && kcache && vcache && rope && pos && B > 0 && T > 0 && n_head > 0 && C % n_head == 0 &&
              (C / n_head) % 2 == 0 && S > 0 && (dt == 0 || dt == 1));
  hipStream_t s = (hipStream_t)stream;
  LLJ_DT(dt, hipLaunchKernelGGL(g_rope_kv_kernel<bf16_t>, dim3(B * T, n_head), dim3(64), 0, s, (const bf16_t*)qkv, (bf16_t*)q_out,
                                (bf16_t*)kcache, (bf16_t*)vcache, rope, pos, T, C, n_head, S),
         hipLaunchKernelGGL(g_rope_kv_kernel<float>, dim3(B * T, n_head), dim3(64), 0, s, (const float*)qkv, (float*)q_out,
                            (float*)kcache, (float*)vcache, rope, pos, T, C, n_head, S));
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_attention(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T, int C,
                    int n_head, int S, int dt, void* stream) {
  LLJ_REQUIRE(q && kcache && vcache && y && pos && B > 0 && T > 0 && n_head > 0 && C % n_head == 0 && S > 0 &&
              (dt == 0 || dt == 1));
  const size_t lds = (size_t)(S + C / n_head) * 4;
  LLJ_REQUIRE(lds <= 64 * 1024);
  hipStream_t s = (hipStream_t)stream;
  // The tiles from 1,024 (row, head) pairs on: below, one workgroup per pair is a shorter chain (us, pairs -> tiles; fp32, heads of 78:
  // 4 rows of 10 heads 4.8 and 7.6, 100 rows 9.2 and 10.4, 128 rows 15.0 and 10.3, 1,000 rows 397 and 74; 301 rows of 32 heads of
  // 128 137 and 37), below 48 rows from 2,048 on: a prompt at the sequence's start then has one short tile of keys (fp32, heads of 80: 36 rows of
  // 32 heads 6.5 and 7.1, 24 of 80 0.89 of the tiles, 64 rows of 32 heads 1.3; from position 200 on the tiles are ahead from some 500
  // pairs, but the host does not know where the rows stand).
  if (T >= kGaRows && (long)B * T * n_head >= (T < 48 ? 2048 : 1024)) {
    const int e = dt == 0 ? ga_launch((const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, (bf16_t*)y, pos, B, T, C, n_head, S, s)
                          : ga_launch((const float*)q, (const float*)kcache, (const float*)vcache, (float*)y, pos, B, T, C, n_head, S, s);
    if (e != 1) return e;
  }
  LLJ_DT(dt, hipLaunchKernelGGL(g_attention_kernel<bf16_t>, dim3(B * T, n_head), dim3(256), lds, s, (const bf16_t*)q,
                                (const bf16_t*)kcache, (const bf16_t*)vcache, (bf16_t*)y, pos, T, C, n_head, S),
         hipLaunchKernelGGL(g_attention_kernel<float>, dim3(B * T, n_head), dim3(256), lds, s, (const float*)q,
                            (const float*)kcache, (const float*)vcache, (float*)y, pos, T, C, n_head, S));
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_silu_mul(const void* a1, const void* a2, void* h, size_t n, int dt, void* stream) {
  LLJ_REQUIRE(a1 && a2 && h && n > 0 && (dt == 0 || dt == 1));
  const size_t blocks = (n + 255) / 256;
  const unsigned g = blocks < 4096 ? (unsigned)blocks : 4096u;
  hipStream_t s = (hipStream_t)stream;
  LLJ_DT(dt, hipLaunchKernelGGL(g_silu_mul_kernel<bf16_t>, dim3(g), dim3(256), 0, s, (const bf16_t*)a1, (const bf16_t*)a2, (bf16_t*)h, n),
         hipLaunchKernelGGL(g_silu_mul_kernel<float>, dim3(g), dim3(256), 0, s, (const float*)a1, (const float*)a2, (float*)h, n));
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_bias_act(int act, void* y, int ldy, const float* bias, void* out, int ldo, int M, int N, float limit, float alpha,
                   int dt, void* stream) {
  LLJ_REQUIRE((act == 0 || act == 2) && y && M > 0 && N > 0 && ldy >= N && (dt == 0 || dt == 1));
  LLJ_REQUIRE(act == 0 ? bias && !out : out && out != y && N % 2 == 0 && ldo >= N / 2);
  const size_t n = (size_t)M * (act ? N / 2 : N), blocks = (n + 255) / 256;
  const unsigned g = blocks < 4096 ? (unsigned)blocks : 4096u;
  hipStream_t s = (hipStream_t)stream;
  LLJ_DT(dt, hipLaunchKernelGGL(g_bias_act_kernel<bf16_t>, dim3(g), dim3(256), 0, s, act, (bf16_t*)y, ldy, bias, (bf16_t*)out, ldo, M, N, limit, alpha),
         hipLaunchKernelGGL(g_bias_act_kernel<float>, dim3(g), dim3(256), 0, s, act, (float*)y, ldy, bias, (float*)out, ldo, M, N, limit, alpha));
  LLJ_CHECK_LAUNCH();
  return 0;
}

size_t llj_g_i8_ws_bytes(int M, int K) { return (((size_t)K + 15) & ~(size_t)15) + (size_t)M * 4; }

int llj_g_i8_linear(const void* x, int ldx, int M, int K, const void* CB, const float* SCB, float threshold, void* ws, int N,
                    void* y, int ldy, const void* resid, int ldr, int dt, void* stream) {
  LLJ_REQUIRE(x && CB && SCB && ws && y && M > 0 && K > 0 && N > 0 && ldx >= K && ldy >= N && (!resid || ldr >= N) &&
              (dt == 0 || dt == 1));
  hipStream_t s = (hipStream_t)stream;
  unsigned char* flags = (unsigned char*)ws;
  float* sca = (float*)((char*)ws + (((size_t)K + 15) & ~(size_t)15));
  const dim3 grid((N + 3) / 4, (M + GL_ROWS - 1) / GL_ROWS);
#define LLJ_GI8(T)                                                                                                   \
  do {                                                                                                                \
    hipLaunchKernelGGL(g_i8_flags_kernel<T>, dim3((K + 255) / 256), dim3(256), 0, s, (const T*)x, ldx, M, K, threshold, \
                       flags);                                                                                        \
    hipLaunchKernelGGL(g_i8_sca_kernel<T>, dim3(M), dim3(256), 0, s, (const T*)x, ldx, K, threshold, sca);            \
    hipLaunchKernelGGL(g_i8_linear_kernel<T>, grid, dim3(256), 0, s, (const T*)x, ldx, M, K, (const int8_t*)CB, SCB,  \
                       flags, sca, N, (T*)y, ldy, (const T*)resid, ldr);                                              \
  } while (0)
  LLJ_DT(dt, LLJ_GI8(bf16_t), LLJ_GI8(float));
#undef LLJ_GI8
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
