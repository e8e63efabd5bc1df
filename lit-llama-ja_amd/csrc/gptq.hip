// GPTQ producer kernels (reference lit_llama/quantization.py:424-614,
// GPTQQuantizer.quantize). The calibration Hessian, its Cholesky factors and the trailing
// block update W[:, i2:] -= Err1 · Hinv[i1:i2, i2:] are plain GEMM / LAPACK work (library calls on
// the device, host side); what is specific to GPTQ is the sequential column loop inside a
// 128-column block (quantization.py:568-596) and the ColBlock packing (pack_weight, 374-388).
//
// llj_gptq_block(_bs): 16 lanes per weight row (rows are independent inside a block: the update of
// row r uses only its own error and the shared Hinv1 rows). The block's 128 columns of each row are in its lanes'
// registers, Hinv1 in LDS; 16 columns at a time are quantized one by one, then the rest of the block takes their 16 updates per
// column. Weights are passed transposed (Wt: K x N, element (k, n) at k * N + n).
// The block is the reference's `blocksize` (557; 16 / 32 / 64 / 128: whole 16-column register
// groups, at most the 128 columns the LDS holds).
// Every arithmetic step is the reference's fp32 op in the reference's order, rounded on its own
// (this file is built with -ffp-contract=off, lit_llama/_build.py), so a block reproduces the torch CPU
// loop bitwise given the same W1 and Hinv1.
#include <utility>

#include "common.h"

namespace llj {

constexpr int kGptqBlock = 128;

constexpr int kGptqSub = 16;          // columns held in registers at a time
constexpr int kHs = kGptqBlock + 4;   // LDS row stride of Hinv1 (rows start on 16 bytes)

// a / b, correctly rounded, from y = 1 / b correctly rounded: two residual steps. The first makes the quotient faithful, the
// second then gives the rounded one (Markstein, "Computation of elementary functions on the IBM RISC System/6000", 1990), for
// operands whose quotient does not overflow and whose residuals do not underflow (a zero's sign is not kept). A third of the division
// sequence's instructions, and no dependent reciprocal.
__device__ __forceinline__ float div_by(float a, float b, float y) {
  float q = __fmul_rn(a, y);
  q = __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
}
__device__ __forceinline__ bool divides(float b) { return fabsf(b) > 0x1p-40f && fabsf(b) < 0x1p40f; }
// The range of the errors e = dq / d seen. From 2^-60 to 2^40, or zero, with divides(d): |dq| is in [2^-100, 2^80), its residuals are
// multiples of 2^-147; and with divides(s) and |z| < 2^30: |w| < 2^81, w / s does not overflow (a small one rounds to code z either way).
struct Errors {
  unsigned hi = 0, lo = ~0u;  // bits of absolute values: NaN's are the largest, a zero's less one too
  __device__ __forceinline__ void add(float e) {
    const unsigned a = __float_as_uint(e) & 0x7fffffffu;
    hi = max(hi, a);
    lo = min(lo, a - 1u);
  }
  __device__ __forceinline__ bool fit() const { return hi < __float_as_uint(0x1p40f) && lo >= __float_as_uint(0x1p-60f) - 1u; }
};

// What a group of 16 columns needs of Hinv1: column l's values in lane l, the diagonal and its reciprocals in every lane
struct Group {
  float h[kGptqSub];
  f32x4 d[kGptqSub / 4], rd[kGptqSub / 4];
  __device__ __forceinline__ void load(const float* hs, const float (*diag)[kGptqBlock], int b, int l) {
#pragma unroll
    for (int u = 0; u < kGptqSub; ++u) h[u] = hs[(b + u) * kHs + b + l];
#pragma unroll
    for (int c = 0; c < kGptqSub / 4; ++c) {
      d[c] = *reinterpret_cast<const f32x4*>(diag[0] + b + 4 * c);
      rd[c] = *reinterpret_cast<const f32x4*>(diag[1] + b + 4 * c);
    }
  }
};

// A group's columns of a row, r: column l in lane l. Every lane of the row forms every column's code and error from the owner's weight.
template <bool FAST>
struct Columns {
  const Group& grp;
  const int l;
  const float s, z, rs, maxq;
  float r, lsum, q_own, e_own;
  float e[kGptqSub];

  template <int U>
  __device__ __forceinline__ int column() {
    const float w = __uint_as_float(dpp_u32<0x150 + U>(__float_as_uint(r)));  // lane U's, of the row's 16
    const float d = grp.d[U / 4][U % 4];
    // quantize_weight (quantization.py:470-473): clamp(round(x / scale) + zero, 0, maxq)
    const float x = FAST ? div_by(w, s, rs) : __fdiv_rn(w, s);
    const float qi = fminf(fmaxf(__fadd_rn(rintf(x), z), 0.f), maxq);
    const float q = __fmul_rn(s, __fsub_rn(qi, z));
    const float dq = __fsub_rn(w, q);
    e[U] = FAST ? div_by(dq, d, grp.rd[U / 4][U % 4]) : __fdiv_rn(dq, d);  // err1 (592)
    // W1[:, i:] -= err1 (x) Hinv1[i, i:] (593) inside the group (columns <= i are never read again)
    r = __fsub_rn(r, __fmul_rn(e[U], grp.h[U]));
    lsum = __fadd_rn(lsum, __fmul_rn(e[U], e[U]));  // Losses1 (590): (w - q)^2 / d^2
    q_own = l == U ? q : q_own;
    e_own = l == U ? e[U] : e_own;
    return U;
  }
  template <int... U>
  __device__ __forceinline__ void all(std::integer_sequence<int, U...>) {
    int done[] = {column<U>()...};
    (void)done;
  }
};

// One block of one row's columns, column 16 i + l in r[i] of lane l (see gptq_block_kernel). FAST: every divisor is in div_by's range; seen: the
// errors of the lane's columns.
template <bool FAST>
__device__ __forceinline__ float gptq_columns(const float* hs, const float (*diag)[kGptqBlock], float (&r)[kGptqBlock / kGptqSub], int l, int blk, float s,
                                              float z, float maxq, bool live, float* __restrict__ q_out, float* __restrict__ e_out, size_t N, Errors& seen) {
  const float rs = __fdiv_rn(1.f, s);
  float lsum = 0.f;
  Group grp;
  grp.load(hs, diag, 0, l);
  for (int b = 0; b < blk; b += kGptqSub) {
    Columns<FAST> c = {grp, l, s, z, rs, maxq, r[0], lsum, 0.f, 0.f};
    c.all(std::make_integer_sequence<int, kGptqSub>());
    lsum = c.lsum;
    if constexpr (FAST) seen.add(c.e_own);
    if (live) {
      q_out[(size_t)(b + l) * N] = c.q_own;
      e_out[(size_t)(b + l) * N] = c.e_own;
    }
    const float* h = hs + b * kHs + b + l;
    if (b + kGptqSub < blk) grp.load(hs, diag, b + kGptqSub, l);
    // the rest of the block: the group's updates of a column in increasing i, as the reference applies them one column i at a time
#pragma unroll
    for (int i = 1; i < kGptqBlock / kGptqSub; ++i) {
      if (b + i * kGptqSub < blk) {
        float hv[kGptqSub];
#pragma unroll
        for (int u = 0; u < kGptqSub; ++u) hv[u] = h[u * kHs + i * kGptqSub];
#pragma unroll
        for (int u = 0; u < kGptqSub; ++u) r[i] = __fsub_rn(r[i], __fmul_rn(c.e[u], hv[u]));
      }
      r[i - 1] = r[i];
    }
  }
  return lsum;
}

// A row's 128 columns are in the registers of 16 lanes, four rows to a wave; a column's weight goes from its lane to the row's others
// (DPP), which all form its code and error (identical inputs, identical fp32 ops) and then update their own columns. Every
// column receives the updates in the reference's order, so results are its bit for bit.
//
// Bound: the chain of dependent instructions of a column, two divisions in it, times 128. A lone wave on a SIMD issues an independent
// instruction every 4.75 cycles and one that waits for the last every 8.1, so length and number both count: 570 a group of 16 columns (890 with a row's 16 columns in every
// lane's registers: 23.6 us at N = 4096; interleaving those updates with the chain, or Hinv1's values a step ahead: no faster). 16 rows put
// N = 4096 on all 256 CUs, one wave per SIMD; above, more rows to a workgroup share Hinv1. us a block with the rows in LDS, Hinv1 waited for
// column by column, and now: N = 256 33 and 17, 4096 35 and 19 (among the producer's other launches
// 39 and 22), 8192 38 and 21, 11008 54 and 31, 35008 171 and 88 (a block with an error out of div_by's range is done twice).
template <int ROWS>
__global__ __launch_bounds__(ROWS * 16) void gptq_block_kernel(const float* __restrict__ hinv, int K, int i1, int blk, float* __restrict__ wt, int N,
                                                               const float* __restrict__ scale, const float* __restrict__ zero, float maxq,
                                                               float* __restrict__ qt, float* __restrict__ err, float* __restrict__ loss) {
  __shared__ __align__(16) float hs[kGptqBlock * kHs];    // hs[i * kHs + j] = Hinv1[i][j]
  __shared__ __align__(16) float diag[2][kGptqBlock];     // Hinv1[i][i], 1 / Hinv1[i][i]
  constexpr int NT = ROWS * 16;
  const int tid = threadIdx.x, t = tid >> 4, l = tid & 15;
  const int n = blockIdx.x * ROWS + t;
  const int nn = n < N ? n : N - 1;  // clamped: loads stay in bounds, stores are guarded
  float r[kGptqBlock / kGptqSub];
  auto stage = [&] {
#pragma unroll
    for (int i = 0; i < kGptqBlock / kGptqSub; ++i) r[i] = i * kGptqSub < blk ? wt[(size_t)(i1 + i * kGptqSub + l) * N + nn] : 0.f;
  };
  stage();
  const float s = scale[nn], z = zero[nn];
  bool fast = divides(s) && fabsf(z) < 0x1p30f;
  if (tid < blk) {
    const float d = hinv[(size_t)(i1 + tid) * K + i1 + tid];
    diag[0][tid] = d;
    diag[1][tid] = __fdiv_rn(1.f, d);
    fast = fast && divides(d);
  }
  if (((K | i1) & 3) == 0 && ((uintptr_t)hinv & 15) == 0) {
    for (int v = tid; v < blk * (blk / 4); v += NT) {
      const int i = v / (blk / 4), j = v % (blk / 4) * 4;
      *reinterpret_cast<f32x4*>(hs + i * kHs + j) = *reinterpret_cast<const f32x4*>(hinv + (size_t)(i1 + i) * K + i1 + j);
    }
  } else {
    for (int v = tid; v < blk * blk; v += NT) hs[v / blk * kHs + v % blk] = hinv[(size_t)(i1 + v / blk) * K + i1 + v % blk];
  }
  bool done = __syncthreads_and(fast);
  const bool live = n < N;
  float* q_out = qt + (size_t)i1 * N + nn;
  float* e_out = err + nn;
  float sum = 0.f;
  Errors seen;
  if (done) {
    sum = gptq_columns<true>(hs, diag, r, l, blk, s, z, maxq, live, q_out, e_out, N, seen);
    done = __syncthreads_and(seen.fit());
    if (!done) stage();  // a quotient out of div_by's range: the block again
  }
  if (!done) sum = gptq_columns<false>(hs, diag, r, l, blk, s, z, maxq, live, q_out, e_out, N, seen);
  if (live && l == 0) loss[n] += sum;
}

// pack_weight (quantization.py:374-388) of reconstructed weights Qt (K x N, fp32):
// code = uint8(clamp(q / scale + zero, 0, 2^bits - 1)) (truncating cast, as the reference's
// .to(torch.uint8)), entries_per_byte = 8 / bits codes per byte, column epb*j + nr in bits
// [nr*bits, (nr+1)*bits) of byte (n, j); quant_weight is column-major: byte (n, j) at j * N + n.
// order: the row of Qt that holds column k (null: k), for a column order that the loop worked in.
__global__ __launch_bounds__(256) void colblock_pack_kernel(const float* __restrict__ qt, const int64_t* __restrict__ order, int N,
                                                            const float* __restrict__ scale,
                                                            const float* __restrict__ zero, int bits,
                                                            unsigned char* __restrict__ qw) {
  const int epb = 8 / bits;
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int j = blockIdx.y;
  if (n >= N) return;
  const float s = scale[n], z = zero[n], maxq = (float)((1 << bits) - 1);
  unsigned v = 0;
  for (int nr = 0; nr < epb; ++nr) {
    const size_t k = order ? (size_t)order[epb * j + nr] : epb * j + nr;
    const float x = qt[k * N + n];
    const float c = fminf(fmaxf(__fadd_rn(__fdiv_rn(x, s), z), 0.f), maxq);
    v += ((unsigned)c) << (nr * bits);
  }
  qw[(size_t)j * N + n] = (unsigned char)v;
}

// find_params_weight's per-row (scale, zero) (quantization.py:475-514) of rows of K weights: one workgroup per row. NaN weights
// give NaN as torch's minimum and maximum do. The quotients are correctly rounded, as the reference's on the CPU.
__global__ __launch_bounds__(256) void gptq_params_kernel(const float* __restrict__ w, int K, float maxq, bool sym, float* __restrict__ scale,
                                                          float* __restrict__ zero) {
  __shared__ float part[2][4];
  const float* row = w + (size_t)blockIdx.x * K;
  float lo = 0.f, hi = 0.f;
  bool nan = false;
#pragma unroll 4
  for (int k = threadIdx.x; k < K; k += 256) {
    const float v = row[k];
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
    nan = nan || v != v;
  }
  lo = -wave_max(-lo);
  hi = wave_max(hi);
  if ((threadIdx.x & 63) == 0) {
    part[0][threadIdx.x >> 6] = lo;
    part[1][threadIdx.x >> 6] = hi;
  }
  nan = __syncthreads_or(nan);
  if (threadIdx.x) return;
  lo = fminf(fminf(part[0][0], part[0][1]), fminf(part[0][2], part[0][3]));
  hi = fmaxf(fmaxf(part[1][0], part[1][1]), fmaxf(part[1][2], part[1][3]));
  if (nan) lo = hi = __builtin_nanf("");
  if (sym) {
    const float neg = lo;
    hi = nan ? hi : fmaxf(fabsf(lo), hi);
    if (neg < 0.f) lo = -hi;
  }
  if (lo == 0.f && hi == 0.f) lo = -1.f, hi = 1.f;
  const float s = __fdiv_rn(__fsub_rn(hi, lo), maxq);
  scale[blockIdx.x] = s;
  zero[blockIdx.x] = sym ? __fmul_rn(__fadd_rn(maxq, 1.f), 0.5f) : rintf(__fdiv_rn(-lo, s));
}

}  // namespace llj

using namespace llj;

extern "C" {

int llj_gptq_block_bs(const float* hinv, int K, int i1, int blocksize, float* wt, int N, const float* scale,
                      const float* zero, int bits, float* qt, float* err, float* loss, void* stream) {
  LLJ_REQUIRE(blocksize >= kGptqSub && blocksize <= kGptqBlock && blocksize % kGptqSub == 0);
  LLJ_REQUIRE(K > 0 && N > 0 && i1 >= 0 && i1 % blocksize == 0 && i1 + blocksize <= K);
  LLJ_REQUIRE(bits == 2 || bits == 4 || bits == 8);
  LLJ_REQUIRE(hinv && wt && scale && zero && qt && err && loss);
  const float maxq = (float)((1 << bits) - 1);
#define LLJ_BLOCK(ROWS)                                                                                                                \
  hipLaunchKernelGGL((gptq_block_kernel<ROWS>), dim3((N + ROWS - 1) / ROWS), dim3(ROWS * 16), 0, (hipStream_t)stream, hinv, K, i1,    \
                     blocksize, wt, N, scale, zero, maxq, qt, err, loss)
  if (N <= 4096) LLJ_BLOCK(16);
  else if (N <= 8192) LLJ_BLOCK(32);
  else LLJ_BLOCK(64);
#undef LLJ_BLOCK
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_gptq_block(const float* hinv, int K, int i1, float* wt, int N, const float* scale, const float* zero,
                   int bits, float* qt, float* err, float* loss, void* stream) {
  return llj_gptq_block_bs(hinv, K, i1, kGptqBlock, wt, N, scale, zero, bits, qt, err, loss, stream);
}

int llj_gptq_params(const float* w, int N, int K, int bits, int sym, float* scale, float* zero, void* stream) {
  LLJ_REQUIRE(w && scale && zero && N > 0 && K > 0 && bits > 0 && bits <= 16);
  hipLaunchKernelGGL(gptq_params_kernel, dim3(N), dim3(256), 0, (hipStream_t)stream, w, K, (float)((1 << bits) - 1), sym != 0, scale, zero);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_colblock_pack_order(const float* qt, const int64_t* order, int K, int N, const float* scale, const float* zero, int bits,
                            unsigned char* qw, void* stream) {
  LLJ_REQUIRE(K > 0 && N > 0 && (bits == 2 || bits == 4 || bits == 8) && K % (8 / bits) == 0);
  LLJ_REQUIRE(qt && scale && zero && qw);
  hipLaunchKernelGGL(colblock_pack_kernel, dim3((N + 255) / 256, K / (8 / bits)), dim3(256), 0, (hipStream_t)stream,
                     qt, order, N, scale, zero, bits, qw);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_colblock_pack(const float* qt, int K, int N, const float* scale, const float* zero, int bits,
                      unsigned char* qw, void* stream) {
  return llj_colblock_pack_order(qt, nullptr, K, N, scale, zero, bits, qw, stream);
}

}  // extern "C"
