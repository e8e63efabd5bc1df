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
#include <algorithm>
#include <utility>

#include "common.h"
#include "gptq_tiles.h"

namespace llj {

constexpr int kGptqBlock = 128;

constexpr int kGptqSub = 16;          // columns held in registers at a time
constexpr int kHs = kGptqBlock + 4;   // LDS row stride of Hinv1 (rows start on 16 bytes)
constexpr int kHsRows = 80;
// Hinv1 in LDS from the diagonal groups on: place of element (b, b), b % 16 == 0, row b + u at + u kHs. The rows of b >= 80 lie in the
// columns that those of 128 - b leave free (42 KB for 68: three workgroups a CU beside the products of gptq_next_kernel).
__device__ __forceinline__ int band(int b) { return b <= 64 ? b * kHs + b : (kGptqBlock - b) * kHs; }

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
    for (int u = 0; u < kGptqSub; ++u) h[u] = hs[band(b) + u * kHs + l];
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
    const float* h = hs + band(b) + l;
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
struct BlockArgs {
  const float* hinv;
  int K, i1, blk, N;  // the block's columns [i1, i1 + blk)
  const float *scale, *zero;
  float maxq;
  float *qt, *err, *loss;
};
struct BlockLds {
  float hs[kHsRows * kHs];     // Hinv1 (band)
  float diag[2][kGptqBlock];  // Hinv1[i][i], 1 / Hinv1[i][i]
};

// The block's columns of rows n = .. + tid / 16. weights(r): this lane's 8 weights, asked for ahead of Hinv1 (EARLY) or behind the barrier after it.
template <int ROWS, bool EARLY, typename F>
__device__ __forceinline__ void gptq_rows(const BlockArgs& p, int n, BlockLds& s_, F weights) {
  constexpr int NT = ROWS * 16;
  const int tid = threadIdx.x, l = tid & 15, K = p.K, i1 = p.i1, blk = p.blk;
  const int nn = n < p.N ? n : p.N - 1;  // clamped: loads stay in bounds, stores are guarded
  float r[kGptqBlock / kGptqSub];
  if (EARLY) weights(r);
  const float s = p.scale[nn], z = p.zero[nn];
  bool fast = divides(s) && fabsf(z) < 0x1p30f;
  if (tid < blk) {
    const float d = p.hinv[(size_t)(i1 + tid) * K + i1 + tid];
    s_.diag[0][tid] = d;
    s_.diag[1][tid] = __fdiv_rn(1.f, d);
    fast = fast && divides(d);
  }
  auto at = [](int i, int j) { return band(i & ~15) + (i & 15) * kHs + j - (i & ~15); };
  if (((K | i1) & 3) == 0 && ((uintptr_t)p.hinv & 15) == 0) {
    for (int v = tid; v < blk * (blk / 4); v += NT) {
      const int i = v / (blk / 4), j = v % (blk / 4) * 4;
      if (j >= (i & ~15)) *reinterpret_cast<f32x4*>(s_.hs + at(i, j)) = *reinterpret_cast<const f32x4*>(p.hinv + (size_t)(i1 + i) * K + i1 + j);
    }
  } else {
    for (int v = tid; v < blk * blk; v += NT) {
      const int i = v / blk, j = v % blk;
      if (j >= (i & ~15)) s_.hs[at(i, j)] = p.hinv[(size_t)(i1 + i) * K + i1 + j];
    }
  }
  bool done = __syncthreads_and(fast);
  if (!EARLY) weights(r);
  const bool live = n < p.N;
  float* q_out = p.qt + (size_t)i1 * p.N + nn;
  float* e_out = p.err + nn;
  float sum = 0.f;
  Errors seen;
  if (done) {
    sum = gptq_columns<true>(s_.hs, s_.diag, r, l, blk, s, z, p.maxq, live, q_out, e_out, p.N, seen);
    done = __syncthreads_and(seen.fit());
    if (!done) weights(r);  // a quotient out of div_by's range: the block again
  }
  if (!done) sum = gptq_columns<false>(s_.hs, s_.diag, r, l, blk, s, z, p.maxq, live, q_out, e_out, p.N, seen);
  if (live && l == 0) p.loss[n] += sum;
}

template <int ROWS>
__global__ __launch_bounds__(ROWS * 16) void gptq_block_kernel(BlockArgs p, const float* __restrict__ wt) {
  __shared__ __align__(16) BlockLds lds;
  const int n = blockIdx.x * ROWS + (threadIdx.x >> 4), nn = n < p.N ? n : p.N - 1, l = threadIdx.x & 15;
  gptq_rows<ROWS, true>(p, n, lds, [&](float (&r)[kGptqBlock / kGptqSub]) {
#pragma unroll
    for (int i = 0; i < kGptqBlock / kGptqSub; ++i) r[i] = i * kGptqSub < p.blk ? wt[(size_t)(p.i1 + i * kGptqSub + l) * p.N + nn] : 0.f;
  });
}

// The update behind one block of 128 and the column loop of the next in one launch. The first workgroups take 16 rows each: they take the
// last block's errors off the next 128 columns -- their own rows of the product, 64 MFMAs a wave, operands from memory as the MFMA
// wants them -- and run the columns; the others meanwhile take the errors off all later columns in 64 x 64 tiles, as gptq_update_kernel
// does. Both form every sum as that kernel does: the same bits.
//
// Bound: the column loop's chain, some 20 us on one wave per SIMD, beside the products (31 us of their own in the mean at
// 4096 x 4096), which fill the matrix cores that the chain leaves idle.
template <bool VEC>
__global__ __launch_bounds__(256) void gptq_next_kernel(BlockArgs p, const float* __restrict__ last, float* __restrict__ wt, int row_groups) {
  typedef AtB<64, 64, float, VEC, false> G;
  struct Rows {
    BlockLds b;
    float w[kGptqBlock * 17];  // the block's columns of the 16 rows
  };
  __shared__ __align__(16) unsigned char lds[sizeof(Rows) > G::kLds * 4 ? sizeof(Rows) : G::kLds * 4];
  const int K = p.K, N = p.N, i0 = p.i1 - kGptqBlock;  // (the last block's first column)
  if ((int)blockIdx.x >= row_groups) {
    const int i3 = p.i1 + kGptqBlock, M = K - i3, mt = (M + 63) / 64, nt = (N + 63) / 64, t = xcd_run(blockIdx.x - row_groups, mt * nt);
    if (t < 0) return;
    const int m0 = t / nt * 64, n0 = t % nt * 64;
    f32x4 acc[G::MI][G::NI], old[G::MI][G::NI];
    G::run(p.hinv + (size_t)i0 * K + i3 + m0, K, M - m0, last + n0, N, N - n0, kGptqBlock, 1.f, reinterpret_cast<float*>(lds), acc, [&] {
      G::load(old, [&](int i, int j) { return wt[(size_t)(i3 + min(m0 + i, M - 1)) * N + min(n0 + j, N - 1)]; });
    });
    G::both(acc, old, [&](int i, int j, float v, float w) {
      const int m = m0 + i, n = n0 + j;
      if (m < M && n < N) wt[(size_t)(i3 + m) * N + n] = w - v;
    });
    return;
  }
  __builtin_amdgcn_s_setprio(3);  // the longest chain of the launch
  Rows& s = *reinterpret_cast<Rows*>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, c = lane & 15, n0 = blockIdx.x * 16;
  {
    // wave: columns 32 wave .. + 32 of the block, lane: rows (of W) n0 + c
    const float* a = p.hinv + (size_t)(i0 + q) * K + p.i1 + 32 * wave + c;
    const float* b = last + (size_t)q * N + min(n0 + c, N - 1);
    const float* w = wt + (size_t)(p.i1 + 32 * wave + 4 * q) * N + min(n0 + c, N - 1);
    constexpr int KS = kGptqBlock / 4;
    float av[KS][2], bv[KS], old[2][4];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      av[k][0] = a[(size_t)4 * k * K];
      av[k][1] = a[(size_t)4 * k * K + 16];
      bv[k] = b[(size_t)4 * k * N];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) old[i][r] = w[(size_t)(16 * i + r) * N];
    f32x4 acc[2] = {};
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = mma4(av[k][i], bv[k], acc[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) s.w[(32 * wave + 16 * i + 4 * q + r) * 17 + c] = old[i][r] - acc[i][r];
  }
  gptq_rows<16, false>(p, n0 + (tid >> 4), s.b, [&](float (&r)[kGptqBlock / kGptqSub]) {
#pragma unroll
    for (int i = 0; i < kGptqBlock / kGptqSub; ++i) r[i] = s.w[(i * kGptqSub + (tid & 15)) * 17 + (tid >> 4)];
  });
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
  const BlockArgs p = {hinv, K, i1, blocksize, N, scale, zero, (float)((1 << bits) - 1), qt, err, loss};
#define LLJ_BLOCK(ROWS) hipLaunchKernelGGL((gptq_block_kernel<ROWS>), dim3((N + ROWS - 1) / ROWS), dim3(ROWS * 16), 0, (hipStream_t)stream, p, wt)
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

int llj_gptq_next(const float* hinv, int K, int i1, const float* last, float* wt, int N, const float* scale, const float* zero, int bits,
                  float* qt, float* err, float* loss, void* stream) {
  LLJ_REQUIRE(K > 0 && N > 0 && i1 >= kGptqBlock && i1 % kGptqBlock == 0 && i1 + kGptqBlock <= K && (bits == 2 || bits == 4 || bits == 8));
  LLJ_REQUIRE(hinv && last && wt && scale && zero && qt && err && err != last && loss);
  const BlockArgs p = {hinv, K, i1, kGptqBlock, N, scale, zero, (float)((1 << bits) - 1), qt, err, loss};
  const bool vec = K % 4 == 0 && N % 4 == 0 && (((uintptr_t)hinv | (uintptr_t)last) & 15) == 0;
  const long M = K - i1 - kGptqBlock, tiles = ((M + 63) / 64) * ((N + 63) / 64), groups = (N + 15) / 16, grid = groups + (tiles + 7) / 8 * 8;
  LLJ_REQUIRE(grid < (1l << 31));
  if (vec) hipLaunchKernelGGL((gptq_next_kernel<true>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, p, last, wt, (int)groups);
  else hipLaunchKernelGGL((gptq_next_kernel<false>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, p, last, wt, (int)groups);
  LLJ_CHECK_LAUNCH();
  return 0;
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
