// Decode-step ops around the weight-streaming GEMVs: token embedding, standalone RMSNorm
// (prefill rows beyond the fused-LDS limit), causal attention over the KV cache, and the
// greedy (top_k = 1) next-token selection.
#include <cstdlib>

#include "common.h"
#include "elem.h"
#include "attention.h"
#ifndef LLJ_NORM_SC1
#define LLJ_NORM_SC1 0
#endif
#include "lit_llama_amd.h"

namespace llj {

// ---- embedding: out[m] = wte[idx[m]]  (reference model.py:110). Optionally bumps the
// device-side decode position (*pos_inc += 1) so a captured decode step is self-advancing.
__global__ __launch_bounds__(256) void embedding_kernel(const int* __restrict__ idx, const uint4* __restrict__ wte,
                                                        uint4* __restrict__ out, int C8, int* pos_inc) {
  const int m = blockIdx.x;
  const size_t r = (size_t)idx[m];
  for (int v = threadIdx.x; v < C8; v += blockDim.x) out[(size_t)m * C8 + v] = wte[r * C8 + v];
  if (pos_inc && m == 0 && threadIdx.x == 0) *pos_inc += 1;
}

// any C (the any-shape path, csrc/generic.hip): bf16 elements
__global__ __launch_bounds__(256) void embedding_any_kernel(const int* __restrict__ idx, const bf16_t* __restrict__ wte,
                                                            bf16_t* __restrict__ out, int C, int* pos_inc) {
  const int m = blockIdx.x;
  const size_t r = (size_t)idx[m];
  for (int v = threadIdx.x; v < C; v += blockDim.x) out[(size_t)m * C + v] = wte[r * C + v];
  if (pos_inc && m == 0 && threadIdx.x == 0) *pos_inc += 1;
}

// ---- RMSNorm with the bf16 rounding points of model.py:281-283 on bf16 tensors. One block
// per row; rows up to 8192 wide are loaded once into registers (x and the scale together,
// before any use), so the kernel is one memory round trip.
// (norm_pair: common.h)

__global__ __launch_bounds__(256) void rmsnorm_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                      float eps, bf16_t* __restrict__ y, int C,
                                                      float* __restrict__ rowsum) {
  constexpr int MAXV = 4;  // 16-byte vectors per thread held in registers
  __shared__ float red[8];
  const int m = blockIdx.x, tid = threadIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)m * C);
  const uint4* g4 = reinterpret_cast<const uint4*>(w);
  uint4* yr = reinterpret_cast<uint4*>(y + (size_t)m * C);
  const int nvec = C >> 3;
  const bool regs = nvec <= MAXV * 256;
  uint4 xa[MAXV], ga[MAXV];
  float ss = 0.f;
  if (regs) {
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
      const int v = tid + 256 * j, vv = v < nvec ? v : 0;
      xa[j] = xr[vv];
      ga[j] = g4[vv];
    }
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
      if (tid + 256 * j < nvec) {
        const uint32_t aw[4] = {xa[j].x, xa[j].y, xa[j].z, xa[j].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) ss += round_bf(bflo(aw[i]) * bflo(aw[i])) + round_bf(bfhi(aw[i]) * bfhi(aw[i]));
      }
    }
  } else {
    for (int v = tid; v < nvec; v += 256) {
      const uint4 a = xr[v];
      const uint32_t aw[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) ss += round_bf(bflo(aw[i]) * bflo(aw[i])) + round_bf(bfhi(aw[i]) * bfhi(aw[i]));
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float r = round_bf(rsqrtf(round_bf(round_bf(tot / (float)C) + eps)));
  float rsum = 0.f;
  auto emit = [&](int v, uint4 a, uint4 g) {
    const uint32_t o0 = norm_pair(a.x, g.x, r), o1 = norm_pair(a.y, g.y, r), o2 = norm_pair(a.z, g.z, r),
                   o3 = norm_pair(a.w, g.w, r);
    rsum += bflo(o0) + bfhi(o0) + bflo(o1) + bfhi(o1) + bflo(o2) + bfhi(o2) + bflo(o3) + bfhi(o3);
#if LLJ_NORM_SC1  // write-through (sc1) 8-byte stores, as the GEMV epilogues (A/B)
    unsigned long long* d8 = reinterpret_cast<unsigned long long*>(yr + v);
    __hip_atomic_store(d8, (unsigned long long)o0 | ((unsigned long long)o1 << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(d8 + 1, (unsigned long long)o2 | ((unsigned long long)o3 << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
    yr[v] = make_uint4(o0, o1, o2, o3);
#endif
  };
  if (regs) {
#pragma unroll
    for (int j = 0; j < MAXV; ++j)
      if (tid + 256 * j < nvec) emit(tid + 256 * j, xa[j], ga[j]);
  } else {
    for (int v = tid; v < nvec; v += 256) emit(v, xr[v], g4[v]);
  }
  if (rowsum) {  // sum of the normalized bf16 row: the int4 GEMV's offset term (gemv.hip header)
    rsum = wave_sum(rsum);
    if ((tid & 63) == 0) red[4 + (tid >> 6)] = rsum;
    __syncthreads();
    if (tid == 0) rowsum[m] = red[4] + red[5] + red[6] + red[7];
  }
}

// ---- attention (attention.h): one block per (head, query row)
// 512 x 4 (128 keys per pass, half the serial score / softmax chain per lane of 256 x 8): 7B
// gptq.int4 decode-only at position ~80, bs=1 847.4 -> 857.8 tok/s, bs=8 4321 -> 4355
// (profiles/r04_attention_block_ab.json; 512 x 8 and 1024 x 2 in between)
#ifndef LLJ_ATT_NTH
#define LLJ_ATT_NTH 512  // threads per (row, head) block
#endif
#ifndef LLJ_ATT_SPEC_BATCH
#define LLJ_ATT_SPEC_BATCH 0  // half speculative pass at any grid size (A/B: option LLJ_OPT_ATT_SPEC_BATCH)
#endif
#ifndef LLJ_ATT_U
#define LLJ_ATT_U 4  // keys per 16-lane group per pass
#endif
template <int HS, int U, int NTH, int SPECU>
__global__ __launch_bounds__(NTH) void attention_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                        const bf16_t* __restrict__ vc, bf16_t* __restrict__ y,
                                                        const int* __restrict__ pos, int T, int S, int nh,
                                                        float scale_log2, uint32_t* st, float thr, uint32_t* clr,
                                                        int clr_words, int spec_ok) {
  __shared__ float lds[attention_lds_floats<HS, NTH>()];
  attention_body<HS, U, NTH, false, SPECU>(q, kc, vc, y, pos, T, S, nh, scale_log2, blockIdx.x, blockIdx.y, lds, 1, 0,
                                           nullptr, st, thr, clr, clr_words, spec_ok != 0);
}

// One decode row's attention with the head's share of attn.c_proj: part[h][n] = sum_d y[h, d] Wp[n, HS h + d], y rounded to bf16 as a
// launch of its own would store it; the next product adds the heads' shares up (rowdot.h, sums). A workgroup takes a head and 64 of Wp's rows, which are on
// their way to registers (HS / 8 lanes and a piece of 16 bytes each to a row) over the attention's own memory trips; the head's other workgroups form
// the same attention again, since a CU takes its 82 KB of Wp no faster than two launches take all of it. For small models, whose launches are
// all latency, where small_step.hip does not take the step: forwards of one token outside a session and models of more than 16 layers. us a token, five
// launches a layer -> four: 19M 340 -> 280, 49M 516 -> 416 (the host's calls), a session's step of 24 layers of 640 434 -> 411 at 30 tokens and 490 -> 482 at
// 300, of 20 layers of 1024 404 -> 397 and 457 -> 449. (A session's step of 10 layers of 640 so, five launches 193: a head's rows in one
// workgroup 201, in two 192, four 188, five 185, ten 183.)
template <int HS, int U, int NTH>
__global__ __launch_bounds__(NTH) void attention_proj_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
                                                             const int* __restrict__ pos, int S, int nh, float scale_log2, const bf16_t* __restrict__ W,
                                                             float* __restrict__ part) {
  constexpr int LR = HS / 8;  // lanes to a row
  static_assert(NTH / LR == 64 && LR == 8);
  __shared__ __align__(16) float lds[attention_lds_floats<HS, NTH>() + HS];
  const int h = blockIdx.x, C = nh * HS, j = threadIdx.x % LR, n = 64 * blockIdx.y + threadIdx.x / LR;
  u32x4 w;
  attention_body<HS, U, NTH, false, U / 2, false, true>(
      q, kc, vc, nullptr, pos, 1, S, nh, scale_log2, h, 0, lds, 1, 0, nullptr, nullptr, 0.f, nullptr, 0, true, nullptr,
      [&] { w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(W + (size_t)n * C + h * HS + 8 * j)); });
  const float* y = lds + attention_lds_floats<HS, NTH>() + 8 * j;
  float a = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    a = fmaf(bflo(w[e]), y[2 * e], a);
    a = fmaf(bfhi(w[e]), y[2 * e + 1], a);
  }
  a += dpp_f32<kDppXor1>(a);
  a += dpp_f32<kDppXor2>(a);
  a += dpp_f32<kDppHalfMirror>(a);
  if (j == 0) __hip_atomic_store(part + (size_t)h * C + n, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// split-K attention over the keys (long contexts): block (head, row, split) -> partial
template <int HS, int U, int NTH>
__global__ __launch_bounds__(NTH) void attention_part_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                             const bf16_t* __restrict__ vc, const int* __restrict__ pos,
                                                             int T, int S, int nh, float scale_log2, int nsplit,
                                                             float* __restrict__ part) {
  __shared__ float lds[attention_lds_floats<HS, NTH>()];
  attention_body<HS, U, NTH, true>(q, kc, vc, nullptr, pos, T, S, nh, scale_log2, blockIdx.x, blockIdx.y, lds, nsplit,
                                   blockIdx.z, part);
}

// attention_part_kernel's key ranges merged by the last block of each (row, head), in one launch and with the bits of the two:
// LLM.int8 logits move by up to 0.03 of their size with the order of these sums. Against the two launches, us in a graph, ranges of
// 256 keys, hs 128: 32 heads, 500 of 512 keys 8.2 -> 7.8; 1010 of 1033 9.9 -> 8.9; 2000 of 2048 15.8 -> 12.1; 100 of 2048 6.6 -> 5.9;
// 40 heads, 1400 keys 13.9 -> 11.1; 8 rows, 900 keys 29.1 -> 27.0. Interleaved ranges gain 1 to 3 % more where few keys are
// in use, and add in another order.
template <int HS, int U, int NTH>
__global__ __launch_bounds__(NTH) void attention_ranges_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                               const bf16_t* __restrict__ vc, bf16_t* __restrict__ y,
                                                               const int* __restrict__ pos, int T, int S, int nh,
                                                               float scale_log2, int nsplit, float* __restrict__ part,
                                                               int* __restrict__ count, uint32_t* st, float thr,
                                                               uint32_t* clr, int clr_words) {
  __shared__ float lds[attention_lds_floats<HS, NTH>()];
  attention_body<HS, U, NTH, true>(q, kc, vc, y, pos, T, S, nh, scale_log2, blockIdx.x, blockIdx.y, lds, nsplit, blockIdx.z, part, st,
                                   thr, clr, clr_words, false, count);
}

// interleaved key splits of a short cache (attention.h ILV), partials merged by the consumer
template <int HS, int U, int NTH, int SPECU>
__global__ __launch_bounds__(NTH) void attention_ilv_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                            const bf16_t* __restrict__ vc, const int* __restrict__ pos,
                                                            int T, int S, int nh, float scale_log2, int nsplit,
                                                            float* __restrict__ part, int spec_ok) {
  __shared__ float lds[attention_lds_floats<HS, NTH>()];
  attention_body<HS, U, NTH, true, SPECU, true>(q, kc, vc, nullptr, pos, T, S, nh, scale_log2, blockIdx.x, blockIdx.y,
                                                lds, nsplit, blockIdx.z, part, nullptr, 0.f, nullptr, 0,
                                                spec_ok != 0);
}

// ---- greedy next token: argmax over bf16 logits (lowest index on ties). Reference
// generate.py:66-74 with top_k = 1 (multinomial over the kept maximum). One workgroup per row: a launch, one trip to memory and
// the compares of one CU. The maximum is found first, two instructions a value; then only a thread that holds it looks where,
// and the place in the row of tokens is read beside the logits. Value and index carried together through every step, us before ->
// now: 32000 bf16 6.1 -> 3.7, 8 rows 6.5 -> 4.0, 100278 20.6 -> 16.2 (a launch that does nothing: 3.6 between events).
template <typename T>
__global__ __launch_bounds__(1024) void argmax_kernel(const T* __restrict__ logits, int ldl, int V,
                                                      int* __restrict__ out_idx, int* __restrict__ tokens_out,
                                                      int tok_stride, const int* __restrict__ pos, int pos_step) {
  __shared__ __attribute__((aligned(16))) float sv[16];
  __shared__ int first;
  const int m = blockIdx.x, tid = threadIdx.x;
  const T* lr = logits + (size_t)m * ldl;
  const int at = tokens_out ? pos[m * pos_step] + 1 : 0;
  if (tid == 0) first = 0x7fffffff;
  float mx = -INFINITY;
  auto take = [&](float x) { mx = x > mx ? x : mx; };  // (a NaN is never taken)
  bool vec = false;
  if constexpr (sizeof(T) == 2) vec = (V & 7) == 0 && (ldl & 7) == 0 && (reinterpret_cast<uintptr_t>(lr) & 15) == 0;
  // 16-byte loads, 4 in flight per thread before any compare (V <= 32768 in one round)
  const uint4* l4 = reinterpret_cast<const uint4*>(lr);
  const int nv = V >> 3;
  uint4 r[4];
  auto fetch = [&](int v0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = l4[v0 + 1024 * u < nv ? v0 + 1024 * u : v0];
  };
  if (vec) {
    for (int v0 = tid; v0 < nv; v0 += 4 * 1024) {
      fetch(v0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // (past the row: v0's once more)
        const uint32_t w[4] = {r[u].x, r[u].y, r[u].z, r[u].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          take(bflo(w[i]));
          take(bfhi(w[i]));
        }
      }
    }
  } else {
#pragma unroll 8
    for (int v = tid; v < V; v += 1024) take(ldv(lr, v));
  }
  const float wmx = wave_max(mx);
  if ((tid & 63) == 0) sv[tid >> 6] = wmx;
  __syncthreads();
  float top = -INFINITY;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 f = reinterpret_cast<const float4*>(sv)[q];
    top = fmaxf(fmaxf(top, fmaxf(f.x, f.y)), fmaxf(f.z, f.w));
  }
  int bi = 0x7fffffff;
  if (mx == top) {
    if (vec) {
      for (int v0 = tid; v0 < nv && bi == 0x7fffffff; v0 += 4 * 1024) {
        if (nv > 4 * 1024) fetch(v0);  // (else the row is still in registers)
#pragma unroll
        for (int u = 3; u >= 0; --u) {
          const int v = v0 + 1024 * u;
          const uint32_t w[4] = {r[u].x, r[u].y, r[u].z, r[u].w};
#pragma unroll
          for (int i = 3; i >= 0; --i) {
            if (v < nv && bfhi(w[i]) == top) bi = 8 * v + 2 * i + 1;
            if (v < nv && bflo(w[i]) == top) bi = 8 * v + 2 * i;
          }
        }
      }
    } else {
      for (int v = tid; v < V && bi == 0x7fffffff; v += 1024)
        if (ldv(lr, v) == top) bi = v;
    }
  }
  if (__any(bi != 0x7fffffff)) {  // (an atomic a lane is a turn a lane: where many hold the maximum, one of 16)
    auto take_first = [&](uint32_t other) { bi = min(bi, (int)other); };
    take_first(dpp_u32<kDppHalfMirror>(bi));
    take_first(dpp_u32<kDppRowMirror>(bi));
    take_first(dpp_u32<kDppXor1>(bi));
    take_first(dpp_u32<kDppXor2>(bi));
    if ((tid & 15) == 0 && bi != 0x7fffffff) atomicMin(&first, bi);
  }
  __syncthreads();
  if (tid == 0) {
    const int chosen = first == 0x7fffffff ? 0 : first;  // all-NaN row: 0
    out_idx[m] = chosen;
    if (tokens_out) tokens_out[(size_t)m * tok_stride + at] = chosen;
  }
}


// ---- sampled next token (generate.py:66-74 with top_k > 1 / None and a temperature):
//   x = bf16(logits * (1 / temperature)) (a bf16 tensor divided by a scalar on the device),
//   keep x >= the top_k-th largest x (torch.topk + where(x < v[-1], -inf): ties at the
//   threshold are kept), probs = bf16(softmax(x)) (fp32 inside), then one draw from probs.
// The draw is the inverse CDF over the kept probabilities in index order at a uniform u in
// [0, 1): the first index whose running sum exceeds u * sum(probs). torch.multinomial draws
// from the same distribution with its own generator (exponential race); u is either given
// (u_in, tests) or a counter-based hash of (seed, decode position, row), so a captured decode
// graph samples a fresh u every step without the host.
// One 1024-thread block per row, bound by its chain of block-wide steps and, the row being one CU's, by the instructions per
// value. The row is read once, as order-preserving keys, into LDS (rows of more than kSampRow bytes are read again by each pass).
// Each thread keeps the largest key it loaded; for top_k <= 1024 the top_k-th largest of those 1024 keys, rounded down to its
// histogram bin, cannot lie above the top_k-th largest key of all, so only keys from there on -- a few hundred -- enter the exact
// radix select (histograms of 11 + 5 bits of the bf16 keys, of 11 + 11 + 10 of the fp32 keys) and the passes after it: the set
// bits of a mask over a thread's range. The running sum over the threads is one chain of additions in thread order, of the threads
// that keep anything (a zero adds nothing), along the lanes of a wave. Where every pass read the row in memory and the chain
// ran through LDS, us a launch, before -> now, V = 32000 bf16: top_k 200 55.1 -> 16.3, 1100 55.2 -> 32.5, all 55.2 -> 29.0;
// V = 35008 bf16: 47.4 -> 17.8; V = 32000 fp32: 62.2 -> 19.9; V = 100278 bf16 (not in LDS): 147 -> 66.
__device__ __forceinline__ uint32_t bf_key(uint32_t b) { return (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u); }
__device__ __forceinline__ float key_bf(uint32_t k) {
  const uint32_t b = (k & 0x8000u) ? (k & 0x7FFFu) : (~k & 0xFFFFu);
  return bf2f((bf16_t)b);
}
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

constexpr int kSampNT = 1024;
// inclusive prefix over the wave in lane order (OP 0: sum, 1: maximum)
template <int OP>
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
#define LLJ_DPP_STEP(ctrl, rows)                                                                  \
  {                                                                                               \
    const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false);  \
    v = OP ? max(v, t) : v + t;                                                                   \
  }
  LLJ_DPP_STEP(0x111, 0xf)  // row_shr 1, 2, 4, 8: within 16 lanes
  LLJ_DPP_STEP(0x112, 0xf)
  LLJ_DPP_STEP(0x114, 0xf)
  LLJ_DPP_STEP(0x118, 0xf)
  LLJ_DPP_STEP(0x142, 0xa)  // the last lane of rows 0, 2 into rows 1, 3; then of the first half into the second
  LLJ_DPP_STEP(0x143, 0xc)
#undef LLJ_DPP_STEP
  return v;
}
constexpr int kSampWaves = kSampNT / 64;
// one value per wave, all read at once
__device__ __forceinline__ void per_wave(const uint32_t* w, uint32_t (&o)[kSampWaves]) {
#pragma unroll
  for (int i = 0; i < kSampWaves / 4; ++i) {
    const uint4 q = reinterpret_cast<const uint4*>(w)[i];
    o[4 * i] = q.x;
    o[4 * i + 1] = q.y;
    o[4 * i + 2] = q.z;
    o[4 * i + 3] = q.w;
  }
}

// The logits type of the sampler: bf16 (the reference's GPU precision: x = bf16(logits * (1/T)),
// probabilities rounded to bf16) or fp32 (its
// float32 model: x = logits / T, fp32 softmax).
template <typename T>
struct SampTraits;
template <>
struct SampTraits<bf16_t> {
  static constexpr int NP = 2;
  static constexpr int SH[3] = {5, 0, 0}, W[3] = {11, 5, 0};
  using Key = uint16_t;
  __device__ static uint32_t key(bf16_t l, float inv_t, float) { return bf_key(f2bf(bf2f(l) * inv_t)); }
  __device__ static float val(uint32_t k) { return key_bf(k); }
  __device__ static float ex(float d) { return __expf(d); }
  __device__ static float prob(float e) { return bf2f(f2bf(e)); }
};
__device__ __forceinline__ uint32_t f_key(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_f(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k); }
template <>
struct SampTraits<float> {
  static constexpr int NP = 3;
  static constexpr int SH[3] = {21, 10, 0}, W[3] = {11, 11, 10};
  using Key = uint32_t;
  __device__ static uint32_t key(float l, float, float t) { return f_key(l / t); }
  __device__ static float val(uint32_t k) { return key_f(k); }
  __device__ static float ex(float d) { return expf(d); }
  __device__ static float prob(float e) { return e; }
};

constexpr size_t kSampRow = 144 * 1024;  // largest row of keys held in LDS

// stride: Keys from one thread's range to the next in LDS (0: not there; more than the range: an odd number of words, so that
// the threads' places lie in different banks, and 16-byte pieces of the row are each one thread's)
template <typename T>
__global__ __launch_bounds__(kSampNT) void sample_kernel(const T* __restrict__ logits, int ldl, int V, float inv_t,
                                                        float temp, int top_k, const float* __restrict__ u_in,
                                                        uint64_t seed, int* __restrict__ out_idx,
                                                        int* __restrict__ tokens_out, int tok_stride,
                                                        const int* __restrict__ pos, int pos_step, int stride) {
  using Tr = SampTraits<T>;
  using Key = typename Tr::Key;
  constexpr int HB = 2048;  // the widest pass: 11 bits
  extern __shared__ __attribute__((aligned(16))) unsigned char samp_row[];
  __shared__ __attribute__((aligned(16))) uint32_t hist[HB];  // the histograms; then the kept threads' sums and what precedes each
  __shared__ __attribute__((aligned(16))) uint32_t ured[2][kSampWaves];
  __shared__ float fred[kSampWaves];
  __shared__ uint32_t sel[4];
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const T* lr = logits + (size_t)m * ldl;
  const int place = pos ? pos[m * pos_step] + 1 : 0;
  // row m of the uniforms of this position (or of the only position without pos)
  const float u = u_in ? u_in[(size_t)place * gridDim.x + m]
                       : (float)(splitmix64(seed ^ ((uint64_t)place << 20) ^ (uint64_t)m) >> 40) * (1.0f / 16777216.0f);
  const int k = top_k < 1 || top_k > V ? V : top_k;
  // each thread owns a contiguous index range (the CDF is taken in index order)
  const int per = (V + kSampNT - 1) / kSampNT;
  const int i0 = min(V, tid * per), i1 = min(V, i0 + per);
  Key* own = reinterpret_cast<Key*>(samp_row) + tid * stride;
  auto key_at = [&](int i) -> uint32_t { return stride ? (uint32_t)own[i - i0] : Tr::key(lr[i], inv_t, temp); };

  // ---- the keys, and this thread's largest (any partition of the row serves for that)
  for (int b = tid; b < HB; b += kSampNT) hist[b] = 0;
  uint32_t tmax = 0;
  constexpr int E = 16 / sizeof(T);
  auto piece = [&](const uint4 w, Key (&ks)[E]) {
    const T* x = reinterpret_cast<const T*>(&w);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint32_t key = Tr::key(x[e], inv_t, temp);
      tmax = max(tmax, key);
      ks[e] = (Key)key;
    }
  };
  const bool ranges = stride > per;
  const int nv = ((uintptr_t)lr & 15) ? 0 : ranges ? (i1 - i0) / E : V / E;
  const uint4* src = reinterpret_cast<const uint4*>(ranges ? lr + i0 : lr);
#pragma unroll 4
  for (int v = ranges ? 0 : tid; v < nv; v += ranges ? 1 : kSampNT) {
    Key ks[E];
    piece(src[v], ks);
    if (ranges) {  // (rows of an odd number of words: 4-byte places)
#pragma unroll
      for (int e = 0; e < 4; ++e) reinterpret_cast<uint32_t*>(own + v * E)[e] = reinterpret_cast<const uint32_t*>(ks)[e];
    } else if (stride) {  // ranges follow each other
      reinterpret_cast<uint4*>(samp_row)[v] = *reinterpret_cast<const uint4*>(ks);
    }
  }
  for (int i = ranges ? i0 + nv * E : nv * E + tid; i < (ranges ? i1 : V); i += ranges ? 1 : kSampNT) {
    const uint32_t key = Tr::key(lr[i], inv_t, temp);
    tmax = max(tmax, key);
    if (ranges) own[i - i0] = (Key)key;
    else if (stride) reinterpret_cast<Key*>(samp_row)[i] = (Key)key;
  }
  const uint32_t wmax = wave_prefix<1>(tmax);
  if (lane == 63) ured[0][wv] = wmax;
  __syncthreads();
  uint32_t each_wave[kSampWaves], kmax = 0;
  per_wave(ured[0], each_wave);
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) kmax = max(kmax, each_wave[w]);
  const float xmax = Tr::val(kmax);

  // ---- the bin of the want-th largest key counted in hist (nbins bins), and the rank within it: sel[0], sel[1]. hist is left
  // cleared: the next pass may count after it.
  auto find = [&](int nbins, uint32_t want) {
    __syncthreads();
    // thread t owns bins [b0, b0 + nb), nb <= 2: counts above them by a suffix sum
    const int nb = nbins > kSampNT ? 2 : (tid < nbins ? 1 : 0), b0 = nb * tid;
    const uint32_t h0 = nb ? hist[b0] : 0, h1 = nb == 2 ? hist[b0 + 1] : 0, c = h0 + h1;
    if (nb) hist[b0] = 0;
    if (nb == 2) hist[b0 + 1] = 0;
    const uint32_t incl = wave_prefix<0>(c);
    if (lane == 63) ured[1][wv] = incl;
    __syncthreads();
    per_wave(ured[1], each_wave);
    uint32_t above = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63) - incl;
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w) above += w > wv ? each_wave[w] : 0;
    if (above < want && want <= above + c) {  // exactly one thread
      const bool upper = nb == 2 && above + h1 >= want;
      sel[0] = (uint32_t)(upper ? b0 + 1 : b0);
      sel[1] = want - (nb == 2 && !upper ? above + h1 : above);
    }
    __syncthreads();
  };
  uint32_t low = 0;  // no candidate lies below
  const bool few = k < V && k <= kSampNT;
  if (few) {
    atomicAdd(&hist[tmax >> Tr::SH[0]], 1u);
    find(1 << Tr::W[0], (uint32_t)k);
    low = sel[0] << Tr::SH[0];
  }
  // ---- candidates: bit e of the mask stands for 1 << qs elements of this thread's range
  int qs = 0;
  while ((per - 1) >> qs > 63) ++qs;
  uint64_t mask = 0;
  if (few && ranges && qs == 0 && sizeof(Key) == 2) {  // two keys per word: the upper decides a comparison of whole words
    if (tmax >= low) {
      const uint32_t* pairs = reinterpret_cast<const uint32_t*>(own);
      const uint32_t bar = low << 16;
      uint32_t half[2] = {0, 0};
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll 8
        for (int i = 16 * h; i < min(per / 2, 16 * h + 16); ++i) {
          const uint32_t w = pairs[i], two = ((w << 16) >= bar ? 1u : 0u) | (w >= bar ? 2u : 0u);
          half[h] |= two << (2 * (i & 15));
        }
      mask = ((uint64_t)half[1] << 32) | half[0];
      if (i1 - i0 < 64) mask &= (1ull << (i1 - i0)) - 1;
    }
  } else if (few && !(ranges && tmax < low)) {
    uint32_t half[2] = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll 8
      for (int i = i0 + (h << (5 + qs)); i < min(i1, i0 + (32 << qs) + (h << (5 + qs))); ++i)
        half[h] |= (key_at(i) >= low ? 1u : 0u) << (((i - i0) >> qs) & 31);
    mask = ((uint64_t)half[1] << 32) | half[0];
  }
  auto each = [&](auto&& f) {  // f(index, key) over the candidates in index order, until it returns false
    if (!few) {
      for (int i = i0; i < i1; ++i)
        if (!f(i, key_at(i))) return;
      return;
    }
    for (uint64_t b = mask; b; b &= b - 1) {
      const int s0 = i0 + ((int)__builtin_ctzll(b) << qs), s1 = min(i1, s0 + (1 << qs));
      for (int i = s0; i < s1; ++i) {
        const uint32_t key = key_at(i);
        if (key >= low && !f(i, key)) return;
      }
    }
  };
  // ---- radix select among them: thr = the k-th largest key; keep key >= thr
  uint32_t thr = 0;
  if (k < V) {
    uint32_t prefix = 0, want = (uint32_t)k;
#pragma unroll
    for (int pass = 0; pass < Tr::NP; ++pass) {
      const int sh = Tr::SH[pass], nbins = 1 << Tr::W[pass];
      auto count = [&](int, uint32_t key) {
        if (pass == 0 || (key >> (sh + Tr::W[pass])) == prefix) atomicAdd(&hist[(key >> sh) & (nbins - 1)], 1u);
        return true;
      };
      if (few || stride) each(count);
      else
        for (int i = tid; i < V; i += kSampNT) count(i, key_at(i));
      find(nbins, want);
      prefix = pass == 0 ? sel[0] : (prefix << Tr::W[pass]) | sel[0];
      want = sel[1];
    }
    thr = prefix;
  }
  // ---- sum of exp over the kept values (fp32, fixed reduction order)
  float esum = 0.f;
  each([&](int, uint32_t key) {
    if (key >= thr) esum += Tr::ex(Tr::val(key) - xmax);
    return true;
  });
  float t = wave_sum(esum);
  if (lane == 0) fred[wv] = t;
  if (tid == 0) sel[2] = sel[3] = 0;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) tot += fred[w];
  const float rinv = 1.f / tot;
  // probabilities, the threads' sums, exclusive scan over the threads that have one (thread order = index order)
  float csum = 0.f;
  int last = -1;
  each([&](int i, uint32_t key) {
    if (key >= thr) {
      csum += Tr::prob(Tr::ex(Tr::val(key) - xmax) * rinv);
      last = i;
    }
    return true;
  });
  if (last >= 0) atomicMax(&sel[2], (uint32_t)last);
  const bool some = csum != 0.f;  // (NaN too)
  const unsigned long long bal = __ballot(some);
  if (lane == 0) ured[0][wv] = (uint32_t)__popcll(bal);
  __syncthreads();
  per_wave(ured[0], each_wave);
  int at = __popcll(bal & ((1ull << lane) - 1ull)), n = 0;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) {
    at += w < wv ? (int)each_wave[w] : 0;
    n += (int)each_wave[w];
  }
  float* sums = reinterpret_cast<float*>(hist);
  float* excl = sums + kSampNT;
  if (some) sums[at] = csum;
  __syncthreads();
  if (wv == 0) {  // one chain of additions: after step j the lanes up to j hold their sum, each its neighbour's plus its own
    float run = 0.f;
    for (int j = 0; j < n; j += 64) {
      const float c = j + lane < n ? sums[j + lane] : 0.f, carry = run;
      float before = carry;
#pragma unroll 8
      for (int e = 0; e < 64; ++e) {
        before = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(carry), __float_as_int(run), 0x138, 0xf, 0xf, false));
        run = before + c;
      }
      excl[j + lane] = before;
      run = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(run), 63));
    }
    if (lane == 0) fred[0] = run;
  }
  __syncthreads();
  const float run = fred[0], target = u * run;
  if (some) {
    const float base = excl[at], next = at + 1 < n ? excl[at + 1] : run;
    if (base <= target && target < next) {  // one thread at most
      float r = base;
      int pick = last;
      each([&](int i, uint32_t key) {
        if (key < thr) return true;
        r += Tr::prob(Tr::ex(Tr::val(key) - xmax) * rinv);
        if (r > target) pick = i;
        return !(r > target);
      });
      sel[3] = (uint32_t)pick + 1;
    }
  }
  __syncthreads();
  if (tid == 0) {
    const int pick = sel[3] ? (int)sel[3] - 1 : (int)sel[2];  // u * sum at the very end (rounding): the last kept index
    out_idx[m] = pick;
    if (tokens_out) tokens_out[(size_t)m * tok_stride + place] = pick;
  }
}

template <typename T>
static int sample_launch(const T* logits, int ldl, int M, int V, float temperature, int top_k, const float* u, uint64_t seed,
                         int* out_idx, int* tokens_out, int tok_stride, const int* pos, int pos_step, hipStream_t s) {
  constexpr int KB = sizeof(typename SampTraits<T>::Key), E = 16 / sizeof(T);
  const int per = (V + kSampNT - 1) / kSampNT;
  // ranges of whole 16-byte pieces lie an even number of words apart: one more word between them
  int stride = per % E == 0 && ((uintptr_t)logits & 15) == 0 && ldl % E == 0 ? per + 4 / KB : per;
  if ((size_t)stride * kSampNT * KB > kSampRow) stride = 0;
  static const hipError_t set =
      hipFuncSetAttribute((const void*)sample_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSampRow);
  if (set != hipSuccess) return (int)set;
  hipLaunchKernelGGL(sample_kernel<T>, dim3(M), dim3(kSampNT), (size_t)stride * kSampNT * KB, s, logits, ldl, V, 1.f / temperature,
                     temperature, top_k, u, seed, out_idx, tokens_out, tok_stride, pos, pos_step, stride);
  LLJ_CHECK_LAUNCH();
  return 0;
}

// Streaming read of n16 16-byte words (the achievable HBM read rate the decode kernels are priced
// against): grid-stride, 4 non-temporal loads in flight per thread, one float per workgroup out so
// the loads stay live.
__global__ __launch_bounds__(256) void stream_read_kernel(const uint4* __restrict__ p, size_t n16, float* out) {
  typedef uint32_t v4u __attribute__((ext_vector_type(4)));
  const v4u* q = reinterpret_cast<const v4u*>(p);
  uint32_t acc = 0;
  const size_t stride = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const v4u a = __builtin_nontemporal_load(q + i), b = __builtin_nontemporal_load(q + i + stride);
    const v4u c = __builtin_nontemporal_load(q + i + 2 * stride), d = __builtin_nontemporal_load(q + i + 3 * stride);
    acc ^= a.x ^ b.y ^ c.z ^ d.w;
  }
  for (; i < n16; i += stride) acc ^= __builtin_nontemporal_load(q + i).x;
  __shared__ uint32_t r[256];
  r[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int k = 0; k < 256; ++k) t ^= r[k];
    out[blockIdx.x] = (float)(t & 0xFFu);
  }
}

}  // namespace llj

using namespace llj;

extern "C" {
LLJ_TRACE_EXPORT(ops)

int llj_stream_read(const void* p, size_t bytes, float* out, int grid, void* stream) {
  LLJ_REQUIRE(p && out && bytes % 16 == 0 && grid > 0);
  hipLaunchKernelGGL(stream_read_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const uint4*)p, bytes / 16, out);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_embedding(const int* idx, const void* wte, void* out, int M, int C, int* pos_inc, void* stream) {
  LLJ_REQUIRE(M > 0 && C > 0);
  if (C % 8) {
    hipLaunchKernelGGL(embedding_any_kernel, dim3(M), dim3(256), 0, (hipStream_t)stream, idx, (const bf16_t*)wte,
                       (bf16_t*)out, C, pos_inc);
    LLJ_CHECK_LAUNCH();
    return 0;
  }
  hipLaunchKernelGGL(embedding_kernel, dim3(M), dim3(256), 0, (hipStream_t)stream, idx, (const uint4*)wte,
                     (uint4*)out, C / 8, pos_inc);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_rmsnorm(const void* x, const void* w, float eps, void* y, int M, int C, void* stream) {
  return llj_rmsnorm_rows(x, w, eps, y, nullptr, M, C, stream);
}

int llj_rmsnorm_rows(const void* x, const void* w, float eps, void* y, float* rowsum, int M, int C, void* stream) {
  LLJ_REQUIRE(M > 0 && C % 8 == 0);
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(M), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)x,
                     (const bf16_t*)w, eps, (bf16_t*)y, C, rowsum);
  LLJ_CHECK_LAUNCH();
  return 0;
}

// decode attention, optionally with the LLM.int8 statistics of y (int8 c_proj) and a block to zero
static int attention_run(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T,
                         int n_head, int head_size, int S, uint32_t* st, float thr, uint32_t* clr, int clr_words,
                         void* stream) {
  LLJ_REQUIRE(B > 0 && T > 0 && n_head > 0 && S > 0);
  const float sl2 = 1.4426950408889634f / sqrtf((float)head_size);
  dim3 grid(n_head, B * T);
  // keys loaded before the position is known at small grids: half a pass (default) or a whole one
  // (option LLJ_OPT_ATT_SPEC_FULL: one memory latency less, more K / V rows read past the position)
  const bool full = opt(LLJ_OPT_ATT_SPEC_FULL) == 1;
  const int sb = opt(LLJ_OPT_ATT_SPEC_BATCH);
  const int spec_ok = (int)grid.x * (int)grid.y <= 64 || (!full && (sb < 0 ? LLJ_ATT_SPEC_BATCH : sb) != 0);
  hipStream_t st_ = (hipStream_t)stream;
#define LLJ_ATT_LAUNCH(HS_, SU_)                                                                                   \
  hipLaunchKernelGGL((attention_kernel<HS_, LLJ_ATT_U, LLJ_ATT_NTH, SU_>), grid, dim3(LLJ_ATT_NTH), 0, st_,         \
                     (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, (bf16_t*)y, pos, T, S, n_head, sl2, \
                     st, thr, clr, clr_words, spec_ok)
  if (head_size == 128) {
    if (full) LLJ_ATT_LAUNCH(128, LLJ_ATT_U); else LLJ_ATT_LAUNCH(128, LLJ_ATT_U / 2);
  } else if (head_size == 64) {
    if (full) LLJ_ATT_LAUNCH(64, LLJ_ATT_U); else LLJ_ATT_LAUNCH(64, LLJ_ATT_U / 2);
  } else {
    return LLJ_EINVAL;
  }
#undef LLJ_ATT_LAUNCH
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_attention(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T,
                  int n_head, int head_size, int S, void* stream) {
  return attention_run(q, kcache, vcache, y, pos, B, T, n_head, head_size, S, nullptr, 0.f, nullptr, 0, stream);
}

// 512 (where one bf16 row goes to rowdot.h) to 1024 values in heads of 64
int llj_attention_proj_ok(int n_head, int head_size, int S) { return head_size == 64 && n_head >= 8 && n_head <= 16 && S > 0; }

int llj_attention_proj(const void* q, const void* kcache, const void* vcache, const int* pos, int n_head, int head_size, int S, const void* W,
                       float* part, void* stream) {
  LLJ_REQUIRE(q && kcache && vcache && pos && W && part && llj_attention_proj_ok(n_head, head_size, S) &&
              (((uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)W) & 15) == 0);
  hipLaunchKernelGGL((attention_proj_kernel<64, LLJ_ATT_U, 512>), dim3(n_head, n_head), dim3(512), 0, (hipStream_t)stream, (const bf16_t*)q,
                     (const bf16_t*)kcache, (const bf16_t*)vcache, pos, S, n_head, 1.4426950408889634f / 8.f, (const bf16_t*)W, part);
  LLJ_CHECK_LAUNCH();
  return 0;
}

size_t llj_attention_ws_bytes(int rows, int n_head, int head_size, int nsplit) {
  return (size_t)rows * n_head * (nsplit < 1 ? 1 : nsplit) * (head_size + 4) * sizeof(float);  // kAttPart
}

static int attention_split_run(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B,
                               int T, int n_head, int head_size, int S, int nsplit, void* part_ws, uint32_t* st,
                               float thr, uint32_t* clr, int clr_words, void* stream) {
  if (nsplit <= 1)
    return attention_run(q, kcache, vcache, y, pos, B, T, n_head, head_size, S, st, thr, clr, clr_words, stream);
  LLJ_REQUIRE(B > 0 && T > 0 && n_head > 0 && S > 0 && part_ws && nsplit <= 1024);
  const float sl2 = 1.4426950408889634f / sqrtf((float)head_size);
  const dim3 grid(n_head, B * T, nsplit), cgrid(n_head, B * T);
  hipStream_t s = (hipStream_t)stream;
  if (head_size == 128) {
    hipLaunchKernelGGL((attention_part_kernel<128, LLJ_ATT_U, LLJ_ATT_NTH>), grid, dim3(LLJ_ATT_NTH), 0, s,
                       (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, pos, T, S, n_head, sl2, nsplit,
                       (float*)part_ws);
    LLJ_CHECK_LAUNCH();
    hipLaunchKernelGGL((attention_combine_kernel<128>), cgrid, dim3(128), 0, s, (const float*)part_ws, (bf16_t*)y,
                       n_head, nsplit, st, thr, clr, clr_words);
  } else if (head_size == 64) {
    hipLaunchKernelGGL((attention_part_kernel<64, LLJ_ATT_U, LLJ_ATT_NTH>), grid, dim3(LLJ_ATT_NTH), 0, s,
                       (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, pos, T, S, n_head, sl2, nsplit,
                       (float*)part_ws);
    LLJ_CHECK_LAUNCH();
    hipLaunchKernelGGL((attention_combine_kernel<64>), cgrid, dim3(64), 0, s, (const float*)part_ws, (bf16_t*)y,
                       n_head, nsplit, st, thr, clr, clr_words);
  } else {
    return LLJ_EINVAL;
  }
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_attention_split(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T,
                        int n_head, int head_size, int S, int nsplit, void* part_ws, void* stream) {
  return attention_split_run(q, kcache, vcache, y, pos, B, T, n_head, head_size, S, nsplit, part_ws, nullptr, 0.f,
                             nullptr, 0, stream);
}

int llj_attention_ranges(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T,
                         int n_head, int head_size, int S, int nsplit, void* part_ws, int* count, void* y_stats, void* clr,
                         int clr_words, float threshold, void* stream) {
  LLJ_REQUIRE(q && kcache && vcache && y && pos && B > 0 && T > 0 && n_head > 0 && S > 0 && nsplit >= 1 && nsplit <= 64 && part_ws &&
              ((uintptr_t)part_ws & 7) == 0 && count && (!y_stats || B * T <= 8) && clr_words >= 0 && (!clr_words || clr));
  const float sl2 = 1.4426950408889634f / sqrtf((float)head_size);
  const dim3 grid(n_head, B * T, nsplit);
#define LLJ_ATT_RANGES(HS_)                                                                                              \
  hipLaunchKernelGGL((attention_ranges_kernel<HS_, LLJ_ATT_U, LLJ_ATT_NTH>), grid, dim3(LLJ_ATT_NTH), 0, (hipStream_t)stream, \
                     (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, (bf16_t*)y, pos, T, S, n_head, sl2, nsplit, \
                     (float*)part_ws, count, (uint32_t*)y_stats, threshold, (uint32_t*)clr, clr_words)
  if (head_size == 128) LLJ_ATT_RANGES(128);
  else if (head_size == 64) LLJ_ATT_RANGES(64);
  else return LLJ_EINVAL;
#undef LLJ_ATT_RANGES
  LLJ_CHECK_LAUNCH();
  return 0;
}

// Decode attention (one-block or split over nsplit key ranges) that also writes the LLM.int8
// statistics of y for the int8 c_proj (i8ws.h; y_stats zeroed beforehand, B * T <= 8 rows) and zeroes
// clr_words words at clr (the previous layer's mlp.c_proj statistics block).
// Decode attention as nsplit interleaved key splits per (row, head) (block s takes the key groups
// s * NG + NG * nsplit * i: a fixed set, loaded before the position is known at small grids), each writing
// its unnormalized partial to part_ws; no combine launch -- llj_linear_resid_attn merges them in its prologue.
int llj_attention_part(const void* q, const void* kcache, const void* vcache, const int* pos, int B, int T,
                       int n_head, int head_size, int S, int nsplit, void* part_ws, void* stream) {
  LLJ_REQUIRE(B > 0 && T > 0 && n_head > 0 && S > 0 && part_ws && nsplit >= 1 && nsplit <= 64);
  const float sl2 = 1.4426950408889634f / sqrtf((float)head_size);
  const dim3 grid(n_head, B * T, nsplit);
  const int spec_ok = (int)(grid.x * grid.y * grid.z) <= 256;
  hipStream_t s = (hipStream_t)stream;
  if (head_size == 128)
    hipLaunchKernelGGL((attention_ilv_kernel<128, LLJ_ATT_U, LLJ_ATT_NTH, LLJ_ATT_U / 2>), grid, dim3(LLJ_ATT_NTH), 0, s,
                       (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, pos, T, S, n_head, sl2, nsplit,
                       (float*)part_ws, spec_ok);
  else if (head_size == 64)
    hipLaunchKernelGGL((attention_ilv_kernel<64, LLJ_ATT_U, LLJ_ATT_NTH, LLJ_ATT_U / 2>), grid, dim3(LLJ_ATT_NTH), 0, s,
                       (const bf16_t*)q, (const bf16_t*)kcache, (const bf16_t*)vcache, pos, T, S, n_head, sl2, nsplit,
                       (float*)part_ws, spec_ok);
  else
    return LLJ_EINVAL;
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_attention_i8(const void* q, const void* kcache, const void* vcache, void* y, const int* pos, int B, int T,
                     int n_head, int head_size, int S, int nsplit, void* part_ws, void* y_stats, void* clr,
                     int clr_words, float threshold, void* stream) {
  LLJ_REQUIRE(y_stats && B * T <= 8 && clr_words >= 0 && (!clr_words || clr));
  return attention_split_run(q, kcache, vcache, y, pos, B, T, n_head, head_size, S, nsplit, part_ws,
                             (uint32_t*)y_stats, threshold, (uint32_t*)clr, clr_words, stream);
}

int llj_sample(const void* logits, int ldl, int M, int V, float temperature, int top_k, const float* u,
               unsigned long long seed, int* out_idx, int* tokens_out, int tok_stride, const int* pos, void* stream) {
  LLJ_REQUIRE(M > 0 && V > 0 && temperature > 0.f && (!tokens_out || pos) && (u || pos));
  return sample_launch((const bf16_t*)logits, ldl, M, V, temperature, top_k, u, (uint64_t)seed, out_idx, tokens_out, tok_stride, pos,
                       0, (hipStream_t)stream);
}

int llj_g_sample(const float* logits, int ldl, int M, int V, float temperature, int top_k, const float* u,
                 unsigned long long seed, int* out_idx, int* tokens_out, int tok_stride, const int* pos, void* stream) {
  LLJ_REQUIRE(logits && out_idx && M > 0 && V > 0 && ldl >= V && temperature > 0.f && (!tokens_out || pos) && (u || pos));
  return sample_launch(logits, ldl, M, V, temperature, top_k, u, (uint64_t)seed, out_idx, tokens_out, tok_stride, pos, 0,
                       (hipStream_t)stream);
}

int llj_argmax(const void* logits, int ldl, int M, int V, int* out_idx, int* tokens_out, int tok_stride,
               const int* pos, void* stream) {
  LLJ_REQUIRE(M > 0 && V > 0 && (!tokens_out || pos));
  hipLaunchKernelGGL(argmax_kernel<bf16_t>, dim3(M), dim3(1024), 0, (hipStream_t)stream, (const bf16_t*)logits, ldl, V,
                     out_idx, tokens_out, tok_stride, pos, 0);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_g_argmax(const float* logits, int ldl, int M, int V, int* out_idx, int* tokens_out, int tok_stride, const int* pos,
                 void* stream) {
  LLJ_REQUIRE(logits && out_idx && M > 0 && V > 0 && ldl >= V && (!tokens_out || pos));
  hipLaunchKernelGGL(argmax_kernel<float>, dim3(M), dim3(1024), 0, (hipStream_t)stream, logits, ldl, V, out_idx, tokens_out,
                     tok_stride, pos, 0);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_next_token(const void* logits, int ldl, int M, int V, float temperature, int top_k, const float* u,
                   unsigned long long seed, int* out_idx, int* tokens_out, int tok_stride, const int* pos, int pos_step,
                   int dt, void* stream) {
  LLJ_REQUIRE(logits && out_idx && M > 0 && V > 0 && ldl >= V && pos && (pos_step == 0 || pos_step == 1) &&
              (dt == 0 || dt == 1) && (top_k == 1 || temperature > 0.f));
  hipStream_t s = (hipStream_t)stream;
  if (top_k == 1) {
    LLJ_DT(dt, hipLaunchKernelGGL(argmax_kernel<bf16_t>, dim3(M), dim3(1024), 0, s, (const bf16_t*)logits, ldl, V, out_idx,
                                  tokens_out, tok_stride, pos, pos_step),
           hipLaunchKernelGGL(argmax_kernel<float>, dim3(M), dim3(1024), 0, s, (const float*)logits, ldl, V, out_idx,
                              tokens_out, tok_stride, pos, pos_step));
  } else if (dt == 0) {
    return sample_launch((const bf16_t*)logits, ldl, M, V, temperature, top_k, u, (uint64_t)seed, out_idx, tokens_out, tok_stride,
                         pos, pos_step, s);
  } else {
    return sample_launch((const float*)logits, ldl, M, V, temperature, top_k, u, (uint64_t)seed, out_idx, tokens_out, tok_stride,
                         pos, pos_step, s);
  }
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
