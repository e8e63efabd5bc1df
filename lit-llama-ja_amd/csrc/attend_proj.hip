// One and two decode rows: the attention over the K / V cache and attn.c_proj with its residual add (reference model.py:172, 218-240) in one
// launch. The first workgroups are the attention's (attention.h), the others own 16 columns of c_proj each and wait for y (handover.h).
// us a pair in a graph, weights and caches from memory, two launches -> this (keys past 512 in ranges, as llj_attention_ranges):
//   one row   int4  4096  8.3 -> 6.2 at 30 keys, 8.5 -> 6.4 at 70, 13.2 -> 11.5 at 500, 14.3 -> 12.6 at 1,000   5120  10.4 -> 7.9   2048  7.6 -> 5.8
//             8-bit 4096  10.1 -> 7.9 at 90 keys, 15.6 -> 14.0 at 1,000
//             bf16  4096  11.7 -> 10.5 at 70 keys, 17.3 -> 15.6 at 1,000   5120  14.9 -> 13.7 at 70, 20.7 -> 19.6 at 1,000   2048  8.1 -> 6.4 at 70
//   two rows  4096  int4 9.3 -> 7.9 at 70 keys, 14.2 -> 13.3 at 500   8-bit 10.1 -> 9.2
// The attention's workgroups may not have started when others wait for them (handover.h: beside three such launches at once, each XCD holding the
// waiting workgroups of two). A workgroup whose wait runs out does the attention that is missing itself, to the same bits, and waits for nobody.
// Three and four rows gain 0.1 to 0.7 (with ranges nothing) and eight lose 2: every workgroup takes all rows past the caches. Of two rows with eight
// ranges 5120 gains nothing any more (int4 2,048 keys 27.5 -> 28.1, 600 keys 17.5 -> 16.6, 8-bit 30.5 -> 30.3 and 19.8 -> 19.6).
// Widths: 4096 and 5120 of 7B and 13B, 2048 of models of that width with heads of 128. 6656 and 8192 (30B, 65B) are left out: one row of codes would
// gain (int4 11.0 -> 9.4 and 13.2 -> 11.8 at 70 keys), two rows and bf16 with long caches would lose (6656: int4 23.8 -> 24.4, bf16 28.6 -> 30.7 at 1,000 keys;
// 8192: two 8-bit rows 32.0 -> 39.0).
#include <algorithm>

#include "attention.h"
#include "common.h"
#include "handover.h"
#include "lit_llama_amd.h"

namespace llj {

enum { AP_W4 = HC_W4, AP_BF16 = 1, AP_W8 = HC_W8 };  // wfmt

struct AttendProjParams {
  const bf16_t *q, *kc, *vc;
  uint32_t* y;      // the rows' words, kNotYet when the launch starts
  uint32_t* clear;  // the next launch's
  const int* pos;
  int S, nh;
  float scale_log2;
  int nsplit;
  float* part;
  int* count;
  const void* W;     // c_proj: bf16 (C, C), W4P or W8P
  const float2* sz;  // W4P, W8P: (scale, 128 or 2176 + zero) per column
  bf16_t* x;         // residual, in place
  float* nstat;      // rows: sums of squares of x', 16 columns a place (llj_linear_resid's nstat_out), or NULL
  int C, M, heads;   // heads: workgroups of the attention
  int waits;         // polls of a wait
};

constexpr int kApNT = 512;
constexpr int kApWaits = 1 << 12;  // some milliseconds
// words [at, at + 2) of y, both there or kNotYet in one of them
__device__ __forceinline__ unsigned long long ap_word2(const uint32_t* y, int at) {
  return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(y + at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool ap_there(unsigned long long w) { return (uint32_t)w != kNotYet && (uint32_t)(w >> 32) != kNotYet; }

// One row of bf16. Wave: two columns; lane: values 512 i + 8 lane .. + 7 of both. false (in every thread), with nothing written: a wait ran out
template <int NI>
__device__ __forceinline__ bool ap_bf16_row(const AttendProjParams& p, int nt, unsigned char* smem) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), C = p.C, n0 = 16 * nt;
  const bf16_t* src = reinterpret_cast<const bf16_t*>(p.W) + (size_t)(n0 + 2 * wave) * C + 8 * lane;
  u32x4 w[2][NI];
  const uint32_t x = reinterpret_cast<const uint32_t*>(p.x)[8 * nt + wave];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c) w[c][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + (size_t)c * C + 512 * i));
  // y once per workgroup: thread t the word pairs t, t + 512, ..
  constexpr int NP = (NI * 128 + kApNT - 1) / kApNT;
  unsigned long long v[NP];
  bool got = false;
  for (int t = 0; t < p.waits; ++t) {
    bool there = true;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      v[i] = ap_word2(p.y, 2 * min(tid + kApNT * i, NI * 128 - 1));
      there = there && ap_there(v[i]);
    }
    got = __all(there);
    if (got) break;
    __builtin_amdgcn_s_sleep(1);
  }
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (tid + kApNT * i < NI * 128) reinterpret_cast<unsigned long long*>(smem)[tid + kApNT * i] = v[i];
  int* all = reinterpret_cast<int*>(smem + NI * 1024);  // [waves]
  if (lane == 0) all[wave] = got;
  __syncthreads();
  int every = 1;
#pragma unroll
  for (int q = 0; q < kApNT / 64; ++q) every &= all[q];
  if (!every) return false;
  float a[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const u32x4 yv = reinterpret_cast<const u32x4*>(smem)[64 * i + lane];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        a[c] = fmaf(bflo(w[c][i][e]), bflo(yv[e]), a[c]);
        a[c] = fmaf(bfhi(w[c][i][e]), bfhi(yv[e]), a[c]);
      }
  }
  const float y0 = round_bf(wave_sum(a[0])), y1 = round_bf(wave_sum(a[1]));
  if (lane == 0) st_out32(p.x + n0 + 2 * wave, pack2bf(bflo(x) + y0, bfhi(x) + y1));
  return true;
}

// The attention's workgroup of row m, head h and range split
template <int HS, bool RANGES>
__device__ __forceinline__ void ap_attend(const AttendProjParams& p, int h, int m, int split, int* count, bool spec, float* lds) {
  attention_body<HS, 4, kApNT, RANGES, 2, false, false, true>(p.q, p.kc, p.vc, reinterpret_cast<bf16_t*>(p.y), p.pos, 1, p.S, p.nh,
                                                              p.scale_log2, h, m, lds, p.nsplit, split, p.part, nullptr, 0.f, nullptr, 0, spec,
                                                              count);
}

// Every head whose words are not all there, as its own workgroups form it (and store it too, when they come to run: the same values at the same
// places). The workgroups start at different heads. All of y is there afterwards. (Its code costs the others: with requests ahead of the position and a loop
// over one range 7B int4 took 1,035 us a step for 1,021.)
template <int HS, bool RANGES>
__device__ __forceinline__ void ap_missing(const AttendProjParams& p, int nt, float* lds) {
  const int n = p.nh * p.M, splits = RANGES ? p.nsplit : 1;
  for (int i = 0; i < n; ++i) {
    const int at = (nt + i) % n, h = at % p.nh, m = at / p.nh;
    const uint32_t w = get_word(p.y, (m * p.C + h * HS) / 2 + (int)(threadIdx.x & (HS / 2 - 1)));
    if (__syncthreads_and(w != kNotYet)) continue;
    for (int s = 0; s < splits; ++s) {
      if (s) __syncthreads();  // (LDS)
      ap_attend<HS, RANGES>(p, h, m, s, nullptr, false, lds);
    }
    if constexpr (RANGES) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partials are out
      __syncthreads();
      if (threadIdx.x < HS) attention_merge<HS, true>(p.part, reinterpret_cast<bf16_t*>(p.y), nullptr, 0.f, h, m, p.nh, p.nsplit);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // y is out
  __syncthreads();
}

// NI: codes: rounds of 8 chunks of 128 that cover C; bf16: steps of 512. MR: most rows.
template <int HS, int WF, int MR, bool RANGES, int NI>
__global__ __launch_bounds__(kApNT) void attend_proj_kernel(AttendProjParams p) {
  constexpr int NW = kApNT / 64, kProj = WF == AP_BF16 ? NI * 1024 + NW * 4 : hand_codes_lds<NW, MR, NI>();
  __shared__ __align__(16) unsigned char smem[std::max(attention_lds_floats<HS, kApNT>() * 4, kProj)];
  if ((int)blockIdx.x < p.heads) {
    const int h = blockIdx.x % p.nh, rest = blockIdx.x / p.nh, m = MR > 1 ? rest % p.M : 0, split = MR > 1 ? rest / p.M : rest;
    ap_attend<HS, RANGES>(p, h, m, split, p.count, p.heads <= 64, reinterpret_cast<float*>(smem));
    return;
  }
  const int nt = blockIdx.x - p.heads;
  // the codes' few bytes wait a microsecond behind the attention's first keys and values (int4, one row, 30 and 70
  // keys: without 6.3 and 7.4 us, with 5.9 and 6.9; bf16's, which take longer than a short attention, do not: 9.6, with 9.9)
  if constexpr (WF != AP_BF16) __builtin_amdgcn_s_sleep(32);
  if ((int)threadIdx.x < 8 * p.M)
    st_out32(p.clear + (size_t)(threadIdx.x >> 3) * (p.C >> 1) + 8 * nt + (threadIdx.x & 7), kNotYet);
  auto product = [&]() __attribute__((always_inline)) {
    if constexpr (WF == AP_BF16) return ap_bf16_row<NI>(p, nt, smem);
    else return hand_codes<WF, NW, MR, NI>(HandCodes{p.y, p.W, p.sz, p.x, p.nstat, p.M, p.C, p.C, p.waits}, nt, smem);
  };
  if (!product()) {  // (a loop around both would hold more registers than either)
    ap_missing<HS, RANGES>(p, nt, reinterpret_cast<float*>(smem));
    product();  // nothing of y is missing
  }
}

template <int WF, int MR, bool RANGES, int NI>
static int attend_proj_go(const AttendProjParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attend_proj_kernel<128, WF, MR, RANGES, NI>), dim3(p.heads + p.C / 16), dim3(kApNT), 0, s, p);
  LLJ_CHECK_LAUNCH();
  return 0;
}
template <int WF, int MR>
static int attend_proj_c(const AttendProjParams& p, hipStream_t s) {
  constexpr int U = WF == AP_BF16 ? 512 : 1024;
#define LLJ_AP(C_) return p.nsplit > 1 ? attend_proj_go<WF, MR, true, C_ / U>(p, s) : attend_proj_go<WF, MR, false, C_ / U>(p, s)
  if (p.C == 2048) LLJ_AP(2048);
  if (p.C == 4096) LLJ_AP(4096);
  if (p.C == 5120) LLJ_AP(5120);
#undef LLJ_AP
  return LLJ_EINVAL;
}
template <int WF>
static int attend_proj_m(const AttendProjParams& p, hipStream_t s) {
  return p.M == 1 ? attend_proj_c<WF, 1>(p, s) : attend_proj_c<WF, 2>(p, s);
}

}  // namespace llj

using namespace llj;

extern "C" {

int llj_attention_resid_ok(int wfmt, int M, int nh, int hs) {
  const int C = nh * hs;
  return (wfmt == AP_W4 || wfmt == AP_W8 || (wfmt == AP_BF16 && M == 1)) && M >= 1 && M <= 2 && hs == 128 && (C == 2048 || C == 4096 || C == 5120);
}

int llj_attention_resid_waits(int wfmt, const void* q, const void* kcache, const void* vcache, void* y, void* y_next, const int* pos, int M, int nh,
                              int hs, int S, int nsplit, void* part, int* count, const void* W, const void* sz, void* x, float* nstat_out, int waits,
                              void* stream) {
  LLJ_REQUIRE(llj_attention_resid_ok(wfmt, M, nh, hs) && q && kcache && vcache && y && y_next && y != y_next && pos && S >= 1 && W && x &&
              (wfmt == AP_BF16 || sz) && nsplit >= 1 && nsplit <= 64 && (nsplit == 1 || (part && count)) && (!nstat_out || M > 1) &&
              (((uintptr_t)W | (uintptr_t)y | (uintptr_t)y_next) & 15) == 0 && ((uintptr_t)x & 3) == 0);
  AttendProjParams p{};
  p.q = (const bf16_t*)q; p.kc = (const bf16_t*)kcache; p.vc = (const bf16_t*)vcache; p.y = (uint32_t*)y; p.clear = (uint32_t*)y_next;
  p.pos = pos; p.S = S; p.nh = nh; p.scale_log2 = 1.4426950408889634f / sqrtf((float)hs); p.nsplit = nsplit; p.part = (float*)part;
  p.count = count; p.W = W; p.sz = (const float2*)sz; p.x = (bf16_t*)x; p.nstat = nstat_out; p.C = nh * hs; p.M = M; p.heads = nh * M * nsplit;
  p.waits = waits > 0 ? waits : kApWaits;
  hipStream_t s = (hipStream_t)stream;
  if (wfmt == AP_BF16) return attend_proj_c<AP_BF16, 1>(p, s);
  return wfmt == AP_W8 ? attend_proj_m<AP_W8>(p, s) : attend_proj_m<AP_W4>(p, s);
}

int llj_attention_resid(int wfmt, const void* q, const void* kcache, const void* vcache, void* y, void* y_next, const int* pos, int M, int nh,
                        int hs, int S, int nsplit, void* part, int* count, const void* W, const void* sz, void* x, float* nstat_out, void* stream) {
  return llj_attention_resid_waits(wfmt, q, kcache, vcache, y, y_next, pos, M, nh, hs, S, nsplit, part, count, W, sz, x, nstat_out, 0, stream);
}

}  // extern "C"
