// A row handed from some workgroups of a launch to the others, whose product it enters: the row is its own signal.
//
// Every 4-byte word of the row holds kNotYet until its two values are there. The workgroups that wait bring their weights to registers
// first and then read the row, past the caches, until no word is kNotYet: one trip through the memory system between the last store and the
// product, where a launch of its own has its start, the trip and the weights' bytes. Words return to kNotYet in the launch before the one that uses
// them next.
//
// The workgroups waited for come first in the grid, but that does not mean that they have started: each XCD starts its share of a launch in that order,
// nothing orders the starts on different XCDs, and waiting workgroups keep their places, so that those of several launches can stand in the
// way of the ones that they wait for. Every wait is bounded, and a launch is right however its waits end: see there.
#pragma once
#include "common.h"

namespace llj {

constexpr uint32_t kNotYet = 0xFFFFFFFFu;  // two NaNs; as outputs they leave as two others
constexpr int kWaits = 1 << 20;  // polls, each a trip past the caches: a second or more

__device__ __forceinline__ uint32_t hand_word(uint32_t w) { return w == kNotYet ? 0x7FFF7FFFu : w; }
__device__ __forceinline__ uint32_t get_word(const uint32_t* y, int at) {
  return __hip_atomic_load(y + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

enum { HC_W4 = 0, HC_W8 = 3 };  // wfmt

// acc += a . one MFMA step of codes (gemv_impl.h: W4P, and W8P as two nibble planes)
template <int WF>
__device__ __forceinline__ void code_mfma(f32x4& acc, bf16x8 a, uint32_t lo, uint32_t hi, uint32_t msk, uint32_t mag, uint32_t mag_hi) {
  auto codes = [&](uint32_t c, uint32_t m) {
    return __builtin_bit_cast(bf16x8, make_uint4(and_or(c, msk, m), and_or(c >> 4, msk, m), and_or(c >> 8, msk, m), and_or(c >> 12, msk, m)));
  };
  acc = mfma_bf16(a, codes(lo, mag), acc);
  if constexpr (WF == HC_W8) acc = mfma_bf16(a, codes(hi, mag_hi), acc);
}

struct HandCodes {
  const uint32_t* y;  // the rows' words, K / 2 a row
  const void* W;      // (N, K) codes, W4P or W8P
  const float2* sz;   // (scale, 128 or 2176 + zero) per column
  bf16_t* x;          // residual (M, N), in place: x += y . W^T in bf16 (model.py:172-173)
  float* nstat;       // sums of squares of x', 16 columns a place (llj_linear_resid's nstat_out), or NULL
  int M, N, K;
  int waits;  // polls of a wait
};
template <int NW, int MR, int NI>
constexpr int hand_codes_lds() { return NW * (MR * (NI * 256 + 16 + 80) + 4); }

// Columns 16 nt .. + 15 for up to MR rows, by NW waves. Wave: chunks wave + NW i of 128 values, at most NI; lane: the codes of column
// lane % 16, 32 of a chunk's values. false (in every thread), with nothing written: a wait ran out.
template <int WF, int NW, int MR, int NI>
__device__ __forceinline__ bool hand_codes(const HandCodes& p, int nt, unsigned char* smem) {
  constexpr int V = WF == HC_W8 ? 2 : 1, RS = NI * 128 + 8;  // (rows on other banks)
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), KW = p.K >> 1;
  const int n0 = 16 * nt, KC = p.K >> 7, g = lane >> 4;
  u32x4 w[NI][V];
  const u32x4* src = reinterpret_cast<const u32x4*>(p.W) + (size_t)nt * KC * 64 * V + lane;
  const int om = min((tid >> 4) & (MR - 1), p.M - 1), on = n0 + (tid & 15);  // the output of a thread: row, column
  const float2 sz = p.sz[on];
  const float x = bf2f(p.x[(size_t)om * p.N + on]);
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int v = 0; v < V; ++v) w[i][v] = __builtin_nontemporal_load(src + (size_t)(min(wave + NW * i, KC - 1) * V + v) * 64);
  // this wave's own values of y: word `lane` of each of its chunks
  bf16_t* ys = reinterpret_cast<bf16_t*>(smem) + wave * MR * RS;
  uint32_t v[MR][NI];
  bool got = false;
  for (int t = 0; t < p.waits; ++t) {
    bool there = true;
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        v[m][i] = get_word(p.y, min(m, p.M - 1) * KW + 64 * min(wave + NW * i, KC - 1) + lane);
        there = there && v[m][i] != kNotYet;
      }
    got = __all(there);
    if (got) break;
    __builtin_amdgcn_s_sleep(1);
  }
  int* all = reinterpret_cast<int*>(smem + NW * MR * (RS * 2 + 80));  // [NW]
  if (lane == 0) all[wave] = got;
  float* red = reinterpret_cast<float*>(smem + NW * MR * RS * 2);  // [NW][MR][16 + 4]
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    float rs = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      reinterpret_cast<uint32_t*>(ys + m * RS)[64 * i + lane] = v[m][i];
      if (wave + NW * i < KC) rs += bflo(v[m][i]) + bfhi(v[m][i]);
    }
    rs = wave_sum(rs);
    if (lane == 0) red[(wave * MR + m) * 20 + 16] = rs;
  }
  uint32_t msk = 0x000F000Fu, mag = 0x43004300u, mag_hi = 0x45004500u;
  asm volatile("" : "+s"(msk));
  asm volatile("" : "+v"(mag), "+v"(mag_hi));
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (wave + NW * i >= KC) break;  // (uniform)
#pragma unroll
    for (int t = 0; t < 4; ++t)  // (the operand's rows past MR are those below again)
      code_mfma<WF>(acc, *reinterpret_cast<const bf16x8*>(ys + (lane & (MR - 1)) * RS + 128 * i + 32 * g + 8 * t), w[i][0][t], w[i][V - 1][t],
                    msk, mag, mag_hi);
  }
  if (lane < 16) {
#pragma unroll
    for (int m = 0; m < MR; ++m) red[(wave * MR + m) * 20 + lane] = acc[m];
  }
  __syncthreads();
  int every = 1;
#pragma unroll
  for (int q = 0; q < NW; ++q) every &= all[q];
  if (!every) return false;
  if (tid >= 64) return true;
  float y = 0.f, r = 0.f;
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    y += red[(q * MR + om) * 20 + (tid & 15)];
    r += red[(q * MR + om) * 20 + 16];
  }
  const bool live = (tid >> 4) < p.M;
  const float xn = round_bf(x + round_bf(sz.x * (y - sz.y * r)));
  const uint32_t o = (uint32_t)f2bf(xn), pr = lane_xor1(o);
  if (live && !(tid & 1)) st_out32(p.x + (size_t)om * p.N + on, o | (pr << 16));
  if (p.nstat) {  // uniform
    const float sq = row16_sum(round_bf(xn * xn));
    if (live && (tid & 15) == 0) st_out32(p.nstat + (size_t)nt * 16 + om, __float_as_uint(sq));
  }
  return true;
}

}  // namespace llj
