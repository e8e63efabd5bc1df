// One activation row times a bf16 weight (N, K): the decode step of a single sequence.
//
// Bound: the weights' bytes. A workgroup owns a range of output columns; each of its NW waves keeps its own slice of the row (SL
// pieces of 512 values, 8 per lane) in registers and streams that slice of column after column -- 1 KiB of consecutive
// bytes per load, two rounds of loads in flight -- into fp32 multiply-adds. The lanes' sums meet over 16 lanes (DPP), the rest
// through LDS once per workgroup, where the epilogue also runs, a thread per column with its operands loaded ahead.
//
// Loads come back in order, and one behind a branch is waited for with all that precede it. So no load here is behind a branch
// (a place past C or a column past the range is a valid one instead, left out of the sums), the row and the epilogue's operands
// are requested before the weights, and the loop's last rounds are written out. A range of one round has a kernel of its own size,
// since loads of columns that are not there cost as much in the caches as others. In a graph, us (TB/s), loads in branches
// -> this:
//   640 -> 1920, norm     4.9 -> 3.8           1792 -> 640            4.5 -> 3.6           640 -> 35008, norm   13.7 -> 10.6 (4.2)
//   2048 -> 6144, norm    8.4 -> 6.6 (3.8)     2048 -> 2048           4.8 -> 4.1           2048 -> 2 x 5632    11.9 -> 10.4 (4.4)
//   4096 -> 12288, norm  20.8 -> 20.0 (5.0)    4096 -> 4096           9.0 -> 8.1 (4.1)     4096 -> 2 x 11008   36.0 -> 34.3 (5.3)
//   11008 -> 4096        19.0 -> 18.6 (4.8)    4096 -> 32000, norm   50.3 -> 48.9 (5.4)    13824 -> 5120       28.4 -> 27.9 (5.1)
// Rounds of 8 columns up to 2048 values: 11.5, 8.4, 11.1 for 10.6, 6.6, 10.4; of 2: 11.8, 6.8, 10.4. The MFMA forms (gemv_impl.h,
// post_gemv.hip), made for several rows, read 16 columns x 64 bytes per load: 21.7 for 11008 -> 4096, 7.0 for 2048 -> 2048.
// (a wave per column, each with the whole row, measured the same without a prologue, but repeats the norm in ten times the
// workgroups.) The grid is about 2048 waves, 8 per CU with 16 KiB in flight each; 256 or 1024 workgroups of the same waves
// lose 1-4 %.
//
// Prologues (the weights' first loads are in flight meanwhile):
//   plain    the row from memory, bf16;
//   norm     RMSNorm with the reference's bf16 rounding points (model.py:281-283);
//   sums     that of the row plus the sum of up to 16 fp32 rows (a product's shares by heads, ops.hip), each rounded to bf16; the row so
//            formed is written once to x';
//   streams  the residual streams after a sublayer, the mixed row and its layer norm (streams.hip), the new streams written
//            once to x'.
#pragma once
#include "common.h"
#include "elem.h"

namespace llj {

enum { RD_PLAIN = 0, RD_NORM = 1, RD_STREAMS = 2, RD_SUMS = 3 /* .. + 16: up to PRO - RD_SUMS rows */ };
// RD_STORE: + bias (fp32 or NULL). RD_RESID: out += . RD_QKV: RoPE, q to out, k / v to the caches. RD_SWIGLU: silu(. W) * (. W2).
// RD_RELU2: max(., 0)^2. RD_GLU: the clamped gated unit of interleaved columns (elem.h), biased.
enum { RD_STORE = 0, RD_RESID = 1, RD_QKV = 2, RD_SWIGLU = 3, RD_RELU2 = 4, RD_GLU = 5 };

struct RowDotParams {
  const bf16_t* A;  // plain, norm: the row
  const bf16_t* w;  // norm, streams: norm weight
  float eps;
  int K, N;         // row stride of the weights; output columns (RD_SWIGLU: both weights' rows, 2 H)
  int C;            // values of the row (<= K, the weights past it are not read)
  const bf16_t* W;
  const bf16_t* W2;
  bf16_t* out;
  const float* bias;
  float limit, alpha;
  const bf16_t* t;  // streams: the sublayer's output; residual in / out
  const float* x;
  float* xo;
  const float* so;  // streams: output weights (S), mix (S, S), input weights (S) or NULL; x, xo: S rows of stride ldx
  const float* sm;
  const float* si;
  int S, ldx;
  const float* parts;  // sums: S rows of C
  bf16_t* ao;          // x'
  bf16_t* kcache;  // RD_QKV
  bf16_t* vcache;
  const float* rope;
  const int* pos;
  int n_head, hs, ring, T, m;  // ring: cache slots; m: row of q (sequence m / T, position pos[m % T])
};

constexpr int kRdStreams = 4;
constexpr int kRdSums = 16;
constexpr int kRdMaxC = 16384;

// ONE: columns of the largest range where a single round of loads holds them, or 0.
template <int NW, int SL, int PRO, int EPI, int ONE>
__global__ __launch_bounds__(NW * 64) void rowdot_kernel(RowDotParams p) {
  extern __shared__ __align__(16) float rd_part[];  // [column][NW * 4]
  __shared__ float red[2][NW];
  constexpr int CB = ONE ? ONE : SL <= 2 ? 4 : 2;  // columns per round of loads
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int units = p.N >> 1;
  const int c0 = 2 * (int)((long)blockIdx.x * units / gridDim.x), c1 = 2 * (int)((long)(blockIdx.x + 1) * units / gridDim.x);
  const int k0 = wave * (SL * 512) + lane * 8;  // slice s: k0 + 512 s
  int kv[SL];  // (past C: a valid place, whose values are left out of the sums)
#pragma unroll
  for (int s = 0; s < SL; ++s) kv[s] = k0 + 512 * s < p.C ? k0 + 512 * s : 0;
  // A wave whose slices are all past the row (8 waves of 1,024 values; C = 5,120 has three): its loads, though unused, would all be
  // issued at once, ahead of the others'. Plain and streams: no loop for it. Norm: no loads; the branch in front of every wave's also
  // holds the range of an output head or a SwiGLU back to what it took before the loads left their branches, which at 5,120 to
  // 5,632 and 8,192 is less. us, loads of all waves / no loop / no loads: 5120 -> 32000 58.7 / 55.8 / 55.8, -> 35008 62.1 / 59.6 / 57.5,
  // -> 2 x 13824 50.5 / 48.4 / 46.5; 5632 -> 35008 67.4 / 66.5 / 63.2; 8192 -> 2 x 22016 117.7 / 117.1 / 114.7; plain 4224 -> 4224
  // 9.4 / 8.8 / 10.0; streams 4224 -> 28000 47.7 / 46.4 / 48.1. With 4 waves, or slices of 512, the test costs 1 to 5 %.
  const bool idle = NW == 8 && SL == 2 && wave * (SL * 512) >= p.C;
  u32x4 wv[2][CB][SL];
  auto fetch = [&](int b, int c) {  // (columns past c1: the last pair again)
    if (idle && PRO == RD_NORM) return;
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      const int n = min(c + (i & ~1), c1 - 2) + (i & 1);
      const bf16_t* r = EPI == RD_SWIGLU ? ((i & 1) ? p.W2 : p.W) + (size_t)(n >> 1) * p.K : p.W + (size_t)n * p.K;
#pragma unroll
      for (int s = 0; s < SL; ++s) wv[b][i][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(r + kv[s]));
    }
  };

  // ---- the epilogue's operands of column c0 + tid: requested with the row, so that no memory trip follows the last barrier
  struct Operand {
    float v;    // RD_RESID: the residual; RD_STORE, RD_GLU: the bias
    float2 cs;  // RD_QKV: the rotation (cos, sin)
    size_t at;  // RD_QKV: place in q / k / v
    int region, odd;
  };
  auto operand = [&](int j) {
    const int n = c0 + j < c1 ? c0 + j : c0;
    Operand o{};
    if constexpr (EPI == RD_RESID) o.v = bf2f(p.out[n]);
    if constexpr (EPI == RD_STORE || EPI == RD_GLU) {
      const float v = (p.bias ? p.bias : reinterpret_cast<const float*>(p.W))[p.bias ? n : 0];
      o.v = p.bias ? v : 0.f;
    }
    if constexpr (EPI == RD_QKV) {  // model.py:204-228: RoPE in fp32 on the bf16 output, k / v to ring slot p % ring
      const int Cd = p.n_head * p.hs, nc = n % Cd, h = nc / p.hs, dd = nc - h * p.hs;
      const int b = p.T == 1 ? p.m : p.m / p.T, ps = p.pos[p.m - b * p.T];
      o.region = n / Cd;
      o.odd = dd & 1;
      o.cs = *reinterpret_cast<const float2*>(p.rope + ((size_t)ps * (p.hs >> 1) + (dd >> 1)) * 2);
      o.at = o.region == 0 ? (size_t)p.m * Cd + nc : (((size_t)b * p.n_head + h) * p.ring + ps % p.ring) * p.hs + dd;
    }
    return o;
  };

  // ---- prologue: this lane's values of the row, fp32 holding bf16 values
  float xf[SL][8];
  Operand first;
  auto block_sum = [&](float v, int which) {
    v = wave_sum(v);
    if (lane == 0) red[which][wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += red[which][i];
    return t;
  };
  if constexpr (PRO != RD_STREAMS) {
    u32x4 xv[SL], gv[SL];
    constexpr int NS = PRO > RD_SUMS ? PRO - RD_SUMS : 1;
    f32x4 pv[SL][NS][2];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      xv[s] = *reinterpret_cast<const u32x4*>(p.A + kv[s]);
      if constexpr (PRO != RD_PLAIN) gv[s] = *reinterpret_cast<const u32x4*>(p.w + kv[s]);
      if constexpr (PRO > RD_SUMS) {
#pragma unroll
        for (int q = 0; q < NS; ++q) {  // (past the last: a copy, not added)
          const f32x4* from = reinterpret_cast<const f32x4*>(p.parts + (size_t)(q < p.S ? q : 0) * p.C + kv[s]);
          pv[s][q][0] = from[0];
          pv[s][q][1] = from[1];
        }
      }
    }
    first = operand(tid);
    fetch(0, c0);
    if constexpr (!ONE) fetch(1, c0 + CB);
#pragma unroll
    for (int s = 0; s < SL; ++s)
      if (k0 + 512 * s >= p.C) xv[s] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < SL; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[s][e] = (e & 1) ? bfhi(xv[s][e >> 1]) : bflo(xv[s][e >> 1]);
    if constexpr (PRO > RD_SUMS) {
#pragma unroll
      for (int s = 0; s < SL; ++s) {
        const int k = k0 + 512 * s;
        float y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < NS; ++q)
          if (q < p.S) {  // (uniform)
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] += pv[s][q][e >> 2][e & 3];
          }
#pragma unroll
        for (int e = 0; e < 8; ++e) xf[s][e] = k < p.C ? round_bf(xf[s][e] + round_bf(y[e])) : 0.f;  // model.py:172
        if (k < p.C && (unsigned)(k >> 3) % gridDim.x == blockIdx.x) {
#pragma unroll
          for (int e = 0; e < 4; ++e) st_out32(p.ao + k + 2 * e, pack2bf(xf[s][2 * e], xf[s][2 * e + 1]));
        }
      }
    }
    if constexpr (PRO != RD_PLAIN) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < SL; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += round_bf(xf[s][e] * xf[s][e]);
      const float r = round_bf(rsqrtf(round_bf(round_bf(block_sum(ss, 0) / (float)p.C) + p.eps)));
#pragma unroll
      for (int s = 0; s < SL; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          xf[s][e] = round_bf(((e & 1) ? bfhi(gv[s][e >> 1]) : bflo(gv[s][e >> 1])) * round_bf(xf[s][e] * r));
    }
  } else {
    u32x4 tv[SL], gv[SL];
    float sv[SL][kRdStreams][8];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      tv[s] = *reinterpret_cast<const u32x4*>(p.t + kv[s]);
      gv[s] = *reinterpret_cast<const u32x4*>(p.w + kv[s]);
#pragma unroll
      for (int q = 0; q < kRdStreams; ++q) ld8(p.x + (size_t)(q < p.S ? q : 0) * p.ldx + kv[s], sv[s][q]);  // (past S: a copy)
    }
    float ot[kRdStreams], mx[kRdStreams][kRdStreams], in[kRdStreams];
#pragma unroll
    for (int t = 0; t < kRdStreams; ++t) {
      const int tt = t < p.S ? t : 0;
      ot[t] = p.so[tt];
      in[t] = (p.si ? p.si : p.so)[tt];
#pragma unroll
      for (int q = 0; q < kRdStreams; ++q) mx[t][q] = p.sm[(q < p.S ? q : 0) * p.S + tt];
    }
    first = operand(tid);
    fetch(0, c0);
    if constexpr (!ONE) fetch(1, c0 + CB);
    float sum = 0.f;
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const int k = k0 + 512 * s;
      const bool mine = k < p.C && (unsigned)(k >> 3) % gridDim.x == blockIdx.x;
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[s][e] = 0.f;
#pragma unroll
      for (int t = 0; t < kRdStreams; ++t) {
        if (t < p.S) {  // (uniform)
          float n[8];
          const float it = p.si ? in[t] : 1.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) n[e] = ot[t] * ((e & 1) ? bfhi(tv[s][e >> 1]) : bflo(tv[s][e >> 1]));
#pragma unroll
          for (int q = 0; q < kRdStreams; ++q) {
            const float a = q < p.S ? mx[t][q] : 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) n[e] += a * sv[s][q][e];
          }
          if (mine) st8(p.xo + (size_t)t * p.ldx + k, n);
#pragma unroll
          for (int e = 0; e < 8; ++e) xf[s][e] += it * n[e];
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += k < p.C ? xf[s][e] : 0.f;
    }
    const float mean = block_sum(sum, 0) / (float)p.C;
    sum = 0.f;
#pragma unroll
    for (int s = 0; s < SL; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xf[s][e] -= mean;
        sum += k0 + 512 * s < p.C ? xf[s][e] * xf[s][e] : 0.f;
      }
    const float r = 1.f / sqrtf(block_sum(sum, 1) / (float)p.C + p.eps);
#pragma unroll
    for (int s = 0; s < SL; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        xf[s][e] = k0 + 512 * s < p.C ? round_bf(xf[s][e] * r * ((e & 1) ? bfhi(gv[s][e >> 1]) : bflo(gv[s][e >> 1]))) : 0.f;
  }

  // ---- the stream
  auto columns = [&](int b, int c) {
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      float a = 0.f;
#pragma unroll
      for (int s = 0; s < SL; ++s) {
        if (k0 + 512 * s >= p.C) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a = fmaf(bflo(wv[b][i][s][e]), xf[s][2 * e], a);
          a = fmaf(bfhi(wv[b][i][s][e]), xf[s][2 * e + 1], a);
        }
      }
      a = row16_sum(a);
      if ((lane & 15) == 0 && c + i < c1) rd_part[(c + i - c0) * (NW * 4) + wave * 4 + (lane >> 4)] = a;
    }
  };
  if constexpr (ONE) {
    columns(0, c0);
  } else if (idle && PRO != RD_NORM) {
    for (int i = lane; i < (c1 - c0) * 4; i += 64) rd_part[(i >> 2) * (NW * 4) + wave * 4 + (i & 3)] = 0.f;
  } else {
    int c = c0;
    for (; c + 3 * CB < c1; c += 2 * CB) {
      columns(0, c);
      fetch(0, c + 2 * CB);
      columns(1, c + CB);
      fetch(1, c + 3 * CB);
    }
    columns(0, c);
    if (c + 2 * CB < c1) {
      fetch(0, c + 2 * CB);
      columns(1, c + CB);
      columns(0, c + 2 * CB);
    } else if (c + CB < c1) {
      columns(1, c + CB);
    }
  }
  __syncthreads();

  // ---- epilogue: thread per column, neighbouring columns in neighbouring lanes (c0 is even)
  const bool pairs = (((uintptr_t)p.out | (uintptr_t)p.kcache | (uintptr_t)p.vcache) & 3) == 0;
  for (int j0 = 0; j0 < c1 - c0; j0 += NW * 64) {
    const int j = j0 + tid, n = c0 + j;
    const bool live = n < c1;
    const f32x4* q = reinterpret_cast<const f32x4*>(rd_part + (live ? j : 0) * (NW * 4));
    float y = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) y += (q[w][0] + q[w][1]) + (q[w][2] + q[w][3]);
    const Operand op = j0 ? operand(j) : first;
    if constexpr (EPI == RD_STORE || EPI == RD_GLU) y += op.v;
    if constexpr (EPI == RD_SWIGLU) {
      const float a = round_bf(y), b = lane_xor1(a);
      if (live && !(n & 1)) p.out[n >> 1] = f2bf(round_bf(a / (1.f + __expf(-a))) * b);  // model.py:258 in bf16
    } else if constexpr (EPI == RD_GLU) {
      const float u = lane_xor1(y);
      if (live && !(n & 1)) p.out[n >> 1] = f2bf(clamped_glu(y, u, p.limit, p.alpha));
    } else {
      float o = y;
      if constexpr (EPI == RD_RELU2) o = fmaxf(y, 0.f) * fmaxf(y, 0.f);
      if constexpr (EPI == RD_RESID) o = round_bf(op.v + round_bf(y));  // model.py:172-173
      bf16_t* dst = p.out + n;
      if constexpr (EPI == RD_QKV) {
        o = round_bf(y);
        const float partner = lane_xor1(o);
        if (op.region < 2) o = op.odd ? o * op.cs.x + partner * op.cs.y : o * op.cs.x - partner * op.cs.y;
        dst = (op.region == 0 ? p.out : op.region == 1 ? p.kcache : p.vcache) + op.at;
      }
      const uint32_t ob = (uint32_t)f2bf(o), pr = lane_xor1(ob);
      if (pairs) {  // columns (n, n + 1) leave as one 4-byte store
        if (live && !(n & 1)) st_out32(dst, ob | (pr << 16));
      } else if (live) {
        *dst = (bf16_t)ob;
      }
    }
  }
}

template <int NW, int SL, int PRO, int EPI>
static int rowdot_go(const RowDotParams& p, hipStream_t s) {
  const int units = p.N / 2;
  int grid = (PRO > RD_SUMS ? 512 : 2048) / NW;  // (every workgroup of a sums prologue reads all of its rows: a session's step of 10 layers of 640 with 2048 198 us, with 512 and 1024 185)
  grid = grid < units ? grid : units;
  // [column][NW * 4] sums of the largest range in 48 KiB (very wide outputs: more workgroups)
  const long most = 48 * 1024 / (NW * 16) - 2;
  if ((long)p.N > most * grid) grid = (int)((p.N + most - 1) / most);
  const size_t lds = (size_t)2 * ((units + grid - 1) / grid) * NW * 16;
  const int range = 2 * ((units + grid - 1) / grid);
#define LLJ_RD(ONE) hipLaunchKernelGGL((rowdot_kernel<NW, SL, PRO, EPI, ONE>), dim3(grid), dim3(NW * 64), lds, s, p)
  if (range <= 2) LLJ_RD(2);
  else if (SL <= 2 && range <= 4) LLJ_RD(SL <= 2 ? 4 : 0);
  else LLJ_RD(0);
#undef LLJ_RD
  LLJ_CHECK_LAUNCH();
  return 0;
}

// The row's slices: as few waves as keep a wave's slice at 1024 values, 8 waves at most (streams, whose prologue reads 20 bytes per
// value in every workgroup: 8 waves and half the workgroups from 2049 on). C <= kRdMaxC (streams: 8192).
template <int PRO, int EPI>
static int rowdot_launch(const RowDotParams& p, hipStream_t s) {
  if (p.C <= 1024) return rowdot_go<2, 1, PRO, EPI>(p, s);
  if (p.C <= 2048) return rowdot_go<4, 1, PRO, EPI>(p, s);
  if (p.C <= 4096) return PRO == RD_STREAMS ? rowdot_go<8, 1, PRO, EPI>(p, s) : rowdot_go<4, 2, PRO, EPI>(p, s);
  if (p.C <= 8192) return rowdot_go<8, 2, PRO, EPI>(p, s);
  if constexpr (PRO <= RD_NORM) {
    if (p.C <= 12288) return rowdot_go<8, 3, PRO, EPI>(p, s);
    if (p.C <= kRdMaxC) return rowdot_go<8, 4, PRO, EPI>(p, s);
  }
  return LLJ_EINVAL;
}

}  // namespace llj
