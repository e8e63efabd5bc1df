// One decode row through all layers of a small bf16 model in one launch (reference model.py:162-175 per layer).
//
// Such a step is all latency: launches of 3 to 5 us for products of 1 to 7 MB. Here a layer's five stages are workgroups of one grid, in the order of
// the data: c_attn with RoPE and the K / V write, the attention (a head each), attn.c_proj, c_fc1 / c_fc2, mlp.c_proj, then the next layer's. Each
// brings its weights (the attention its first keys and values) to registers and waits for its row, which is its own signal (handover.h);
// as workgroups end, those of later layers start, so that the weights arrive layers ahead. What bounds it is a stage's trip through the caches, 2.5 us
// from row to row with the dot product and the lanes' sums; a wave owns four neighbouring columns, whole.
// Requests for the same lines delay one another and the stores to them: a row that many wait for is written in kSmCopies places (49M, two
// columns a wave in the feed-forward, us a step: 1 / 2 / 4 / 8 / 16 places 182 / 165 / 158 / 155 / 162), fewer and larger workgroups' waves ask for it
// (144 with four columns), and a workgroup first waits on one word of the row before its own.
// us a step in a graph, with the embedding, the head and the next token, launches of their own -> this: 19M 111 -> 85, 220 tokens in the cache 118 -> 102;
// 49M 182 -> 144, at 450 tokens 223 -> 194; 125M (heads of 78) at 100 tokens 245 -> 207, at 300 267 -> 256.
#include <algorithm>

#include "attention.h"
#include "common.h"
#include "handover.h"
#include "lit_llama_amd.h"

namespace llj {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
constexpr int kSmLayers = 16, kSmNT = 256, kSmNW = 4;
constexpr int kSmCopies = 8;  // of a row that many workgroups wait for
constexpr int kSmUp = 4, kSmDown = 4;  // columns a wave of the feed-forward's products (of two each 155 us a step of 49M and 89 of 19M, for 144 and 86)
constexpr int kSmU = 8;                // keys to 16 lanes and pass: 128 keys a pass

struct SmallLayer {
  const bf16_t *n1, *wa, *wp, *n2, *w1, *w2, *wd;
  bf16_t *kc, *vc;
};
struct SmallParams {
  SmallLayer layer[kSmLayers];
  bf16_t* x;       // the row, in and out
  uint32_t* hand;  // per layer the words of q, k, v; y; x after the attention; h; x after the layer
  const float* rope;
  const int* pos;
  int L, C, H, nh, hs, S;
  float eps, scale_log2;
  int ta, tp, tu, td, per;  // workgroups of the stages (the attention: nh), of a layer
};

// the words of a row that this thread takes (thread + 256 i). plain: from an earlier launch
template <int NWD>
__device__ __forceinline__ void sm_wait(const uint32_t* row, int words, bool plain, uint32_t (&v)[NWD]) {
  const int tid = threadIdx.x;
  for (int t = 0; t < kWaits; ++t) {
    bool there = true;
#pragma unroll
    for (int i = 0; i < NWD; ++i) {
      v[i] = get_word(row, min(tid + kSmNT * i, words - 1));
      there = there && v[i] != kNotYet;
    }
    if (plain || __all(there)) break;
  }
}
// until a word of `row` (or NULL) is there
__device__ __forceinline__ void sm_early(const uint32_t* row, int words, int b) {
  if (!row) return;  // uniform
  if (threadIdx.x < 64) {
    const uint32_t* at = row + (unsigned)(b * 7) % (unsigned)words;
    for (int t = 0; t < kWaits; ++t) {
      if (get_word(at, 0) != kNotYet) break;
      __builtin_amdgcn_s_sleep(16);
    }
  }
  __syncthreads();
}

// NC weight rows (columns n .. of K values), pieces of 4 values: 256 p + 4 lane
template <int NC, int P>
struct SmDot {
  u32x2 w[NC][P];
  __device__ __forceinline__ void load(const bf16_t* W, int n, int K) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = 256 * p + 4 * (threadIdx.x & 63);
        w[c][p] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(W + (size_t)(n + c) * K + (k < K ? k : 0)));
      }
  }
  // xf: this lane's values of the row (zeros past K)
  __device__ __forceinline__ void sums(const float (&xf)[P][4], int K, float (&s)[NC]) const {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float a = 0.f;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const bool in = 256 * p + 4 * (int)(threadIdx.x & 63) < K;
        const uint32_t lo = in ? w[c][p][0] : 0u, hi = in ? w[c][p][1] : 0u;
        a = fmaf(bflo(lo), xf[p][0], a);
        a = fmaf(bfhi(lo), xf[p][1], a);
        a = fmaf(bflo(hi), xf[p][2], a);
        a = fmaf(bfhi(hi), xf[p][3], a);
      }
      s[c] = wave_sum(a);  // (column by column: the four together, with three lane swaps for eight, take 155 us a step for 144)
    }
  }
};

// the row from LDS as this lane's pieces
template <int P>
__device__ __forceinline__ void sm_pieces(const uint32_t* lds, int K, float (&xf)[P][4]) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int k = 256 * p + 4 * (threadIdx.x & 63);
    const u32x2 v = *reinterpret_cast<const u32x2*>(lds + (k < K ? k >> 1 : 0));
    const bool in = k < K;
    xf[p][0] = in ? bflo(v[0]) : 0.f;
    xf[p][1] = in ? bfhi(v[0]) : 0.f;
    xf[p][2] = in ? bflo(v[1]) : 0.f;
    xf[p][3] = in ? bfhi(v[1]) : 0.f;
  }
}

// waits for a row, leaves this lane's pieces of it, with NORM of its RMSNorm (the reference's bf16 rounding points, model.py:281-283); g: the scale's
// pieces
template <bool NORM, int NWD, int P>
__device__ __forceinline__ void sm_row(const uint32_t* row, int K, bool plain, const u32x2 (&g)[NORM ? P : 1], float eps, uint32_t* lds, float* red,
                                       float (&xf)[P][4]) {
  const int tid = threadIdx.x, words = K >> 1;
  uint32_t v[NWD];
  sm_wait<NWD>(row, words, plain, v);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NWD; ++i) {
    if (tid + kSmNT * i < words) {
      lds[tid + kSmNT * i] = v[i];
      if (NORM) ss += round_bf(bflo(v[i]) * bflo(v[i])) + round_bf(bfhi(v[i]) * bfhi(v[i]));
    }
  }
  if constexpr (NORM) {
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
  }
  __syncthreads();
  sm_pieces<P>(lds, K, xf);
  if constexpr (NORM) {
    const float r = round_bf(rsqrtf(round_bf(round_bf((red[0] + red[1] + red[2] + red[3]) / (float)K) + eps)));
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gv = (e & 1) ? bfhi(g[p][e >> 1]) : bflo(g[p][e >> 1]);
        xf[p][e] = 256 * p + 4 * (tid & 63) < K ? round_bf(gv * round_bf(xf[p][e] * r)) : 0.f;
      }
  }
}

template <int P>
__device__ __forceinline__ void sm_scale(const bf16_t* w, int K, u32x2 (&g)[P]) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int k = 256 * p + 4 * (threadIdx.x & 63);
    g[p] = *reinterpret_cast<const u32x2*>(w + (k < K ? k : 0));
  }
}

// PK, PH: pieces of 256 values that cover C and H. WPL: pairs of a head's values to one of 16 lanes.
template <int PK, int PH, int WPL>
__global__ __launch_bounds__(kSmNT) void small_step_kernel(SmallParams p) {
  __shared__ __align__(16) uint32_t lds[PH * 128];
  __shared__ float red[2 * kSmNW + kSmNW * 32 * WPL];
  constexpr int WK = (PK * 128 + kSmNT - 1) / kSmNT, WH = (PH * 128 + kSmNT - 1) / kSmNT;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), b = blockIdx.x;
  const int l = b / p.per, C = p.C, H = p.H;
  int r = b - l * p.per;
  const SmallLayer& W = p.layer[l];
  const int stride = 3 * C + (H >> 1);  // words of a layer
  const size_t copy = (size_t)p.L * stride;
  uint32_t* const qkv = p.hand + (size_t)l * stride;  // (one copy: a head's workgroup alone waits for its q, k and v)
  uint32_t* const yw = qkv + 3 * (C >> 1) + (b % kSmCopies) * copy;
  const ptrdiff_t to = (ptrdiff_t)copy * -(b % kSmCopies);  // to the first copy
  uint32_t* const x1 = yw + (C >> 1);
  uint32_t* const hw = x1 + (C >> 1);
  uint32_t* const x2 = hw + (H >> 1);
  const bool first = l == 0;
  const uint32_t* const xin = first ? reinterpret_cast<const uint32_t*>(p.x) : x2 - stride;
  const int ps = p.pos[0];

  if (r < p.ta) {  // ---- c_attn: 4 columns a wave
    const int n = 4 * (r * kSmNW + wave), nn = n < 3 * C ? n : 0;
    SmDot<4, PK> d;
    u32x2 g[PK];
    d.load(W.wa, nn, C);
    sm_scale<PK>(W.n1, C, g);
    // lane & 1: a pair of columns
    const int nc = nn + 2 * (lane & 1), region = nc / C, c = nc - region * C, h = c / p.hs, dd = c - h * p.hs;
    const float2 cs = *reinterpret_cast<const float2*>(p.rope + ((size_t)ps * (p.hs >> 1) + (dd >> 1)) * 2);
    float xf[PK][4], s[4];
    sm_early(first ? nullptr : hw - stride, H >> 1, b);
    sm_row<true, WK, PK>(xin, C, first, g, p.eps, lds, red, xf);
    d.sums(xf, C, s);
    float v0 = round_bf((lane & 1) ? s[2] : s[0]), v1 = round_bf((lane & 1) ? s[3] : s[1]);
    if (region < 2) {
      const float a = v0 * cs.x - v1 * cs.y;
      v1 = v1 * cs.x + v0 * cs.y;
      v0 = a;
    }
    if (lane < 2 && n < 3 * C) {
      const uint32_t w = pack2bf(v0, v1);
      st_out32(qkv + (nc >> 1), hand_word(w));
      if (region > 0) {
        bf16_t* cache = region == 1 ? W.kc : W.vc;
        st_out32(cache + ((size_t)h * p.S + (ps < p.S ? ps : ps % p.S)) * p.hs + dd, w);
      }
    }
    return;
  }
  r -= p.ta;
  if (r < p.nh) {  // ---- the attention of head r: 16 lanes a key, lane: word pairs sub + 16 i
    const int sub = lane & 15, kg = tid >> 4, HW = p.hs >> 1, nvalid = ps < p.S ? ps + 1 : p.S, slot = ps < p.S ? ps : ps % p.S;
    const uint32_t* kc = reinterpret_cast<const uint32_t*>(W.kc) + (size_t)r * p.S * HW;
    const uint32_t* vc = reinterpret_cast<const uint32_t*>(W.vc) + (size_t)r * p.S * HW;
    uint32_t kw[kSmU][WPL], vw[kSmU][WPL];
    auto pass = [&](int j0) {
#pragma unroll
      for (int u = 0; u < kSmU; ++u) {
        const int j = j0 + 16 * u < nvalid ? j0 + 16 * u : 0;
#pragma unroll
        for (int i = 0; i < WPL; ++i) {
          const int at = j * HW + min(sub + 16 * i, HW - 1);
          kw[u][i] = kc[at];
          vw[u][i] = vc[at];
        }
      }
    };
    pass(kg);
    sm_early(first ? nullptr : x2 - stride, C >> 1, b);
    uint32_t nq[WPL], nk[WPL], nv[WPL];
    for (int t = 0; t < kWaits; ++t) {
      bool there = true;
#pragma unroll
      for (int i = 0; i < WPL; ++i) {
        const int at = r * HW + min(sub + 16 * i, HW - 1);
        nq[i] = get_word(qkv, at);
        nk[i] = get_word(qkv, (C >> 1) + at);
        nv[i] = get_word(qkv, C + at);
        there = there && nq[i] != kNotYet && nk[i] != kNotYet && nv[i] != kNotYet;
      }
      if (__all(there)) break;
    }
    float qf[2 * WPL], o[2 * WPL], mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
      const bool in = sub + 16 * i < HW;
      qf[2 * i] = in ? bflo(nq[i]) * p.scale_log2 : 0.f;
      qf[2 * i + 1] = in ? bfhi(nq[i]) * p.scale_log2 : 0.f;
      o[2 * i] = o[2 * i + 1] = 0.f;
    }
    for (int j0 = kg; j0 < nvalid; j0 += 16 * kSmU) {
      if (j0 != kg) pass(j0);
#pragma unroll
      for (int u = 0; u < kSmU; ++u) {
        const int j = j0 + 16 * u;
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < WPL; ++i) {
          kw[u][i] = j == slot ? nk[i] : kw[u][i];
          vw[u][i] = j == slot ? nv[i] : vw[u][i];
          if (sub + 16 * i < HW) s += qf[2 * i] * bflo(kw[u][i]) + qf[2 * i + 1] * bfhi(kw[u][i]);
        }
        s = row16_sum(s);
        if (j >= nvalid) continue;
        const float mn = fmaxf(mx, s), corr = exp2f(mx - mn), pj = exp2f(s - mn);
        sum = sum * corr + pj;
#pragma unroll
        for (int i = 0; i < WPL; ++i) {
          o[2 * i] = o[2 * i] * corr + pj * bflo(vw[u][i]);
          o[2 * i + 1] = o[2 * i + 1] * corr + pj * bfhi(vw[u][i]);
        }
        mx = mn;
      }
    }
    float mlo, mhi, llo, lhi, olo[2 * WPL], ohi[2 * WPL];
    auto merge = [&](auto wide) {
      constexpr bool WIDE = decltype(wide)::value;
      lane_halves<WIDE>(mx, mlo, mhi);
      lane_halves<WIDE>(sum, llo, lhi);
#pragma unroll
      for (int i = 0; i < 2 * WPL; ++i) lane_halves<WIDE>(o[i], olo[i], ohi[i]);
      softmax_merge<2 * WPL>(mx, sum, o, mlo, mhi, llo, lhi, olo, ohi);
    };
    merge(std::false_type{});
    merge(std::true_type{});
    float *sm = red, *sl = red + kSmNW, *so = red + 2 * kSmNW;  // [wave], [wave], [wave][32 WPL]
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < WPL; ++i)
        *reinterpret_cast<float2*>(so + wave * 32 * WPL + 2 * (sub + 16 * i)) = make_float2(o[2 * i], o[2 * i + 1]);
      if (lane == 0) {
        sm[wave] = mx;
        sl[wave] = sum;
      }
    }
    __syncthreads();
    if (tid < HW) {
      const float M = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
      float Ls = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int w = 0; w < kSmNW; ++w) {
        const float f = sm[w] == -INFINITY ? 0.f : exp2f(sm[w] - M);
        Ls += sl[w] * f;
        o0 += so[w * 32 * WPL + 2 * tid] * f;
        o1 += so[w * 32 * WPL + 2 * tid + 1] * f;
      }
      const uint32_t w = hand_word(pack2bf(o0 / Ls, o1 / Ls));
#pragma unroll
      for (int k = 0; k < kSmCopies; ++k) st_out32(yw + to + k * copy + r * HW + tid, w);
    }
    return;
  }
  r -= p.nh;
  if (r < p.tp) {  // ---- attn.c_proj + residual: 4 columns a wave
    const int n = 4 * (r * kSmNW + wave), nn = n < C ? n : 0;
    SmDot<4, PK> d;
    d.load(W.wp, nn, C);
    const u32x2 none[1] = {};
    float xf[PK][4], s[4];
    sm_early(qkv, 3 * (C >> 1), b);
    const int at = (nn >> 1) + (lane & 1);
    uint32_t xw = get_word(xin, at);
    sm_row<false, WK, PK>(yw, C, false, none, 0.f, lds, red, xf);
    d.sums(xf, C, s);
    for (int t = 0; t < kWaits && !first && !__all(xw != kNotYet); ++t) xw = get_word(xin, at);
    const float a = bflo(xw) + round_bf((lane & 1) ? s[2] : s[0]), c = bfhi(xw) + round_bf((lane & 1) ? s[3] : s[1]);
    if (lane < 2 * kSmCopies && n < C) st_out32(x1 + to + (lane >> 1) * copy + at, hand_word(pack2bf(a, c)));
    return;
  }
  r -= p.tp;
  if (r < p.tu) {  // ---- c_fc1, c_fc2, silu * mul: kSmUp columns a wave
    const int n = kSmUp * (r * kSmNW + wave), nn = n < H ? n : 0;
    SmDot<kSmUp, PK> d1, d2;
    u32x2 g[PK];
    d1.load(W.w1, nn, C);
    d2.load(W.w2, nn, C);
    sm_scale<PK>(W.n2, C, g);
    float xf[PK][4], s1[kSmUp], s2[kSmUp];
    sm_early(yw, C >> 1, b);
    sm_row<true, WK, PK>(x1, C, false, g, p.eps, lds, red, xf);
    d1.sums(xf, C, s1);
    d2.sums(xf, C, s2);
    const int pair = lane % (kSmUp / 2), to_copy = lane / (kSmUp / 2);
    float o[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {  // model.py:258 in bf16
      float u = s1[e], v = s2[e];
#pragma unroll
      for (int q = 1; q < kSmUp / 2; ++q) {
        u = pair == q ? s1[2 * q + e] : u;
        v = pair == q ? s2[2 * q + e] : v;
      }
      const float a = round_bf(u);
      o[e] = round_bf(a / (1.f + __expf(-a))) * round_bf(v);
    }
    if (to_copy < kSmCopies && n < H) st_out32(hw + to + to_copy * copy + (nn >> 1) + pair, hand_word(pack2bf(o[0], o[1])));
    return;
  }
  r -= p.tu;
  {  // ---- mlp.c_proj + residual: kSmDown columns a wave
    const int n = kSmDown * (r * kSmNW + wave), nn = n < C ? n : 0;
    SmDot<kSmDown, PH> d;
    d.load(W.wd, nn, H);
    const u32x2 none[1] = {};
    float xf[PH][4], s[kSmDown];
    sm_early(x1, C >> 1, b);
    const int pair = lane % (kSmDown / 2), to_copy = lane / (kSmDown / 2), at = (nn >> 1) + pair;
    uint32_t xw = get_word(x1, at);
    sm_row<false, WH, PH>(hw, H, false, none, 0.f, lds, red, xf);
    d.sums(xf, H, s);
    for (int t = 0; t < kWaits && !__all(xw != kNotYet); ++t) xw = get_word(x1, at);
    float u = s[0], v = s[1];
#pragma unroll
    for (int q = 1; q < kSmDown / 2; ++q) {
      u = pair == q ? s[2 * q] : u;
      v = pair == q ? s[2 * q + 1] : v;
    }
    const uint32_t w = pack2bf(bflo(xw) + round_bf(u), bfhi(xw) + round_bf(v));
    if (to_copy < kSmCopies && n < C) {
      if (l < p.L - 1) st_out32(x2 + to + to_copy * copy + at, hand_word(w));
      else if (to_copy == 0) st_out32(p.x + 2 * at, w);
    }
  }
}

// The step's first launch: the token's embedding, the position, and every word of the rows to come as not there yet.
__global__ __launch_bounds__(256) void small_begin_kernel(const int* __restrict__ idx, const uint32_t* __restrict__ wte, uint32_t* __restrict__ x, int words,
                                                          int* pos_inc, uint32_t* __restrict__ hand, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < words) x[i] = wte[(size_t)idx[0] * words + i];
  if (i == 0) *pos_inc += 1;
  for (int k = i; k < n; k += gridDim.x * 256) hand[k] = kNotYet;
}

template <int PK, int PH>
static int small_go(const SmallParams& p, hipStream_t s) {
  const dim3 grid(p.per * p.L), nt(kSmNT);
  if (p.hs <= 64) hipLaunchKernelGGL((small_step_kernel<PK, PH, 2>), grid, nt, 0, s, p);
  else if (p.hs <= 96) hipLaunchKernelGGL((small_step_kernel<PK, PH, 3>), grid, nt, 0, s, p);
  else hipLaunchKernelGGL((small_step_kernel<PK, PH, 4>), grid, nt, 0, s, p);
  LLJ_CHECK_LAUNCH();
  return 0;
}

}  // namespace llj

using namespace llj;

extern "C" {

// (up to 512 cache slots and from 512 values: what was measured, always for the better)
int llj_small_step_ok(int L, int C, int H, int nh, int S) {
  return L >= 1 && L <= kSmLayers && nh >= 1 && C % nh == 0 && (C / nh) % 2 == 0 && C / nh <= 128 && C / nh >= 32 && C % 4 == 0 && C >= 512 && C <= 1024 &&
         H % 4 == 0 && H >= 2 * C && H <= 2816 && S >= 1 && S <= 512;
}
size_t llj_small_step_words(int L, int C, int H) { return (size_t)kSmCopies * L * (3 * C + (H >> 1)); }

int llj_small_begin(const int* idx, const void* wte, void* x, int C, int* pos, void* hand, int words, void* stream) {
  LLJ_REQUIRE(idx && wte && x && C >= 2 && C % 2 == 0 && C <= 64 * 1024 && pos && hand && words >= 0 && (((uintptr_t)wte | (uintptr_t)x | (uintptr_t)hand) & 3) == 0);
  const int blocks = std::max((C / 2 + 255) / 256, std::min((words + 255) / 256, 128));
  hipLaunchKernelGGL(small_begin_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, idx, (const uint32_t*)wte, (uint32_t*)x, C / 2, pos, (uint32_t*)hand, words);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_small_step(const void* const* layers, int L, int C, int H, int nh, int S, float eps, const float* rope, const int* pos, void* x, void* hand,
                   void* stream) {
  LLJ_REQUIRE(llj_small_step_ok(L, C, H, nh, S) && layers && rope && pos && x && hand && ((uintptr_t)x & 3) == 0 && ((uintptr_t)hand & 3) == 0);
  SmallParams p{};
  for (int l = 0; l < L; ++l) {
    for (int i = 0; i < 9; ++i) LLJ_REQUIRE(layers[9 * l + i] && ((uintptr_t)layers[9 * l + i] & (i < 7 ? 7 : 3)) == 0);
    const void* const* t = layers + 9 * l;
    p.layer[l] = SmallLayer{(const bf16_t*)t[0], (const bf16_t*)t[1], (const bf16_t*)t[2], (const bf16_t*)t[3], (const bf16_t*)t[4],
                            (const bf16_t*)t[5], (const bf16_t*)t[6], (bf16_t*)t[7], (bf16_t*)t[8]};
  }
  p.x = (bf16_t*)x; p.hand = (uint32_t*)hand; p.rope = rope; p.pos = pos;
  p.L = L; p.C = C; p.H = H; p.nh = nh; p.hs = C / nh; p.S = S; p.eps = eps;
  p.scale_log2 = 1.4426950408889634f / sqrtf((float)p.hs);
  auto groups = [](int columns, int a_wave) { return (columns + a_wave * kSmNW - 1) / (a_wave * kSmNW); };
  p.ta = groups(3 * C, 4);
  p.tp = groups(C, 4);
  p.tu = groups(H, kSmUp);
  p.td = groups(C, kSmDown);
  p.per = p.ta + nh + p.tp + p.tu + p.td;
  hipStream_t s = (hipStream_t)stream;
  const int pk = (C + 255) / 256, ph = (H + 255) / 256;
  if (pk <= 2) return ph <= 6 ? small_go<2, 6>(p, s) : small_go<4, 11>(p, s);
  if (pk == 3) return ph <= 7 ? small_go<3, 7>(p, s) : ph == 8 ? small_go<3, 8>(p, s) : small_go<4, 11>(p, s);
  return ph <= 9 ? small_go<4, 9>(p, s) : small_go<4, 11>(p, s);
}

}  // extern "C"
