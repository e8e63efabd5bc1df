// One decode row through all layers of a small bf16 model in one launch (reference model.py:162-175 per layer).
//
// Such a step is all latency: launches of 3 to 5 us for products of 1 to 7 MB. Here a layer's five stages are workgroups of one grid, in the order of
// the data: c_attn with RoPE and the K / V write, the attention (a head each), attn.c_proj, c_fc1 / c_fc2, mlp.c_proj, then the next layer's. Each
// brings its weights (the attention its first keys and values) to registers and waits for its row, which is its own signal (handover.h);
// as workgroups end, those of later layers start, so that the weights arrive layers ahead. That order holds on each XCD, not between them: beside another
// launch whose workgroups wait, one's next workgroups can find their XCD full of the other's and both stand still. So a workgroup that has
// waited long writes nothing and ends, and a second launch does what the first left undone, with places in the order of the starts (small_again_kernel).
// What bounds it is a stage's trip through the caches, 2.5 us from row to row with the dot product and the lanes' sums; a wave owns four neighbouring columns, whole.
// Requests for the same lines delay one another and the stores to them: a row that many wait for is written in kSmCopies places (49M, two
// columns a wave in the feed-forward, us a step: 1 / 2 / 4 / 8 / 16 places 182 / 165 / 158 / 155 / 162), fewer and larger workgroups' waves ask for it
// (144 with four columns), and a workgroup first waits on one word of the row before its own.
// us a step in a graph, with the embedding, the head and the next token, launches of their own -> this: 19M 111 -> 88, 49M 182 -> 145, 125M (heads of 78) at
// 100 tokens 245 -> 207; before the second launch, which finds nothing to do in 1 to 3 us of them: 19M at 220 tokens 118 -> 102, 49M at 450 223 -> 194, 125M at 300 267 -> 256.
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

constexpr int kSmWaits = 1 << 11;  // polls of the first launch's waits: a few milliseconds
constexpr int kSmAgain = 128;      // workgroups of the second launch
constexpr int kSmLine = 32;        // words of a line

struct SmallLayer {
  const bf16_t *n1, *wa, *wp, *n2, *w1, *w2, *wd;
  bf16_t *kc, *vc;
};
struct SmallParams {
  SmallLayer layer[kSmLayers];
  bf16_t* x;           // the row, out
  const uint32_t* x0;  // the row, in
  uint32_t* hand;      // per layer the words of q, k, v; y; x after the attention; h; x after the layer
  uint32_t* undone;    // kNotYet while no wait of the first launch has run out
  uint32_t* taken;     // the second launch's places taken, less one
  const uint32_t* stop;  // the waits end when this is no longer kNotYet (undone; for the second launch a word that stays)
  int* failed;         // set if a wait of the second launch ran out
  int waits;           // polls of a wait
  const float* rope;
  const int* pos;
  int L, C, H, nh, hs, S;
  float eps, scale_log2;
  int ta, tp, tu, td, per;  // workgroups of the stages (the attention: nh), of a layer
};

// polls there() until it is true in every lane of the wave; false: it was not after p.waits polls, or the launch has given up
template <typename F>
__device__ __forceinline__ bool sm_until(const SmallParams& p, F there) {
  for (int t = 1; t <= p.waits; ++t) {
    if (__all(there())) return true;
    if (t % 64 == 0 && uniform(get_word(p.stop, 0)) != (int)kNotYet) break;
  }
  return false;
}
// the words of a row that this thread takes (thread + 256 i). plain: from an earlier launch
template <int NWD>
__device__ __forceinline__ bool sm_wait(const SmallParams& p, const uint32_t* row, int words, bool plain, uint32_t (&v)[NWD]) {
  const int tid = threadIdx.x;
  return sm_until(p, [&] {
    bool there = true;
#pragma unroll
    for (int i = 0; i < NWD; ++i) {
      v[i] = get_word(row, min(tid + kSmNT * i, words - 1));
      there = there && v[i] != kNotYet;
    }
    return plain || there;
  });
}
// until a word of `row` (or NULL) is there, or for as long as a wait lasts
__device__ __forceinline__ void sm_early(const SmallParams& p, const uint32_t* row, int words, int b) {
  if (!row) return;  // uniform
  if (threadIdx.x < 64) {
    const uint32_t* at = row + (unsigned)(b * 7) % (unsigned)words;
    sm_until(p, [&] {
      const bool there = get_word(at, 0) != kNotYet;
      if (!there) __builtin_amdgcn_s_sleep(16);
      return there;
    });
  }
  __syncthreads();
}
// A wave's wait ended (got) or ran out. Behind a barrier, all(): whether every wave's did. AGAIN: goes on without its row, the launch failed.
template <bool AGAIN>
struct SmGot {
  int* s;  // [kSmNW]
  __device__ __forceinline__ void put(const SmallParams& p, bool got) const {
    if constexpr (AGAIN) {
      if (!got) st_out32(p.failed, 1u);
    } else if ((threadIdx.x & 63) == 0) {
      s[threadIdx.x >> 6] = got;
      if (!got) st_out32(p.undone, 1u);
    }
  }
  __device__ __forceinline__ bool all() const {
    if constexpr (AGAIN) return true;
    static_assert(kSmNW == 4);
    return s[0] & s[1] & s[2] & s[3];
  }
};

// word `at` of a row, asked for before (w): false if it did not come (the wave's own: no other wave needs it)
template <bool AGAIN>
__device__ __forceinline__ bool sm_own(const SmallParams& p, const uint32_t* row, int at, uint32_t& w) {
  if (__all(w != kNotYet) || sm_until(p, [&] { return (w = get_word(row, at)) != kNotYet; })) return true;
  st_out32(AGAIN ? (void*)p.failed : (void*)p.undone, 1u);
  return AGAIN;
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
// pieces. false (in every thread): it did not come
template <bool NORM, int NWD, int P, typename G>
__device__ __forceinline__ bool sm_row(const SmallParams& p, const uint32_t* row, int K, bool plain, const u32x2 (&g)[NORM ? P : 1], uint32_t* lds,
                                       float* red, G got, float (&xf)[P][4]) {
  const int tid = threadIdx.x, words = K >> 1;
  uint32_t v[NWD];
  got.put(p, sm_wait<NWD>(p, row, words, plain, v));
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
  if (!got.all()) return false;
  sm_pieces<P>(lds, K, xf);
  if constexpr (NORM) {
    const float r = round_bf(rsqrtf(round_bf(round_bf((red[0] + red[1] + red[2] + red[3]) / (float)K) + p.eps)));
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gv = (e & 1) ? bfhi(g[i][e >> 1]) : bflo(g[i][e >> 1]);
        xf[i][e] = 256 * i + 4 * (tid & 63) < K ? round_bf(gv * round_bf(xf[i][e] * r)) : 0.f;
      }
  }
  return true;
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
struct SmallLds {
  uint32_t row[PH * 128];
  float red[2 * kSmNW + kSmNW * 32 * WPL];
  int got[kSmNW];
};
// place b of the step
template <int PK, int PH, int WPL, bool AGAIN>
__device__ __forceinline__ void small_place(const SmallParams& p, int b, SmallLds<PK, PH, WPL>& shared) {
  uint32_t* const lds = shared.row;
  float* const red = shared.red;
  const SmGot<AGAIN> got{shared.got};
  constexpr int WK = (PK * 128 + kSmNT - 1) / kSmNT, WH = (PH * 128 + kSmNT - 1) / kSmNT;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
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
  const uint32_t* const xin = first ? p.x0 : x2 - stride;
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
    sm_early(p, first ? nullptr : hw - stride, H >> 1, b);
    if (!sm_row<true, WK, PK>(p, xin, C, first, g, lds, red, got, xf)) return;
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
    sm_early(p, first ? nullptr : x2 - stride, C >> 1, b);
    uint32_t nq[WPL], nk[WPL], nv[WPL];
    got.put(p, sm_until(p, [&] {
      bool there = true;
#pragma unroll
      for (int i = 0; i < WPL; ++i) {
        const int at = r * HW + min(sub + 16 * i, HW - 1);
        nq[i] = get_word(qkv, at);
        nk[i] = get_word(qkv, (C >> 1) + at);
        nv[i] = get_word(qkv, C + at);
        there = there && nq[i] != kNotYet && nk[i] != kNotYet && nv[i] != kNotYet;
      }
      return there;
    }));
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
    if (tid < HW && got.all()) {
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
    sm_early(p, qkv, 3 * (C >> 1), b);
    const int at = (nn >> 1) + (lane & 1);
    uint32_t xw = get_word(xin, at);
    if (!sm_row<false, WK, PK>(p, yw, C, false, none, lds, red, got, xf)) return;
    d.sums(xf, C, s);
    if (!first && !sm_own<AGAIN>(p, xin, at, xw)) return;
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
    sm_early(p, yw, C >> 1, b);
    if (!sm_row<true, WK, PK>(p, x1, C, false, g, lds, red, got, xf)) return;
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
    sm_early(p, x1, C >> 1, b);
    const int pair = lane % (kSmDown / 2), to_copy = lane / (kSmDown / 2), at = (nn >> 1) + pair;
    uint32_t xw = get_word(x1, at);
    if (!sm_row<false, WH, PH>(p, hw, H, false, none, lds, red, got, xf)) return;
    d.sums(xf, H, s);
    if (!sm_own<AGAIN>(p, x1, at, xw)) return;
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

template <int PK, int PH, int WPL>
__global__ __launch_bounds__(kSmNT) void small_step_kernel(SmallParams p) {
  __shared__ __align__(16) SmallLds<PK, PH, WPL> lds;
  small_place<PK, PH, WPL, false>(p, blockIdx.x, lds);
}

// What the first launch left undone, and again what it did, to the same values (its input x0 is not its output). A workgroup's place is the order of its
// start, from a counter: it waits for places taken before its own, so that the lowest unfinished one is running and waits for nobody, whatever else is
// on the device. Not the way of the first launch, since the counter takes 51 ns a workgroup, one after the other (49M 144 -> 178 us, 125M 207 -> 251).
template <int PK, int PH, int WPL>
__global__ __launch_bounds__(kSmNT) void small_again_kernel(SmallParams p) {
  __shared__ __align__(16) SmallLds<PK, PH, WPL> lds;
  __shared__ int place;
  if (get_word(p.undone, 0) == kNotYet) return;
  for (;;) {
    __syncthreads();  // (every wave is done with the last place's LDS)
    if (threadIdx.x == 0) place = (int)__hip_atomic_fetch_add(p.taken, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    __syncthreads();
    const int b = uniform(place);
    if ((unsigned)b >= (unsigned)(p.per * p.L)) return;
    small_place<PK, PH, WPL, true>(p, b, lds);
  }
}

// The step's first launch: the token's embedding, the position, and every word of the rows to come as not there yet, with the line behind x0.
__global__ __launch_bounds__(256) void small_begin_kernel(const int* __restrict__ idx, const uint32_t* __restrict__ wte, int words, int* pos_inc,
                                                          uint32_t* __restrict__ hand, int n, uint32_t* __restrict__ x0) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < words) x0[i] = wte[(size_t)idx[0] * words + i];
  if (i == 0) *pos_inc += 1;
  if (i < kSmLine) hand[n + i] = kNotYet;
  for (int k = i; k < n; k += gridDim.x * 256) hand[k] = kNotYet;
}

template <int PK, int PH>
static int small_go(SmallParams p, hipStream_t s) {
  SmallParams again = p;
  again.waits = p.waits < 0 ? -p.waits : kWaits;
  again.stop = p.undone + 2;
  p.waits = p.waits < 0 ? -p.waits : p.waits > 0 ? p.waits : kSmWaits;
  auto go = [&](auto step, auto rest) {
    hipLaunchKernelGGL(step, dim3(p.per * p.L), dim3(kSmNT), 0, s, p);
    LLJ_CHECK_LAUNCH();
    hipLaunchKernelGGL(rest, dim3(kSmAgain), dim3(kSmNT), 0, s, again);
    LLJ_CHECK_LAUNCH();
    return 0;
  };
  if (p.hs <= 64) return go(small_step_kernel<PK, PH, 2>, small_again_kernel<PK, PH, 2>);
  if (p.hs <= 96) return go(small_step_kernel<PK, PH, 3>, small_again_kernel<PK, PH, 3>);
  return go(small_step_kernel<PK, PH, 4>, small_again_kernel<PK, PH, 4>);
}

}  // namespace llj

using namespace llj;

extern "C" {

// Up to 512 cache slots: a head's one workgroup walks all keys. us a session's step, this for launches of their own (those with heads of 64 as ops.hip's
// shares), heads of 64 unless said:
//   10 layers of 640  139 / 204 at 30 keys, 204 / 220 at 600 (640 slots), 222 / 221 at 740, 259 / 225 at 1,000   12 of 1024  185 / 267, 272 / 298, 292 / 303, 331 / 305
//   12 layers of 780 (heads of 78)  194 / 234 at 30, 268 / 272 at 480, 290 / 278 at 600, 364 / 318 at 1,000   16 of 512, heads of 32  193 / 237, 272 / 266 at 480
// From 512 values on, where one bf16 row's products run on rowdot.h. Any number of layers, though the second launch and the first one's clearing are 4 us of a step:
// one layer takes 0.96 to 1.16 of its launches, two 0.88 to 1.14, three 0.84 to 1.12, six and more 0.75 to 1.03, the larger ones past 400 keys.
int llj_small_step_ok(int L, int C, int H, int nh, int S) {
  return L >= 1 && L <= kSmLayers && nh >= 1 && C % nh == 0 && (C / nh) % 2 == 0 && C / nh <= 128 && C / nh >= 32 && C % 4 == 0 && C >= 512 && C <= 1024 &&
         H % 4 == 0 && H >= 2 * C && H <= 2816 && S >= 1 && S <= 512;
}
// the rows' words, a line (undone, taken), x0
static size_t small_rows(int L, int C, int H) { return ((size_t)kSmCopies * L * (3 * C + (H >> 1)) + kSmLine - 1) / kSmLine * kSmLine; }
size_t llj_small_step_words(int L, int C, int H) { return small_rows(L, C, H) + kSmLine + (C >> 1); }

int llj_small_begin(const int* idx, const void* wte, int L, int C, int H, int* pos, void* hand, void* stream) {
  LLJ_REQUIRE(idx && wte && L >= 1 && L <= kSmLayers && C >= 2 && C % 2 == 0 && C <= 1024 && H >= 2 && H <= 2816 && pos && hand &&
              (((uintptr_t)wte | (uintptr_t)hand) & 3) == 0);
  const int words = (int)small_rows(L, C, H), blocks = std::min((words + 255) / 256, 128);  // (more than x0's: words >= 24 C)
  hipLaunchKernelGGL(small_begin_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, idx, (const uint32_t*)wte, C / 2, pos, (uint32_t*)hand, words,
                     (uint32_t*)hand + words + kSmLine);
  LLJ_CHECK_LAUNCH();
  return 0;
}

int llj_small_step(const void* const* layers, int L, int C, int H, int nh, int S, float eps, const float* rope, const int* pos, void* x, void* hand,
                   int* failed, int waits, void* stream) {
  LLJ_REQUIRE(llj_small_step_ok(L, C, H, nh, S) && layers && rope && pos && x && hand && failed && ((uintptr_t)x & 3) == 0 && ((uintptr_t)hand & 3) == 0);
  SmallParams p{};
  for (int l = 0; l < L; ++l) {
    for (int i = 0; i < 9; ++i) LLJ_REQUIRE(layers[9 * l + i] && ((uintptr_t)layers[9 * l + i] & (i < 7 ? 7 : 3)) == 0);
    const void* const* t = layers + 9 * l;
    p.layer[l] = SmallLayer{(const bf16_t*)t[0], (const bf16_t*)t[1], (const bf16_t*)t[2], (const bf16_t*)t[3], (const bf16_t*)t[4],
                            (const bf16_t*)t[5], (const bf16_t*)t[6], (bf16_t*)t[7], (bf16_t*)t[8]};
  }
  p.x = (bf16_t*)x; p.hand = (uint32_t*)hand; p.undone = p.hand + small_rows(L, C, H); p.stop = p.undone; p.taken = p.undone + 1; p.x0 = p.undone + kSmLine;
  p.failed = failed; p.waits = waits; p.rope = rope; p.pos = pos;
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
