// Up to 8 rows of the any-shape path on dense weights (generic.hip's llj_g_linear, llj_g_norm_linear, llj_g_norm_swiglu), and the
// attention of decode rows with their rotary positions and cache writes (llj_g_rope_attention).
//
// Decode of these models (780 wide, 3.6 MB per matrix) is bound by latency: what counts is how many dependent memory trips and
// launches a layer has. A wave takes one output column (four where there are columns enough for every CU), its lanes
// consecutive pieces of K. The residual's RMSNorm is computed by every workgroup for itself (a read of a few KB) in the order of
// g_rmsnorm_kernel, so a layer is 5 launches instead of 10. Loads come back in order, so each wave requests first what it needs
// first: the norm's row and weights (up to 1,024 values; beyond that they are read again), the residual, then the weights' pieces,
// and all without a branch, from clamped addresses whose values go unused; so a round has as many pieces as K needs (gr_pieces).
// us per launch, one row, weights first and all loads in branches -> this with 4 a round: bf16, K = 780: rms_1 and c_attn 4.6 -> 4.0, c_proj 2.8 -> 2.6, rms_2, c_fc1, c_fc2 and silu * mul 5.8 -> 4.6,
// mlp.c_proj (K = 2,080) 3.2 -> 3.0, lm_head 14.7 -> 11.0 (5.1 TB/s); four rows 10.6 -> 8.3, 4.7 -> 4.5, 13.1 -> 9.7, 5.7 -> 5.5,
// 35.1 -> 29.4; fp32, K = 512: the same to 0.2 less, lm_head 15.2 -> 12.6; bf16, K = 2,100: 12.2 -> 11.2, 16.4 -> 14.3. Two
// sets of 4 pieces by turns instead: 4.1, 2.7, 4.8, 3.5, 11.2.
#pragma once
#include <type_traits>

#include "common.h"
#include "elem.h"

namespace llj {

constexpr int GL_ROWS = 8;
constexpr int kGrNormLds = 48 * 1024;  // the rows' normalized copy of the norm-fused forms

enum { GR_PLAIN = 0, GR_NORM = 1, GR_SWIGLU = 2 };

// y[m, n] = x[m] . W[n] (+ resid), x through an RMSNorm in the fused forms; GR_SWIGLU: silu(x . W[n]) * (x . W2[n]). VE elements
// per load: a divisor of K (and of ldx), with x and W aligned to it. MB: 1 or 8 rows' accumulators; NC: columns per wave; U: pieces of 64
// lanes x VE elements per round (gr_pieces). APART: the last round's code by itself.
template <typename T, int VE, int MB, int NC, int MODE, int U, bool APART>
__global__ __launch_bounds__(256) void g_rows_kernel(const T* __restrict__ x, int ldx, const T* __restrict__ nw, float eps, int M,
                                                     int K, const T* __restrict__ W, const T* __restrict__ W2, int N,
                                                     T* __restrict__ y, int ldy, const T* resid, int ldr) {
  extern __shared__ __align__(16) char gr_lds[];
  typedef T vec __attribute__((ext_vector_type(VE)));
  constexpr int NT = MODE == GR_SWIGLU ? 2 : NC;
  const int tid = threadIdx.x, lane = tid & 63, n0 = (blockIdx.x * 4 + (tid >> 6)) * NC;
  const T* wr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = MODE == GR_SWIGLU ? n0 : n0 + t;
    wr[t] = (MODE == GR_SWIGLU && t ? W2 : W) + (size_t)(n < N ? n : N - 1) * K;
  }
  constexpr int RU = MODE == GR_PLAIN ? 1 : 4;
  T xf[MB][RU], nf[RU], rv[MB];
  if constexpr (MODE != GR_PLAIN) {
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int k = min(tid + 256 * u, K - 1);
      nf[u] = nw[k];
#pragma unroll
      for (int r = 0; r < MB; ++r) xf[r][u] = x[(size_t)min(r, M - 1) * ldx + k];
    }
  }
  if constexpr (MODE != GR_SWIGLU) {
    const T* rp = resid ? resid + min(n0 + min(lane, NC - 1), N - 1) : x;
#pragma unroll
    for (int r = 0; r < MB; ++r) rv[r] = rp[resid ? (size_t)min(r, M - 1) * ldr : 0];
  }
  vec wv[NT][U];
  // piece u at k: from a valid address whatever k is; of 8 vectors, the last 4 behind branches
  auto piece = [&](const T* p, int k, int u) {
    if (U < 8 || VE == 1 || u < 4 || k < K) return *reinterpret_cast<const vec*>(p + min(k, K - VE));
    return vec(0);
  };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t) wv[t][u] = piece(wr[t], k0 + (u * 64 + lane) * VE, u);
  };
  fetch(0);
  T* xs = reinterpret_cast<T*>(gr_lds);
  if constexpr (MODE != GR_PLAIN) {
    __shared__ float red[MB][4];
#pragma unroll
    for (int r = 0; r < MB; ++r) {
      if (r < M) {
        float ss = 0.f;
        auto add = [&](float v) { ss += rnd<T>(v * v); };
#pragma unroll
        for (int u = 0; u < RU; ++u)
          if (tid + 256 * u < K) add(ldv(&xf[r][u], 0));
        for (int k = tid + 256 * RU; k < K; k += 256) add(ldv(x, (size_t)r * ldx + k));
        ss = wave_sum(ss);
        if (lane == 0) red[r][tid >> 6] = ss;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < MB; ++r) {
      if (r < M) {
        const float tot = red[r][0] + red[r][1] + red[r][2] + red[r][3];
        const float s = rnd<T>(rsqrtf(rnd<T>(rnd<T>(tot / (float)K) + eps)));
#pragma unroll
        for (int u = 0; u < RU; ++u)
          if (tid + 256 * u < K) stv(xs, r * K + tid + 256 * u, ldv(&nf[u], 0) * rnd<T>(ldv(&xf[r][u], 0) * s));
        for (int k = tid + 256 * RU; k < K; k += 256) stv(xs, r * K + k, ldv(nw, k) * rnd<T>(ldv(x, (size_t)r * ldx + k) * s));
      }
    }
    __syncthreads();
  }
  float acc[MB][NT];
#pragma unroll
  for (int r = 0; r < MB; ++r)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[r][t] = 0.f;
  // One round; only the last asks of each piece whether it is past K (asked in every round, single elements, 8 rows of K = 6,400, bf16,
  // -> 20,000: 145 us for 101). Its code is apart from the others', or with theirs in the loop, which one column of 2 to 8 rows prefers
  // where K is a single round (fp32, K = 780 -> 780, norm: 4 rows 6.4 us apart, 5.5 in the loop; several rounds, bf16, 8 rows of 6,400 ->
  // 3,000 21.3 and 24.0).
  auto round = [&](int k0, bool last) {
#pragma unroll
    for (int r = 0; r < MB; ++r) {
      if (r < M) {
        const T* xr = MODE == GR_PLAIN ? x + (size_t)r * ldx : xs + r * K;
        vec xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = k0 + (u * 64 + lane) * VE;
          xv[u] = APART && !last ? *reinterpret_cast<const vec*>(xr + k) : piece(xr, k, u);
        }
        auto add = [&](int u) {
#pragma unroll
          for (int e = 0; e < VE; ++e) {
            T xe = xv[u][e];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              T we = wv[t][u][e];
              acc[r][t] += ldv(&xe, 0) * ldv(&we, 0);
            }
          }
        };
        if (last) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (k0 + (u * 64 + lane) * VE < K) add(u);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) add(u);
        }
      }
    }
  };
  int k0 = 0;
  if constexpr (APART) {
    for (; k0 + U * 64 * VE < K; k0 += U * 64 * VE) {
      round(k0, false);
      fetch(k0 + U * 64 * VE);
    }
    round(k0, true);
  } else {
    for (; k0 < K; k0 += U * 64 * VE) {
      if (k0) fetch(k0);
      round(k0, k0 + U * 64 * VE > K);
    }
  }
#pragma unroll
  for (int r = 0; r < MB; ++r) {
    if (r < M) {
      float s[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) s[t] = rnd<T>(wave_sum(acc[r][t]));
      if constexpr (MODE == GR_SWIGLU) {
        if (lane == 0 && n0 < N) stv(y, (size_t)r * ldy + n0, rnd<T>(s[0] / (1.f + expf(-s[0]))) * s[1]);
      } else {
#pragma unroll
        for (int t = 0; t < NC; ++t) {
          if (lane == t && n0 + t < N) {
            float v = s[t];
            if (resid) v = ldv(&rv[r], 0) + v;
            stv(y, (size_t)r * ldy + n0 + t, v);
          }
        }
      }
    }
  }
}

// A pair in rotary position (c, s), rounded the same in every kernel that forms it
__device__ __forceinline__ float2 gr_rotate(float x0, float x1, float c, float s) {
  const float a = x1 * s, b = x1 * c;
  return make_float2(__builtin_fmaf(x0, c, -a), __builtin_fmaf(x0, s, b));
}

// One token per sequence: rotary positions of q and k (g_rope_kv_kernel), k and v into cache slot p % S, and causal attention over
// the cache (g_attention_kernel). Block (row, head) of 512 threads -- a few tens of blocks with a chain of memory trips each: 16
// lanes per key and 128 keys at a time, then the values with the threads split over dimension pairs and up to kGrKeyGroups
// interleaved groups of keys. The first keys and values are loaded before the rotation, without a branch around any of them but in MASK. For heads
// of more than 128 (fp32 with many workgroups: 64); the others below. LDS: S + hs (3 + groups) floats.
constexpr int kGrThreads = 512, kGrKeyGroups = 14;
__host__ __device__ inline int gr_groups(int P) { return P > kGrThreads ? 1 : P * kGrKeyGroups > kGrThreads ? kGrThreads / P : kGrKeyGroups; }
// MASK: only what is seen is loaded, behind branches.
template <typename T, bool MASK>
__global__ __launch_bounds__(kGrThreads) void g_rope_attention_kernel(const T* __restrict__ qkv, T* __restrict__ kc, T* __restrict__ vc,
                                                               const float* __restrict__ rope, const int* __restrict__ pos,
                                                               T* __restrict__ y, int C, int nh, int S) {
  extern __shared__ __align__(16) char gr_lds[];
  __shared__ float red[kGrThreads / 64];
  typedef T pair __attribute__((ext_vector_type(2)));
  constexpr int NQ = 4;  // pairs of a key for each of its 16 lanes, at a time
  const int m = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int hs = C / nh, P = hs / 2, p = pos[0], slot = p % S, nvis = p < S ? p + 1 : S;
  float* sc = reinterpret_cast<float*>(gr_lds);  // [S] scores, then weights
  float* sq = sc + S;                            // [hs] the scaled query
  float* sk = sq + hs;                           // [hs] the new key
  float* sv = sk + hs;                           // [hs] and value
  float* so = sv + hs;                           // [groups][hs] partial outputs
  const float scale = 1.f / sqrtf((float)hs);
  const T* row = qkv + (size_t)m * 3 * C + h * hs;
  const size_t cb = ((size_t)m * nh + h) * S * hs, cbase = cb + (size_t)slot * hs;
  // keys j0 + 32 u of this group of 16 lanes, 16 NQ pairs from i0 on: up to 16 loads in flight
  const int sub = tid & 15, kg = tid >> 4;
  pair kw[4][NQ];
  auto keys = [&](int j0, int i0) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int j = min(j0 + 32 * u, S - 1), i = min(i0 + 16 * q + sub, P - 1);  // (a valid pair, not used past the last: no branch)
        if (MASK && !(j0 + 32 * u < nvis && i0 + 16 * q + sub < P)) kw[u][q] = pair(0);
        else kw[u][q] = reinterpret_cast<const pair*>(kc + cb + (size_t)j * hs)[i];
      }
  };
  const int G = gr_groups(P), g = P > kGrThreads ? 0 : tid / P;
  const int pi = P > kGrThreads ? tid : tid % P;  // this thread's (first) pair of the values, keys g + G u
  const pair* vr = reinterpret_cast<const pair*>(vc + cb) + pi;
  constexpr int VU = 12;
  pair vw[VU];
  keys(kg, 0);
#pragma unroll
  for (int u = 0; u < VU; ++u) {
    if (MASK && !(g < G && g + G * u < nvis)) vw[u] = pair(0);
    else vw[u] = vr[(size_t)min(min(g, G - 1) + G * u, S - 1) * P];
  }
  // in flight while q and k are rotated; the rows that this workgroup writes come from LDS
  for (int i = tid; i < P; i += kGrThreads) {
    const float c = rope[((size_t)p * P + i) * 2], s = rope[((size_t)p * P + i) * 2 + 1];
    const float q0 = ldv(row, 2 * i), q1 = ldv(row, 2 * i + 1), k0 = ldv(row, C + 2 * i), k1 = ldv(row, C + 2 * i + 1);
    const float2 q = gr_rotate(q0, q1, c, s), k = gr_rotate(k0, k1, c, s);
    sq[2 * i] = rnd<T>(q.x) * scale;
    sq[2 * i + 1] = rnd<T>(q.y) * scale;
    const float r0 = rnd<T>(k.x), r1 = rnd<T>(k.y);
    sk[2 * i] = r0;
    sk[2 * i + 1] = r1;
    sv[2 * i] = ldv(row, 2 * C + 2 * i);
    sv[2 * i + 1] = ldv(row, 2 * C + 2 * i + 1);
    stv(kc, cbase + 2 * i, r0);
    stv(kc, cbase + 2 * i + 1, r1);
    vc[cbase + 2 * i] = row[2 * C + 2 * i];
    vc[cbase + 2 * i + 1] = row[2 * C + 2 * i + 1];
  }
  __syncthreads();
  float mx = -INFINITY;
  for (int j0 = kg; j0 < nvis; j0 += 128) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < P; i0 += 16 * NQ) {
      if (j0 != kg || i0) keys(j0, i0);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int i = i0 + 16 * q + sub;
        if (i >= P) continue;
        const float q0 = sq[2 * i], q1 = sq[2 * i + 1];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          T k0 = kw[u][q][0], k1 = kw[u][q][1];
          const bool own = j0 + 32 * u == slot;
          s[u] += q0 * (own ? sk[2 * i] : ldv(&k0, 0)) + q1 * (own ? sk[2 * i + 1] : ldv(&k1, 0));
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s[u] = row16_sum(s[u]);
      if (j0 + 32 * u < nvis) {
        if (sub == 0) sc[j0 + 32 * u] = s[u];
        mx = fmaxf(mx, s[u]);
      }
    }
  }
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kGrThreads / 64; ++w) mx = fmaxf(mx, red[w]);
  __syncthreads();
  float l = 0.f;
  for (int j = tid; j < nvis; j += kGrThreads) {
    const float e = __expf(sc[j] - mx);
    sc[j] = e;
    l += e;
  }
  l = wave_sum(l);
  if ((tid & 63) == 0) red[tid >> 6] = l;
  __syncthreads();
  l = 0.f;
#pragma unroll
  for (int w = 0; w < kGrThreads / 64; ++w) l += red[w];
  const float inv = 1.f / l;
  for (int i = pi; i < P && g < G; i += P > kGrThreads ? kGrThreads : P) {
    float o0 = 0.f, o1 = 0.f;
    auto add = [&](int j, pair v) {
      T v0 = v[0], v1 = v[1];
      o0 += sc[j] * (j == slot ? sv[2 * i] : ldv(&v0, 0));
      o1 += sc[j] * (j == slot ? sv[2 * i + 1] : ldv(&v1, 0));
    };
    int j = g;
    if (i == pi) {
#pragma unroll
      for (int u = 0; u < VU; ++u, j += G)
        if (j < nvis) add(j, vw[u]);
    }
#pragma unroll 8
    for (; j < nvis; j += G) add(j, vr[(i - pi) + (size_t)j * P]);
    so[g * hs + 2 * i] = o0;
    so[g * hs + 2 * i + 1] = o1;
  }
  __syncthreads();
  for (int d = tid; d < hs; d += kGrThreads) {
    float o = 0.f;
    for (int k = 0; k < G; ++k) o += so[k * hs + d];
    stv(y, (size_t)m * C + h * hs + d, o * inv);
  }
}


// The same for heads of up to 128, in registers: lane l of 16 holds pairs l, l + 16 .. of the query, of its keys and of the outputs, so the rotation needs
// no LDS, keys and values pass once (running maximum and sum per 16 lanes, key group + 32 i) and the workgroup meets once, at the end.
// A chain of three memory trips: the first 128 keys and values with the position (not in MASK), then its rotary pairs, then (from 128 keys on) the next
// keys, a pass ahead.
// us with the scores in LDS (the kernel above) and so, bf16: 10 heads of 78, 40 keys 5.4 and 3.9, 110 keys 5.7 and 4.0, 500 keys 18.7 and 7.0 (launches one after the
// other; in a decode step 110 keys take 5.0); 8 rows
// of 32 heads of 80, 500 keys 28.4 and 11.9; fp32: 10 heads of 78, 110 keys 5.7 and 5.1, 500 keys 12.9 and 9.5; heads of
// 100 and 128 in the first some 50 keys 6.2 to 6.6 and 6.4 to 6.9, later 1.1 to 1.3 times as fast. 10 workgroups: bound by the chain, not by the 16 KB a
// head.
template <typename T, int NQ, int U, bool MASK>
__global__ __launch_bounds__(kGrThreads) void g_rope_attention16_kernel(const T* __restrict__ qkv, T* __restrict__ kc, T* __restrict__ vc,
                                                                 const float* __restrict__ rope, const int* __restrict__ pos,
                                                                 T* __restrict__ y, int C, int nh, int S) {
  constexpr int kWaves = kGrThreads / 64, kGroups = kGrThreads / 16, kMost = 32 * NQ;
  __shared__ float so[kWaves][kMost], sm[kWaves], sl[kWaves];
  typedef T pair __attribute__((ext_vector_type(2)));
  typedef pair __attribute__((aligned(sizeof(T)))) any_pair;
  const int m = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, sub = tid & 15, kg = tid >> 4;
  const int hs = C / nh, P = hs / 2;
  const size_t cb = ((size_t)m * nh + h) * S * hs;
  const T* row = qkv + (size_t)m * 3 * C + h * hs;
  int at[NQ];  // this lane's pairs (past the last: a valid one, not used)
#pragma unroll
  for (int q = 0; q < NQ; ++q) at[q] = min(16 * q + sub, P - 1);
  constexpr int kBufs = MASK ? 1 : 2;  // (many workgroups: two to a CU instead of a pass ahead)
  pair kw[kBufs][U][NQ], vw[kBufs][U][NQ];
  auto load = [&](int b, int j0, int lim) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t r = cb + (size_t)min(j0 + kGroups * u, lim - 1) * hs;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        kw[b][u][q] = reinterpret_cast<const pair*>(kc + r)[at[q]];
        vw[b][u][q] = reinterpret_cast<const pair*>(vc + r)[at[q]];
      }
    }
  };
  pair qw[NQ], nk[NQ], nv[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    qw[q] = *reinterpret_cast<const any_pair*>(row + 2 * at[q]);
    nk[q] = *reinterpret_cast<const any_pair*>(row + C + 2 * at[q]);
    nv[q] = *reinterpret_cast<const any_pair*>(row + 2 * C + 2 * at[q]);
  }
  if constexpr (!MASK) load(0, kg, S);
  const int p = pos[0], slot = p % S, nvis = p < S ? p + 1 : S;
  typedef float any_rope __attribute__((ext_vector_type(2), aligned(4)));
  any_rope cs[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) cs[q] = *reinterpret_cast<const any_rope*>(rope + ((size_t)p * P + at[q]) * 2);
  if constexpr (MASK) load(0, kg, nvis);
  const float scale = 1.f / sqrtf((float)hs);
  float q0[NQ], q1[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    T a0 = qw[q][0], a1 = qw[q][1], b0 = nk[q][0], b1 = nk[q][1];
    const float c = cs[q].x, s = cs[q].y, x0 = ldv(&a0, 0), x1 = ldv(&a1, 0), k0 = ldv(&b0, 0), k1 = ldv(&b1, 0);
    const bool mine = 16 * q + sub < P;
    const float2 rq = gr_rotate(x0, x1, c, s), rk = gr_rotate(k0, k1, c, s);
    q0[q] = mine ? rnd<T>(rq.x) * scale : 0.f;
    q1[q] = mine ? rnd<T>(rq.y) * scale : 0.f;
    stv(&b0, 0, rk.x);
    stv(&b1, 0, rk.y);
    nk[q] = pair{b0, b1};
    if (kg == 0 && mine) {
      reinterpret_cast<pair*>(kc + cb + (size_t)slot * hs)[at[q]] = nk[q];
      reinterpret_cast<pair*>(vc + cb + (size_t)slot * hs)[at[q]] = nv[q];
    }
  }
  float mx = -INFINITY, l = 0.f, o[2 * NQ] = {};
  auto pass = [&](int b, int base) {  // keys base + group + 32 u
    if constexpr (MASK) {
      if (base) load(0, base + kg, nvis);
    } else if (base + kGroups * U < nvis) {
      load(b ^ 1, base + kGroups * U + kg, nvis);
    }
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = base + kg + kGroups * u;
      s[u] = 0.f;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if (j == slot) kw[b][u][q] = nk[q], vw[b][u][q] = nv[q];
        T k0 = kw[b][u][q][0], k1 = kw[b][u][q][1];
        float v0 = ldv(&k0, 0), v1 = ldv(&k1, 0);
        if (q == NQ - 1) {  // (a pair of another lane: no part of this one's sum, whatever it holds)
          v0 = 16 * q + sub < P ? v0 : 0.f;
          v1 = 16 * q + sub < P ? v1 : 0.f;
        }
        s[u] += q0[q] * v0 + q1[q] * v1;
      }
      s[u] = row16_sum(s[u]);
      s[u] = j < nvis ? s[u] : -INFINITY;
    }
    float mn = mx;
#pragma unroll
    for (int u = 0; u < U; ++u) mn = fmaxf(mn, s[u]);
    const float ref = mn == -INFINITY ? 0.f : mn, corr = __expf(mx - ref);  // (nothing seen yet: weights of zero)
    mx = mn;
    l *= corr;
#pragma unroll
    for (int i = 0; i < 2 * NQ; ++i) o[i] *= corr;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (base + kg + kGroups * u >= nvis) continue;
      const float w = __expf(s[u] - ref);
      l += w;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        T v0 = vw[b][u][q][0], v1 = vw[b][u][q][1];
        o[2 * q] += w * ldv(&v0, 0);
        o[2 * q + 1] += w * ldv(&v1, 0);
      }
    }
  };
  for (int base = 0; base < nvis; base += 2 * kGroups * U) {
    pass(0, base);
    if (base + kGroups * U < nvis) pass(kBufs - 1, base + kGroups * U);
  }
  auto merge = [&](auto wide) {  // two groups of 16 lanes, in every lane of both
    constexpr bool W = decltype(wide)::value;
    float mlo, mhi, llo, lhi;
    lane_halves<W>(mx, mlo, mhi);
    lane_halves<W>(l, llo, lhi);
    const float M = fmaxf(mlo, mhi), flo = mlo == -INFINITY ? 0.f : __expf(mlo - M), fhi = mhi == -INFINITY ? 0.f : __expf(mhi - M);
    mx = M;
    l = llo * flo + lhi * fhi;
#pragma unroll
    for (int i = 0; i < 2 * NQ; ++i) {
      float lo, hi;
      lane_halves<W>(o[i], lo, hi);
      o[i] = lo * flo + hi * fhi;
    }
  };
  merge(std::false_type());
  merge(std::true_type());
  const int wave = tid >> 6;
  if ((tid & 63) < 16) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) *reinterpret_cast<float2*>(&so[wave][2 * (16 * q + sub)]) = make_float2(o[2 * q], o[2 * q + 1]);
    if (sub == 0) sm[wave] = mx, sl[wave] = l;
  }
  __syncthreads();
  if (tid < hs) {
    float M = sm[0], L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) M = fmaxf(M, sm[w]);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = sm[w] == -INFINITY ? 0.f : __expf(sm[w] - M);
      L += sl[w] * f;
      O += so[w][tid] * f;
    }
    stv(y, (size_t)m * C + h * hs + tid, O / L);
  }
}

}  // namespace llj
