// Causal attention of a prompt's rows over the cache for any head size (generic.hip's llj_g_attention), on the fp32 matrix cores.
//
// A workgroup owns 16 consecutive rows of one sequence and head; keys come 64 at a time. Four waves score 16 keys each, the rows'
// running maxima and sums go over LDS, then each wave takes the outputs' 16-column blocks w, w + 4, ..: operands are fp32 in LDS
// whatever the cache holds, one operand read of 16 bytes a lane is four v_mfma_f32_16x16x4_f32 (the order over the reduced index is
// free as long as both operands agree). Keys and values take turns in one LDS buffer; the values' loads are in flight while the
// scores are formed, the next keys' while the values are used. A tile of either is one contiguous piece of the cache, loaded in
// vectors that a row holds a whole number of.
//
// fp32 heads of 129 to 256 keep 9 of their registers in scratch; with one wave per SIMD instead of two there is no scratch, and heads of
// 256 take 52 us for 56 (301 rows, 16 heads), but heads of 160 41 for 36.
//
// Bound: at some hundred rows by the chain of a few tiles (loads, two barriers, softmax). One row per workgroup and one key per
// thread, which this replaces for all but short prompts, read a key's elements one by one, a row apart from lane to lane.
#pragma once
#include "common.h"
#include "elem.h"

namespace llj {

constexpr int kGaRows = 16, kGaKeys = 64, kGaPs = kGaKeys + 4;
constexpr int kGaMaxD = 256;
constexpr int kGaLoads = 16;  // most vectors of a tile per thread

__host__ __device__ inline int ga_stride(int hs) { return ((hs + 15) & ~15) + 4; }  // fp32 LDS row: 16 rows on 16 groups of 4 banks
inline size_t ga_lds(int hs) { return ((size_t)(kGaRows + kGaKeys) * ga_stride(hs) + kGaRows * kGaPs + 8 * kGaRows) * 4; }
inline int ga_vectors(int hs, int ve) { return (kGaKeys * hs / ve + 255) / 256; }  // per thread and tile

// One row by g_attention_kernel's steps: y = softmax(q . K) V over its n keys and no other. q: the scaled row, lds: 264 floats.
template <typename T>
__device__ __forceinline__ void ga_row(const float* q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ y, int n, int hs, float* lds, int tid) {
  const int lane = tid & 63, wave = tid >> 6;
  float *sc = lds, *top = lds + 256, *sum = lds + 260;
  auto score = [&](int j) {
    float s = 0.f;
    for (int d = 0; d < hs; ++d) s += q[d] * ldv(k, (size_t)j * hs + d);
    return s;
  };
  float mx = -INFINITY, l = 0.f, o = 0.f;
  for (int j = tid; j < n; j += 256) mx = fmaxf(mx, score(j));
  mx = wave_max(mx);
  if (lane == 0) top[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
  for (int j0 = 0; j0 < n; j0 += 256) {
    const float p = j0 + tid < n ? __expf(score(j0 + tid) - mx) : 0.f;
    l += p;
    sc[tid] = p;
    __syncthreads();
    if (tid < hs)
      for (int j = 0; j < min(256, n - j0); ++j) o += sc[j] * ldv(v, (size_t)(j0 + j) * hs + tid);
    __syncthreads();
  }
  l = wave_sum(l);
  if (lane == 0) sum[wave] = l;
  __syncthreads();
  if (tid < hs) stv(y, tid, o * (1.f / (sum[0] + sum[1] + sum[2] + sum[3])));
}

template <typename T, int VE, int NL>
__global__ __launch_bounds__(256, 2) void g_attention_tiles_kernel(const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc,
                                                                   T* __restrict__ y, const int* __restrict__ pos, int T_, int C, int nh, int S) {
  extern __shared__ __align__(16) float ga_lds_mem[];
  typedef T vec __attribute__((ext_vector_type(VE)));
  const int hs = C / nh, ST = ga_stride(hs), DB = (hs + 15) >> 4;
  float* Qs = ga_lds_mem;               // [16][ST]
  float* KV = Qs + kGaRows * ST;        // [64][ST]
  float* Ps = KV + kGaKeys * ST;        // [16][kGaPs]
  float* red = Ps + kGaRows * kGaPs;    // [4][16]
  int* s_n = reinterpret_cast<int*>(red + 4 * kGaRows);  // [16] visible keys of a row
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c16 = lane & 15, g4 = lane >> 4;
  const int QT = (T_ + kGaRows - 1) / kGaRows, b = blockIdx.x / QT, t0 = (QT - 1 - (int)blockIdx.x % QT) * kGaRows, h = blockIdx.y;
  const float scale = 1.f / sqrtf((float)hs);
  const size_t base = ((size_t)b * nh + h) * S * hs;
  auto load = [&](__amdgpu_buffer_rsrc_t buf, int at) -> vec {  // (outside the buffer: zeros, with no branch around a load)
    if constexpr (sizeof(vec) == 16) return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(buf, at, 0, 0));
    else if constexpr (sizeof(vec) == 8) return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b64(buf, at, 0, 0));
    else if constexpr (sizeof(vec) == 4) return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b32(buf, at, 0, 0));
    else return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b16(buf, at, 0, 0));
  };
  // The rows, the first keys (all of the cache's: which are seen is not known yet, the others' scores are replaced) and the positions
  // are on their way together.
  constexpr int NQ = (NL + 3) / 4;
  const int rows = min(kGaRows, T_ - t0);
  const __amdgpu_buffer_rsrc_t qbuf =
      __builtin_amdgcn_make_buffer_rsrc((void*)(q + ((size_t)b * T_ + t0) * C + h * hs), 0, ((rows - 1) * C + hs) * (int)sizeof(T), 0x00020000);
  const __amdgpu_buffer_rsrc_t kbuf = __builtin_amdgcn_make_buffer_rsrc((void*)(kc + base), 0, S * hs * (int)sizeof(T), 0x00020000);
  const int p0 = pos[min(t0 + c16, T_ - 1)];
  vec qr[NQ], kr[NL], vr[NL];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int e = (tid + 256 * i) * VE, r = e / hs;
    qr[i] = load(qbuf, r < rows ? (r * C + e - r * hs) * (int)sizeof(T) : 0x7ffffff0);
  }
  auto fetch = [&](vec (&w)[NL], __amdgpu_buffer_rsrc_t buf, int k0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) w[i] = load(buf, ((tid + 256 * i) * VE + k0 * hs) * (int)sizeof(T));
  };
  fetch(kr, kbuf, 0);
  if (tid < kGaRows) s_n[tid] = p0 < S ? p0 + 1 : S;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int e = (tid + 256 * i) * VE, r = e / hs, d = e - r * hs;
    if (r < kGaRows) {
#pragma unroll
      for (int j = 0; j < VE; ++j) {
        T v = qr[i][j];
        Qs[r * ST + d + j] = ldv(&v, 0) * scale;
      }
    }
  }
  for (int i = tid; i < kGaRows * (ST - hs); i += 256) {
    const int r = i / (ST - hs);
    Qs[r * ST + hs + i - r * (ST - hs)] = 0.f;
  }
  for (int i = tid; i < kGaKeys * (ST - hs); i += 256) {  // the padding of the reduced index
    const int r = i / (ST - hs);
    KV[r * ST + hs + i - r * (ST - hs)] = 0.f;
  }
  __syncthreads();
  int nrow[4], nmax = 0;
#pragma unroll
  for (int r = 0; r < kGaRows; ++r) nmax = max(nmax, s_n[r]);
#pragma unroll
  for (int r = 0; r < 4; ++r) nrow[r] = s_n[4 * g4 + r];
  nmax = uniform(nmax);

  const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc((void*)(vc + base), 0, nmax * hs * (int)sizeof(T), 0x00020000);
  auto put = [&](const vec (&w)[NL]) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (tid + 256 * i) * VE, r = e / hs, d = e - r * hs;
      if (r < kGaKeys) {
#pragma unroll
        for (int j = 0; j < VE; ++j) {
          T v = w[i][j];
          KV[r * ST + d + j] = ldv(&v, 0);
        }
      }
    }
  };
  f32x4 o[kGaMaxD / 64];
#pragma unroll
  for (int i = 0; i < kGaMaxD / 64; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mx[4], l[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) mx[r] = -3.402823466e38f, l[r] = 0.f;  // (finite: a first tile of scores of minus infinity has weights of 0)
  for (int k0 = 0; k0 < nmax; k0 += kGaKeys) {
    put(kr);
    fetch(vr, vbuf, k0);
    __syncthreads();  // the keys are there
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int d = 0; d < DB; ++d) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(Qs + c16 * ST + 16 * d + 4 * g4);
      const f32x4 k = *reinterpret_cast<const f32x4*>(KV + (16 * wave + c16) * ST + 16 * d + 4 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], k[e], s, 0, 0, 0);
    }
    const int key = k0 + 16 * wave + c16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (key >= nrow[r]) s[r] = -INFINITY;
      const float m = row16_max(s[r]);
      if (c16 == 0) red[wave * kGaRows + 4 * g4 + r] = m;
    }
    __syncthreads();  // the keys are read, the maxima are there
    put(vr);
    if (k0 + kGaKeys < nmax) fetch(kr, kbuf, k0 + kGaKeys);
    f32x4 keep;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g4 + r;
      const float m = fmaxf(fmaxf(fmaxf(red[i], red[kGaRows + i]), fmaxf(red[2 * kGaRows + i], red[3 * kGaRows + i])), mx[r]);
      keep[r] = __expf(mx[r] - m);
      mx[r] = m;
      const float p = __expf(s[r] - m);
      l[r] = l[r] * keep[r] + p;
      Ps[i * kGaPs + 16 * wave + c16] = p;
    }
    __syncthreads();  // the values and the weights are there
#pragma unroll
    for (int i = 0; i < kGaMaxD / 64; ++i) {
      const int d = wave + 4 * i;
      if (d >= DB) break;
      f32x4 a = o[i] * keep;
#pragma unroll
      for (int g = 0; g < kGaKeys / 16; ++g) {
        const f32x4 p = *reinterpret_cast<const f32x4*>(Ps + c16 * kGaPs + 16 * g + 4 * g4);
        const float* v = KV + (16 * g + 4 * g4) * ST + 16 * d + c16;
#pragma unroll
        for (int e = 0; e < 4; ++e) a = __builtin_amdgcn_mfma_f32_16x16x4f32(p[e], v[e * ST], a, 0, 0, 0);
      }
      o[i] = a;
    }
    __syncthreads();  // the values are read
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float v = row16_sum(l[r]);
    if (c16 == 0) red[wave * kGaRows + 4 * g4 + r] = v;
  }
  int* odd = reinterpret_cast<int*>(Ps);  // [16] rows with an output that is not finite
  if (tid < kGaRows) odd[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * g4 + r;
    const float inv = 1.f / ((red[i] + red[kGaRows + i]) + (red[2 * kGaRows + i] + red[3 * kGaRows + i]));
    if (t0 + i >= T_) continue;
#pragma unroll
    for (int n = 0; n < kGaMaxD / 64; ++n) {
      const int d = 16 * (wave + 4 * n) + c16;
      const float v = o[n][r] * inv;
      if (d < hs) stv(y, ((size_t)b * T_ + t0 + i) * C + h * hs + d, v);
      if (d < hs && !(fabsf(v) < INFINITY)) odd[i] = 1;
    }
  }
  // A row that does not see a key takes 0 times its value above, and that is not 0 for a value that is not finite: where an output is
  // not, its row again from its own keys alone. (lane2: the lane without a register held through the loop, which cost fp32 heads of 78
  // their third wave per SIMD. Told apart in the loop, it took 10 registers.)
  __syncthreads();
  const int lane2 = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
  unsigned again = (unsigned)__ballot(lane2 < kGaRows && odd[lane2 & (kGaRows - 1)]);
  for (; again; again &= again - 1) {
    const int i = __builtin_ctz(again);
    ga_row(Qs + i * ST, kc + base, vc + base, y + ((size_t)b * T_ + t0 + i) * C + h * hs, uniform(s_n[i]), hs, KV, wave * 64 + lane2);
    __syncthreads();
  }
}

// Launches the tiled form for head sizes it takes; 1: not one of them.
template <typename T>
static int ga_launch(const T* q, const T* kc, const T* vc, T* y, const int* pos, int B, int T_, int C, int nh, int S, hipStream_t s) {
  const int hs = C / nh;
  const int ve = hs % 4 == 0 && (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) % (4 * sizeof(T))) == 0   ? 4
                 : hs % 2 == 0 && (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) % (2 * sizeof(T))) == 0 ? 2
                                                                                             : 1;
  const int nl = ga_vectors(hs, ve);
  const long blocks = (long)B * ((T_ + kGaRows - 1) / kGaRows);
  if (hs > kGaMaxD || nl > kGaLoads || (long)S * hs * (long)sizeof(T) > 0x7fffff00 || (long)kGaRows * C * (long)sizeof(T) > 0x7fffff00 || blocks >= (1l << 31)) return 1;
  const size_t lds = ga_lds(hs);
  auto go = [&](auto kern) -> int {
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, nh), dim3(256), lds, s, q, kc, vc, y, pos, T_, C, nh, S);
    LLJ_CHECK_LAUNCH();
    return 0;
  };
  if (ve == 4) return nl <= 4 ? go(g_attention_tiles_kernel<T, 4, 4>) : nl <= 8 ? go(g_attention_tiles_kernel<T, 4, 8>) : go(g_attention_tiles_kernel<T, 4, 16>);
  if (ve == 2) return nl <= 10 ? go(g_attention_tiles_kernel<T, 2, 10>) : go(g_attention_tiles_kernel<T, 2, 16>);
  return nl <= 4 ? go(g_attention_tiles_kernel<T, 1, 4>) : go(g_attention_tiles_kernel<T, 1, 16>);
}

}  // namespace llj
