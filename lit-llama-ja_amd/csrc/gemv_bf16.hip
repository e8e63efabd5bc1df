// Instantiations of the GEMV kernels for weight format WF_BF16 (gemv_impl.h), one row on rowdot.h.
#include "gemv_impl.h"
#include "rowdot.h"

namespace llj {

// One row: rowdot.h where its 16-byte loads are aligned and nothing asks for what only the MFMA form does (a bias, the norm
// statistics hand-off, merged attention partials, more than kRdMaxC values). It is the faster one at every width measured, from 512
// (c_proj 4.6 us for 6.5) to 13,824; products of narrower rows or less than 512 x 512 are a launch's latency in both.
static bool rowdot_takes(int am, int ep, const GemvParams& p) {
  return p.M == 1 && !p.apart && !p.nstat && !p.nstat_out && !p.bias && p.K <= kRdMaxC && p.K >= 512 && (long)p.N * p.K >= 512 * 512 && p.N % 2 == 0 && am != AM_SNORM &&
         (ep == EP_STORE || ep == EP_RESID || p.norm_w) && !(ep == EP_RESID && p.norm_w) &&
         (((uintptr_t)p.A | (uintptr_t)p.W | (uintptr_t)p.W2 | (uintptr_t)p.norm_w) & 15) == 0;
}

int gemv_launch_bf16(int am, int ep, const GemvParams& p, hipStream_t s) {
  if (!rowdot_takes(am, ep, p)) return launch_fmt<WF_BF16>(am, ep, p, s);
  RowDotParams r{};
  r.A = p.A; r.w = p.norm_w; r.eps = p.eps; r.K = r.C = p.K; r.N = ep == EP_SWIGLU ? 2 * p.N : p.N;
  r.W = (const bf16_t*)p.W; r.W2 = (const bf16_t*)p.W2; r.out = ep == EP_QKV ? p.q_out : p.C;
  r.kcache = p.kcache; r.vcache = p.vcache; r.rope = p.rope; r.pos = p.pos; r.n_head = p.n_head; r.hs = p.head_size;
  r.ring = p.S; r.T = p.T; r.m = p.m0;
  switch (ep) {
    case EP_STORE: return p.norm_w ? rowdot_launch<RD_NORM, RD_STORE>(r, s) : rowdot_launch<RD_PLAIN, RD_STORE>(r, s);
    case EP_RESID: return rowdot_launch<RD_PLAIN, RD_RESID>(r, s);
    case EP_QKV: return rowdot_launch<RD_NORM, RD_QKV>(r, s);
    case EP_SWIGLU: return rowdot_launch<RD_NORM, RD_SWIGLU>(r, s);
  }
  return LLJ_EINVAL;
}
}  // namespace llj

using namespace llj;

extern "C" {
LLJ_TRACE_EXPORT(bf16)

int llj_sums_swiglu(const void* x, const float* parts, int nparts, void* x_out, const void* norm_w, float eps, const void* W1, const void* W2, void* h,
                    int H, int C, void* stream) {
  LLJ_REQUIRE(x && parts && nparts >= 1 && nparts <= kRdSums && x_out && x_out != x && norm_w && W1 && W2 && h && H > 0 && C > 0 && C % 8 == 0 && C <= 1024 &&
              (((uintptr_t)x | (uintptr_t)parts | (uintptr_t)norm_w | (uintptr_t)W1 | (uintptr_t)W2) & 15) == 0 && ((uintptr_t)x_out & 3) == 0);
  RowDotParams r{};
  r.A = (const bf16_t*)x; r.parts = parts; r.S = nparts; r.ao = (bf16_t*)x_out; r.w = (const bf16_t*)norm_w; r.eps = eps; r.K = r.C = C; r.N = 2 * H;
  r.W = (const bf16_t*)W1; r.W2 = (const bf16_t*)W2; r.out = (bf16_t*)h;
  if (nparts <= 8) return rowdot_go<2, 1, RD_SUMS + 8, RD_SWIGLU>(r, (hipStream_t)stream);
  if (nparts <= 10) return rowdot_go<2, 1, RD_SUMS + 10, RD_SWIGLU>(r, (hipStream_t)stream);
  return rowdot_go<2, 1, RD_SUMS + kRdSums, RD_SWIGLU>(r, (hipStream_t)stream);
}
}
