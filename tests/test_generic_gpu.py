"""The any-shape path (csrc/generic.hip via LLaMA._blocks_generic / _head): configurations outside
the streaming kernels' tiling, which the reference runs and the fast path cannot --
  * the JA fork's own 125M (n_layer 12, n_head 10, n_embd 780: head 78, n_hidden 2304, vocab 35000;
    reference lit_llama/model.py:48-51);
  * the reference test's n_embd 32 / n_head 16 (head 2), 16 layers, block 64
    (reference tests/test_model.py:108-112, test_bfloat16_llama_init).
Logits against the oracle on the same weights, prefill rows and teacher-forced decode steps, bf16
weights and gptq.int4 (the ColBlockQuantizedLinear buffers used as stored, no repack).

Tolerance, as in tests/test_model_7b_gpu.py: twice the measured bf16 noise floor, i.e. the oracle
against ITSELF with its Linears / RMSNorm means summed in another valid order, on these very weights,
ids and steps (tools/noise_floor.py --generic, profiles/r03_noise_floor_generic.json). Deeper models
carry more of it than the 2-layer width tests: n_embd 32 x 16 layers floor max 2.87e-2 / mean
2.9e-3; 125M (12 layers) max 1.71e-2 (bf16) / 1.88e-2 (int4), mean <= 1.56e-2. Every row / step is
held to 2x the max and the mean over rows to 2x the floor mean."""
import math

import numpy as np
import pytest
import torch

from oracle import llama_np as O
from oracle.weights import Cfg, make_params
from tests.test_model_7b_gpu import _check, _gpu_steps, _oracle_steps, oracle_linears

pytestmark = pytest.mark.gpu

REF_TEST = Cfg(block_size=64, vocab_size=32000, n_layer=16, n_head=16, n_embd=32)
C125 = Cfg(block_size=128, n_layer=12, n_head=10, n_embd=780, vocab_size=35000)
# (max per row, mean over rows): 2x profiles/r03_noise_floor_generic.json
TOL_REF_TEST = (5.8e-2, 5.8e-3)
TOL_125M = (3.8e-2, 3.2e-2)
# llm.int8 re-quantizes every Linear input per row, so the same flips move whole int8 steps: floor max
# 3.12e-2 / mean 2.16e-2 (profiles/r04_noise_floor_generic.json, with the GPU-formula variant)
TOL_125M_I8 = (6.3e-2, 4.4e-2)


def _check_mean(got, ref, tol, what):
    worst = _check(got, ref, tol[0], what)
    B, n = got.shape[:2]
    mean = float(np.mean([np.linalg.norm(got[b, s] - ref[b, s]) / np.linalg.norm(ref[b, s])
                          for b in range(B) for s in range(n)]))
    assert mean < tol[1], f"{what}: mean rel err {mean:.3e}"
    return worst


def _setup(cfg: Cfg, mode, seed):
    from lit_llama import LLaMA, LLaMAConfig
    from lit_llama.utils import EmptyInitOnDevice

    pb, sd, lin = oracle_linears(make_params(cfg, seed), mode)
    with EmptyInitOnDevice(device=torch.device("cuda"), dtype=torch.bfloat16, quantization_mode=mode):
        m = LLaMA(LLaMAConfig(block_size=cfg.block_size, vocab_size=cfg.vocab_size, n_layer=cfg.n_layer,
                              n_head=cfg.n_head, n_embd=cfg.n_embd))
    m.load_state_dict({k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in sd.items()})
    assert m._generic(), "this config should take the any-shape path"
    return m.eval(), O.OracleLLaMA(cfg, pb, linears=lin, act_bf16=True)


def test_reference_test_config_no_cache_vs_oracle():
    """The reference test's model (n_embd 32, head 2, 16 layers) at its batch 3 x 64 tokens,
    no-cache forward (all rows); then the cache path gives the same logits."""
    m, orc = _setup(REF_TEST, None, 32)
    idx = np.random.default_rng(3).integers(0, REF_TEST.vocab_size, (3, 64))
    out = m(torch.from_numpy(idx).cuda()).float().cpu().numpy()
    ref = orc.forward(idx)
    _check_mean(out, ref, TOL_REF_TEST, "ref-test config no-cache")
    m.reset_cache()
    out2 = m(torch.from_numpy(idx).cuda(), 64, torch.arange(64).cuda()).float().cpu().numpy()
    np.testing.assert_allclose(out2, out, rtol=0, atol=1e-6)


@pytest.mark.parametrize("mode", [None, "gptq.int4", "llm.int8"])
def test_125m_prefill_and_decode_vs_oracle(mode):
    """125M: a 12-token prompt (every row) then 4 teacher-forced decode steps, batch 2. llm.int8:
    Linear8bitLt at K = 780 / 2304 on the any-shape LLM.int8 kernels (llj_g_i8_linear)."""
    m, orc = _setup(C125, mode, 125)
    ids = np.random.default_rng(12).integers(3, C125.vocab_size, (2, 12 + 5))
    got, got_rows = _gpu_steps(m, ids, t_prompt=12, steps=4, s=32, all_rows=True)
    ref, ref_rows = _oracle_steps(orc, ids, t_prompt=12, steps=4, s=32, all_rows=True)
    tol = TOL_125M_I8 if mode == "llm.int8" else TOL_125M
    _check_mean(got_rows, ref_rows, tol, f"125M {mode} prompt rows")
    _check_mean(got, ref, tol, f"125M {mode} steps")


def test_125m_generate_graph_matches_eager_and_wraps():
    """generate() on 125M (greedy, the captured decode graph on the any-shape kernels): the same ids
    as a decode session stepped eagerly, past a ring wrap (max_seq_length 16 < 8 + 20 tokens)."""
    from lit_llama.engine import DecodeSession

    m, _ = _setup(C125, "gptq.int4", 7)
    prompt = torch.from_numpy(np.random.default_rng(5).integers(3, C125.vocab_size, 8)).cuda()
    outs = []
    for graph in (True, False):
        s = DecodeSession(m, 1, 16, 28, use_graph=graph)
        s.prefill(prompt.view(1, -1))
        s.decode(19)
        outs.append(s.output()[0].cpu().numpy())
    np.testing.assert_array_equal(outs[0], outs[1])
    assert outs[0].shape == (28,) and ((outs[0] >= 0) & (outs[0] < C125.vocab_size + 64)).all()


@pytest.mark.parametrize("odd", ["keys", "values"])
def test_decode_over_caches_at_odd_places(odd):
    """Caches that the caller laid out, starting at an odd element (decode rows on the fused launch read pairs): the same logits
    as over the model's own, to the rounding of the separate launches."""
    m, _ = _setup(REF_TEST, None, 9)
    ids = torch.from_numpy(np.random.default_rng(4).integers(0, REF_TEST.vocab_size, (2, 9))).cuda()
    outs = []
    for own in (True, False):
        m.reset_cache()
        if not own:
            for k, v in m._alloc_kv(2, 16, ids.device):
                at = torch.zeros(k.numel() + 1, dtype=k.dtype, device=k.device)[1:].view(k.shape)
                m.kv_caches.append((at, v) if odd == "keys" else (k, at))
        m(ids[:, :8], 16, torch.arange(8).cuda())
        outs.append(m(ids[:, 8:], 16, torch.tensor([8]).cuda()).float())
    m.reset_cache()
    assert float((outs[0] - outs[1]).norm() / outs[0].norm()) < 2e-2


def test_decode_on_a_device_full_of_cached_blocks(monkeypatch):
    """A step that allocates where everything the process may use lies in the allocator's cache (after a large prompt): the capture
    makes room, and the tokens are those of eager steps."""
    from lit_llama.engine import DecodeSession

    m, _ = _setup(REF_TEST, None, 7)
    prompt = torch.from_numpy(np.random.default_rng(5).integers(3, REF_TEST.vocab_size, (2, 8))).cuda()
    plain, attempts = DecodeSession._step, []

    def step(self):
        attempts.append(1)
        room = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")  # (a step's own buffers)
        plain(self)
        del room

    monkeypatch.setattr(DecodeSession, "_step", step)
    outs = []
    try:
        for graph in (False, True):
            s = DecodeSession(m, 2, 32, 32, use_graph=graph)
            s.prefill(prompt)
            if graph:
                torch.cuda.empty_cache()
                full = torch.empty(256 << 20, dtype=torch.uint8, device="cuda")
                del full
                total = torch.cuda.get_device_properties(0).total_memory
                torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (16 << 20)) / total)
                attempts.clear()
            s.decode(12)
            outs.append(s.output().cpu().numpy())
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert len(attempts) == 2  # captured at the second attempt, then replayed
    np.testing.assert_array_equal(outs[0], outs[1])


def test_generic_linear_grouped_int8_codes_vs_numpy():
    """llj_g_linear on ColBlock bits=8 codes with groups (tile_cols 256 over K 780 -> 4 groups, the
    last partial) and the residual form, against numpy (q - z) * s in fp32."""
    from lit_llama import _hip

    rng = np.random.default_rng(1)
    M, K, N, g = 5, 780, 36, 256
    G = (K + g - 1) // g
    q = rng.integers(0, 256, (N, K)).astype(np.uint8)
    sc = (rng.random((N, G)) * 0.01 + 0.001).astype(np.float32)
    zr = rng.integers(100, 156, (N, G)).astype(np.float32)
    x = O.bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    res = O.bf16_round(rng.standard_normal((M, N)).astype(np.float32))
    Wd = (q.astype(np.float32) - np.repeat(zr, g, 1)[:, :K]) * np.repeat(sc, g, 1)[:, :K]
    ref = O.bf16_round(res + O.bf16_round(x @ Wd.T))
    dev = torch.device("cuda")
    qw = torch.from_numpy(q.T.copy()).to(dev)  # column-major (N, K) bytes: byte (n, k) at k*N + n
    xt = torch.from_numpy(x).to(dev).to(torch.bfloat16)
    y = torch.from_numpy(res).to(dev).to(torch.bfloat16)
    sct, zrt = torch.from_numpy(sc).to(dev), torch.from_numpy(zr).to(dev)
    _hip.call("llj_g_linear", 0, xt.data_ptr(), K, M, K, qw.data_ptr(), sct.data_ptr(), zrt.data_ptr(), 8, g, N,
              y.data_ptr(), N, y.data_ptr(), N, 0, _hip.stream())
    got = y.float().cpu().numpy()
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"[generic] grouped int8 linear + residual: max err {err:.2e} of max|y|")
    assert err < 1e-2


@pytest.mark.parametrize("outliers", [0, 5, 200])
@pytest.mark.parametrize("M,K,N", [(1, 780, 2340), (7, 2304, 780), (40, 780, 36)])
def test_generic_int8_linear_vs_oracle(M, K, N, outliers):
    """llj_g_i8_linear (LLM.int8 for K % 128 != 0: the 125M's 780 / 2304) against the oracle's
    restatement of bitsandbytes' MatMul8bitLt (parity unpinned: bitsandbytes is absent), with and
    without outlier columns, plain and with the residual add."""
    from lit_llama import _hip
    from tests.helpers import assert_bf16_close

    rng = np.random.default_rng(M + K + outliers)
    W = O.bf16_round((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    cb, scb = O.int8_quantize_weight(W)
    x = rng.standard_normal((M, K)).astype(np.float32)
    if outliers:
        x[:, rng.choice(K, outliers, replace=False)] *= 25.0
    x = O.bf16_round(x)
    res = O.bf16_round(rng.standard_normal((M, N)).astype(np.float32))
    dev = torch.device("cuda")
    xt = torch.from_numpy(x).to(dev).to(torch.bfloat16)
    cbt, scbt = torch.from_numpy(cb).to(dev), torch.from_numpy(scb).to(dev)
    ws = torch.empty(_hip.lib().llj_g_i8_ws_bytes(M, K), dtype=torch.uint8, device=dev)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    yr = torch.from_numpy(res).to(dev).to(torch.bfloat16)
    _hip.call("llj_g_i8_linear", xt.data_ptr(), K, M, K, cbt.data_ptr(), scbt.data_ptr(), 6.0, ws.data_ptr(), N,
              y.data_ptr(), N, None, 0, 0, _hip.stream())
    _hip.call("llj_g_i8_linear", xt.data_ptr(), K, M, K, cbt.data_ptr(), scbt.data_ptr(), 6.0, ws.data_ptr(), N,
              yr.data_ptr(), N, yr.data_ptr(), N, 0, _hip.stream())
    ref = O.int8_linear(x, cb, scb)
    assert_bf16_close(y.float().cpu().numpy(), ref, f"generic int8 M={M} K={K} outliers={outliers}", rel=1e-2)
    assert_bf16_close(yr.float().cpu().numpy(), O.bf16_round(res + O.bf16_round(ref)), "generic int8 resid", rel=1e-2)
    # fp32 activations (a float32 model under llm.int8): f16(x) in, the fp16 result back as fp32
    x32 = x + O.bf16_round(rng.standard_normal((M, K)).astype(np.float32) * 1e-3)  # not bf16-representable
    xt32 = torch.from_numpy(x32).to(dev)
    y32 = torch.empty(M, N, dtype=torch.float32, device=dev)
    r32 = torch.from_numpy(res).to(dev)
    _hip.call("llj_g_i8_linear", xt32.data_ptr(), K, M, K, cbt.data_ptr(), scbt.data_ptr(), 6.0, ws.data_ptr(), N,
              y32.data_ptr(), N, None, 0, 1, _hip.stream())
    yr32 = r32.clone()
    _hip.call("llj_g_i8_linear", xt32.data_ptr(), K, M, K, cbt.data_ptr(), scbt.data_ptr(), 6.0, ws.data_ptr(), N,
              yr32.data_ptr(), N, yr32.data_ptr(), N, 1, _hip.stream())
    ref32 = O.int8_linear(x32, cb, scb)
    got = y32.cpu().numpy()
    assert np.array_equal(got, got.astype(np.float16).astype(np.float32))  # fp16 values, cast back
    err = np.abs(got - ref32)
    assert (err <= 2e-3 * np.abs(ref32) + 1e-3 * np.abs(ref32).max()).all(), err.max()
    np.testing.assert_allclose(yr32.cpu().numpy(), res + got, rtol=0, atol=1e-6)


# ---- matrix products of more than 8 rows (generic_gemm.h)
def _g_linear_operands(kind, bits, group, dt, M, K, N, ldx, seed):
    rng = np.random.default_rng(seed)
    dtype = torch.float32 if dt else torch.bfloat16
    buf = torch.from_numpy(rng.standard_normal(M * ldx + 1).astype(np.float32)).cuda().to(dtype)
    G = -(-K // group)
    if kind == 1:
        w = torch.from_numpy(rng.standard_normal((N, K)).astype(np.float32)).cuda().to(dtype)
        return buf, w, None, None, w.double()
    q = torch.from_numpy(rng.integers(0, 1 << bits, (N, K)).astype(np.uint8)).cuda()
    sc = torch.from_numpy((rng.random((N, G)) * 0.01 + 0.001).astype(np.float32)).cuda()
    zr = torch.from_numpy(rng.integers(0, 1 << bits, (N, G)).astype(np.float32)).cuda()
    epb = 8 // bits
    packed = sum(q[:, r::epb].int() << (r * bits) for r in range(epb)).to(torch.uint8).t().contiguous()
    cols = torch.arange(K, device="cuda") // group
    return buf, packed, sc, zr, (q.double() - zr[:, cols].double()) * sc[:, cols].double()


@pytest.mark.parametrize("kind,bits", [(1, 16), (0, 4), (0, 8)])
def test_generic_gemm_fp32_halves_need_no_scratch(kind, bits):
    """fp32, short K: the sums of the two halves of K are kept apart inside one workgroup (the same bits as the two halves' own
    products, 7 tiles each, added), so large outputs take no scratch: twice the output's size for a head's logits otherwise."""
    from lit_llama import _hip

    for M in (1000, 2048, 16384):
        assert _hip.lib().llj_g_linear_ws_bytes(kind, M, 35008, 780, 1) == 0
    M, N, K, group = 77, 300, 448, 32
    buf, w, sc, zr, _ = _g_linear_operands(kind, bits, group, 1, M, K, N, K, 5)
    x = buf[:M * K].view(M, K)

    def product(a, w, sc, zr):
        y = torch.empty(M, N, device="cuda")
        _hip.call("llj_g_linear", kind, a.data_ptr(), a.stride(0), M, a.shape[1], w.data_ptr(), _hip.ptr(sc), _hip.ptr(zr), bits, group, N,
                  y.data_ptr(), N, None, 0, 1, _hip.stream())
        return y

    half = []
    for lo, hi in ((0, 224), (224, 448)):
        ww = w[:, lo:hi] if kind == 1 else w[lo * bits // 8:hi * bits // 8]
        s = (None, None) if kind == 1 else (sc[:, lo // group:hi // group].contiguous(), zr[:, lo // group:hi // group].contiguous())
        half.append(product(x[:, lo:hi], ww.contiguous(), *s))
    assert torch.equal(product(x, w, sc, zr), half[0] + half[1])


@pytest.mark.parametrize("kind,bits,group", [(1, 16, 0), (0, 2, 0), (0, 4, 0), (0, 8, 0), (0, 4, 100)])
@pytest.mark.parametrize("dt", [0, 1])
@pytest.mark.parametrize("M,N,K,pad,off", [(9, 1, 4, 0, 0), (9, 127, 32, 0, 0), (64, 128, 36, 4, 0), (65, 129, 780, 0, 0),
                                           (129, 255, 1028, 1, 1), (33, 780, 2304, 8, 0), (70, 36, 4100, 0, 1)])
def test_generic_gemm_edges_vs_float64(kind, bits, group, dt, M, N, K, pad, off):
    """Partial tiles, the K tail, loads of 16 / 8 / 4 / 2 bytes (strides and pointers off the alignment), the K split, groups,
    and the residual in place. Bound: fp32 sums over chains of at most 32, 8, K / 128 and 16 (splits) terms lose half an
    ulp of sum |x w| per term; a weight element from codes two more; bf16 results (8 significant bits) round by 2^-8, once more with the
    residual."""
    from lit_llama import _hip

    group = group or K
    ldx = K + pad
    buf, w, sc, zr, w64 = _g_linear_operands(kind, bits, group, dt, M, K, N, ldx, M * N + K)
    x = buf[off:off + M * ldx].view(M, ldx)
    x64 = x[:, :K].double()
    res = torch.randn(M, N, device="cuda", generator=torch.Generator("cuda").manual_seed(K)).to(x.dtype)
    want, mass = x64 @ w64.T, x64.abs() @ w64.abs().T
    bound = mass * 2.0 ** -24 * (32 + 8 + K // 128 + 16 + 4)
    half = 0.0 if dt else 2.0 ** -8 * 1.01
    for resid in (None, res):
        ref = want if resid is None else want + resid.double()
        lim = bound + half * want.abs() + (0.0 if resid is None else (half + 2.0 ** -24) * (ref.abs() + half * want.abs()))
        y = torch.empty(M, N, dtype=x.dtype, device="cuda") if resid is None else resid.clone()
        _hip.g_linear(kind, x, M, K, w, sc, zr, bits, group, N, y, None if resid is None else y, dt, _hip.stream())
        one = torch.empty_like(y) if resid is None else resid.clone()
        _hip.call("llj_g_linear", kind, x.data_ptr(), ldx, M, K, w.data_ptr(), _hip.ptr(sc), _hip.ptr(zr), bits, group, N,
                  one.data_ptr(), N, None if resid is None else one.data_ptr(), 0 if resid is None else N, dt, _hip.stream())
        for got in (y, one):
            bad = (got.double() - ref).abs() > lim + 1e-30
            assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside the bound"


@pytest.mark.parametrize("M,N,K,pad,ws", [
    (9, 1, 3104, 0, True), (9, 129, 3104, 4, False), (64, 128, 4096, 0, True), (65, 129, 3104, 12, True), (65, 780, 4096, 0, False),
    (301, 1000, 3104, 0, True), (37, 12288, 4096, 0, True), (301, 13200, 3104, 4, False), (513, 11000, 3104, 0, False),
    (64, 16500, 3072, 0, False), (70, 256, 32 * 113, 0, True), (1000, 7900, 3104, 0, False), (301, 5000, 3104, 4, True),
    (33, 1100, 800, 0, True), (33, 4100, 780, 4, True), (100, 6000, 780, 0, True), (65, 11008, 800, 4, True), (384, 2304, 780, 0, True),
    (301, 4096, 4100, 0, True), (90, 8200, 3108, 0, True), (70, 12288, 780, 0, False), (40, 500, 288, 0, False), (20, 2000, 260, 8, False),
    (9, 1100, 36, 0, False)])
def test_generic_gemm_direct_tiles_equal_staged_ones(M, N, K, pad, ws):
    """fp32 rows in 16-byte loads (K a multiple of 32, and of 4 alone) against the same product in loads from any element on (x one element off the
    alignment): the same sums bit for bit, with and without the residual in place. Tiles of every height, fewer than eight column tiles and
    more, column and row remainders, padded rows, K in ranges (32 x 113: of unequal length), in one piece and in halves, one tile, odd and even
    counts of them."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(M + N + K)
    ldx = K + pad
    w, res = torch.randn(N, K, device="cuda", generator=g), torch.randn(M, N, device="cuda", generator=g)
    x = torch.randn(M, K, device="cuda", generator=g)
    rows = []
    for off in (0, 1):
        buf = torch.full((M * ldx + 4,), float("nan"), device="cuda")
        rows.append(buf[off:off + M * ldx].view(M, ldx))
        rows[-1][:, :K] = x
    nbytes = _hip.lib().llj_g_linear_ws_bytes(1, M, N, K, 1) if ws else 0
    scratch = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
    for resid in (False, True):
        outs = []
        for r in rows:
            y = res.clone() if resid else torch.full_like(res, float("nan"))
            _hip.call("llj_g_linear_ws", 1, r.data_ptr(), ldx, M, K, w.data_ptr(), None, None, 16, K, N, y.data_ptr(), N,
                      y.data_ptr() if resid else None, N if resid else 0, 1, scratch.data_ptr() if nbytes else None, nbytes, _hip.stream())
            outs.append(y)
        assert torch.equal(*outs)
        if M * N < 200000:  # (the bound of the test above)
            want, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
            ref = want + res.double() if resid else want
            lim = mass * 2.0 ** -24 * (32 + 8 + K // 128 + 16 + 4) + (2.0 ** -24 * ref.abs() if resid else 0.0)
            assert ((outs[0].double() - ref).abs() <= lim + 1e-30).all()


@pytest.mark.parametrize("M", [9, 17, 40, 64, 80, 96, 100])
@pytest.mark.parametrize("N,K,off", [(260, 3104, 0), (260, 3104, 1), (1200, 1028, 0), (130, 775, 1), (9, 40, 0)])
def test_generic_gemm_fp32_sums_and_values_out_of_range(M, N, K, off):
    """fp32 products as sums of bf16 ones, all three kinds of loads (every height of a tile: the tests below). Rows of ordinary values are as near to
    float64 as fp32 sums (the 2-norm of half an ulp for the result and one for the sums of a tile, of eight and of the rest); infinities, NaN, values that
    round to infinity in bf16, large and very small ones give what fp32 sums give: non-finite outputs where float64 has them, the bound of the tests
    above where no partial sum can overflow."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(M + N + K)
    x = torch.randn(M * K + 1, device="cuda", generator=g)[off:off + M * K].view(M, K)
    w = torch.randn(N, K, device="cuda", generator=g)

    def product():
        y = torch.empty(M, N, device="cuda")
        _hip.g_linear(1, x, M, K, w, None, None, 16, K, N, y, None, 1, _hip.stream())
        return y.double()

    want = x.double() @ w.double().T
    assert ((product() - want).norm() / want.norm()).item() < 2.0 ** -24 * (0.5 + 3 * 0.5)
    x[1, 5], x[2, 7], x[3, K - 1], w[7, 5], w[8, 3] = math.inf, -math.inf, math.nan, 0.0, math.inf
    x[4] *= 1e34
    x[5, 2], w[:, 2] = 3.4e38, 1.2e-38 * torch.sign(w[:, 2])  # above bf16's largest, the products 4
    x[6] *= 1e-30
    want, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    got = product()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    safe = mass < 1e38
    lim = mass * 2.0 ** -24 * (32 + 8 + K // 128 + 16 + 4)
    assert safe[0, :7].all() and safe[4:7, :7].all() and ((got - want).abs()[safe] <= lim[safe]).all()


# (rows, columns, K, K ranges): tiles of 16, 32 .. 96 rows in this order, then K in one piece (its halves kept apart at 780), then longer sums. The
# ranges are asserted: a plan that chooses others has other heights as well, and shapes for it are to be looked for
GEMM_HEIGHTS = [(9, 260, 800, 13), (9, 260, 780, 13), (33, 1100, 800, 13), (33, 1100, 780, 13), (33, 4100, 800, 9), (33, 4100, 780, 9),
                (100, 6000, 800, 5), (100, 6000, 780, 5), (65, 11008, 800, 5), (65, 11008, 780, 5), (384, 2304, 800, 5), (384, 2304, 780, 5),
                (70, 12288, 780, 1), (301, 11008, 800, 1), (301, 12288, 4096, 1), (301, 4096, 4096, 4), (90, 8200, 3108, 7)]


def _gemm_heights_operands(M, N, K, ranges, off):
    """fp32 x (M, K), `off` elements past an aligned address, w (N, K), a call of their product."""
    from lit_llama import _hip

    assert _hip.lib().llj_g_linear_ws_bytes(1, M, N, K, 1) == (ranges * M * N * 4 if ranges > 1 else 0)
    g = torch.Generator("cuda").manual_seed(M + N + K)
    x = torch.randn(M * K + 1, device="cuda", generator=g)[off:off + M * K].view(M, K)
    w = torch.randn(N, K, device="cuda", generator=g)

    def product():
        y = torch.full((M, N), math.nan, device="cuda")
        _hip.g_linear(1, x, M, K, w, None, None, 16, K, N, y, None, 1, _hip.stream())
        return y.double()

    return x, w, product


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("M,N,K,ranges", GEMM_HEIGHTS)
def test_generic_gemm_fp32_outputs_formed_again(M, N, K, ranges, off):
    """Finite values that bf16 parts cannot hold (3.4e38, times weights of 1e-38, and the other way round) and infinities, the last one in
    W's last element (whose place past K is read with x's zeros). Bound of the finite outputs in the 2-norm: random roundings of 2^-24 / sqrt(3), for
    the 8 values of a chain 4.5 of them, the pairs 2, eight of these 4.5 and the rest of K / 256 half as many."""
    x, w, product = _gemm_heights_operands(M, N, K, ranges, off)
    x[::2, 3], w[::3, K - 2] = 3.4e38, -3.4e38
    w[:, 3], x[:, K - 2] = 1.2e-38 * torch.sign(w[:, 3]), 1.2e-38 * torch.sign(x[:, K - 2])
    bound = 2.0 ** -24 / 3 ** 0.5 * (11 + (K / 256 + 1) / 2) ** 0.5
    for step in range(2):
        want, got = x.double() @ w.double().T, product()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        for rows, cols in ((slice(0, None, 2), slice(None)), (slice(1, None, 2), slice(0, None, 3)), (slice(1, None, 2), slice(1, None, 3))):
            a, b = got[rows, cols], want[rows, cols]
            fin = torch.isfinite(b)
            assert fin.all() if step == 0 else fin.any()
            assert (((a - b)[fin].norm() / b[fin].norm()).item()) < bound
        x[1, 0], x[2, 7], w[5, K - 1] = math.nan, -math.inf, math.inf


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("M,N,K,ranges", GEMM_HEIGHTS)
def test_generic_gemm_fp32_small_values(M, N, K, ranges, off):
    """Operands down to fp32's smallest: as near to float64 as ordinary ones (the 2-norm of half an ulp for the result and one for the sums of a tile,
    of eight and of the rest)."""
    x, w, product = _gemm_heights_operands(M, N, K, ranges, off)
    x0, w0 = x.clone(), w.clone()
    for a, b in ((1.0, 1.0), (1e-34, 1.0), (1e-36, 1.0), (1.0, 1e-37), (1e-18, 1e-18), (1e-41, 1e11), (1e12, 1e-42)):
        x.copy_(x0 * a), w.copy_(w0 * b)
        want = x.double() @ w.double().T
        assert ((product() - want).norm() / want.norm()).item() < 2.0 ** -24 * (0.5 + 3 * 0.5), (a, b)


@pytest.mark.parametrize("M,N,K", [(29, 1, 512), (10, 8, 512), (256, 1, 700), (128, 2, 4096), (18, 14, 3109), (15, 17, 1030), (13, 20, 310), (9, 28, 96),
                                   (64, 130, 17), (70, 300, 1), (33, 129, 63)])
@pytest.mark.parametrize("off", [0, 1])
def test_generic_gemm_fp32_small_outputs(M, N, K, off):
    """K in ranges of one tile and of several whose sums fit one workgroup of the second launch (all on its XCD: up to 256 outputs) and just do not, and
    K of a tile's part, whole and one more; the residual in place, nothing outside the output. Bound as in the first test."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(M + N + K)
    x = torch.randn(M * K + 1, device="cuda", generator=g)[off:off + M * K].view(M, K)
    w, res = torch.randn(N, K, device="cuda", generator=g), torch.randn(M, N, device="cuda", generator=g)
    want, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    lim = mass * 2.0 ** -24 * (32 + 8 + K // 128 + 16 + 4)
    for resid in (False, True):
        buf = torch.full((M + 1, N + 3), 7.0, device="cuda")
        y = buf[:M, :N]
        if resid:
            y.copy_(res)
        _hip.g_linear(1, x, M, K, w, None, None, 16, K, N, y, y if resid else None, 1, _hip.stream())
        ref = want + res.double() if resid else want
        assert ((y.double() - ref).abs() <= lim + (2.0 ** -24 * ref.abs() if resid else 0.0)).all()
        assert (buf[M] == 7.0).all() and (buf[:M, N:] == 7.0).all()


# ---- up to 8 rows (generic_rows.h)
@pytest.mark.parametrize("dt", [0, 1])
@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K,off", [(1, 1, 0), (5, 6, 0), (780, 780, 0), (36, 2304, 0), (129, 4100, 1), (8200, 260, 0), (8193, 40, 0),
                                     (70, 500, 0), (70, 700, 0), (70, 900, 0), (70, 1500, 0), (40, 5200, 0), (36, 1283, 0), (36, 1285, 1),
                                     (8200, 700, 0), (8200, 1000, 0), (8200, 701, 0), (8195, 1030, 0), (8200, 2600, 0), (8200, 3300, 0),
                                     (8200, 101, 0), (8200, 201, 0), (8195, 321, 0), (8200, 1020, 0)])
def test_generic_rows_vs_float64_and_fused_forms(dt, M, N, K, off):
    """Rows of x at and off the loads' alignment, columns in ones and fours, K of 1 to 8 pieces a round and of several rounds, K tails, the
    residual in place. Bound: a lane
    sums ceil(K / 64) + 7 products, six more additions over the lanes, half an ulp of sum |x w| each; bf16 as above. The
    norm-fused forms give bitwise what the separate calls give: the same sums in the same order."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(M * N + K)
    dtype = torch.float32 if dt else torch.bfloat16
    x = torch.randn(M * K + 1, device="cuda", generator=g).to(dtype)[off:off + M * K].view(M, K)
    w, w2 = (torch.randn(N, K, device="cuda", generator=g).to(dtype) for _ in range(2))
    nw = (1 + 0.1 * torch.randn(K, device="cuda", generator=g)).to(dtype)
    res = torch.randn(M, N, device="cuda", generator=g).to(dtype)
    want, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    half = 0.0 if dt else 2.0 ** -8 * 1.01
    st = _hip.stream()
    for resid in (None, res):
        ref = want if resid is None else want + resid.double()
        lim = mass * 2.0 ** -24 * (K // 64 + 14) + half * want.abs()
        lim = lim if resid is None else lim + (half + 2.0 ** -24) * (ref.abs() + half * want.abs())
        y = torch.empty_like(res) if resid is None else resid.clone()
        _hip.g_linear(1, x, M, K, w, None, None, 16, K, N, y, None if resid is None else y, dt, st)
        assert ((y.double() - ref).abs() <= lim + 1e-30).all()
    assert _hip.lib().llj_g_norm_ok(M, K, dt) == (M * K * (4 if dt else 2) <= 48 * 1024)
    if not _hip.lib().llj_g_norm_ok(M, K, dt):
        return
    xn, one, two, sep = torch.empty(M, K, dtype=dtype, device="cuda"), *(torch.empty_like(res) for _ in range(3))
    _hip.call("llj_g_rmsnorm", x.data_ptr(), K, nw.data_ptr(), 1e-5, xn.data_ptr(), K, M, K, dt, st)
    _hip.g_linear(1, xn, M, K, w, None, None, 16, K, N, one, None, dt, st)
    _hip.g_linear(1, xn, M, K, w2, None, None, 16, K, N, two, None, dt, st)
    fused = torch.empty_like(one)
    _hip.call("llj_g_norm_linear", x.data_ptr(), K, nw.data_ptr(), 1e-5, M, K, w.data_ptr(), N, fused.data_ptr(), N, dt, st)
    assert torch.equal(fused, one)
    _hip.call("llj_g_silu_mul", one.data_ptr(), two.data_ptr(), sep.data_ptr(), M * N, dt, st)
    _hip.call("llj_g_norm_swiglu", x.data_ptr(), K, nw.data_ptr(), 1e-5, M, K, w.data_ptr(), w2.data_ptr(), N, fused.data_ptr(), N,
              dt, st)
    assert torch.equal(fused, sep)


@pytest.mark.parametrize("dt", [0, 1])
@pytest.mark.parametrize("B,nh,hs,S,p", [(1, 10, 78, 132, 0), (3, 10, 78, 132, 131), (2, 2, 2, 16, 40), (1, 3, 64, 300, 17),
                                         (8, 2, 128, 1000, 999), (1, 1, 600, 40, 20), (1, 1, 1100, 40, 39), (1, 5, 32, 40, 10),
                                         (2, 3, 34, 50, 49), (1, 2, 96, 200, 150), (33, 8, 16, 20, 7), (26, 10, 78, 132, 131), (13, 20, 128, 64, 100),
                                         (300, 1, 66, 30, 0)])
def test_generic_rope_attention_vs_separate_calls(dt, B, nh, hs, S, p):
    """First position, a full cache, a wrapped ring, head sizes from one pair to more pairs than threads, few and many (more than
    256) rows and heads: the caches bitwise as
    llj_g_rope_kv leaves them, the output against attention in float64 over them. Bound: scores and weighted sums
    lose half an ulp per term of hs and S (exp: 2 more), relative to sum |p v|; bf16 results round by 2^-8."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(B * S + p)
    dtype, C, st = torch.float32 if dt else torch.bfloat16, nh * hs, _hip.stream()
    qkv = torch.randn(B, 3 * C, device="cuda", generator=g).to(dtype)
    kc, vc = (torch.randn(B, nh, S, hs, device="cuda", generator=g).to(dtype) for _ in range(2))
    ang = torch.rand(p + 1, hs // 2, device="cuda", generator=g) * 6
    rope = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    pos = torch.tensor([p], dtype=torch.int32, device="cuda")
    k2, v2, q, y = kc.clone(), vc.clone(), torch.empty(B, C, dtype=dtype, device="cuda"), torch.empty(B, C, dtype=dtype, device="cuda")
    assert _hip.lib().llj_g_rope_attention_ok(S, hs) == 1
    _hip.call("llj_g_rope_attention", qkv.data_ptr(), kc.data_ptr(), vc.data_ptr(), rope.data_ptr(), pos.data_ptr(), y.data_ptr(),
              B, C, nh, S, dt, st)
    _hip.call("llj_g_rope_kv", qkv.data_ptr(), q.data_ptr(), k2.data_ptr(), v2.data_ptr(), rope.data_ptr(), pos.data_ptr(), B, 1, C,
              nh, S, dt, st)
    assert torch.equal(kc, k2) and torch.equal(vc, v2)
    n = min(p + 1, S)
    s = (k2[:, :, :n].double() * q.view(B, nh, 1, hs).double()).sum(-1) * hs ** -0.5
    size = (k2[:, :, :n].double() * q.view(B, nh, 1, hs).double()).abs().sum(-1) * hs ** -0.5
    w = torch.softmax(s, -1)
    want, mass = ((w[..., None] * t).sum(2).reshape(B, C) for t in (v2[:, :, :n].double(), v2[:, :, :n].double().abs()))
    loss = 2.0 ** -24 * (n + 16 + 2 * (hs // 2 + 8) * float(size.max()))
    assert ((y.double() - want).abs() <= mass * loss + (0.0 if dt else 2.0 ** -8 * 1.01) * want.abs() + 1e-30).all()


@pytest.mark.parametrize("dt", [0, 1])
@pytest.mark.parametrize("B,nh,hs,S,p", [(1, 2, 78, 300, 100), (2, 3, 30, 400, 255), (1, 2, 126, 400, 256), (33, 8, 50, 200, 5), (1, 2, 66, 140, 500)])
def test_generic_rope_attention_unseen_slots(dt, B, nh, hs, S, p):
    """Slots that hold nothing yet (NaN) and the slot that the token takes (NaN before it) are no part of the result:
    the same bits as over a cache of zeros there; one pass of 128 keys, several, the last one partial, a ring that has gone round."""
    from lit_llama import _hip

    g = torch.Generator("cuda").manual_seed(p)
    dtype, C = torch.float32 if dt else torch.bfloat16, nh * hs
    qkv = torch.randn(B, 3 * C, device="cuda", generator=g).to(dtype)
    ang = torch.rand(p + 1, hs // 2, device="cuda", generator=g)
    rope, pos = torch.stack([ang.cos(), ang.sin()], -1).contiguous(), torch.tensor([p], dtype=torch.int32, device="cuda")
    kv = [torch.randn(B, nh, S, hs, device="cuda", generator=g).to(dtype) for _ in range(2)]
    outs = []
    for fill in (float("nan"), 0.0):
        k, v = (t.clone() for t in kv)
        for t in (k, v):
            t[:, :, p + 1:] = fill
            t[:, :, p % S] = fill
        y = torch.empty(B, C, dtype=dtype, device="cuda")
        _hip.call("llj_g_rope_attention", qkv.data_ptr(), k.data_ptr(), v.data_ptr(), rope.data_ptr(), pos.data_ptr(), y.data_ptr(), B, C, nh, S, dt,
                  _hip.stream())
        outs.append(y)
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,nh,hs,S,p0", [(1, 301, 32, 128, 301, 0), (2, 67, 10, 78, 80, 5), (1, 130, 8, 1, 130, 0), (3, 49, 8, 13, 64, 40),
                                            (1, 1030, 1, 256, 1030, 0), (2, 129, 5, 101, 200, 0), (1, 70, 16, 64, 72, 60), (1, 128, 9, 250, 128, 0),
                                            (1, 130, 8, 17, 130, 0), (1, 140, 8, 63, 150, 7), (1, 131, 8, 82, 131, 0), (1, 129, 8, 126, 140, 9),
                                            (1, 130, 8, 132, 130, 0), (1, 36, 32, 80, 36, 0), (4, 36, 16, 80, 40, 2), (1, 48, 22, 64, 48, 0)])
def test_prompt_attention_tiles(hip, dtype, B, T, nh, hs, S, p0):
    """llj_g_attention on tiles of 16 rows and 64 keys, any head size (also one whose vectors are too many for the tiles), remainders of
    both, rows whose positions have gone round the cache, unseen slots that hold NaN. Against float64: the output's own rounding, and in
    fp32 the scores' (values of some units, sums of hs products)."""
    from lit_llama import _hip

    g = torch.Generator(device="cuda").manual_seed(T)
    C = nh * hs
    q, k, v = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((B, T, C), (B, nh, S, hs), (B, nh, S, hs)))
    pos = torch.arange(p0, p0 + T, dtype=torch.int32, device="cuda")
    seen = (pos + 1).clamp(max=S)
    k[:, :, int(seen.max()):], v[:, :, int(seen.max()):] = float("nan"), float("nan")
    y = torch.full((B, T, C), float("nan"), dtype=dtype, device="cuda")
    _hip.call("llj_g_attention", q.data_ptr(), k.data_ptr(), v.data_ptr(), y.data_ptr(), pos.data_ptr(), B, T, C, nh, S,
              int(dtype == torch.float32), _hip.stream())
    torch.cuda.synchronize()
    mask = torch.arange(S, device="cuda")[None] < seen[:, None]
    s = q.double().view(B, T, nh, hs).transpose(1, 2).contiguous() @ k.double().nan_to_num().transpose(2, 3).contiguous() * hs ** -0.5
    want = (torch.softmax(s.masked_fill(~mask, float("-inf")), -1) @ v.double().nan_to_num()).transpose(1, 2).reshape(B, T, C)
    assert (y.double() - want).norm() <= (2e-6 if dtype == torch.float32 else 2.0 ** -8) * want.norm()


def _prompt_attention(dtype, B, T, nh, hs, S, p0, seed):
    """(q, k, v, positions, a call of llj_g_attention)."""
    from lit_llama import _hip

    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((B, T, nh * hs), (B, nh, S, hs), (B, nh, S, hs)))
    pos = torch.arange(p0, p0 + T, dtype=torch.int32, device="cuda")

    def run():
        y = torch.empty(B, T, nh * hs, dtype=dtype, device="cuda")
        _hip.call("llj_g_attention", q.data_ptr(), k.data_ptr(), v.data_ptr(), y.data_ptr(), pos.data_ptr(), B, T, nh * hs, nh, S,
                  int(dtype == torch.float32), _hip.stream())
        torch.cuda.synchronize()
        return y.view(B, T, nh, hs).transpose(1, 2)

    return q.view(B, T, nh, hs).transpose(1, 2), k, v, pos, run


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,nh,hs,dead", [(200, 8, 64, 64), (200, 8, 78, 70), (150, 8, 16, 128)])
def test_prompt_attention_first_scores_minus_infinity(hip, dtype, T, nh, hs, dead):
    """The first `dead` keys score minus infinity in every row: the rows that see a later one average the later ones."""
    q, k, v, pos, run = _prompt_attention(dtype, 1, T, nh, hs, T, 0, dead)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, :, :dead, 0] = float("-inf")
    y = run()
    assert not y[:, :, :dead].isfinite().any()  # no score but minus infinity: as a softmax of those
    s = (q.double() @ k.double().transpose(2, 3).contiguous()) * hs ** -0.5
    s = s.masked_fill(pos[None, :] > pos[:, None], float("-inf"))[:, :, dead:]
    want = torch.softmax(s, -1) @ v.double()
    assert (y[:, :, dead:].double() - want).norm() <= (2e-6 if dtype == torch.float32 else 2.0 ** -8) * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("T,nh,hs,p0,at", [(130, 8, 64, 0, 37), (130, 10, 78, 3, 64), (100, 12, 13, 0, 99), (129, 8, 200, 2, 0)])
def test_prompt_attention_values_of_later_tokens(hip, dtype, value, T, nh, hs, p0, at):
    """One value of key `at` is not finite: the rows before it give what they give without it (to the order of their sums), the rows
    that see it one output that is not finite."""
    q, k, v, pos, run = _prompt_attention(dtype, 1, T, nh, hs, T + p0, p0, at)
    want = run()
    v[0, 1, at, hs // 2] = value
    got = run()
    sees = (pos >= at).nonzero().flatten()
    assert not got[0, 1, sees, hs // 2].isfinite().any()
    got, want = got.clone(), want.clone()
    got[0, 1, sees, hs // 2] = want[0, 1, sees, hs // 2] = 0
    assert got.isfinite().all()
    assert (got.double() - want.double()).norm() <= (2e-6 if dtype == torch.float32 else 2.0 ** -8) * want.double().norm()
