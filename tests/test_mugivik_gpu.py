"""Mugivik on the device against oracle/mugivik_np.py (float64, recomputed from the first token): whole
prompts, token by token, portions, batches of unequal requests, slots used again, window edges, the first
tokens, long decoding, greedy generation. float32 models are held to rounding (5e-5 of the logits' rms),
bfloat16 ones to a few bf16 roundings per layer."""
import copy

import numpy as np
import pytest
import torch

from tests.mugivik_cases import CONFIGS, TOL, build, check, config, errors, gla, oracle, prompts, weights

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]
_cache = {}


def case(name, dtype, sharp=1.0, seed=0):
    key = (name, dtype, sharp, seed)
    if key not in _cache:
        cfg = CONFIGS[name]
        w = weights(cfg, seed, sharp=sharp)
        _cache[key] = (cfg, w, build(cfg, w, dtype))
    return _cache[key]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_whole_prompts(hip, name, dtype):
    cfg, w, m = case(name, dtype)
    for n in (1, 2, 3, 17, 64, 65, 150, 300):
        toks = prompts(cfg, [n], seed=n)[0]
        st = m.new_state(1)
        got = m.extend(st, st.alloc(1), [0], [toks])
        check(got, oracle(cfg, w, toks), dtype, (name, n))


def test_norms_off_16_bytes(hip):
    """Norm weights that are views 8 bytes into a larger buffer: few rows close them in a launch of their own, to the bits of the products that close aligned
    ones (one row: to a few roundings, its two forms add in other orders)."""
    from lit_llama.mugivik import Mugivik, MugivikConfig

    cfg = config(2048, 512, [gla(8, 64, 128), gla(8, 64, 128)], 4096)
    t = {k: torch.from_numpy(v).to("cuda", torch.bfloat16) for k, v in weights(cfg, 4).items()}
    moved = {k: torch.cat([v.new_zeros(4), v])[4:] if k.endswith((".norm1", ".norm2")) else v for k, v in t.items()}
    toks, out = prompts(cfg, [8], seed=6)[0], []
    for tensors in (t, moved):
        m = Mugivik.from_tensors(MugivikConfig.from_dict(cfg), tensors)
        assert all((w.data_ptr() % 16 != 0) == (tensors is moved) for w in m.norm1 + m.norm2)
        assert m.mlps[0].up.takes_post(2, 2048, m.norm1[0]) == (tensors is t)
        out.append([])
        for n in (1, 2, 3, 8):
            st = m.new_state(1)
            out[-1].append(m.extend(st, st.alloc(1), [0], [toks[:n]]).float())
    for a, b in list(zip(*out))[1:]:
        assert torch.equal(a, b)
    assert (out[0][0] - out[1][0]).norm() <= 2.0 ** -6 * out[0][0].norm()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_residual_after_every_layer(hip, name, dtype):
    from oracle import mugivik_np as O

    cfg, w, m = case(name, dtype)
    toks = prompts(cfg, [90], seed=5)[0]
    taps, want = [], []
    st = m.new_state(1)
    got = m.extend(st, st.alloc(1), [0], [toks], taps=taps)
    ref = O.forward(toks, cfg, w, want)
    assert len(taps) == len(want) == len(cfg["layers"])
    for i, (a, b) in enumerate(zip(taps, want)):
        assert np.abs(a.cpu().numpy() - b).max() < (5e-5 if dtype == torch.float32 else 0.1) * np.abs(b).max(), i
    check(got, ref, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_token_by_token_equals_prompt(hip, name, dtype):
    """Decode steps (the session's captured graph) from the first token on, past every window."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case(name, dtype)
    n = 160
    toks = prompts(cfg, [n], seed=2)[0]
    ref = oracle(cfg, w, toks)
    s = DecodeSession(m, 1, None, None, keep_tokens=False)
    out = [s.prefill([toks[:1]], want=[[0]]).clone()]
    for t in toks[1:]:
        out.append(s.feed([t]).clone())
    check(torch.cat(out), ref, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "tiled", "wide"])
@pytest.mark.parametrize("portion", [2, 7, 64, 100])
def test_portions(hip, name, dtype, portion):
    cfg, w, m = case(name, dtype)
    toks = prompts(cfg, [40 if portion == 2 else 210], seed=3)[0]
    ref = oracle(cfg, w, toks)
    st = m.new_state(1)
    slot = st.alloc(1)
    got = [m.extend(st, slot, [p], [toks[p:p + portion]]) for p in range(0, len(toks), portion)]
    check(torch.cat(got), ref, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "tiled", "wide"])
def test_unequal_batch_and_early_ends(hip, name, dtype):
    """Prompts of different lengths in one call, decoded together, ending one by one; the freed slots serve
    a second batch."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case(name, dtype)
    state = m.new_state(4)
    for turn in range(2):
        lens = [1, 150, 37, 70] if turn == 0 else [66, 2, 129]
        extra = [3, 9, 6, 9] if turn == 0 else [5, 12, 1]
        toks = prompts(cfg, [a + b for a, b in zip(lens, extra)], seed=10 + turn)
        refs = [oracle(cfg, w, t) for t in toks]
        s = DecodeSession(m, len(lens), None, None, state=state, keep_tokens=False)
        want = [sorted({0, n // 2, n - 1}) for n in lens]
        got = s.prefill([t[:n] for t, n in zip(toks, lens)], want=want)
        check(got, np.concatenate([r[k] for r, k in zip(refs, want)]), dtype)
        live, at, outs, wants = list(range(len(lens))), list(lens), [], []
        while live:
            outs.append(s.feed([toks[i][at[i]] for i in live]).clone())
            wants += [refs[i][at[i]] for i in live]
            for i in live:
                at[i] += 1
            done = [k for k, i in enumerate(live) if at[i] == len(toks[i])]
            if done:
                s.finish(done)
                live = [i for k, i in enumerate(live) if k not in done]
        check(torch.cat(outs), np.stack(wants), dtype)
        assert len(state._free) == 4


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch", [2, 5, 8, 11, 19, 40])
def test_batched_decode_rows(hip, dtype, batch):
    """Every batch size class of the decode kernels: rows equal their own sequences."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case("tiled", dtype)
    toks = prompts(cfg, [30 + (7 * b) % 11 for b in range(batch)], seed=batch)
    s = DecodeSession(m, batch, None, None, keep_tokens=False)
    s.prefill([t[:-3] for t in toks])
    for k in (3, 2, 1):
        out = s.feed([t[-k] for t in toks])
        want = np.stack([oracle(cfg, w, t[:len(t) - k + 1])[-1] for t in toks])
        check(out, want, dtype, k)


def _mutant(cfg, layer, delta):
    c = copy.deepcopy(cfg)
    c["layers"][layer]["mixer"]["mask"]["size"] += delta
    return c


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("layer", [1, 3])
def test_window_edges_show(hip, dtype, layer):
    """Sharp scores (single keys stand out): a window one key wider or narrower in either latent layer would
    show far above the tolerance, in prompts and in decoding."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case("tiled", dtype, sharp=6.0, seed=4)
    f = 1.5 if dtype == torch.bfloat16 else 1.0
    toks = prompts(cfg, [120], seed=6)[0]
    ref = oracle(cfg, w, toks)
    for delta in (-1, 1):
        e = errors(oracle(_mutant(cfg, layer, delta), w, toks), ref)
        assert e[0] > 2 * f * TOL[dtype][0], e
    st = m.new_state(1)
    check(m.extend(st, st.alloc(1), [0], [toks]), ref, dtype, factor=f)
    s = DecodeSession(m, 1, None, None, keep_tokens=False)
    s.prefill([toks[:10]])
    out = torch.stack([s.feed([t])[0].clone() for t in toks[10:]])
    check(out, ref[10:], dtype, factor=f)


@pytest.mark.parametrize("dtype", DTYPES)
def test_first_tokens_and_bigram_row(hip, dtype):
    """The first token takes the bigram table's last row: made large, it would show anywhere else."""
    cfg = CONFIGS["tiled"]
    w = dict(weights(cfg, 3))
    w["bigram"] = w["bigram"].copy()
    w["bigram"][-1] *= 8.0
    m = build(cfg, w, dtype)
    toks = prompts(cfg, [1, 2, 9], seed=8)
    st = m.new_state(3)
    slots = st.alloc(3)
    got = m.extend(st, slots, [0, 0, 0], toks)
    check(got, np.concatenate([oracle(cfg, w, t) for t in toks]), dtype)
    # a slot used again starts like new
    st.release(slots[1:2])
    again = st.alloc(1)
    assert again == slots[1:2]
    check(m.extend(st, again, [0], [toks[2]]), oracle(cfg, w, toks[2]), dtype)


def test_large_bigram_factors(hip):
    """Row numbers need 64-bit products."""
    cfg = config(64, 4096, [gla(1, 16, 16)], 64, buckets=1009, mul_prev=1000003, mul_cur=2147483647)
    w = weights(cfg, 1)
    m = build(cfg, w, torch.float32)
    toks = [4095, 4094, 7, 4095, 4095, 0, 4093]
    st = m.new_state(1)
    check(m.extend(st, st.alloc(1), [0], [toks]), oracle(cfg, w, toks), torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(hip, dtype):
    """Hundreds of decoded tokens with slow decays: the state neither drifts nor leaks."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case("odd", dtype)
    toks = prompts(cfg, [700], seed=9)[0]
    ref = oracle(cfg, w, toks)
    s = DecodeSession(m, 1, None, None, keep_tokens=False)
    s.prefill([toks[:50]])
    out = torch.stack([s.feed([t])[0].clone() for t in toks[50:]])
    check(out, ref[50:], dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tau", [0.25, 1.0, 64.0])
def test_decay_extremes(hip, dtype, tau):
    """Decays from almost none to (sigmoid(-30))^4 per token: nothing overflows in chunks of any size."""
    cfg = config(128, 90, [gla(2, 32, 64, tau), gla(2, 16, 32, tau)], 128)
    w = dict(weights(cfg, 2))
    for i in range(2):
        b = w[f"l{i}.mix.a2.b"] = w[f"l{i}.mix.a2.b"].copy()
        b[::3], b[1::3] = 12.0, -30.0
    m = build(cfg, w, dtype)
    toks = prompts(cfg, [260], seed=4)[0]
    st = m.new_state(1)
    slot = st.alloc(1)
    ref = oracle(cfg, w, toks)
    got = m.extend(st, slot, [0], [toks[:257]])
    assert torch.isfinite(got.float()).all()
    check(torch.cat([got, m.extend(st, slot, [257], [toks[257:]])]), ref, dtype)


def test_greedy_generation_float32(hip):
    """generate(), generate_batch() on unequal prompts and sampled sessions go through the framework's own
    loop; greedy ids equal the oracle's."""
    import generate as G

    cfg, w, m = case("tiled", torch.float32)
    toks = prompts(cfg, [23, 5, 61], seed=12)
    want = []
    for t in toks:
        t = list(t)
        for _ in range(12):
            t.append(int(oracle(cfg, w, t)[-1].argmax()))
        want.append(t)
    for t, r in zip(toks, want):
        got = G.generate(m, torch.tensor(t).cuda(), 12, top_k=1)
        assert got.tolist() == r
    rows = G.generate_batch(m, [torch.tensor(t) for t in toks], 12)
    assert [r.tolist() for r in rows] == want
    eos = want[0][-4]
    cut = G.generate(m, torch.tensor(toks[0]).cuda(), 12, top_k=1, eos_id=eos).tolist()
    first = want[0].index(eos, len(toks[0]))
    assert cut == want[0][:first]
    torch.manual_seed(3)
    a = G.generate(m, torch.tensor(toks[1]).cuda(), 20, top_k=7, temperature=0.9)
    torch.manual_seed(3)
    b = G.generate(m, torch.tensor(toks[1]).cuda(), 20, top_k=7, temperature=0.9)
    assert a.tolist() == b.tolist() and max(a.tolist()) < cfg["vocab"]


def test_graph_replays_equal_eager_steps(hip):
    """Replays of the captured step, with eager work in between, give the eager steps' ids."""
    from lit_llama.engine import DecodeSession

    cfg, w, m = case("wide", torch.bfloat16)
    toks = prompts(cfg, [20, 33], seed=13)
    runs = []
    for graph in (True, False):
        s = DecodeSession(m, 2, 200, 200, use_graph=graph)
        s.prefill(toks)
        for n in (1, 5, 2, 40):
            s.decode(n)
            torch.cuda.synchronize()
            torch.ones(1000, device="cuda").sum().item()
        runs.append([r.tolist() for r in s.output()])
    assert runs[0] == runs[1]


def test_model_folder_forward_and_cli(hip, tmp_path, capsys):
    """A folder (config.json + model.safetensors) through load_model, LLaMA-style forward and generate.py."""
    import json

    import generate as G
    from lit_llama import load_model
    from safetensors.torch import save_file

    cfg, w, m = case("odd", torch.float32)
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    save_file({k: torch.from_numpy(v).to(torch.bfloat16).contiguous() for k, v in w.items()},
              str(tmp_path / "model.safetensors"))
    f = load_model(tmp_path, torch.float32)
    idx = torch.tensor(prompts(cfg, [30, 30], seed=20)).cuda()
    ref = np.stack([oracle(cfg, w, t) for t in idx.tolist()])
    check(f(idx).reshape(60, -1), ref.reshape(60, -1), torch.float32)
    got = [f(idx[:, :12], 40, torch.arange(12)), f(idx[:, 12:13], 40, torch.tensor([12])), f(idx[:, 13:], 40, torch.arange(13, 30))]
    check(torch.cat(got, 1).reshape(60, -1), ref.reshape(60, -1), torch.float32)
    f.reset_cache()
    G.main(checkpoint_path=tmp_path, prompt_tokens=idx[0].tolist(), max_new_tokens=6, top_k=1, dtype="float32")
    out = [int(x) for x in capsys.readouterr().out.split()]
    assert out == G.generate(m, idx[0], 6, top_k=1).tolist()
