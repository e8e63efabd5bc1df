"""A finished decode session is freed at once, not by the garbage collector: its captured graph may not be freed while
another session captures (freeing one synchronizes the device)."""
import gc
import types
import weakref

import pytest
import torch

from lit_llama.engine import DecodeSession, HybridProgram, LLaMAProgram


class _Model:
    """What a session reads of a model before its first prompt."""

    device = torch.device("cpu")
    config = types.SimpleNamespace(block_size=64, padded_vocab_size=128, vocab_size=100)

    def __init__(self, program):
        self.session_program = program

    def act_dtype(self):
        return torch.bfloat16

    def new_state(self, slots, max_length):
        return object()


@pytest.mark.parametrize("program", [HybridProgram, LLaMAProgram])
def test_session_is_freed_without_the_collector(program, monkeypatch):
    monkeypatch.setattr("lit_llama._hip.require_device", lambda *a: None)
    model = _Model(program)
    model.transformer = types.SimpleNamespace(wte=types.SimpleNamespace(weight=torch.zeros(1)))
    gc.disable()
    try:
        sess = DecodeSession(model, 2, 16, 16)
        assert sess.program.sess is sess
        gone = weakref.ref(sess)
        del sess
        assert gone() is None
    finally:
        gc.enable()


def test_dropped_graphs_wait_for_the_next_capture(monkeypatch):
    """A session's graph outlives it until a capture has ended -- freeing one inside a capture aborts -- and at most two are kept;
    every few captures the allocator gives back what the freed graphs' steps had allocated. A step that raises ends its capture."""
    import contextlib

    from lit_llama import engine

    log = []

    class Graph:
        def capture_begin(self):
            log.append("begin")

        def capture_end(self):
            log.append("end")

    monkeypatch.setattr(engine, "_retired", type(engine._retired)(maxlen=2))
    monkeypatch.setattr(engine, "_captures", engine.itertools.count(1))
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "Stream", lambda dev: None)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: log.append("trim"))
    monkeypatch.setattr(DecodeSession, "_step", lambda self: log.append("step"))
    for _ in range(3):
        sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
        sess.graph = Graph()
        gone = weakref.ref(sess.graph)
        weakref.finalize(sess.graph, log.append, "free")
        del sess
    assert gone() is not None and log == ["free"]
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    sess.capture()
    assert log == ["free", "begin", "step", "end", "free", "free"] and gone() is None and sess.graph is not None
    sess.capture()
    assert len(log) == 6  # captured already
    for _ in range(engine._TRIM - 1):
        DecodeSession(_Model(HybridProgram), 1, 16, 16).capture()
    assert log.count("trim") == 1 and log[-1] == "trim"
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    monkeypatch.setattr(DecodeSession, "_step", lambda self: 1 / 0)
    with pytest.raises(ZeroDivisionError):
        sess.capture()
    assert log[-2:] == ["begin", "end"] and sess.graph is None


def test_capture_makes_room_once(monkeypatch):
    """A step whose buffers find no room during its capture: what the allocator and the dropped graphs hold is given back, with the
    first attempt's graph, and the step captured again; the second time the error is the caller's."""
    import contextlib

    from lit_llama import engine

    log = []

    class Graph:
        def __init__(self):
            weakref.finalize(self, log.append, "free")

        def capture_begin(self):
            log.append("begin")

        def capture_end(self):
            log.append("end")

    monkeypatch.setattr(engine, "_retired", type(engine._retired)(maxlen=2))
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "Stream", lambda dev: None)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: log.append("wait"))
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: log.append("trim"))
    failures = [1]

    def step(self):
        if failures:
            failures.pop()
            raise torch.OutOfMemoryError("no room")
        log.append("step")

    monkeypatch.setattr(DecodeSession, "_step", step)
    old = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    old.graph = Graph()
    del old
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    sess.capture()
    assert log == ["begin", "end", "free", "free", "wait", "trim", "begin", "step", "end"] and sess.graph is not None
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    failures += [1, 1]
    with pytest.raises(torch.OutOfMemoryError):
        sess.capture()
    assert sess.graph is None and log.count("begin") == log.count("end") == 4


def test_graphs_dropped_during_a_capture_wait_for_its_end(monkeypatch):
    """Sessions that end while another one captures, in its own thread (the garbage collector) or in others: their graphs are freed
    after the capture, however many; two threads' captures follow each other."""
    import contextlib
    import threading

    from lit_llama import engine

    log, inside = [], []

    class Graph:
        def __init__(self):
            weakref.finalize(self, lambda: log.append("freed inside" if inside else "free"))

        def capture_begin(self):
            assert not inside
            inside.append(1)

        def capture_end(self):
            inside.pop()

    def drop(n):
        for _ in range(n):
            sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
            sess.graph = Graph()
            del sess

    monkeypatch.setattr(engine, "_retired", type(engine._retired)(maxlen=2))
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "Stream", lambda dev: None)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: None)
    other = [DecodeSession(_Model(HybridProgram), 1, 16, 16)]
    threads = []

    def step(self):
        if not threads:
            drop(4)
            t = threading.Thread(target=drop, args=(4,))
            t.start()
            t.join(20)
            assert not t.is_alive()  # (a drop does not wait for the capture)
            threads.append(threading.Thread(target=other[0].capture))
            threads[0].start()
            threads[0].join(0.2)
        log.append("step")

    monkeypatch.setattr(DecodeSession, "_step", step)
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    sess.capture()
    threads[0].join(20)
    assert sess.graph is not None and other[0].graph is not None
    assert log.count("free") == 8 and log.count("step") == 2 and "freed inside" not in log
    drop(3)
    assert log.count("free") == 9  # two are kept


def test_failed_step_raises(monkeypatch):
    """A step that says on the device that it failed (a wait ran out): check() and the reads that wait for the steps raise, until the next prompt; a
    program without such steps has nothing to check."""
    import generate

    monkeypatch.setattr("lit_llama._hip.require_device", lambda *a: None)
    monkeypatch.setattr(DecodeSession, "decode", lambda self, n: None)
    monkeypatch.setattr(DecodeSession, "prefill", lambda self, prompts: None)
    model = _Model(LLaMAProgram)
    model.transformer = types.SimpleNamespace(wte=types.SimpleNamespace(weight=torch.zeros(1)))
    sess = DecodeSession(model, 1, 16, 16)
    sess.lens, sess.steps_done, ids = [3], 2, torch.arange(3)
    eos = int(sess.tokens[0, 3])
    reads = [sess.check, lambda: sess.feed([1]), lambda: generate._run_session(sess, ids, 2, None), lambda: generate._run_session(sess, ids, 2, eos)]
    for read in reads:
        read()
    sess.program.small = types.SimpleNamespace(failed=torch.zeros(1, dtype=torch.int32))
    for read in reads:
        read()
    sess.program.small.failed.fill_(1)
    for read in reads:
        with pytest.raises(RuntimeError, match="waited too long"):
            read()
    DecodeSession(_Model(HybridProgram), 1, 16, 16).check()


def test_small_step_keeps_what_it_points_to():
    """A small model's step holds addresses of weights, norms and caches: it keeps them all alive when the model lets go of them."""
    from lit_llama.model import LLaMA, LLaMAConfig, _SmallStep

    model = LLaMA(LLaMAConfig(block_size=32, vocab_size=64, n_layer=2, n_head=8, n_embd=512)).to(torch.bfloat16)
    model.kv_caches = [tuple(torch.zeros(1, 8, 32, 64, dtype=torch.bfloat16) for _ in range(2)) for _ in range(2)]
    lins = [(b.attn.c_attn, b.attn.c_proj, b.mlp.c_fc1, b.mlp.c_fc2, b.mlp.c_proj) for b in model.transformer.h]
    specs = {"layers": [[(1, lin.weight, None) for lin in layer] for layer in lins]}
    step = _SmallStep(model, specs, 32)
    at = [int(p) for p in step.layers]
    held = [weakref.ref(t) for b, kv in zip(model.transformer.h, model.kv_caches) for t in (b.rms_1.scale, b.mlp.c_proj.weight, *kv)]
    assert len(at) == 18 and {r().data_ptr() for r in held} <= set(at)
    del model, specs, lins
    gc.collect()
    assert all(r() is not None for r in held)
