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
    """A session's graph outlives it until the next capture, and at most two are kept."""
    from lit_llama import engine

    class Graph:
        pass

    monkeypatch.setattr(engine, "_retired", type(engine._retired)(maxlen=2))
    refs = []
    for _ in range(3):
        sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
        sess.graph = Graph()
        refs.append(weakref.ref(sess.graph))
        del sess
    assert refs[0]() is None and len(engine._retired) == 2
    sess = DecodeSession(_Model(HybridProgram), 1, 16, 16)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: 1 / 0)
    with pytest.raises(ZeroDivisionError):
        sess.capture()
    assert refs[1]() is None and refs[2]() is None
