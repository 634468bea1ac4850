"""What stays out of the way of a recording: garbage collections (a decoder that is no longer used is part of a cycle, and what it recorded must not be destroyed then), and waits
that nothing needs."""
import contextlib
import gc
import threading
import types

import pytest
import torch


@pytest.fixture
def recorded(monkeypatch):
    """torch.cuda.graph without a device; whether the collector was on in each recording."""
    seen = []

    @contextlib.contextmanager
    def graph(g, **where):
        seen.append(gc.isenabled())
        yield
    stream = types.SimpleNamespace(synchronize=lambda: None)
    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: types.SimpleNamespace(replay=lambda: None))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    return seen


def test_a_prompt_pass_and_a_loop(recorded):
    from poptransformer_amd.engine import loop, prompt
    p = prompt.PromptPass.__new__(prompt.PromptPass)
    p.spec, p.rows, p.first, p.graph, p.pool, p._warm, p._layers = types.SimpleNamespace(max_len=8), 4, torch.zeros(()), None, None, True, lambda: recorded.append(gc.isenabled())
    p.run(0)
    d = loop.DecodeLoop.__new__(loop.DecodeLoop)
    d.spec, d._stream, d.reset, d.step_fn = types.SimpleNamespace(batch=1, max_len=8), None, lambda ids: None, lambda: None
    d.capture()
    assert recorded == [False, False, False] and gc.isenabled()


def test_it_is_on_again_as_it_was(recorded):
    from poptransformer_amd.engine import loop
    with pytest.raises(ValueError):
        with loop.recording(None):
            raise ValueError
    assert gc.isenabled()
    gc.disable()
    try:
        with loop.recording(None):
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()


def test_with_two_threads_it_waits_for_the_last(recorded):
    from poptransformer_amd.engine import loop
    inside, leave = threading.Event(), threading.Event()

    def other():
        with loop.recording(None):
            inside.set()
            leave.wait(10)
    t = threading.Thread(target=other)
    with loop.recording(None):
        t.start()
        assert inside.wait(10)
    assert not gc.isenabled()
    leave.set()
    t.join(10)
    assert gc.isenabled()


@pytest.mark.parametrize("answer, plain", [(0, True), (1, False)])
def test_an_answer_that_is_there_is_not_waited_for(monkeypatch, answer, plain):
    """A wait for an event ends what another thread may be recording: F8Weight.plain waits only as long as its byte holds 2."""
    from poptransformer_amd import kernels as K
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for there in (True, False):
        host, waits = torch.full((1,), answer if there else 2, dtype=torch.uint8), []
        w = K.F8Weight.__new__(K.F8Weight)
        w._plain, w._asked = False, (host, types.SimpleNamespace(synchronize=lambda: (waits.append(1), host.fill_(answer))))
        assert w.plain is plain and w.plain is plain and len(waits) == (not there)
