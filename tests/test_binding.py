"""The Python binding's handling of memory that a GPU stream may still use,
on the CPU: the library call and torch's device functions are stood in for."""
import contextlib
import gc
import types
import weakref

import pytest
import torch

import bmx


class _Stream:
    def __init__(self, handle):
        self.cuda_stream = handle


@pytest.fixture
def fake(monkeypatch):
    """torch with CPU tensors for CUDA ones and a current stream that can be
    asked for; library calls go to fake.calls, which may refuse them."""
    state = types.SimpleNamespace(current=_Stream(0), calls=[], refuse=False, during=lambda: None)

    @contextlib.contextmanager
    def use(s):
        before, state.current = state.current, s
        try:
            yield
        finally:
            state.current = before

    shim = types.SimpleNamespace(
        bfloat16=torch.bfloat16, float32=torch.float32,
        empty=lambda *shape, dtype=None, device=None: torch.empty(*shape, dtype=dtype),
        cuda=types.SimpleNamespace(Stream=_Stream, stream=use))

    def call(name, *args):
        state.during()
        if state.refuse:
            raise bmx.BmxError(bmx.BMX_E_SHAPE, name)
        state.calls.append(name)

    monkeypatch.setattr(bmx, "_torch", lambda: shim)
    monkeypatch.setattr(bmx, "call", call)
    return state


def _model():
    m = bmx.Qwen3.__new__(bmx.Qwen3)
    m.cfg, m.h, m.max_tokens = types.SimpleNamespace(vocab=16), None, 8
    return m, types.SimpleNamespace(h=None)


def test_forward_outputs_live_until_the_stream_has_written_them(fake):
    """On the null stream an output that the caller dropped is given back only
    after a call has waited for the forward after it: not before that call
    has returned, not for a refused one, at once where a call waits for the
    whole stream."""
    m, cache = _model()
    null, refs = _Stream(0), []

    def forward():
        out = m.forward(cache, [1, 2], all_logits=True, stream=null)
        refs.append(weakref.ref(out))

    def alive():
        gc.collect()
        return [r() is not None for r in refs]

    forward()
    forward()
    assert alive() == [True, True]
    seen = []
    fake.during = lambda: seen.append(alive())
    fake.refuse = True
    with pytest.raises(bmx.BmxError):
        m.forward(cache, [1] * 9, all_logits=True, stream=null)
    assert seen.pop() == [True, True] and alive() == [True, True]
    fake.refuse = False
    forward()
    assert seen.pop() == [True, True] and alive() == [False, True, True]
    m.decode_step(cache, 1, stream=_Stream(64))  # another stream's end
    assert alive() == [False, True, True]
    m.decode_step(cache, 1, stream=null)
    assert alive() == [False, False, False]
    forward()
    m.generate_greedy(cache, [1, 2], 4, stream=null)
    assert alive() == [False] * 4


def test_forward_on_a_given_stream_holds_nothing(fake):
    m, cache = _model()
    out = m.forward(cache, [1, 2], all_logits=True, stream=_Stream(64))
    ref = weakref.ref(out)
    del out
    gc.collect()
    assert ref() is None


def test_attention_workspace_of_a_call_belongs_to_its_stream(fake, monkeypatch):
    """A call on a given stream allocates and clears its own workspace there:
    freed on return, it goes to that stream's later allocations only.  (The
    many-token path writes its key-split partials there too.)"""
    made = []
    monkeypatch.setattr(bmx, "_require_cuda", lambda *ts: None)
    monkeypatch.setattr(bmx, "attention_workspace",
                        lambda Hq, M, device: made.append(fake.current) or torch.zeros(8))
    q, kc = torch.empty(8, 70, 128, dtype=torch.bfloat16), torch.empty(2, 80, 128, dtype=torch.bfloat16)
    side = _Stream(64)
    bmx.attention(q, kc, kc, 3, stream=side)
    t, norm = torch.empty(1, 1024, dtype=torch.bfloat16), torch.empty(128, dtype=torch.bfloat16)
    bmx.qk_norm_rope_kv_attention(t, t, t, norm, norm, kc, kc, 3, stream=side)
    assert made == [side, side]
    monkeypatch.setattr(bmx, "_stream", lambda s: 0)
    bmx.attention(q, kc, kc, 3)
    assert made[2] is fake.current
    bmx.attention(q, kc, kc, 3, workspace=torch.zeros(8), stream=side)
    assert len(made) == 3
