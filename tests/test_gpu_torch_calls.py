"""GPU tier: the C++ host side of the public calls against the general path.

Every public call first offers its arguments to _torch_calls, which takes the
plain case and declines (returns None) anything else. The outputs and gradients
have to be those of the general path bit for bit, and what only the general
path knows -- tensor subclasses, transforms, dispatch modes, forward-mode AD --
has to reach it, with saved-tensor hooks, streams and double use of a graph as
before.
"""

from __future__ import annotations

import contextlib
import types

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.checkpoint import checkpoint

from gpu_util import note
from pallas_flash import (_lib, flash_attention, flash_attention_decode, flash_attention_decode_step,
                          flash_attention_rope, paged_flash_attention, precompute_rope)

pytestmark = pytest.mark.gpu

NAMES = ("attention", "rope", "decode", "paged", "step")


@contextlib.contextmanager
def _declining():
    """The general path alone."""
    real = _lib.calls()
    _lib._calls = types.SimpleNamespace(**{n: (lambda *a: None) for n in NAMES})
    try:
        yield
    finally:
        _lib._calls = real


@contextlib.contextmanager
def _recording(seen):
    """The C++ host side; notes which function was offered a call and whether it took it."""
    real = _lib.calls()

    def noting(name):
        def call(*args):
            o = getattr(real, name)(*args)
            seen.append((name, o is not None))
            return o
        return call

    _lib._calls = types.SimpleNamespace(**{n: noting(n) for n in NAMES})
    try:
        yield
    finally:
        _lib._calls = real


def _r(*shape, dt=torch.bfloat16, seed=0):
    return torch.randn(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda").to(dt)


def _qkv(dt, B=2, Hq=4, Hkv=2, S=130, D=64):
    return [_r(B, h, S, D, dt=dt, seed=i) for i, h in enumerate((Hq, Hkv, Hkv))]


def _calls(dt):
    """name -> a call with fresh arguments, returning a tuple of tensors."""
    q, k, v = _qkv(dt)
    d, n = q.shape[3], q.shape[2]
    cos, sin = (t.cuda() for t in precompute_rope(n, d, 10000.0))
    q1 = q[:, :, :1]
    table = torch.tensor([[1, 0], [1, 2]], dtype=torch.int32, device="cuda")
    lens = torch.tensor([20, 32], dtype=torch.int32, device="cuda")
    pages = [_r(3, 2, 16, d, dt=dt, seed=s) for s in (5, 6)]

    def train():
        ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = flash_attention(*ts, causal=True, sm_scale=0.2, kv_len=100)
        return (o, *torch.autograd.grad(o.sum(), ts))

    def step():
        qs, ks, vs = _qkv(dt, S=64, D=128)
        c, s = (t.cuda() for t in precompute_rope(200, 128, 10000.0))
        pos = torch.tensor([3, 190], dtype=torch.int32, device="cuda")
        o = flash_attention_decode_step(qs[:, :, :1], ks[:, :, 5:6], vs[:, :, 7:8], ks, vs, pos, c, s, ring=True)
        return o, ks, vs

    return {
        "forward": lambda: (flash_attention(q, k, v, kv_len=77),),
        "transposed": lambda: (flash_attention(*(t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)),
                                               causal=True),),
        "train": train,
        "rope": lambda: (flash_attention_rope(q, k, v, cos, sin, causal=True),),
        "rope own tables": lambda: (flash_attention_rope(q1, k, v, cos[:1], sin[:1], cos, sin),),
        "decode": lambda: (flash_attention_decode(q1, k, v, 99),),
        "paged": lambda: (paged_flash_attention(q1, *pages, table, lens, sm_scale=0.3),),
        "step": step,
    }


DTYPES = (torch.bfloat16, torch.float16, torch.float32)
TAKEN_BY = {"forward": "attention", "transposed": "attention", "train": "attention", "rope": "rope",
            "rope own tables": "rope", "decode": "decode", "paged": "paged", "step": "step"}


@pytest.mark.parametrize("name,dt", [(n, dt) for n in TAKEN_BY for dt in DTYPES
                                     if n != "step" or dt != torch.float32])  # the step is 16-bit
def test_same_as_the_general_path(name, dt):
    note(f"calls: {name} {dt}")
    call = _calls(dt)[name]
    seen = []
    with _recording(seen):
        got = call()
    assert seen == [(TAKEN_BY[name], True)]
    with _declining():
        want = call()
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


def test_takes_the_plain_case():
    q, k, v = _qkv(torch.bfloat16)
    c = _lib.calls()
    assert c.attention(q, k, v, True, None, None) is not None
    assert c.decode(q[:, :, :1], k, v, 5, None) is not None


def test_declines_what_it_does_not_know():
    """Nothing is computed, accepted or refused for these: the caller's general
    path decides."""
    note("calls: declines")
    c = _lib.calls()
    q, k, v = _qkv(torch.bfloat16)

    class Sub(torch.Tensor):
        pass

    ok = (q, k, v, True, None, None)
    for bad in ((q.cpu(), k, v), (q.as_subclass(Sub), k, v), (q, k.float(), v), (q[0], k, v), (q, k[:, :, :5], v),
                (q[..., :48], k[..., :48], v[..., :48]), (q.double(), k.double(), v.double()), (q[:, :3], k, v),
                (q[:0], k[:0], v[:0]), (None, k, v)):
        assert c.attention(*bad, *ok[3:]) is None
    for bad in ((1, None, None), (True, "1", None), (True, float("nan"), None), (True, None, 0), (True, None, 131),
                (True, None, 1.0), (True, None, 1 << 70)):
        assert c.attention(q, k, v, *bad) is None
    assert c.attention(q, k, v) is None
    q1 = q[:, :, :1]
    assert c.decode(q, k, v, 5, None) is None
    assert c.decode(q1, k, v, 131, None) is None
    assert c.decode(q1.clone().requires_grad_(True), k, v, 5, None) is None
    table, lens = torch.zeros((2, 1), dtype=torch.int32, device="cuda"), torch.ones(2, dtype=torch.int32, device="cuda")
    pages = [_r(3, 2, 16, 64), _r(3, 2, 16, 64)]
    assert c.paged(q1, *pages, table, lens, None) is not None
    assert c.paged(q1, *pages, table.cpu(), lens, None) is None
    assert c.paged(q1, *pages, table.long(), lens, None) is None
    assert c.paged(q1, *(p.transpose(1, 2) for p in pages), table, lens, None) is None

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert c.attention(*ok) is None
    seen = []
    torch.func.vmap(lambda x: seen.append(c.attention(x, k, v, True, None, None)) or x)(q[None])
    torch.func.grad(lambda x: seen.append(c.attention(x, k, v, True, None, None)) or x.float().sum())(q)
    with torch.autograd.forward_ad.dual_level():
        seen.append(c.attention(torch.autograd.forward_ad.make_dual(q, q), k, v, True, None, None))
    assert seen == [None, None, None]


def test_tracer_and_function_mode_reach_the_general_path():
    note("calls: jit tracer, function mode")
    c = _lib.calls()
    q, k, v = _qkv(torch.bfloat16)
    want = flash_attention(q, k, v, causal=True)
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        seen.append(c.attention(q, k, v, True, None, None))
        assert torch.equal(flash_attention(q, k, v, causal=True), want)
    torch.jit.trace(lambda x: seen.append(c.attention(x, k, v, True, None, None)) or x * 1, (q,), check_trace=False)
    assert seen == [None, None]
    assert c.attention(q, k, v, True, None, None) is not None  # and afterwards it is taken again


def test_create_graph_and_checkpoint():
    """create_graph: the gradients are as the general path's, which are not
    differentiable again. Checkpointing: the recomputation ends with an exception
    that its pack hook throws through the C++ function."""
    note("calls: create_graph, checkpoint")
    ts = [t.requires_grad_(True) for t in _qkv(torch.float32)]
    call = lambda *a: flash_attention(*a, causal=True)

    def create_graph():
        o = call(*ts)
        return (o, *torch.autograd.grad(o.sum(), ts, create_graph=True))

    got = create_graph()
    with _declining():
        want = create_graph()
    for a, b in zip(got, want):
        assert torch.equal(a, b) and a.requires_grad == b.requires_grad
    assert not got[1].requires_grad
    seen = []
    with _recording(seen):
        grads = torch.autograd.grad(checkpoint(call, *ts, use_reentrant=False).sum(), ts)
    assert ("attention", True) in seen
    assert all(torch.equal(a, b) for a, b in zip(grads, want[1:]))


def test_saved_tensor_hooks_and_graph_reuse():
    note("calls: saved-tensor hooks")
    ts = [t.requires_grad_(True) for t in _qkv(torch.float32)]
    packed = []

    def pack(t):
        packed.append(tuple(t.shape))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        o = flash_attention(*ts, causal=True)
    assert len(packed) == 5  # q, k, v, o, lse
    do = _r(*o.shape, dt=torch.float32, seed=9)
    first = torch.autograd.grad(o, ts, do, retain_graph=True)
    again = torch.autograd.grad(o, ts, do)
    want = torch.autograd.grad(flash_attention(*ts, causal=True), ts, do)
    for a, b, c in zip(first, again, want):
        assert torch.equal(a, b) and torch.equal(a, c)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, ts, do)


def test_side_stream_and_no_grad():
    note("calls: side stream")
    ts = [t.requires_grad_(True) for t in _qkv(torch.bfloat16)]
    want = flash_attention(*ts, causal=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        o = flash_attention(*ts, causal=True)
        grads = torch.autograd.grad(o.float().sum(), ts)
    torch.cuda.current_stream().wait_stream(s)
    ref = torch.autograd.grad(want.float().sum(), ts)
    assert torch.equal(o, want) and all(torch.equal(a, b) for a, b in zip(grads, ref))
    with torch.no_grad():
        o2 = flash_attention(*ts, causal=True)
    assert not o2.requires_grad and torch.equal(o2, want)
