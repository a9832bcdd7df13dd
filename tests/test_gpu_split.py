"""GPU tier: forward and backward with split work items.

A launch with few work items cuts each into chunks of keys (forward, dQ) or
runs of query blocks (dK/dV) whose float32 partials a second kernel merges.
These shapes split (asserted through the workspace queries) at the places
where a cut can go wrong: lengths around a chunk and a tile, causal blocks that
need one chunk only beside ones that need several, chunks that start past a
query block, key blocks with no step at all (kv_len, Sq < Sk), one to four
heads per workgroup, and -inf scores over a whole chunk. Oracle:
flash_attention.py:61-159 and :354-442.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import TORCH_DT, check_fwd, check_grad, dev, host, note, qkv
from oracle import attention_bwd_ref, attention_ref, rope_attention_ref
from pallas_flash import _lib, flash_attention, flash_attention_rope, flash_attention_with_lse, precompute_rope

pytestmark = pytest.mark.gpu

SHAPES = [  # B, Hq, Hkv, Sq, Sk, kv_len, causal
    (1, 4, 1, 257, 1025, 1025, False),
    (1, 2, 1, 33, 2000, 1873, False),
    (2, 1, 1, 1, 700, 700, False),
    (1, 4, 2, 900, 900, 900, True),
    (1, 1, 1, 1153, 1153, 1153, True),
    (1, 4, 1, 640, 1400, 1101, True),
    (1, 8, 2, 1300, 400, 389, True),
]


def _args(dt, B, Hq, Hkv, Sq, Sk, kv_len, causal, D):
    tag = _lib.PF_DTYPE[TORCH_DT[dt]]
    tail = (B, Hq, Hkv, Sq, Sk, D, kv_len, int(causal), 0.1, tag)
    return _lib.FwdArgs(8, 8, 8, 8, 8, *tail), _lib.BwdArgs(*[8] * 10, *tail)


@pytest.mark.parametrize("dt,D", [("f32", 64), ("f32", 128), ("bf16", 64), ("f16", 128), ("bf16", 256)])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_forward_backward(shape, dt, D):
    B, Hq, Hkv, Sq, Sk, kv_len, causal = shape
    note(f"split {dt} D={D} {shape}")
    fwd, bwd = _args(dt, *shape, D)
    L = _lib.lib()
    assert L.pf_attn_bwd_workspace_size(bwd) > 0
    assert L.pf_attn_fwd_workspace_size(fwd) > 0 or dt != "f32"
    q, k, v = qkv(np.random.default_rng(Sq + Sk), B, Hq, Hkv, Sq, Sk, D)
    do = np.random.default_rng(3).standard_normal(q.shape)
    tq, tk, tv = (dev(x, dt).requires_grad_(True) for x in (q, k, v))
    tdo = dev(do, dt)
    o = flash_attention(tq, tk, tv, causal=causal, kv_len=kv_len)
    dq, dk, dv = torch.autograd.grad(o, (tq, tk, tv), tdo)
    hq, hk, hv = host(tq), host(tk), host(tv)
    ref, lse_ref = attention_ref(hq, hk, hv, causal=causal, kv_len=kv_len)
    check_fwd(host(o), ref, dt)
    _, lse = flash_attention_with_lse(tq.detach(), tk.detach(), tv.detach(), causal=causal, kv_len=kv_len)
    # one rounding of each score and sum: 1e-5 of the largest (float32 dot of D terms)
    assert np.abs(host(lse) - lse_ref).max() <= 1e-5 * max(1.0, np.abs(lse_ref).max())
    grads = attention_bwd_ref(hq, hk, hv, host(tdo), causal=causal, kv_len=kv_len)
    for name, got, want in zip(("dq", "dk", "dv"), (dq, dk, dv), grads):
        check_grad(host(got), want, dt, name)
    assert not host(dk)[:, :, kv_len:].any() and not host(dv)[:, :, kv_len:].any()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_split_rope(dt):
    note(f"split rope {dt}")
    B, Hq, Hkv, S, D = 1, 4, 1, 1500, 128
    q, k, v = qkv(np.random.default_rng(1), B, Hq, Hkv, S, S, D)
    cos, sin = precompute_rope(S, D, 10000.0)
    tq, tk, tv = dev(q, dt), dev(k, dt), dev(v, dt)
    out = flash_attention_rope(tq, tk, tv, cos.cuda(), sin.cuda(), causal=True)
    ref = rope_attention_ref(host(tq), host(tk), host(tv), cos.numpy().astype(np.float64),
                             sin.numpy().astype(np.float64), causal=True)
    check_fwd(host(out), ref, dt)


def test_chunk_of_minus_infinity_scores():
    """Keys whose scores are all -inf drop out, a whole chunk of them too."""
    note("split: -inf chunk")
    q = torch.ones((1, 1, 64, 128), device="cuda")
    k = torch.randn((1, 1, 1024, 128), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    v = torch.randn_like(k)
    args = _args("f32", 1, 1, 1, 64, 1024, 1024, False, 128)[0]
    assert _lib.lib().pf_attn_fwd_workspace_size(args) > 0
    k[:, :, 512:, 0] = -float("inf")
    out = flash_attention(q, k, v)
    want = flash_attention(q, k, v, kv_len=512)
    check_fwd(host(out), host(want), "f32")


@pytest.mark.parametrize("dt,D", [("f32", 64), ("f32", 128), ("bf16", 128)])
@pytest.mark.parametrize("causal", [False, True])
def test_minus_infinity_rows_do_not_depend_on_the_split(dt, D, causal):
    """Rows whose scores are -inf throughout, over the first block of keys, or
    over later ones give what whole work items give: NaN for the first two
    (the running max starts at -inf), the finite scores' result for the last."""
    note(f"split: -inf rows {dt} D={D} causal={causal}")
    S = 2048
    fwd = _args(dt, 1, 1, 1, S, S, S, causal, D)[0]
    L = _lib.lib()
    ws_bytes = L.pf_attn_fwd_workspace_size(fwd)
    assert ws_bytes > 0
    g = torch.Generator("cuda").manual_seed(4)
    q, k, v = (torch.randn((1, 1, S, D), device="cuda", generator=g).to(TORCH_DT[dt]) for _ in range(3))
    q[0, 0, :, 0] = 1.0  # every row meets column 0 of K, -inf for some keys
    for lo, hi, nan_rows in ((0, S, slice(0, S)), (0, 64, slice(0, S)), (64, S, slice(0, 0)), (600, 1400, slice(0, 0))):
        k2 = k.clone()
        k2[0, 0, lo:hi, 0] = -float("inf")
        o, lse = [], []
        for split in (False, True):
            o.append(torch.empty_like(q))
            lse.append(torch.empty((1, 1, S), dtype=torch.float32, device="cuda"))
            a = _lib.FwdArgs(q.data_ptr(), k2.data_ptr(), v.data_ptr(), o[-1].data_ptr(), lse[-1].data_ptr(), 1, 1, 1,
                             S, S, D, S, int(causal), 0.1, _lib.dtype_tag(q))
            st = torch.cuda.current_stream().cuda_stream
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda")
            assert (L.pf_attn_fwd_ws(a, ws.data_ptr(), ws_bytes, st) if split else L.pf_attn_fwd(a, st)) == 0
        torch.cuda.synchronize()
        for whole, cut in (o, lse):
            assert torch.equal(torch.isnan(whole), torch.isnan(cut)), (lo, hi)
        assert torch.isnan(o[0][0, 0, nan_rows]).all() and torch.isnan(o[0]).any() == (nan_rows.stop > 0)
        if nan_rows.stop == 0:
            check_fwd(host(o[1]), host(o[0]), dt)


@pytest.mark.parametrize("B,H,S", [(8, 12, 1000), (5, 13, 1100), (3, 11, 1025)])
def test_resident_causal_items(B, H, S):
    """16-bit head_dim 64, causal, 257-768 work items (no split, every other
    round of 256 back to front; whole and partial last rounds): every row against
    the float32 product."""
    n_work = B * H * -(-S // 128)
    assert 256 < n_work <= 768
    note(f"resident causal items B={B} H={H} S={S}")
    g = torch.Generator("cuda").manual_seed(S)
    q, k, v = (torch.randn((B, H, S, 64), device="cuda", generator=g).half() for _ in range(3))
    out = flash_attention(q, k, v, causal=True)
    mask = torch.ones((S, S), dtype=torch.bool, device="cuda").triu_(1)
    for b in range(B):
        s = torch.matmul(q[b].float(), k[b].float().transpose(1, 2).contiguous()) * 0.125
        ref = torch.matmul(torch.softmax(s.masked_fill_(mask, -float("inf")), -1), v[b].float())
        check_fwd(host(out[b]), host(ref), "f16")
