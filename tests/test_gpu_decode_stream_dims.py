"""GPU tier: the streaming decode at head_dim 64 and 256 and in float32.

The same partition logic as the 16-bit head_dim 128 kernel
(test_gpu_decode_stream.py) over other row lengths: 128-byte rows (two to a
LDS bank window, 8 rows a load), 512-byte rows (16-key stages) and float32
products, at the edges of their stages and page groups, on grids that leave
sequences whole, cut in a few pieces and cut in one piece per stage (each
combine form), and at the ends of the form that gives a short sequence a
workgroup of its own. Oracle: flash_attention.py:555-589 decode on the cache prefix,
paged.py:45-99 over the gathered pages.
"""

from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch

from gpu_util import check_fwd, dev, host, note
from oracle import decode_ref, paged_ref
from pallas_flash import (_lib, flash_attention_decode, flash_attention_decode_step, paged_flash_attention,
                          precompute_rope)

pytestmark = pytest.mark.gpu

FORMS = [("bf16", 64), ("f16", 64), ("bf16", 256), ("f16", 256), ("f32", 64), ("f32", 128)]


def _waves(w):
    return contextlib.nullcontext() if w is None else _lib.tuning(decode_waves=w)


@pytest.mark.parametrize("w", [None, 1, 7])
@pytest.mark.parametrize("dt,D", FORMS + [("bf16", 128)])
@pytest.mark.parametrize("B,Hq,Hkv,cap,L", [
    (3, 8, 2, 70, 1),       # one key; g = 4
    (2, 10, 2, 64, 15),     # g = 5: 16 query rows, a short 16-key stage
    (2, 32, 2, 64, 33),     # g = 16: every query row; one key past a stage
    (1, 1, 1, 1300, 1299),  # one sequence cut in dozens of pieces
    (2, 8, 2, 400, 192),    # 12 stages of 16 keys: the last length of a workgroup per sequence there
    (2, 8, 2, 400, 384),    # 12 stages of 32 keys
    (2, 8, 2, 400, 385),    # one key more: the persistent grid
    (2, 34, 2, 40, 17),     # g = 17: the generic kernel
])
def test_decode(w, dt, D, B, Hq, Hkv, cap, L):
    note(f"stream decode waves={w} {dt} D={D} B={B} Hq={Hq} Hkv={Hkv} cap={cap} L={L}")
    rng = np.random.default_rng(L)
    q = rng.standard_normal((B, Hq, 1, D))
    k, v = rng.standard_normal((2, B, Hkv, cap, D))
    k[:, :, L:] = v[:, :, L:] = np.nan
    tq, tk, tv = dev(q, dt), dev(k, dt), dev(v, dt)
    with _waves(w):
        out = host(flash_attention_decode(tq, tk, tv, L))
    check_fwd(out, decode_ref(host(tq), host(tk), host(tv), L), dt)


@pytest.mark.parametrize("w", [None, 5])
@pytest.mark.parametrize("dt,D", FORMS)
@pytest.mark.parametrize("page", [4, 8, 12, 16, 48, 64])
def test_paged(w, dt, D, page):
    note(f"stream paged waves={w} {dt} D={D} page={page}")
    rng = np.random.default_rng(page)
    B, Hq, Hkv, pps = 6, 8, 2, 20
    lens = np.array([0, 1, 15, 33, 5 * page + 3, pps * page], np.int32)
    used = -(-lens // page)
    npages = int(used.sum()) + 3
    perm = rng.permutation(npages)
    table = np.full((B, pps), -1, np.int32)
    cur = 0
    for b, n in enumerate(used):
        table[b, :n] = perm[cur:cur + n]
        cur += n
    q = rng.standard_normal((B, Hq, 1, D))
    kp, vp = rng.standard_normal((2, npages, Hkv, page, D))
    kp[perm[cur:]] = vp[perm[cur:]] = np.nan  # pages of no sequence
    for b, n in enumerate(used):
        if lens[b] % page:
            kp[table[b, n - 1], :, lens[b] % page:] = np.nan
            vp[table[b, n - 1], :, lens[b] % page:] = np.nan
    tq, tk, tv = dev(q, dt), dev(kp, dt), dev(vp, dt)
    with _waves(w):
        out = host(paged_flash_attention(tq, tk, tv, torch.as_tensor(table), torch.as_tensor(lens)))
    clean = lambda t: np.nan_to_num(host(t))
    check_fwd(out, paged_ref(host(tq), clean(tk), clean(tv), np.where(table < 0, 0, table), lens), dt)
    assert (out[0] == 0).all()


@pytest.mark.parametrize("w", [None, 7])
@pytest.mark.parametrize("B,Hq,Hkv,L", [
    (20, 16, 4, 409),  # 80 x 13 stages of 32 keys: more than there are waves, 16-key stages
    (20, 16, 4, 416),  # whole stages
    (27, 10, 2, 593),  # g = 5: 16 query rows; one key past a 16-key stage
    (20, 12, 3, 545),  # 60 x 18, one key into the last
    (16, 8, 4, 512),   # 64 x 16: a 32-key stage each still
])
def test_f32_fine_stages(w, B, Hq, Hkv, L):
    note(f"fine stages waves={w} B={B} Hq={Hq} Hkv={Hkv} L={L}")
    rng = np.random.default_rng(L)
    q = rng.standard_normal((B, Hq, 1, 64))
    k, v = rng.standard_normal((2, B, Hkv, L + 3, 64))
    k[:, :, L:] = v[:, :, L:] = np.nan
    tq, tk, tv = dev(q, "f32"), dev(k, "f32"), dev(v, "f32")
    with _waves(w):
        out = host(flash_attention_decode(tq, tk, tv, L))
    check_fwd(out, decode_ref(host(tq), host(tk), host(tv), L), "f32")


@pytest.mark.parametrize("Hq", [4, 12])
@pytest.mark.parametrize("page", [4, 8, 12, 16, 48, 64])
def test_f32_fine_stages_paged(Hq, page):
    """60 sequences x up to 576 keys, g = 2 and 6."""
    note(f"fine stages paged Hq={Hq} page={page}")
    rng = np.random.default_rng(page)
    B, Hkv, pps = 30, 2, 576 // page
    lens = rng.integers(0, 577, B).astype(np.int32)
    lens[:6] = [0, 1, 15, 17, 33, 576]
    table = rng.permutation(B * pps).reshape(B, pps).astype(np.int32)
    q = rng.standard_normal((B, Hq, 1, 64))
    kp, vp = rng.standard_normal((2, B * pps, Hkv, page, 64))
    for b, n in enumerate(lens):
        for j in range(pps):
            kp[table[b, j], :, max(n - j * page, 0):] = vp[table[b, j], :, max(n - j * page, 0):] = np.nan
    tq, tk, tv = dev(q, "f32"), dev(kp, "f32"), dev(vp, "f32")
    out = host(paged_flash_attention(tq, tk, tv, torch.as_tensor(table), torch.as_tensor(lens)))
    clean = lambda t: np.nan_to_num(host(t))
    check_fwd(out, paged_ref(host(tq), clean(tk), clean(tv), table, lens), "f32")
    assert (out[0] == 0).all()


@pytest.mark.parametrize("dt,D", [("f16", 64), ("bf16", 256), ("f32", 128), ("bf16", 128)])
def test_unaligned_cache_keeps_the_generic_kernel(dt, D):
    """A contiguous cache that starts between two 16-byte boundaries: the
    streaming kernel's loads want aligned rows, so the generic kernel reads it."""
    note(f"unaligned cache {dt} D={D}")
    rng = np.random.default_rng(D)
    B, Hq, Hkv, cap, L = 2, 8, 2, 300, 290
    tq = dev(rng.standard_normal((B, Hq, 1, D)), dt)
    caches = []
    for _ in range(2):
        x = dev(rng.standard_normal((B, Hkv, cap, D)), dt)
        flat = torch.empty(x.numel() + 8, dtype=x.dtype, device="cuda")
        view = flat[1:1 + x.numel()].view(x.shape)
        view.copy_(x)
        assert view.is_contiguous() and view.data_ptr() % 16 != 0
        caches.append(view)
    out = host(flash_attention_decode(tq, *caches, L))
    check_fwd(out, decode_ref(host(tq), host(caches[0]), host(caches[1]), L), dt)


def _skewed(x):
    """x's values in a contiguous tensor that starts between two 16-byte boundaries."""
    flat = torch.empty(x.numel() + 8, dtype=x.dtype, device="cuda")
    view = flat[1:1 + x.numel()].view(x.shape)
    view.copy_(x)
    assert view.is_contiguous() and view.data_ptr() % 16 != 0
    return view


@pytest.mark.parametrize("B,Hq,Hkv,w", [(3, 8, 2, 0), (11, 8, 2, 4), (5, 40, 2, 1)])
@pytest.mark.parametrize("what", ["decode", "paged"])
def test_unaligned_operands_at_16bit_head_dim_128(what, B, Hq, Hkv, w):
    """The form whose workspace has one size: with a grid of a few waves (w) that
    size holds the partials of a few batches, and the generic kernel runs
    slice after slice (11 batches by 4; 5 by 1)."""
    note(f"unaligned 16-bit head_dim 128 {what} B={B} Hq={Hq} w={w}")
    rng = np.random.default_rng(B)
    D, page, n = 128, 16, 60
    tq = _skewed(dev(rng.standard_normal((B, Hq, 1, D)), "bf16"))
    with _lib.tuning(decode_waves=w):
        if what == "decode":
            tk, tv = (_skewed(dev(rng.standard_normal((B, Hkv, page * n, D)), "bf16")) for _ in range(2))
            out = host(flash_attention_decode(tq, tk, tv, 901))
            want = decode_ref(host(tq), host(tk), host(tv), 901)
        else:
            tk, tv = (_skewed(dev(rng.standard_normal((B * n, Hkv, page, D)), "bf16")) for _ in range(2))
            lens = rng.integers(0, page * n + 1, B).astype(np.int32)
            table = rng.permutation(B * n).reshape(B, n).astype(np.int32)
            out = host(paged_flash_attention(tq, tk, tv, torch.as_tensor(table), torch.as_tensor(lens)))
            want = paged_ref(host(tq), host(tk), host(tv), table, lens)
    check_fwd(out, want, "bf16")


@pytest.mark.parametrize("skew", ["q", "k", "v", "all"])
def test_unaligned_decode_step(skew):
    """The fused step through the public call: as with aligned operands, the
    caches written in place; the C entry refuses them."""
    note(f"unaligned decode step {skew}")
    rng = np.random.default_rng(7)
    B, Hq, Hkv, C, D = 3, 8, 2, 500, 128
    ops = [dev(rng.standard_normal(s), "bf16") for s in ((B, Hq, 1, D), (B, Hkv, C, D), (B, Hkv, C, D))]
    k_new, v_new = (dev(rng.standard_normal((B, Hkv, 1, D)), "bf16") for _ in range(2))
    cos, sin = (t.cuda() for t in precompute_rope(1200, D, 10000.0))
    pos = torch.tensor([3, 499, 1150], dtype=torch.int32, device="cuda")
    own = [_skewed(t) if skew in (name, "all") else t.clone() for name, t in zip("qkv", ops)]
    ptrs = [t.data_ptr() for t in own]
    got = flash_attention_decode_step(own[0], k_new, v_new, own[1], own[2], pos, cos, sin, ring=True)
    want = flash_attention_decode_step(ops[0], k_new, v_new, ops[1], ops[2], pos, cos, sin, ring=True)
    assert ptrs == [t.data_ptr() for t in own]
    assert torch.equal(got, want) and torch.equal(own[1], ops[1]) and torch.equal(own[2], ops[2])
    args = _lib.DecodeStepArgs(ptrs[0], k_new.data_ptr(), v_new.data_ptr(), ptrs[1], ptrs[2], got.data_ptr(),
                               pos.data_ptr(), 1, None, None, 0, B, Hq, Hkv, C, D, 1, 0.1, _lib.dtype_tag(k_new),
                               None, 0)
    L = _lib.lib()
    ws = torch.empty(L.pf_attn_decode_step_workspace_size(args), dtype=torch.uint8, device="cuda")
    args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
    assert L.pf_attn_decode_step(args, None) == _lib.PF_ERR_INVALID
