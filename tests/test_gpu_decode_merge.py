"""GPU tier: the streaming decode's work list over many sequences and the merge
of those that wave boundaries cut.

Batches past 64 (a lane then holds several) and past 4096 (a lane's share is
itself searched in steps), sequences without keys, one long sequence in dozens
of pieces among short ones, two head slices, the fused step; against the
oracle (paged.py:45-99; model.py:475-491). And the time of a call whose heads
are many: mostly the attention's, not the merge's.
"""

from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch

from gpu_util import check_fwd, dev, host, note
from oracle import decode_step_ref, paged_ref, precompute_rope_ref
from pallas_flash import _lib, flash_attention_decode_step, paged_flash_attention

pytestmark = pytest.mark.gpu


def _waves(w):
    return contextlib.nullcontext() if w is None else _lib.tuning(decode_waves=w)


@pytest.mark.parametrize("w", [None, 1, 100])
@pytest.mark.parametrize("dt,D,B,Hq,Hkv,page,short,long", [
    ("bf16", 64, 64, 8, 2, 8, 70, 300),
    ("bf16", 64, 65, 8, 2, 8, 70, 300),
    ("f32", 64, 130, 16, 1, 16, 40, 700),
    ("f32", 128, 71, 3, 3, 4, 90, 500),
    ("bf16", 128, 129, 34, 2, 16, 70, 900),  # g = 17
    ("f16", 256, 66, 12, 2, 16, 50, 400),
    ("bf16", 64, 4100, 2, 1, 8, 80, 80),
])
def test_many_sequences(w, dt, D, B, Hq, Hkv, page, short, long):
    note(f"decode merge {dt} D={D} B={B} Hq={Hq} Hkv={Hkv} waves={w}")
    rng = np.random.default_rng(B)
    lens = rng.integers(0, short + 1, B).astype(np.int32)
    lens[[0, B // 2, B - 1]] = 0
    lens[B // 3] = long
    pps = -(-long // page)
    used = -(-lens // page)
    table = np.full((B, pps), -1, np.int32)
    perm = rng.permutation(int(used.sum())).astype(np.int32)
    first = np.concatenate([[0], np.cumsum(used)])
    for b in range(B):
        table[b, :used[b]] = perm[first[b]:first[b + 1]]
    tq = dev(rng.standard_normal((B, Hq, 1, D)), dt)
    tk, tv = (dev(rng.standard_normal((len(perm), Hkv, page, D)), dt) for _ in range(2))
    with _waves(w):
        out = host(paged_flash_attention(tq, tk, tv, torch.as_tensor(table), torch.as_tensor(lens)))
    check_fwd(out, paged_ref(host(tq), host(tk), host(tv), np.where(table < 0, 0, table), lens), dt)
    assert not out[lens == 0].any()


@pytest.mark.parametrize("w", [None, 60])
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (34, 2)])
def test_step_over_many_sequences(w, Hq, Hkv):
    note(f"decode merge: step Hq={Hq} waves={w}")
    rng = np.random.default_rng(Hq)
    B, C, D = 150, 400, 128
    pos = rng.integers(0, 60, B)
    pos[[3, 140]] = -1
    pos[70] = 390
    cos, sin = precompute_rope_ref(C, D, 10000.0)
    tq, kn, vn = (dev(rng.standard_normal((B, h, 1, D)), "bf16") for h in (Hq, Hkv, Hkv))
    kc, vc = (dev(rng.standard_normal((B, Hkv, C, D)), "bf16") for _ in range(2))
    kc0, vc0 = host(kc), host(vc)
    tcos, tsin = dev(cos, "f32"), dev(sin, "f32")
    with _waves(w):
        out = host(flash_attention_decode_step(tq, kn, vn, kc, vc, dev(pos, "f32").to(torch.int32), tcos, tsin))
    store = lambda x: torch.as_tensor(np.asarray(x)).to(torch.bfloat16).double().numpy()
    want, _, _ = decode_step_ref(host(tq), host(kn), host(vn), kc0, vc0, pos, host(tcos), host(tsin), store=store)
    check_fwd(out, want, "bf16")
    assert not out[pos < 0].any()


def test_the_merge_of_many_heads_is_a_small_part():
    """4096 x 16 heads of 8-64 keys, a little over half of the pool's 268 MB: less
    than 6 copies of its K half (about 50 us each). The kernels take 47 us; with
    a search per head in the merge they took 945."""
    note("decode merge: time")
    B, Hq, Hkv, page, D = 4096, 16, 4, 64, 64
    gen = torch.Generator("cuda").manual_seed(1)
    k, v = (torch.randn((B, Hkv, page, D), device="cuda", generator=gen).bfloat16() for _ in range(2))
    q = torch.randn((B, Hq, 1, D), device="cuda", generator=gen).bfloat16()
    table = torch.arange(B, dtype=torch.int32, device="cuda").view(B, 1)
    lens = torch.randint(8, page + 1, (B,), device="cuda", generator=gen, dtype=torch.int32)
    copy = torch.empty_like(k)

    def us(call):
        best = float("inf")
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                call()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best

    assert us(lambda: paged_flash_attention(q, k, v, table, lens)) < 6 * us(lambda: copy.copy_(k))
