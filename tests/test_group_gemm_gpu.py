"""Grouped products whose k-steps are fewer than, as many as and more than the
ring that is filled ahead of them, and off its turns, against 64 bits.

The limit is that of the same products at other sizes: two bf16 roundings of
the gated columns and one of the result.
"""

import pytest
import torch

from .test_timisun_gpu import C, F64, err, moe_case, moe_weights, rand  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 11])
@pytest.mark.parametrize("T", [1, 33])
def test_expert_depths(C, T, steps):  # noqa: F811
    H, F, Fs = 64 * steps, 64 * (12 - steps) - 16, 64 * steps
    d, ids, wts, lim, slim, parts = moe_case(T, H, 3, 2, F, Fs, torch.bfloat16)
    w, dn, ws, dns = moe_weights(d, H, F, Fs)
    for tm in (32, 64, 128):
        perm, tiles = C.moe_group(ids.to(DEV), 3, tm)
        mid, mids = C.moe_up(d["h"].to(DEV), perm, tiles, 2, w, lim, 1.702, ws, slim, tm)
        slab = torch.full((3, T, H), 7.0, dtype=torch.bfloat16, device=DEV)
        C.moe_down(mid, mids, perm, tiles, wts.to(DEV), dn, dns, slab, tm)
        assert err(slab, parts) < 6e-3


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 11])
def test_head_depths(C, steps):  # noqa: F811
    M, G, N, K = 70, 3, 144, 64 * steps
    a, w = rand(M, G * K, seed=1).bfloat16(), rand(G, N, K, seed=2).bfloat16()
    want = torch.einsum("mgk,gnk->mgn", a.to(F64).reshape(M, G, K), w.to(F64)).reshape(M, -1)
    for tm in (32, 64, 128):
        assert err(C.batch_linear(a.to(DEV), w.to(DEV), tm), want) < 4e-3
