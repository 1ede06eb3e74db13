"""Decode attention of few sequences on MFMA against 64 bits and the VALU kernel:
weights in two bf16 terms are off by 2^-17, a hundredth of the result's rounding.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("nh,n_kv", [(4, 2), (32, 8), (8, 1)])
@pytest.mark.parametrize("splits", [1, 3, 4, 32, 200])
@pytest.mark.parametrize("last", [0, 30, 31, 32, 128, 911])
def test_few_sequences(B, nh, n_kv, splits, last):
    from llm_sharding_demo_amd import _C as C

    hd, S = 128, 920
    gen = torch.Generator().manual_seed(last)
    kc, vc = (torch.randn(B + 1, n_kv, S, hd, generator=gen).bfloat16() for _ in range(2))
    q = (2 * torch.randn(B, nh * hd, generator=gen)).bfloat16()
    slots, pos = list(range(B, 0, -1)), [max(0, last - 5 * b) for b in range(B)]
    for s, p in zip(slots, pos):
        kc[s, :, p + 1:], vc[s, :, p + 1:] = float("nan"), float("nan")
    i32 = dict(dtype=torch.int32, device=DEV)
    args = (q.to(DEV), kc.to(DEV), vc.to(DEV), torch.tensor(slots, **i32), torch.tensor(pos, **i32), nh, splits)
    got = C.attn_decode(*args).cpu().double().reshape(B, nh, hd)
    C.attn_set_mfma_min(0)
    try:
        valu = C.attn_decode(*args).cpu().double().reshape(B, nh, hd)
    finally:
        C.attn_set_mfma_min(256)
    want = torch.empty(B, nh, hd, dtype=torch.float64)
    for b in range(B):
        k, v = (c[slots[b], :, :pos[b] + 1].double().repeat_interleave(nh // n_kv, 0) for c in (kc, vc))
        w = torch.softmax((k @ q[b].double().reshape(nh, hd, 1))[..., 0] * hd ** -0.5, -1)
        want[b] = (w[:, None] @ v)[:, 0]
    rms = lambda x: float(x.pow(2).mean().sqrt())  # noqa: E731
    if B * n_kv * splits < 256:  # (more waves take their weights in one term)
        assert rms(got - want) <= 1.02 * rms(valu - want) + 2 ** -16 * rms(want)
    assert rms(got - want) < 2 ** -9 * rms(want)
