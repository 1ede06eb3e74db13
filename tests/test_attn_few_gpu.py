"""Decode attention of few sequences on MFMA against 64 bits and the VALU kernel: weights in
three bf16 terms are those of fp32.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("nh,n_kv", [(4, 2), (32, 8), (8, 1)])
@pytest.mark.parametrize("splits", [1, 3, 4, 32, 200])
@pytest.mark.parametrize("last", [0, 30, 31, 32, 128, 911])
@pytest.mark.parametrize("keys", [0, 912])  # (known: ranges are taken in parts)
def test_few_sequences(B, nh, n_kv, splits, last, keys):
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
    got = C.attn_decode(*args, keys).cpu().double().reshape(B, nh, hd)
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


@pytest.mark.parametrize("nh,n_kv", [(4, 2), (32, 8), (8, 1)])
@pytest.mark.parametrize("splits", [1, 2])
def test_weights_keep_their_bits(nh, n_kv, splits):
    """Values that nearly cancel, so that the result shows the weights' last bits.  Scores are
    exact, so a weight is off by the rounding of the scaled score (at most 1.3, and its maximum
    alike: 2^-22 of the weight) and of exp2 and the sums (2^-22 each).  Two terms are off by
    up to 2^-17."""
    from llm_sharding_demo_amd import _C as C

    hd, n = 128, 24
    gen = torch.Generator().manual_seed(nh + splits)
    score = torch.randint(0, 40, (nh, n), generator=gen).float() * 0.25
    G = nh // n_kv
    # keys pick a query's columns, one per key: a head's score of key j is its column j
    q = torch.zeros(1, nh, hd)
    q[0, :, :n] = score
    kc = torch.zeros(1, n_kv, 64, hd)
    kc[0, :, :n] = torch.eye(n, hd)
    w = torch.softmax(score.double() * hd ** -0.5, -1)
    vc = torch.zeros(1, n_kv, 64, hd)
    for h in range(n_kv):  # column c: the group's head c % G is the one whose sum cancels
        for c in range(hd):
            wt, rest = w[h * G + c % G], 0.0
            for j in torch.randperm(n, generator=gen).tolist():
                v = (torch.tensor(-rest / float(wt[j])) if rest else torch.tensor(1.0 + c / 128)).bfloat16()
                vc[0, h, j, c] = v
                rest += float(v) * float(wt[j])
    i32 = dict(dtype=torch.int32, device=DEV)
    got = C.attn_decode(q.bfloat16().reshape(1, -1).to(DEV), kc.bfloat16().to(DEV), vc.bfloat16().to(DEV),
                        torch.zeros(1, **i32), torch.tensor([n - 1], **i32), nh, splits).cpu().double().reshape(nh, hd)
    v = vc[0, :, :n].double().repeat_interleave(G, 0)
    want, size = (w[:, None] @ v)[:, 0], (w[:, None] @ v.abs())[:, 0]
    own = (torch.arange(hd) % G) == (torch.arange(nh)[:, None] % G)  # (cancelled for the head itself)
    assert float((want.abs() / size)[own].max()) < 2.0 ** -16
    assert bool(((got - want).abs() <= 2.0 ** -19 * size + 2.0 ** -8 * want.abs())[own].all())
