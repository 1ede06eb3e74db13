"""One row through gemv_stream_kernel gives the bits that two equal rows get from gemv_kernel:
the same sums in the same order, whatever the units a wave goes through."""

import pytest
import torch

from .test_gemv_gpu import C, bf  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


def both(x):
    return x.expand(2, -1).contiguous()


# items of two rows: as many as waves, one and more a wave, a last one that is not there
@pytest.mark.parametrize("N,K", [(8224, 1032), (8224, 2048), (12320, 2056), (28672, 4096), (4128, 4096)])
@pytest.mark.parametrize("glu", [0, 1])
def test_gated(C, N, K, glu):  # noqa: F811
    x, g, w = torch.randn(1, K, device=DEV), bf(K, seed=1), bf(N, K, scale=0.05, seed=2)
    outs = [torch.empty(m, N // 2, dtype=torch.bfloat16, device=DEV) for m in (1, 2)]
    for o, rows in zip(outs, (x, both(x))):
        C.gemv_into(rows, w, 2, 2, g, None, 1e-5, o, glu, 1.0)
    assert torch.equal(outs[0][0], outs[1][0])


# items of eight rows, with a part of one at the end, and their maxima
@pytest.mark.parametrize("N,K", [(16384, 2056), (16392, 4096), (32768 + 8, 3072), (50257, 4088)])
@pytest.mark.parametrize("norm", [1, 2])
def test_head(C, N, K, norm):  # noqa: F811
    x, g, w = torch.randn(1, K, device=DEV), bf(K, seed=1), bf(N, K, scale=0.05, seed=2)
    beta, bias = (bf(K, seed=3) if norm == 1 else None), bf(N, seed=4)
    args = (w, bias, 3, norm, g, beta, 1e-5, None, None, None, None, None, 0, 0, 0, None)
    one, two = C.gemv(x, *args), C.gemv(both(x), *args)
    assert torch.equal(one[0], two[0])
    if N % 8 == 0:
        seg = torch.empty(1, N // 8, device=DEV)
        out = C.gemv_logits(x, w, norm, g, beta, 1e-5, seg)
        assert torch.equal(seg[0], out[0].view(-1, 8).amax(1))


@pytest.mark.parametrize("N", [4096, 4097, 8194])
@pytest.mark.parametrize("K", [2056, 4096, 8200, 11264, 14336])
@pytest.mark.parametrize("bias", [False, True])
def test_residual(C, N, K, bias):  # noqa: F811
    a, w, b = bf(1, K, seed=1), bf(N, K, scale=0.05, seed=2), bf(N, seed=3) if bias else None
    x = torch.randn(1, N, device=DEV)
    one, two = x.clone(), both(x)
    for rows, r in ((a, one), (both(a), two)):
        C.gemv(rows, w, b, 4, 0, None, None, 0.0, r, None, None, None, None, 0, 0, 0, None)
    assert torch.equal(one[0], two[0])


@pytest.mark.parametrize("K", [2056, 4096])
@pytest.mark.parametrize("norm,rope,bias", [(1, False, True), (2, True, False), (2, True, True)])
def test_qkv(C, K, norm, rope, bias):  # noqa: F811
    q, kv, hd = 3072, 768, 128
    N = q + 2 * kv
    x, g, w = torch.randn(1, K, device=DEV), bf(K, seed=1), bf(N, K, scale=0.05, seed=2)
    beta, b = (bf(K, seed=3) if norm == 1 else None), bf(N, seed=4) if bias else None
    table = torch.randn(64, hd // 2, 2, device=DEV) if rope else None
    got = []
    for rows in (x, both(x)):
        m = rows.shape[0]
        caches = [torch.zeros(3, kv // hd, 64, hd, dtype=torch.bfloat16, device=DEV) for _ in "kv"]
        slot = torch.tensor([2, 0][:m], dtype=torch.int32, device=DEV)
        pos = torch.full((m,), 37, dtype=torch.int32, device=DEV)
        out = C.gemv(rows, w, b, 6, norm, g, beta, 1e-5, None, *caches, slot, pos, q, kv, hd, table)
        got.append([out[0]] + [c[2, :, 37] for c in caches])
    for one, two in zip(*got):
        assert torch.equal(one, two) and bool(one.any())
