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


# the line of the rule: its blocks' last round, the slots behind K, one item a wave
RULE = [(28672, 4096, 2, 2, True), (11264, 1664, 2, 2, True), (11264, 1536, 2, 2, False), (11232, 2048, 2, 2, False),
        (16384, 3072, 2, 2, True), (16384, 2688, 2, 2, False), (14336, 4096, 2, 2, False), (28672, 4096, 2, 0, False),
        (16384, 2560, 3, 2, True), (16384, 2552, 3, 1, False), (50304, 4096, 3, 2, False), (128256, 4096, 3, 2, True),
        (6144, 3584, 6, 2, True), (6144, 3456, 6, 2, False), (8192, 4096, 6, 2, False), (5120, 4096, 6, 1, False),
        (4096, 4096, 4, 0, True), (8192, 4096, 4, 0, False), (12288, 4096, 4, 0, True), (4608, 14336, 4, 0, False),
        (8192, 11072, 4, 0, True), (8192, 11008, 4, 0, False), (4096, 5120, 4, 0, False), (4094, 4096, 4, 0, False)]


@pytest.mark.parametrize("N,K,epi,norm,want", RULE)
def test_rule(C, N, K, epi, norm, want):  # noqa: F811
    assert C.gemv_on_stream(N, K, epi, norm) == want


# launches of the rule, ragged: rows behind the last item, items behind the last wave's, slots behind K
@pytest.mark.parametrize("N,K", [(11296, 1664), (11264, 2040), (16448, 3072), (28704, 3208), (22016, 4096)])
def test_gated_of_the_rule(C, N, K):  # noqa: F811
    assert C.gemv_on_stream(N, K, 2, 2)
    test_gated(C, N, K, 0)


@pytest.mark.parametrize("N,K", [(31997, 2560), (28674, 3208), (57400, 4096), (65531, 2568)])
def test_head_of_the_rule(C, N, K):  # noqa: F811
    assert C.gemv_on_stream(N, K, 3, 2)
    test_head(C, N, K, 2)


@pytest.mark.parametrize("N", [4096, 5633, 6143, 11265])
@pytest.mark.parametrize("K", [3584, 3592, 4096, 11072, 11080, 14328, 14336])
def test_residual_of_the_rule(C, N, K):  # noqa: F811
    assert C.gemv_on_stream(N, K, 4, 0)
    test_residual(C, N, K, True)


@pytest.mark.parametrize("heads,kv", [(32, 6), (70, 12)])
@pytest.mark.parametrize("K", [3584, 3592, 4096])
def test_qkv_of_the_rule(C, heads, kv, K):  # noqa: F811
    q, kvs, hd = heads * 128, kv * 128, 128
    N = q + 2 * kvs
    assert C.gemv_on_stream(N, K, 6, 2)
    x, g, w, table = torch.randn(1, K, device=DEV), bf(K, seed=1), bf(N, K, scale=0.05, seed=2), torch.randn(64, hd // 2, 2, device=DEV)
    got = []
    for rows in (x, both(x)):
        m = rows.shape[0]
        caches = [torch.zeros(3, kv, 64, hd, dtype=torch.bfloat16, device=DEV) for _ in "kv"]
        slot, pos = torch.tensor([2, 0][:m], dtype=torch.int32, device=DEV), torch.full((m,), 37, dtype=torch.int32, device=DEV)
        out = C.gemv(rows, w, None, 6, 2, g, None, 1e-5, None, *caches, slot, pos, q, kvs, hd, table)
        got.append([out[0]] + [c[2, :, 37] for c in caches])
    for one, two in zip(*got):
        assert torch.equal(one, two) and bool(one.any())
