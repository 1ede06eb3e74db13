"""The prompt GEMM on four waves: each of its tiles and epilogues at edges of rows, columns and K-tiles, against
the 256 x 256 kernel bit for bit (the same products, summed in the same order) and against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


@pytest.fixture(scope="module")
def C():
    from llm_sharding_demo_amd import _C as C

    return C


def both(C, call):
    got = call()
    C.gemm_set_big_min(1)
    try:
        return got, call()
    finally:
        C.gemm_set_big_min(160)


def operands(M, N, K, lda=0, ldw=0):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    wide = [torch.randn(r, K + x, generator=g, device=DEV).bfloat16()[:, :K] for r, x in ((M, lda), (N, ldw))]
    return wide[0], wide[1] * K ** -0.5 if ldw == 0 else wide[1], torch.randn(N, generator=g, device=DEV).bfloat16(), g


# 1, 3, 5, 7 K-tiles and even ones; one row, one block of columns behind a tile; row strides of their own
@pytest.mark.parametrize("tile,M,N,K", [(222, 257, 5472, 64), (222, 641, 3040, 128), (222, 2003, 1504, 64), (322, 1030, 7200, 64),
                                        (322, 577, 6944, 320), (331, 1030, 7200, 128), (331, 2003, 4128, 192), (331, 2003, 4256, 448),
                                        (422, 3333, 7200, 64), (422, 3333, 8416, 448),
                                        (431, 1000, 8224, 448), (431, 2003, 4448, 512), (341, 257, 24608, 512), (341, 380, 25472, 576)])
@pytest.mark.parametrize("wide", [0, 72])
def test_epilogues(C, tile, M, N, K, wide):
    """An fp32 sum of K products is off by K + 2 ulp of their sizes, a bf16 result by half a bf16 step more."""
    assert C.gemm_on_wave4(M, N, K, 0, 1) == tile
    a, w, b, g = operands(M, N, K, wide, wide)
    acc, off = a.to(F64) @ w.to(F64).T, (K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T)
    got, same = both(C, lambda: C.linear(a, w, None, 0, 1, 1, None))
    assert torch.equal(got, same) and bool(((got.to(F64) - acc).abs() <= off + 2.0 ** -8 * acc.abs()).all())
    for call in (lambda: C.linear(a, w, b, 0, 1, 1, None), lambda: C.linear(a, w, b, 1, 1, 1, None),
                 *(lambda k=k: C.linear(a, w, None, k, 1, 1, None, None, 1.25) for k in (2, 3, 4))):
        assert torch.equal(*both(C, call))
    x = torch.randn(M, N, generator=g, device=DEV)

    def add():
        y = x.clone()
        C.linear_residual(a, w, b, y, 1, 1, None, False)
        return y
    got, same = both(C, add)
    want = x.to(F64) + b.to(F64) + acc
    assert torch.equal(got, same) and bool(((got.to(F64) - want).abs() <= off + 2.0 ** -22 * (want.abs() + x.abs() + b.abs())).all())
    assert torch.equal(*both(C, lambda: C.linear_residual(a, w, None, x, 1, 1, None, True)))


# splits of unequal lengths; a split's sums end in front of columns 2^30 times as large
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("tile,M,N,K,S", [(222, 257, 2720, 128, 2), (222, 700, 1696, 192, 2), (222, 257, 3360, 320, 3),
                                          (322, 385, 8224, 128, 2), (322, 300, 7776, 320, 3), (331, 641, 5408, 320, 2),
                                          (331, 257, 7200, 448, 3), (422, 1030, 6432, 128, 2), (422, 1030, 7392, 320, 3)])
def test_slabs(C, tile, M, N, K, S, fp32):
    assert C.gemm_on_wave4(M, N, K, 5, S) == tile
    a, w, _, _ = operands(M, N, K)
    at = [K // 64 * s // S * 64 for s in range(S + 1)]
    a[:, at[1]:] *= 2.0 ** 30
    x = torch.zeros(M, N, device=DEV)
    C.gemm_set_slab_bf16(int(not fp32))
    try:
        got, same = both(C, lambda: C.linear_residual(a, w, None, x, S, 1, None, False))
    finally:
        C.gemm_set_slab_bf16(1)
    assert got.shape[0] == S and got.dtype == (torch.float32 if fp32 else torch.bfloat16) and torch.equal(got, same)
    for s in range(S):
        p, q = a[:, at[s]:at[s + 1]].to(F64), w[:, at[s]:at[s + 1]].to(F64)
        y = p @ q.T
        step = 0 if fp32 else 2.0 ** -8
        assert bool(((got[s].to(F64) - y).abs() <= (K + 3) * 2.0 ** -24 * (p.abs() @ q.abs().T) + step * y.abs()).all())


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("tile,M,heads,kv,hd,K", [(222, 2003, 55, 5, 16, 64), (222, 1030, 19, 5, 64, 64), (222, 257, 47, 5, 96, 64),
                                                  (322, 1500, 47, 5, 96, 64), (322, 1030, 47, 5, 128, 64), (331, 2003, 55, 5, 64, 192),
                                                  (331, 1500, 53, 2, 96, 192), (422, 2003, 39, 5, 256, 64), (431, 2003, 43, 2, 96, 448),
                                                  (431, 1000, 55, 5, 128, 448), (431, 577, 48, 2, 256, 448), (431, 1030, 117, 5, 64, 448),
                                                  (341, 370, 251, 5, 96, 640), (341, 300, 97, 2, 256, 640)])
def test_qkv(C, tile, M, heads, kv, hd, K, rope):
    N, seq = (heads + 2 * kv) * hd, 40
    assert C.gemm_on_wave4(M, N, K, 6, 1) == tile
    a, w, b, g = operands(M, N, K)
    slot, pos = torch.randperm(M, generator=g, device=DEV).int(), (torch.arange(M, device=DEV) * 7 % seq).int()
    table = torch.randn(seq, hd // 2, 2, generator=g, device=DEV) if rope else None

    def call():
        kc, vc = (torch.zeros(M + 1, kv, seq, hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        return (C.linear_qkv(a, w, b, kc, vc, slot, pos, heads * hd, kv * hd, hd, table, 1, 1, None), kc, vc)
    for got, same in zip(*both(C, call)):
        assert torch.equal(got, same)


def test_line(C):
    """Nothing else is taken: few rows, few tiles, part K-tiles, fp32 results, splits without slabs, far rows."""
    M, N, K = 2003, 4256, 448
    assert C.gemm_on_wave4(M, N, K, 0, 1) == 331 and C.gemm_on_wave4(M, N, K, 5, 2) == 322
    for call in ((256, N, K, 0, 1), (1000, 2048, K, 0, 1), (M, N, 432, 0, 1), (M, N, K, 3, 1), (M, N, K, 0, 2), (M, N, K, 5, 8),
                 (4096, 4096, 4096, 0, 1)):
        assert C.gemm_on_wave4(*call) == 0
