"""Epilogues of the 256 x 256 GEMM at edges of its tile and k-ring, against 64
bits: an fp32 sum of K products is off by (K + 2) ulp of their sizes, and a bf16
result by half a bf16 step more.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


@pytest.fixture(scope="module")
def C():
    from llm_sharding_demo_amd import _C as C

    C.gemm_set_big_min(1)
    yield C
    C.gemm_set_big_min(160)


def near(got, want, slack):
    got = got.cpu().to(F64)
    step = 2.0 ** -8 if slack is not None else 0.0
    return bool(((got - want).abs() <= slack + step * want.abs()).all())


# (256 rows: the deep ring)
@pytest.mark.parametrize("M,N,K", [(256, 64, 64), (256, 256, 128), (257, 288, 192), (300, 1600, 64), (511, 544, 448),
                                   (512, 64, 64), (512, 256, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_epilogues(C, M, N, K, bias):
    assert C.gemm_on_deep(M, N, K, 0, 1, 1) == (M <= 256)
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g).bfloat16() if bias else None
    x = torch.randn(M, N, generator=g)
    bd = b.to(DEV) if bias else None
    acc = a.to(F64) @ w.to(F64).T
    off = (K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T)
    y = acc + (b.to(F64) if bias else 0)
    at = (a.to(DEV), w.to(DEV))
    assert near(C.linear(*at, bd, 0, 1, 1, None), y, off + 2.0 ** -23 * y.abs())
    gelu = y * 0.5 * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (y + 0.044715 * y ** 3)))
    assert near(C.linear(*at, bd, 1, 1, 1, None), gelu, 2 * off + 2.0 ** -20)  # |gelu'| < 1.13
    xd = x.to(DEV)
    C.linear_residual(*at, bd, xd, 1, 1, None, False)
    assert bool(((xd.cpu().to(F64) - x.to(F64) - y).abs() <= off + 2.0 ** -22 * (y.abs() + x.abs())).all())
    if bias:
        return
    assert bool(((C.linear_f32(*at, 1, 1, None).cpu().to(F64) - acc).abs() <= off).all())
    gate, up = (acc.reshape(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1))
    size = off.reshape(M, N // 32, 2, 16).amax(2).reshape(M, N // 2)
    both = (1.1 * up.abs() + gate.abs() + 1) * size + 2.0 ** -20 * (1 + gate.abs() * up.abs())
    assert near(C.linear(*at, None, 2, 1, 1, None), gate / (1 + torch.exp(-gate)) * up, both)
    slab = C.linear_residual(*at, None, xd, 1, 1, None, True)
    slab = slab[0] if slab.dim() == 3 else slab
    assert near(slab, acc, off)


# 1 .. 8 K-tiles a split, which ends in front of columns that are 2^30 times as large: nothing
# that is staged behind a split's last tile may reach its sum
@pytest.mark.parametrize("kind", [4, 1])
@pytest.mark.parametrize("tiles", range(1, 9))
def test_k_tiles(C, kind, tiles):
    M, N, K = 300, 288, 128 * tiles
    g = torch.Generator().manual_seed(tiles)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    a[:, K // 2:] *= 2.0 ** 30
    C.gemm_set_big_kind(kind)
    try:
        slabs = C.linear_residual(a.to(DEV), w.to(DEV), None, torch.zeros(M, N, device=DEV), 2, 1, None, False)
    finally:
        C.gemm_set_big_kind(4)
    assert slabs.shape[0] == 2
    for h, got in enumerate(slabs):
        part = slice(h * K // 2, (h + 1) * K // 2)
        x, y = a[:, part].to(F64), w[:, part].to(F64)
        assert near(got.float(), x @ y.T, (K + 3) * 2.0 ** -24 * (x.abs() @ y.abs().T))


# 512 and 520 tiles of 128 x 128: one round of two a CU, and 132 tiles of 256 x 256
@pytest.mark.parametrize("N", [8192, 8320])
def test_more_than_a_round(C, N):
    M, K = 1000, 192
    g = torch.Generator().manual_seed(N)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    acc = a.to(F64) @ w.to(F64).T
    off = (K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T)
    C.gemm_set_big_min(160)
    try:
        assert C.gemm_big_tiles(M, N, K, 1) == (N > 8192)
        assert near(C.linear(a.to(DEV), w.to(DEV), None, 0, 1, 1, None), acc, off)
        x = torch.randn(M, N, generator=g)
        xd = x.to(DEV)
        C.linear_residual(a.to(DEV), w.to(DEV), None, xd, 1, 1, None, False)
    finally:
        C.gemm_set_big_min(1)
    assert bool(((xd.cpu().to(F64) - x.to(F64) - acc).abs() <= off + 2.0 ** -22 * (acc.abs() + x.abs())).all())
