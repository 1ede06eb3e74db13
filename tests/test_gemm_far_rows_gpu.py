"""bf16 products of rows that lie so far apart that a tile's byte offsets pass 32 bits (views of much
wider rows), against 64 bits: an fp32 sum of K products is off by (K + 2) ulp of their sizes, a
bf16 result by half a bf16 step more.
"""

import pytest
import torch

DEV, F64 = "cuda:0", torch.float64
NEAR, FAR = (1 << 22) - 8, 1 << 22  # row strides on both sides of the line


@pytest.fixture(scope="module")
def C():
    from llm_sharding_demo_amd import _C as C

    return C


# a tile's last row, of 256, and its last k-step are within a resource's 2^31 - 1 bytes, or the call is far
@pytest.mark.parametrize("K", [64, 2048, 16384])
def test_line(C, K):
    for ld in (K, NEAR // 2, NEAR - K // 8, NEAR, FAR, 1 << 24, 1 << 33):
        far = 255 * ld * 2 + 2 * K >= (1 << 31) - 1
        for M, N, rows in ((300, 64, (ld, K)), (1024, 64, (K, ld))):
            got = C.gemm_far_rows(M, N, K, *rows)
            assert got or not far
            assert not got or 257 * ld * 2 + 2 * K >= 1 << 31
    assert not C.gemm_far_rows(1, 64, K, 1 << 33, K)  # one row lies nowhere else


@pytest.mark.gpu
@pytest.mark.parametrize("kind,splits", [(1, 1), (2, 1), (3, 1), (2, 2), (3, 2)])
@pytest.mark.parametrize("step", [NEAR, FAR, 1 << 23, 1 << 24, (1 << 24) + 8, 1 << 25])
@pytest.mark.parametrize("operand", ["a", "w"])
def test_rows_far_apart(C, kind, splits, step, operand):
    M, N, K = (300, 144, 256) if operand == "a" else (264, 272, 256)
    g = torch.Generator().manual_seed(M + kind)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    assert not C.gemm_on_deep(M, N, K, 0, kind, splits)
    src = a if operand == "a" else w
    room = torch.empty((src.shape[0] - 1) * step + K, dtype=torch.bfloat16, device=DEV).as_strided(src.shape, (step, 1))
    room.copy_(src)
    ad, wd = (room, w.to(DEV)) if operand == "a" else (a.to(DEV), room)
    acc = a.to(F64) @ w.to(F64).T
    off = (K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T)
    tickets = torch.zeros(1024, dtype=torch.int32, device=DEV)
    for big in (1, 160, 1 << 16):  # 256 x 256 tiles, by size, 128 x 128 tiles
        C.gemm_set_big_min(big)
        try:
            y = C.linear(ad, wd, None, 0, kind, splits, tickets).cpu().to(F64)
            slabs = C.linear_residual(ad, wd, None, torch.zeros(M, N, device=DEV), 2, kind, tickets, True).cpu().to(F64)
        finally:
            C.gemm_set_big_min(160)
        assert bool(((y - acc).abs() <= off + 2.0 ** -8 * acc.abs()).all())
        for h, got in enumerate(slabs):
            part = slice(h * K // 2, (h + 1) * K // 2)
            want = a[:, part].to(F64) @ w[:, part].to(F64).T
            assert bool(((got - want).abs() <= off + 2.0 ** -8 * want.abs()).all())
    assert not tickets.any()
