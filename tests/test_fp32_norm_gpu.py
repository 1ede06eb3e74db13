"""RMS norms of fp32 rows with slabs, against 64 bits: rows of whole 16 bytes in registers up to
8192 columns, others and unaligned ones column by column.

A row's sum of S slabs is off by S ulp (2^-24) of their sizes, a sum of H squares relatively by
the longest chain of its additions (H / 256 in a thread, six and four between them)."""

import pytest
import torch

from .test_timisun_gpu import C, rand  # noqa: F811,F401

pytestmark = pytest.mark.gpu
DEV, F64, ULP = "cuda:0", torch.float64, 2.0 ** -24


@pytest.mark.parametrize("H", [4, 10, 1020, 1024, 1028, 2052, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("S", [0, 1, 4, 5, 9])
@pytest.mark.parametrize("off", [0, 1])
def test_rows(C, H, S, off):  # noqa: F811
    T, eps = 3, 1e-3
    x, w, slab = rand(T, H, seed=1), rand(H, seed=2), rand(max(S, 1), T, H, seed=3)
    room = torch.empty(T * H + off, device=DEV)
    xd = room[off:].view(T, H)
    xd.copy_(x)
    out = C.norm_fp32(xd, slab.to(DEV) if S else None, w.to(DEV), eps, None, True, 0, 0.5).cpu().to(F64)
    got = xd.cpu().to(F64)
    want, size = x.to(F64), x.to(F64).abs()
    if S:
        want, size = want + slab.to(F64).sum(0), size + slab.to(F64).abs().sum(0)
    assert bool(((got - want).abs() <= S * ULP * size).all())
    y = got / torch.sqrt(got.pow(2).mean(1, keepdim=True) + eps) * (w.to(F64) + 0.5)
    assert bool(((out - y).abs() <= (H // 256 + 20) * ULP * (y.abs() + 2.0 ** -20)).all())
    rows = torch.tensor([2, 0], dtype=torch.int32, device=DEV)
    few = C.norm_fp32(xd, None, w.to(DEV), eps, rows, True, 0, 0.5).cpu()
    assert torch.equal(few.to(F64), C.norm_fp32(xd, None, w.to(DEV), eps, None, True, 0, 0.5).cpu().to(F64)[[2, 0]])


def test_slabs_alone(C):  # noqa: F811
    x, slab = rand(5, 2048, seed=1), rand(3, 5, 2048, seed=2)
    xd = x.to(DEV)
    assert C.norm_fp32(xd, slab.to(DEV), None, 1e-5, None, False, 0, 0.0) is None
    assert torch.equal(xd.cpu(), ((x + slab[0]) + slab[1]) + slab[2])


# both sides of the line for rows with slabs, and rows without
@pytest.mark.parametrize("H", [64, 380, 384, 388])
@pytest.mark.parametrize("S", [0, 1, 5])
def test_narrow_rows(C, H, S):  # noqa: F811
    test_rows(C, H, S, 0)
