"""Decode products of wide outputs: blocks of 128 columns, and column tiles that start their sums at places of K of their own."""

import pytest
import torch

from .test_gemm_deep_gpu import C  # noqa: F401

DEV, F64 = "cuda:0", torch.float64
BF16, GELU, SILU, F32 = 0, 1, 2, 3

# rows and columns of a block: M, N, K.  K of 2048 and 4096 is turned, the others' sums start at the first k
WIDE = [((16, 128), 1, 28672, 2048), ((16, 128), 16, 28640, 2048), ((32, 128), 17, 32000, 2048), ((32, 128), 32, 22528, 64),
        ((48, 128), 40, 28656, 4096), ((48, 128), 48, 50304, 192), ((64, 128), 64, 28672, 2048), ((64, 128), 49, 32016, 2112),
        ((96, 128), 65, 32000, 2048), ((96, 128), 96, 28688, 192), ((128, 128), 97, 32000, 2048), ((128, 128), 128, 29008, 2048),
        ((32, 64), 30, 16384, 4096), ((48, 64), 33, 11264, 2048), ((48, 96), 96, 11264, 2048)]


@pytest.mark.parametrize("shape,M,N,K", WIDE)
def test_rule(shape, M, N, K):
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    for epi in (BF16, GELU, F32) + ((SILU,) if N % 32 == 0 else ()):
        assert _C.gemm_on_deep(M, N, K, epi, 1, 1) and _C.gemm_deep_shape(M, N, K, epi, 1) == shape
    assert _C.gemm_deep_shape(48, 40960, 1600, F32, 1) == (48, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,M,N,K", WIDE)
def test_products(C, shape, M, N, K):  # noqa: F811
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g).bfloat16()
    ad, wd = a.to(DEV), w.to(DEV)
    acc = (a.to(DEV).to(F64) @ wd.to(F64).T).cpu()
    off = (K + 3) * 2.0 ** -24 * (ad.to(F64).abs() @ wd.to(F64).abs().T).cpu()

    def near(got, want, slack, step=2.0 ** -8):
        return bool(((got.cpu().to(F64) - want).abs() <= slack + step * want.abs()).all())
    assert near(C.linear_f32(ad, wd, 1, 1, None), acc, off, 0.0)
    y = acc + b.to(F64)
    assert near(C.linear(ad, wd, b.to(DEV), BF16, 1, 1, None), y, off + 2.0 ** -23 * y.abs())
    gelu = y * 0.5 * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (y + 0.044715 * y ** 3)))
    assert near(C.linear(ad, wd, b.to(DEV), GELU, 1, 1, None), gelu, 2 * off + 2.0 ** -20)
    if N % 32 == 0:
        gate, up = (acc.reshape(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1))
        size = off.reshape(M, N // 32, 2, 16).amax(2).reshape(M, N // 2)
        both = (1.1 * up.abs() + gate.abs() + 1) * size + 2.0 ** -20 * (1 + gate.abs() * up.abs())
        assert near(C.linear(ad, wd, None, SILU, 1, 1, None), gate / (1 + torch.exp(-gate)) * up, both)


@pytest.mark.gpu
def test_rows_of_w_in_a_wider_tensor(C):  # noqa: F811
    """Rows 4 KB apart of which fewer k's are taken, and whole rows at another stride: not turned, the same results."""
    g = torch.Generator().manual_seed(5)
    a, w = torch.randn(20, 4096, generator=g).bfloat16(), (torch.randn(16384, 4096, generator=g) / 64).bfloat16().to(DEV)
    for k in (2112, 2048):
        ak, wk = a[:, :k].contiguous().to(DEV), w[:, :k]
        want = (ak.to(F64) @ wk.to(F64).T).cpu()
        off = (k + 3) * 2.0 ** -24 * (ak.to(F64).abs() @ wk.to(F64).abs().T).cpu()
        assert bool(((C.linear_f32(ak, wk, 1, 1, None).cpu().to(F64) - want).abs() <= off).all())
