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


def test_turned():
    """Rows whole 4 KB apart, all blocks under way at once, blocks of 64 columns and more."""
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    for shape, M, N, K in WIDE:
        assert _C.gemm_deep_turned(M, N, K, K, F32, 1) == (K in (2048, 4096))
    for M, N, K, ldw in ((20, 16384, 2112, 4096), (20, 16384, 2048, 2112), (20, 128256, 4096, 4096), (20, 6144, 4096, 4096)):
        assert not _C.gemm_deep_turned(M, N, K, ldw, F32, 1)
    assert _C.gemm_deep_turned(20, 16384, 2048, 4096, F32, 1) and not _C.gemm_deep_turned(20, 16384, 2048, 2048, 5, 2)


def test_wide_blocks_all_start_at_once():
    """Blocks of 96 and 128 rows by 128 columns, one of which a CU holds: never more than CUs."""
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    for M in range(65, 129):
        for N in range(32, 70000, 32 * 13):
            if _C.gemm_on_deep(M, N, 2048, F32, 1, 1) and _C.gemm_deep_shape(M, N, 2048, F32, 1)[1] == 128:
                assert (N + 127) // 128 <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("k,stride", [(2112, 4096), (2048, 4096), (2048, 2112), (2048, 2048)])
def test_rows_of_w_in_a_wider_tensor(C, k, stride):  # noqa: F811
    """Rows 4 KB apart of which fewer k's are taken, turned where those are whole 4 KB too, and rows at another stride."""
    g = torch.Generator().manual_seed(5)
    a, w = torch.randn(20, k, generator=g).bfloat16(), (torch.randn(16384, stride, generator=g) / 64).bfloat16().to(DEV)
    assert C.gemm_deep_turned(20, 16384, k, stride, F32, 1) == (k == 2048 and stride != 2112)
    ak, wk = a.to(DEV), w[:, :k]
    want = (ak.to(F64) @ wk.to(F64).T).cpu()
    off = (k + 3) * 2.0 ** -24 * (ak.to(F64).abs() @ wk.to(F64).abs().T).cpu()
    assert bool(((C.linear_f32(ak, wk, 1, 1, None).cpu().to(F64) - want).abs() <= off).all())
