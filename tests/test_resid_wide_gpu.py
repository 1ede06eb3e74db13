"""Residual rows around 2^21 columns, from where 256 of them pass what the 256 x 256 kernel's resource holds."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2 ** 21 - 64, 2 ** 21])
def test_wide_rows(N):
    """Two fp32 sums of K products, off by K + 3 ulp of their sizes each."""
    from llm_sharding_demo_amd import _C as C

    M, K = 300, 64
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    x = torch.ones(M, N, device="cuda")
    assert C.gemm_big_tiles(M, N, K, 1)
    C.linear_residual(a, w, None, x, 1, 1, None, False)
    for c in range(0, N, 2 ** 18):
        part = w[c: c + 2 ** 18].float()
        off = 2 * (K + 3) * 2.0 ** -24 * (a.float().abs() @ part.abs().T + 1)
        assert bool(((x[:, c: c + 2 ** 18] - 1 - a.float() @ part.T).abs() <= off).all()), c
