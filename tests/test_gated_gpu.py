"""Gated activations in the products' epilogues, each kind at each kernel, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.mark.parametrize("glu", [0, 1, 2])
@pytest.mark.parametrize("M,kind", [(1, 0), (17, 0), (17, 1), (130, 0), (130, 1), (256, 0), (300, 1), (513, 1)])
def test_gated(glu, M, kind):
    """A sum of K products is off by K + 3 ulp of their sizes, the activation's slope is below
    1.13, its own functions' error some 2^-20, the result's rounding 2^-8."""
    from llm_sharding_demo_amd import _C as C

    N, K, s = 384, 192, 1.25
    g = torch.Generator().manual_seed(M + glu)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * 2 * K ** -0.5).bfloat16()
    split = lambda t: (t.reshape(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1))  # noqa: E731
    gate, up = split(a.to(F64) @ w.to(F64).T)
    eg, eu = split((K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T))
    if glu == 2:
        gc, uc = gate.clamp(max=s), up.clamp(-s, s) + 1
        want = gc * torch.sigmoid(1.702 * gc) * uc
    else:
        x, uc, eg, eu = s * gate, s * up, s * eg, s * eu
        want = (x * torch.sigmoid(x) if glu == 0 else torch.nn.functional.gelu(x, approximate="tanh")) * uc
    C.gemm_set_big_min(1 if M > 512 else 160)
    try:
        if M == 513:
            assert C.gemm_big_tiles(M, N, K, 1)
        got = C.linear(a.cuda(), w.cuda(), None, 2 + glu, kind, 1, None, None, s).cpu().to(F64)
    finally:
        C.gemm_set_big_min(160)
    slack = 1.13 * uc.abs() * eg + (want / uc).abs().nan_to_num(0) * eu + 2.0 ** -20 * (1 + want.abs()) + 2.0 ** -8 * want.abs()
    assert bool(((got - want).abs() <= slack).all())
