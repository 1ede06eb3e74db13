"""Decode GEMM of up to 256 rows (csrc/kernels/gemm_deep.hip) against float64: every row class
and tile width, partial tiles of rows and columns, K down to one k-step and one k-step a split.

Bound per element: sums of K products in fp32 in any order are at most K 2^-24 sum |a w| off;
what is stored in bf16 is rounded once more (2^-8 of the value covers it and the activation)."""
import pytest
import torch

from llm_sharding_demo_amd.ops import reference as ref
from llm_sharding_demo_amd.ops.hip import interleave_gate_up

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def C():
    from llm_sharding_demo_amd import _C
    return _C


@pytest.fixture(scope="module")
def CNT():
    return torch.zeros(1 << 16, dtype=torch.int32, device=DEV)


def data(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * 1000 + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    return rnd(M, K).bfloat16(), (rnd(N, K) * 0.05).bfloat16(), (rnd(N) * 0.1).bfloat16()


def check(got, want, a, w, rounded=True, more=0.0):
    spread = (a.double().abs() @ w.double().abs().T) * (a.shape[1] + 8) * 2.0 ** -24
    bound = spread + more + (2.0 ** -8 * want.abs() if rounded else 2.0 ** -23 * want.abs())
    over = ((got.double() - want).abs() - bound).max()
    assert float(over) <= 0, float(over)


# columns: 16-wide tiles with a ragged end, 32- and 64-wide ones, K with and without 128-wide steps
@pytest.mark.parametrize("M", [9, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K", [(64, 64), (1616, 128), (4160, 192), (2624, 1024), (10304, 320), (20000, 128)])
def test_epilogues(C, CNT, M, N, K):
    a, w, b = data(M, N, K)
    y = a.double() @ w.double().T
    check(C.linear_f32(a, w, True, 1, CNT), y, a, w, rounded=False)
    check(C.linear(a, w, b, 0, True, 1, CNT), y + b.double(), a, w)
    x = torch.randn(M, N, device=DEV)
    want = x.double() + y + b.double()
    if N % 64 == 0:
        C.linear_residual(a, w, b, x, 3 if K >= 256 else 1, False, CNT, False)
        check(x, want, a, w, rounded=False)
    if N % 32 == 0:
        n = N // 2
        got = C.linear(a, interleave_gate_up(w, n), None, 2, True, 1, CNT)
        g, u = y.split(n, 1)
        # d silu <= 1.1, so the product moves by the sums' error times the other factor
        spread = (a.double().abs() @ w.double().abs().T) * (K + 8) * 2.0 ** -24
        more = 1.1 * (spread[:, :n] * u.abs() + spread[:, n:] * g.abs()) + 1e-6
        want = torch.nn.functional.silu(g) * u
        assert bool(((got.double() - want).abs() <= more + 2.0 ** -7 * want.abs()).all())
    assert int(CNT.abs().sum()) == 0


@pytest.mark.parametrize("M", [9, 40, 64, 96, 128, 150, 193])
@pytest.mark.parametrize("N,K,S", [(64, 64, 1), (1664, 128, 2), (2048, 1024, 4), (4096, 1024, 8), (768, 768, 6), (768, 768, 12)])
def test_slabs(C, CNT, M, N, K, S):
    a, w, _ = data(M, N, K)
    x = torch.zeros(M, N, device=DEV)
    prev = C.gemm_slab_bf16()
    C.gemm_set_slab_bf16(0)
    try:
        slab = C.linear_residual(a, w, None, x, S, True, CNT, True)
    finally:
        C.gemm_set_slab_bf16(int(prev))
    assert tuple(slab.shape) == (S, M, N)
    check(slab.double().sum(0), a.double() @ w.double().T, a, w, rounded=False)


@pytest.mark.parametrize("M", [9, 33, 64, 96, 128, 129, 256])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("heads,kv,hd,K", [(4, 2, 64, 128), (25, 25, 64, 320), (32, 8, 128, 256)])
def test_qkv(C, CNT, M, rope, heads, kv, hd, K):
    N = (heads + 2 * kv) * hd
    a, w, b = data(M, N, K)
    slots, seq = M + 1, 40
    kc, vc = (torch.zeros(slots, kv, seq, hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    slot = torch.randperm(M, device=DEV).int()
    pos = (torch.arange(M, device=DEV) * 7 % seq).int()
    table = torch.randn(seq, hd // 2, 2, device=DEV) if rope else None
    q = C.linear_qkv(a, w, b, kc, vc, slot, pos, heads * hd, kv * hd, hd, table, True, 1, CNT)
    y = a.double() @ w.double().T + b.double()
    if rope:
        t = y[:, : (heads + kv) * hd].reshape(M, heads + kv, hd // 2, 2)
        c, s = (table[pos.long()].double()[:, None, :, i] for i in (0, 1))
        turned = torch.stack([t[..., 0] * c - t[..., 1] * s, t[..., 1] * c + t[..., 0] * s], -1)
        y = torch.cat([turned.reshape(M, -1), y[:, (heads + kv) * hd:]], 1)
    got = torch.cat([q] + [t[slot.long(), :, pos.long()].reshape(M, -1) for t in (kc, vc)], 1)
    tol = 2.0 ** -7 * y.abs() + 16 * (K + 8) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - y).abs() <= tol + 1e-5).all())
    used = torch.zeros(slots, seq, dtype=torch.bool, device=DEV)
    used[slot.long(), pos.long()] = True
    assert int((kc.abs().sum((1, 3)) > 0).logical_and(~used).sum()) == 0  # nothing else is written


def test_segment_maxima_and_reference(C, CNT):
    a, w, _ = data(40, 20032, 256)
    seg = torch.empty(40, 20032 // 8, device=DEV)
    y = C.linear_f32(a, w, True, 1, CNT, seg)
    assert torch.equal(seg, y.reshape(40, -1, 8).amax(-1))
    check(y, ref.linear(a, w).double(), a, w, rounded=False, more=1e-4)


def test_same_bits_twice(C, CNT):
    a, w, b = data(40, 2624, 2048)
    y = C.linear(a, w, b, 1, True, 1, CNT)
    assert all(torch.equal(C.linear(a, w, b, 1, True, 1, CNT), y) for _ in range(4))


@pytest.mark.parametrize("M,N,K,S,want", [(40, 4096, 14336, 8, 4), (40, 4096, 4096, 5, 4), (64, 2048, 2048, 4, 4),
                                          (8, 4096, 4096, 5, 5), (129, 4096, 4096, 5, 5), (40, 768, 96, 2, 2), (40, 768, 384, 4, 1), (9, 64, 128, 1, 1)])
def test_slab_splits(M, N, K, S, want):
    from llm_sharding_demo_amd.ops.routing import Routing

    assert Routing.slab_splits(M, N, K, S) == want
