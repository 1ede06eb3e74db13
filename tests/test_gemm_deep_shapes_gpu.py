"""Products of 50 to 256 rows, of more than 64 in blocks of fewer rows, at edges of rows, columns and the k-ring,
against 64 bits: an fp32 sum of K products is off by (K + 2) ulp of their sizes, and a bf16 result
by half a bf16 step more.
"""

import pytest
import torch

DEV, F64 = "cuda:0", torch.float64
BF16, GELU, SILU, F32, SLAB = 0, 1, 2, 3, 5

# (rows, columns of a block): (M, N) that take them
SHAPES = [((64, 32), 50, 2624), ((64, 32), 64, 2608), ((48, 32), 65, 3072), ((48, 32), 96, 3056), ((48, 64), 96, 6464),
          ((48, 64), 130, 4064), ((48, 80), 81, 8512), ((48, 80), 140, 5888), ((48, 96), 96, 11264), ((48, 96), 70, 11232),
          ((48, 64), 97, 4800), ((64, 64), 255, 4064), ((64, 64), 250, 3616), ((64, 80), 256, 4800), ((64, 80), 193, 4784),
          ((64, 96), 112, 11264), ((64, 96), 200, 5888)]


@pytest.mark.parametrize("shape,M,N", SHAPES)
def test_rule(shape, M, N):
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert _C.gemm_on_deep(M, N, 192, BF16, 1, 1)
    assert _C.gemm_deep_shape(M, N, 192, BF16, 1) == shape


# beside another lane's launches 160 rows and more stay in blocks that hold all of them
@pytest.mark.parametrize("M,N,lanes,shape", [(256, 4800, 2, (128, 64)), (256, 4800, 1, (64, 80)), (160, 4800, 2, (96, 64)),
                                             (159, 4800, 2, (48, 80)), (128, 4800, 2, (48, 64)), (256, 11264, 3, (128, 64)),
                                             (64, 2624, 2, (64, 32))])
def test_rule_with_lanes(M, N, lanes, shape):
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert _C.gemm_deep_shape(M, N, 192, BF16, 1, lanes) == shape


def test_shapes_that_have_no_kernel():
    """All of 65 rows and more in blocks of 32 columns: 96 rows in slabs only, 128 not at all."""
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    for M, rows in ((65, 96), (96, 96), (97, 128), (128, 128)):
        for epi, splits in ((BF16, [1]), (SILU, [1]), (SLAB, range(1, 65))):
            for S in splits:
                some = {_C.gemm_deep_shape(M, N, 4096, epi, S) for N in range(32, 32768 // S + 32, 16 if epi != SILU else 32)
                        if _C.gemm_on_deep(M, N, 4096, epi, 1, S)}
                assert (rows, 32) not in some or (epi == SLAB and rows == 96), (M, epi, S)


def test_launches_know_their_lanes():
    """Every product of a forward that shares the chip says so."""
    pytest.importorskip("llm_sharding_demo_amd._C")
    from llm_sharding_demo_amd.ops.hip import HipBackend, Residual

    seen = []

    class Calls:
        def __getattr__(self, name):
            def call(*args, lanes=1):
                seen.append((name, args[SIGNATURE[name]] if len(args) > SIGNATURE[name] else lanes))
                return torch.zeros(1)
            return call

    be = HipBackend.__new__(HipBackend)
    be.C, be.concurrency, be.fp32, be.lane, be._counters, be.decode, be._rope = Calls(), 2, False, 0, None, True, None
    a, w, x = torch.zeros(200, 1600).bfloat16(), torch.zeros(4800, 1600).bfloat16(), torch.zeros(200, 4800)

    class Meta:
        token_slots = token_pos = None
        q_size, kv_size, head_dim = 1600, 1600, 64

    be.linear(a, w)
    be.linear(a, w, out=x)
    be._linear_f32(a, w)
    be.logits(a, w)
    be.linear_residual(a, w, None, Residual(x))
    be._slabs(a, w, x)
    be.qkv_kv_append(a, w, None, None, None, Meta, Meta)
    assert len(seen) == 7 and all(n == 2 for _, n in seen), seen


SIGNATURE = {"linear": 9, "linear_f32": 6, "linear_residual": 9, "linear_qkv": 14}  # where lanes come by position


def near(got, want, slack, step):
    got = got.cpu().to(F64)
    return bool(((got - want).abs() <= slack + step * want.abs()).all())


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 192, 448])
@pytest.mark.parametrize("shape,M,N", SHAPES)
def test_products(shape, M, N, K):
    from llm_sharding_demo_amd import _C as C

    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    b, at = torch.randn(N, generator=g).bfloat16(), None
    at = (a.to(DEV), w.to(DEV))
    acc = a.to(F64) @ w.to(F64).T
    off = (K + 3) * 2.0 ** -24 * (a.to(F64).abs() @ w.to(F64).abs().T)
    y = acc + b.to(F64)
    assert near(C.linear(*at, b.to(DEV), BF16, 1, 1, None), y, off + 2.0 ** -23 * y.abs(), 2.0 ** -8)
    assert torch.equal(C.linear(*at, b.to(DEV), BF16, 1, 1, None, lanes=2), C.linear(*at, b.to(DEV), BF16, 1, 1, None))
    gelu = y * 0.5 * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (y + 0.044715 * y ** 3)))
    assert near(C.linear(*at, b.to(DEV), GELU, 1, 1, None), gelu, 2 * off + 2.0 ** -20, 2.0 ** -8)
    assert near(C.linear_f32(*at, 1, 1, None), acc, off, 0.0)
    x = torch.randn(M, N, generator=g)
    xd = x.to(DEV)
    C.linear_residual(*at, None, xd, 1, 1, None, False)
    assert near(xd, x.to(F64) + acc, off + 2.0 ** -22 * (acc.abs() + x.abs()), 0.0)
    if N % 32 == 0:
        gate, up = (acc.reshape(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1))
        size = off.reshape(M, N // 32, 2, 16).amax(2).reshape(M, N // 2)
        both = (1.1 * up.abs() + gate.abs() + 1) * size + 2.0 ** -20 * (1 + gate.abs() * up.abs())
        assert near(C.linear(*at, None, SILU, 1, 1, None), gate / (1 + torch.exp(-gate)) * up, both, 2.0 ** -8)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,S", [(256, 1600, 3), (128, 768, 6), (96, 1600, 2), (66, 1312, 2), (140, 800, 5)])
def test_slabs(M, N, S):
    from llm_sharding_demo_amd import _C as C

    K = 64 * (2 * S + 1)
    assert C.gemm_on_deep(M, N, K, SLAB, 1, S) and C.gemm_deep_shape(M, N, K, SLAB, S)[0] < min(M, 96)
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    slabs = C.linear_residual(a.to(DEV), w.to(DEV), None, torch.zeros(M, N, device=DEV), S, 1, None, True)
    ends = [K // 64 * s // S * 64 for s in range(S + 1)]
    for s, got in enumerate(slabs):
        x, y = (t[:, ends[s]: ends[s + 1]].to(F64) for t in (a, w))
        off = (K + 3) * 2.0 ** -24 * (x.abs() @ y.abs().T)
        assert near(got.float(), x @ y.T, off, 2.0 ** -8)
