"""fp32 products as sums of three bf16 terms against 64 bits.

A sum of K products in fp32 is off by at most (K + 2) ulp of the sum of the products'
sizes, in any order (ulp: 2^-24); the products of terms that are left out are 2^-26 each.
"""

import pytest
import torch

from .test_timisun_gpu import C, rand  # noqa: F401

DEV, F64, ULP = "cuda:0", torch.float64, 2.0 ** -24


def near(got, a, w, extra=0.0):
    want, size = a.to(F64) @ w.to(F64).T, a.to(F64).abs() @ w.to(F64).abs().T
    return bool(((got.cpu().to(F64) - want - extra).abs() <= (a.shape[1] + 4) * ULP * size + 2 * ULP * abs(extra)).all())


# every tile: its edges, parts of K that are empty, uneven and whole
TILES = [(17, 40, (32, 64, 4)), (33, 1985, (32, 64, 4)), (81, 5952, (48, 64, 4)), (193, 3264, (48, 64, 4)), (500, 1985, (64, 64, 2)),
         (561, 2048, (80, 64, 3)), (561, 2560, (48, 128, 1)), (961, 2048, (64, 128, 1)), (801, 2600, (80, 128, 1)),
         (561, 4160, (96, 128, 1))]


def test_tiles():
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert [_C.fp32_tile(M, N) for M, N, _ in TILES] == [t for _, _, t in TILES]


@pytest.mark.gpu
@pytest.mark.parametrize("K", [544, 576, 608, 672, 928])
@pytest.mark.parametrize("M,N,tile", TILES)
def test_products(C, M, N, tile, K):  # noqa: F811
    a, w, b = rand(M, K, seed=1), rand(N, K, seed=2), rand(N, seed=3)
    got = C.linear_fp32(a.to(DEV), w.to(DEV), None, b.to(DEV))
    want, size = a.to(F64) @ w.to(F64).T + b.to(F64), a.to(F64).abs() @ w.to(F64).abs().T + b.to(F64).abs()
    assert bool(((got.cpu().to(F64) - want).abs() <= (K + 4) * ULP * size).all())


# what leaves the range of bf16's normal numbers goes to fp32 MFMAs: sums as in fp32, and no other rows change
@pytest.mark.gpu
@pytest.mark.parametrize("K", [544, 576])
@pytest.mark.parametrize("scale,back", [(2.0 ** -120, 2.0 ** 60), (2.0 ** 120, 2.0 ** -60), (3.4e38, 2.0 ** -100), (2.0 ** -115, 2.0 ** 100),
                                        (2.0 ** 80, 2.0 ** -115)])
def test_sizes(C, K, scale, back):  # noqa: F811
    a, w = rand(70, K, seed=1).clamp(-1, 1) * scale, rand(100, K, seed=2) * back
    assert near(C.linear_fp32(a.to(DEV), w.to(DEV)), a, w)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("side", ["a", "w"])
def test_not_finite(C, side, value):  # noqa: F811
    a, w = rand(70, 576, seed=1), rand(130, 576, seed=2)
    (a if side == "a" else w)[40, 50] = value
    w[3, 50] = a[5, 50] = 1.0  # no middle and low terms: infinity times them is not a number
    want, got = a @ w.T, C.linear_fp32(a.to(DEV), w.to(DEV)).cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    ok = want.isfinite()
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    assert bool(((got - want).abs()[ok] <= 600 * ULP * 576).all())


# experts whose fp32 tiles are fewer than the CUs stay on fp32 MFMAs, 18 rows a tile of the table and more or not
@pytest.mark.gpu
@pytest.mark.parametrize("T,E", [(300, 3), (129, 5), (64, 1), (30, 9)])
def test_experts(C, T, E):  # noqa: F811
    H, F, top = 128, 192, min(2, E)
    h, up, dn = rand(T, H, seed=1), rand(E, 2 * F, H, seed=2) * 0.2, rand(E, H, F, seed=3) * 0.2
    shared_up, shared_dn = rand(2 * F, H, seed=4) * 0.2, rand(H, F, seed=5) * 0.2
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int()
    ids[: T // 2, 0], ids[: T // 2, 1:] = 0, min(1, E - 1)  # uneven
    wts = torch.rand(T, top)
    order, tiles = C.moe_group(ids.to(DEV), E, 64)
    on = T * top >= 18 * tiles.shape[0]
    assert on == (T > 30)
    mid, mids = C.moe_up(h.to(DEV), order, tiles, top, up.to(DEV), 0.0, 1.0, shared_up.to(DEV), 0.0, 64)

    def gated(x, w):
        y = (x.to(F64) @ w.to(F64).T).reshape(len(x), F // 16, 2, 16)
        g, u = y[:, :, 0].reshape(len(x), F), y[:, :, 1].reshape(len(x), F)
        return g * torch.sigmoid(g) * u

    perm = order.cpu().long()[: T * top]
    want = torch.stack([gated(h[e // top][None], up[ids[e // top, e % top]])[0] for e in perm.tolist()])
    assert float((mid.cpu().to(F64)[: T * top] - want).abs().max()) < 1e-5 * float(want.abs().max())
    assert float((mids.cpu().to(F64) - gated(h, shared_up)).abs().max()) < 1e-5 * float(want.abs().max())
    slab = torch.empty(top + 1, T, H, device=DEV)
    C.moe_down(mid, mids, order, tiles, wts.to(DEV), dn.to(DEV), shared_dn.to(DEV), slab, 64)
    m = mid.cpu().to(F64)
    for s, e in enumerate(perm.tolist()):
        y = wts[e // top, e % top].to(F64) * (dn[ids[e // top, e % top]].to(F64) @ m[s])
        assert float((slab[e % top, e // top].cpu().to(F64) - y).abs().max()) < 1e-5 * max(1.0, float(y.abs().max()))
    y = mids.cpu().to(F64) @ shared_dn.to(F64).T
    assert float((slab[top].cpu().to(F64) - y).abs().max()) < 1e-5 * float(y.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,tile", [(193, 3264, (48, 64, 4)), (961, 2048, (64, 128, 1)), (561, 4160, (96, 128, 1))])
def test_recomputed_sums(C, M, N, tile):  # noqa: F811
    """A tile with a value past the terms' range is summed as few rows are, by fp32 MFMAs in two chains: to the bit where
    a block has all of K."""
    a, w = rand(M, 576, seed=1), rand(N, 576, seed=2)
    assert C.fp32_tile(M, N) == tile
    few = C.linear_fp32(a[:16].to(DEV), w.to(DEV)).cpu()
    a[9, 3] = 2.0 ** 60
    got = C.linear_fp32(a.to(DEV), w.to(DEV)).cpu()[:16]
    got[9] = few[9]
    if tile[2] == 1:
        assert torch.equal(got, few)
    else:
        assert bool(((got - few).abs() <= 580 * ULP * (a[:16].abs() @ w.abs().T)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(70, 100), (300, 2048), (561, 2560)])
def test_operands_behind_the_terms(C, M, N):  # noqa: F811
    """Operands without a bf16 term, in rows of their own: the sums are zero until they are computed again; columns
    of zeros stay zeros."""
    a, w = rand(M, 576, seed=1).clamp(-1, 1), rand(N, 576, seed=2) * 2.0 ** 50
    a[::3] *= 2.0 ** -140
    w[5:90:7] = 0
    assert int(a[::3].count_nonzero()) > 100 and float(a[::3].abs().max()) < 2.0 ** -134
    got = C.linear_fp32(a.to(DEV), w.to(DEV))
    assert near(got, a, w) and int(got[:, 5:90:7].count_nonzero()) == 0 and int(got[::3, :5].count_nonzero()) > 0


# where experts change kernels: fp32 tiles more than the CUs, rows a tile of the table, K
RULE = [(200, 2, 14, 1024, 1024, 512, False), (300, 2, 25, 1024, 1024, 512, True), (300, 2, 25, 1024, 1024, 352, False),
        (565, 4, 67, 1024, 1024, 128, True), (200, 4, 45, 1024, 1024, 512, False), (200, 4, 44, 1024, 1024, 512, True),
        (200, 4, 44, 1024, 1024, 352, False), (1000, 2, 39, 256, 0, 256, False), (120, 2, 11, 2048, 0, 2048, True)]


def test_experts_rule():
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert [_C.moe_on_split(*r[:-1]) for r in RULE] == [r[-1] for r in RULE]


# experts on split operands: 28 rows a tile of the table and more, their last tiles part full, and short K
@pytest.mark.gpu
@pytest.mark.parametrize("T,E,H,F", [(290, 9, 128, 1024), (129, 2, 64, 2080), (300, 3, 448, 1200), (1, 1, 64, 16)])
def test_experts_on_split(C, T, E, H, F):  # noqa: F811
    top = min(2, E)
    h, up = rand(T, H, seed=1), rand(E, 2 * F, H, seed=2) * 0.2
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int()
    order, tiles = C.moe_group(ids.to(DEV), E, 64)
    assert C.moe_on_split(T, top, tiles.shape[0], 2 * F, 0, H) == (T > 1)
    mid, _ = C.moe_up(h.to(DEV), order, tiles, top, up.to(DEV), 0.0, 1.0, None, 0.0, 64)
    perm = order.cpu().long()[: T * top]
    for s, e in enumerate(perm.tolist()):
        y = (up[ids[e // top, e % top]].to(F64) @ h[e // top].to(F64)).reshape(F // 16, 2, 16)
        g, u = y[:, 0].reshape(F), y[:, 1].reshape(F)
        want = g * torch.sigmoid(g) * u
        assert float((mid[s].cpu().to(F64) - want).abs().max()) < 1e-5 * max(1.0, float(want.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(70, 100), (561, 2560), (961, 2048), (561, 4160)])
def test_weights_behind_the_terms(C, M, N):  # noqa: F811
    """Columns of W without a bf16 term, and rows that are all of a tile."""
    a, w = rand(M, 576, seed=1).clamp(-1, 1) * 2.0 ** 50, rand(N, 576, seed=2).clamp(-1, 1)
    w[3:90:7] *= 2.0 ** -140
    got = C.linear_fp32(a.to(DEV), w.to(DEV))
    assert near(got, a, w) and bool((got[:, 3:90:7] != 0).all())
    got = C.linear_fp32(w[3:90:7].repeat(6, 1).to(DEV), a.to(DEV))
    assert near(got, w[3:90:7].repeat(6, 1), a) and bool((got != 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,H,F,Fs", [(290, 9, 1280, 1024, 192), (65, 2, 4224, 2752, 64)])
def test_experts_and_shared_on_split(C, T, E, H, F, Fs):  # noqa: F811
    """Both products, beside a shared expert: sums of K products and a gated one in front of them, against 64 bits."""
    top = 2
    h, up, dn = rand(T, H, seed=1), rand(E, 2 * F, H, seed=2) * 0.05, rand(E, H, F, seed=3) * 0.05
    shared_up, shared_dn = rand(2 * Fs, H, seed=4) * 0.05, rand(H, Fs, seed=5) * 0.05
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int()
    wts = torch.rand(T, top)
    order, tiles = C.moe_group(ids.to(DEV), E, 64)
    for N, Ns, K in ((2 * F, 2 * Fs, H), (H, H, F)):
        assert C.moe_on_split(T, top, tiles.shape[0], N, Ns, K)
    mid, mids = C.moe_up(h.to(DEV), order, tiles, top, up.to(DEV), 0.0, 1.0, shared_up.to(DEV), 0.0, 64)
    slab = torch.empty(top + 1, T, H, device=DEV)
    C.moe_down(mid, mids, order, tiles, wts.to(DEV), dn.to(DEV), shared_dn.to(DEV), slab, 64)

    def gated(x, w):
        y = (x @ w.to(F64).T).reshape(len(x), -1, 2, 16)
        return (y[:, :, 0] * torch.sigmoid(y[:, :, 0]) * y[:, :, 1]).reshape(len(x), -1)

    def close(got, want):
        assert float((got.cpu().to(F64) - want).abs().max()) < 1e-5 * float(want.abs().max())
    perm, x = order.cpu().long()[: T * top], h.to(F64)
    token, expert = perm // top, ids.reshape(-1)[perm]
    close(mids, gated(x, shared_up))
    close(slab[top], mids.cpu().to(F64) @ shared_dn.to(F64).T)
    for e in range(E):
        mine = (expert == e).nonzero()[:, 0]
        close(mid.cpu()[mine], gated(x[token[mine]], up[e]))
        want = wts.reshape(-1)[perm[mine]].to(F64)[:, None] * (mid.cpu()[mine].to(F64) @ dn[e].to(F64).T)
        close(slab[:top].cpu()[perm[mine] % top, token[mine]], want)
