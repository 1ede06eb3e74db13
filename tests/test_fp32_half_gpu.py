"""fp32 products on two fp16 terms against 64 bits.

A sum of K products in fp32 is off by at most (K + 2) ulp of the sum of the products' sizes, in any order (ulp:
2^-24); the terms leave out three ulp of each product.  Of values too small for them they leave out more, 3 K / 4 ulp of the
sizes at most where such sums are not computed again; an fp32 MFMA adds 32 products in a few roundings, so sums stay in K + 14.
"""

import pytest
import torch

from .test_timisun_gpu import C, rand  # noqa: F401

DEV, F64, ULP = "cuda:0", torch.float64, 2.0 ** -24


def near(got, a, w):
    want, size = a.to(F64) @ w.to(F64).T, a.to(F64).abs() @ w.to(F64).abs().T
    return bool(((got.cpu().to(F64) - want).abs() <= (a.shape[1] + 14) * ULP * size).all())


# every tile: its edges, parts of K that are even and uneven
TILES = [(500, 1985, 1376, (64, 64, 2)), (449, 2048, 2080, (64, 64, 2)), (561, 2048, 2048, (80, 64, 3)), (565, 2000, 2144, (80, 64, 3)),
         (961, 2048, 1024, (64, 128, 1)), (513, 2600, 1056, (64, 128, 1)), (561, 4160, 1024, (96, 128, 1)),
         (222, 11264, 1088, (128, 128, 1))]


def test_tiles():
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert [_C.fp32_tile(M, N, K) for M, N, K, _ in TILES] == [t for *_, t in TILES]
    # short K and sums that would be in fewer parts stay on three terms
    assert _C.fp32_tile(961, 2100, 992) == _C.fp32_tile(961, 2100) and _C.fp32_tile(100, 2048, 2048) == (32, 64, 4)
    assert _C.fp32_tile(300, 2048, 2048) == (48, 64, 4) and _C.fp32_tile(565, 2048, 1024) == (80, 64, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile", TILES)
def test_products(C, M, N, K, tile):  # noqa: F811
    a, w, b = rand(M, K, seed=1), rand(N, K, seed=2) * 0.02, rand(N, seed=3)
    got = C.linear_fp32(a.to(DEV), w.to(DEV)).cpu()
    assert near(got, a, w)
    want = a.to(F64) @ w.to(F64).T
    # not behind three bf16 terms, whose sums are 1.3e-7 to 2e-7 of the result off here
    assert float((got.to(F64) - want).norm() / want.norm()) < 2e-7
    x = rand(M, N, seed=4)
    y = x.to(DEV).clone()
    C.linear_fp32(a.to(DEV), w.to(DEV), y)
    assert float((y.cpu().to(F64) - x.to(F64) - want).abs().max()) < (K + 14) * ULP * float((a.abs() @ w.abs().T).max())
    assert torch.equal(C.linear_fp32(a.to(DEV), w.to(DEV), None, b.to(DEV)).cpu(), got + b)


# rows and columns that leave the terms' range, alone and beside others, are computed again
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile", [TILES[0], TILES[2], TILES[4], TILES[6], TILES[7]])
@pytest.mark.parametrize("scale", [2.0 ** -140, 2.0 ** -40, 2.0 ** -16, 2.0 ** 13, 2.0 ** 60])
def test_sizes(C, M, N, K, tile, scale):  # noqa: F811
    a, w = rand(M, K, seed=1).clamp(-1, 1), rand(N, K, seed=2).clamp(-1, 1) * 0.02
    a[5:100:30] *= scale
    big = w * (2.0 ** 50 if scale < 2.0 ** -100 else 1.0)
    assert near(C.linear_fp32(a.to(DEV), big.to(DEV)), a, big)
    w[3:90:29] *= scale
    w[7] = 0
    a[5:100:30] = rand(4, K, seed=3) * (2.0 ** 50 if scale < 2.0 ** -100 else 1.0)
    got = C.linear_fp32(a.to(DEV), w.to(DEV))
    rows = slice(5, 100, 30) if scale < 2.0 ** -100 else slice(None)  # (products of the others are below fp32's numbers)
    assert near(got[rows], a[rows], w) and int(got[:, 7].count_nonzero()) == 0


@pytest.mark.gpu
def test_lone_small_values(C):  # noqa: F811
    """Small values of a row beside which the weights are zeros: sums of their own size."""
    M, N, K, _ = TILES[4]
    a, w = rand(M, K, seed=1), torch.zeros(N, K)
    a[:, 100], w[:, 100] = 2.0 ** -45, 1.0
    got = C.linear_fp32(a.to(DEV), w.to(DEV))
    assert near(got, a, w)


# 2^-16 and 2^-22 are where terms of A and of W begin to keep fewer than 22 bits
SMALL = torch.tensor([m * 2.0 ** -e for e in range(12, 46) for m in (1.7, 1.05, 1.3)])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile", TILES)
def test_lone_products(C, M, N, K, tile):  # noqa: F811
    """Values far below the others of their row of A or column of W, whose partners are zeros but for one or for few:
    their sums are of their own size, and as near as any."""
    n = len(SMALL)
    a, w = rand(M, K, seed=1), rand(N, K, seed=2) * 0.02
    a[:n, 100] = SMALL
    for column, partner in ((7, 1.0), (33, -2.0 ** -6), (60, 128.0), (1980, 0.3)):
        w[column] = 0
        w[column, 100] = partner
    w[200: 200 + n, K - 5] = SMALL * 2.0 ** -6
    for row, partner in ((110, 8192.0), (111, 1.0), (200, -0.01)):
        a[row] = 0
        a[row, K - 5] = partner
    a[20, 300], a[70, 301], w[210, 302], w[290, 303] = 20000.0, 2.0 ** 40, 300.0, 2.0 ** 30  # (beside them lost sooner)
    w[[7, 33, 60, 1980], 300:304] = 0
    for row, e in ((120, 20), (150, 26), (180, 34)):  # many such products
        a[row, : K // 2] *= 2.0 ** -e
    w[61, K // 2:] = 0
    got = C.linear_fp32(a.to(DEV), w.to(DEV))
    assert near(got, a, w)


@pytest.mark.gpu
def test_lone_products_of_experts(C):  # noqa: F811
    """The same of one expert's and a shared expert's down product, beside an expert with few rows."""
    T, H, F, n = 200, 2176, 1024, len(SMALL)
    mid, mids, dn = rand(T, F, seed=1), rand(T, F, seed=2), rand(2, H, F, seed=3) * 0.02
    shared = rand(H, F, seed=4) * 0.02
    ids = (torch.arange(T)[:, None] >= T - 3).int()  # the last three tokens to the second expert
    order, tiles = C.moe_group(ids.to(DEV), 2, 64)
    assert C.moe_on_split(T, 1, tiles.shape[0], H, H, F)
    for x in (mid, mids):
        x[:n, 100] = SMALL
        x[110], x[110, F - 5] = 0, 8192.0
    for w in (dn[0], shared):
        w[7], w[7, 100] = 0, 1.0
        w[60], w[60, 100] = 0, 128.0
        w[100: 100 + n, F - 5] = SMALL * 2.0 ** -6
    slab = torch.empty(2, T, H, device=DEV)
    C.moe_down(mid.to(DEV), mids.to(DEV), order, tiles, torch.ones(T, 1).to(DEV), dn.to(DEV), shared.to(DEV), slab, 64)
    at = order.cpu().long()[:T]
    assert near(slab[1], mids, shared)
    assert near(slab[0][at[: T - 3].to(DEV)], mid[: T - 3], dn[0]) and near(slab[0][at[T - 3:].to(DEV)], mid[T - 3:], dn[1])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile,rows,value,weight", [
    *((*case, slice(None, None, step), value, weight) for case in (TILES[2], TILES[4]) for step in (1, 40) for value, weight in (
        (16376.0, 0.0), (3e9, 0.0), (2.0 ** 59, 0.0), (2.0 ** 70, 0.0), (20000.0, 300.0), (2.0 ** 50, 2.0 ** 50))),
    *((*case, slice(None, None, step), 20000.0, 0.0) for case in TILES for step in (1, 40))])
def test_large_values(C, M, N, K, tile, rows, value, weight):  # noqa: F811
    """Rows that the terms cannot hold are summed again with other scales, or by fp32 MFMAs behind 2^60, as near to 64 bits as on three
    bf16 terms (a value of 20000 2.4e-7 and 2.9e-7 of the result; by fp32 MFMAs in two chains, as few rows are, 4.6e-7 and 5.5e-7)."""
    a, w = rand(M, K, seed=1), rand(N, K, seed=2) * 0.02
    a[rows, 50] = value
    if weight:
        w[::3, K - 2] = weight
    got, want = C.linear_fp32(a.to(DEV), w.to(DEV)).cpu().to(F64), a.to(F64) @ w.to(F64).T
    assert near(got, a, w)
    if not weight:  # (with it products of a few large values, which round less)
        assert float((got - want)[rows].norm() / want[rows].norm()) < 3.5e-7


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 65504.0, -3e38])
@pytest.mark.parametrize("side", ["a", "w"])
def test_not_finite(C, side, value):  # noqa: F811
    M, N, K, _ = TILES[0]
    a, w = rand(M, K, seed=1), rand(N, K, seed=2)
    (a if side == "a" else w)[40, 50] = value
    w[3, 50] = a[5, 50] = 0.5
    want, got = a @ w.T, C.linear_fp32(a.to(DEV), w.to(DEV)).cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    ok = want.isfinite()
    size = a.nan_to_num(0, 0, 0).abs() @ w.nan_to_num(0, 0, 0).abs().T
    assert bool(((got - want).abs()[ok] <= 2 * (K + 14) * ULP * size[ok]).all())


# where column tiles start their sums elsewhere: tokens, choices, tiles of the table, columns, the shared expert's, K
TURNED = [(300, 4, 50, 2048, 4096, 2048, True), (300, 4, 50, 2048, 2048, 1024, True), (700, 4, 75, 2048, 0, 1024, True),
          (800, 4, 82, 2048, 0, 1024, False), (300, 4, 50, 2176, 4224, 2112, False), (300, 4, 50, 2048, 2048, 1088, False),
          (300, 2, 17, 5120, 0, 2560, False), (300, 4, 50, 2048, 0, 4096, False), (300, 2, 25, 2048, 0, 4096, True),
          (300, 2, 25, 2048, 2048, 4096, False), (300, 2, 25, 2048, 0, 3072, True)]


def test_turned():
    _C = pytest.importorskip("llm_sharding_demo_amd._C")
    assert [_C.moe_turned(*r[:-1]) for r in TURNED] == [r[-1] for r in TURNED]


# experts of 1024 columns and more: full and part full tiles, beside a shared expert; the third ones turned
@pytest.mark.gpu
@pytest.mark.parametrize("T,E,H,F,Fs", [(290, 3, 1024, 1088, 1024), (150, 2, 1056, 1024, 0), (290, 9, 1024, 1088, 1024), (150, 8, 3072, 1024, 0)])
def test_experts(C, T, E, H, F, Fs):  # noqa: F811
    H = (H + 63) // 64 * 64
    h, up, dn = rand(T, H, seed=1), rand(E, 2 * F, H, seed=2) * 0.05, rand(E, H, F, seed=3) * 0.05
    top = 2
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int()
    ids[: T // 3, 0], ids[: T // 3, 1] = 0, 1
    wts = torch.rand(T, top)
    shared_up, shared_dn = (rand(2 * Fs, H, seed=4) * 0.05, rand(H, Fs, seed=5) * 0.05) if Fs else (None, None)
    order, tiles = C.moe_group(ids.to(DEV), E, 64)
    for N, Ns, K in ((2 * F, 2 * Fs, H), (H, H if Fs else 0, F)):
        assert C.moe_on_split(T, top, tiles.shape[0], N, Ns, K) or K < 2 * F
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    mid, mids = C.moe_up(h.to(DEV), order, tiles, top, up.to(DEV), 0.0, 1.0, dev(shared_up), 0.0, 64)
    slab = torch.empty(top + bool(Fs), T, H, device=DEV)
    C.moe_down(mid, mids if Fs else None, order, tiles, wts.to(DEV), dn.to(DEV), dev(shared_dn), slab, 64)

    def gated(x, w):
        y = (x @ w.to(F64).T).reshape(len(x), -1, 2, 16)
        return (y[:, :, 0] * torch.sigmoid(y[:, :, 0]) * y[:, :, 1]).reshape(len(x), -1)

    def close(got, want):  # sums of some thousand products: 1e-6 of the largest, and twice in front of a gate
        assert float((got.cpu().to(F64) - want).abs().max()) < 4e-6 * float(want.abs().max())
    perm, x = order.cpu().long()[: T * top], h.to(F64)
    token, expert = perm // top, ids.reshape(-1)[perm]
    if Fs:
        close(mids, gated(x, shared_up))
        close(slab[top], mids.cpu().to(F64) @ shared_dn.to(F64).T)
    for e in range(E):
        mine = (expert == e).nonzero()[:, 0]
        close(mid.cpu()[mine], gated(x[token[mine]], up[e]))
        want = wts.reshape(-1)[perm[mine]].to(F64)[:, None] * (mid.cpu()[mine].to(F64) @ dn[e].to(F64).T)
        close(slab[:top].cpu()[perm[mine] % top, token[mine]], want)
