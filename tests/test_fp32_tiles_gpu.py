"""fp32 products and latent attention on matrix tiles against 64 bits.

A sum of K products in fp32 is off by at most (K + 2) ulp of the sum of the
products' sizes, in any order (ulp: 2^-24).
"""

import pytest
import torch

from . import timisun_oracle as orc
from .test_timisun_gpu import C, latent_tokens, paged, rand  # noqa: F401

pytestmark = pytest.mark.gpu
DEV, F64, ULP = "cuda:0", torch.float64, 2.0 ** -24


@pytest.mark.parametrize("K", [16, 32, 48, 64, 96, 128, 160])
@pytest.mark.parametrize("M,N", [(1, 1), (1, 65), (15, 64), (16, 63), (17, 130), (64, 3), (65, 129), (200, 32),
                                 (1000, 4097), (513, 8100)])
def test_linear_fp32_edges(C, M, N, K):  # noqa: F811
    a, w, x, b = rand(M, K, seed=1), rand(N, K, seed=2), rand(M, N, seed=3), rand(N, seed=4)
    want, size = a.to(F64) @ w.to(F64).T, a.to(F64).abs() @ w.to(F64).abs().T
    got = C.linear_fp32(a.to(DEV), w.to(DEV), None, b.to(DEV)).cpu().to(F64)
    assert bool(((got - want - b.to(F64)).abs() <= (K + 3) * ULP * (size + b.abs())).all())
    if N % 4 == 0:
        xd = x.to(DEV)
        C.linear_fp32(a.to(DEV), w.to(DEV), xd)
        assert bool(((xd.cpu().to(F64) - want - x.to(F64)).abs() <= (K + 3) * ULP * (size + x.abs())).all())


def test_weights_off_16_bytes(C):  # noqa: F811
    a, w = rand(70, 64, seed=1), rand(1, 80, 64, seed=2)
    dev = torch.empty(80 * 64 + 1, device=DEV)[1:].view(1, 80, 64)
    dev.copy_(w)
    assert dev.data_ptr() % 16 == 4
    want, size = a.to(F64) @ w[0].to(F64).T, a.to(F64).abs() @ w[0].to(F64).abs().T
    for x in (w.to(DEV), dev):
        got = C.batch_linear(a.to(DEV), x, 64).cpu().to(F64)
        assert bool(((got - want).abs() <= 66 * ULP * size).all())


@pytest.mark.parametrize("H", [1, 15, 16, 33])
@pytest.mark.parametrize("rank,value", [(64, 64), (128, 40), (192, 192), (512, 448), (576, 512)])
def test_latent_values_and_sinks_fp32(C, rank, value, H):  # noqa: F811
    """Heads off the 16-head tile, fewer value than key columns, sinks; a stale
    row behind the last key that is not a number."""
    n, W, scale = 70, 45, rank ** -0.5
    c, q, sink = rand(n, rank, seed=1), rand(n, H, rank, seed=2), rand(H, seed=3)
    pool, table = paged(torch.cat([c, torch.full((1, rank), float("nan"))]), torch.float32, rank)
    i32 = dict(dtype=torch.int32, device=DEV)
    cols = rank - 64 if value <= rank - 64 else rank
    got = C.latent_decode(q.reshape(n, -1).to(DEV), pool, table, torch.ones(n, **i32), torch.arange(n, **i32), H, W,
                          scale, 1, value, sink.to(DEV)).reshape(n, H, cols).cpu().to(F64)
    s = torch.einsum("thr,kr->thk", q.to(F64), c.to(F64)) * scale
    seen = torch.tensor([[orc.visible(p, k, W) for k in range(n)] for p in range(n)])
    s = torch.cat([s.masked_fill(~seen[:, None], float("-inf")), sink.to(F64).expand(n, H)[..., None]], -1)
    p = torch.softmax(s, -1)[..., :-1]
    # a score is off by 4 ulp of its products' sizes at most (their roundings are
    # independent: sqrt(rank) of the worst case), which weights share relatively
    assert float((got - p @ c[:, :cols].to(F64)).pow(2).mean().sqrt()) < 2e-6


@pytest.mark.parametrize("H,rank", [(1, 64), (16, 512), (33, 576)])
def test_latent_without_keys_fp32(C, H, rank):  # noqa: F811
    """A row at position -1 has no key and reads none: its sink takes all the weight."""
    n = 3
    c, q, sink = rand(n, rank, seed=1), rand(2, H, rank, seed=2), rand(H, seed=3)
    pool, table = paged(c, torch.float32, rank)
    i32 = dict(dtype=torch.int32, device=DEV)
    got = C.latent_decode(q.reshape(2, -1).to(DEV), pool, table, torch.ones(2, **i32), torch.tensor([-1, n - 1], **i32), H,
                          1 << 30, rank ** -0.5, 1, rank, sink.to(DEV)).reshape(2, H, -1).cpu().to(F64)
    assert not got[0].any()
    s = torch.cat([q[1].to(F64) @ c.to(F64).T * rank ** -0.5, sink.to(F64)[:, None]], -1)
    assert float((got[1] - (torch.softmax(s, -1)[:, :-1] @ c.to(F64))[:, : got.shape[2]]).abs().max()) < 1e-5


# rows that a tile of 64 reaches in 32 bits, and the next wider ones
@pytest.mark.parametrize("K,step", [(64, (1 << 24) - 4), (64, 1 << 24)])
@pytest.mark.parametrize("far", ["a", "w"])
def test_rows_far_apart(C, K, step, far):  # noqa: F811
    n = 65
    a, w = rand(n, K, seed=1), rand(n, K, seed=2)
    room = torch.empty(n * step, device=DEV).as_strided((n, K), (step, 1))
    room.copy_(a if far == "a" else w)
    got = C.linear_fp32(*((room, w.to(DEV)) if far == "a" else (a.to(DEV), room))).cpu().to(F64)
    size = a.to(F64).abs() @ w.to(F64).abs().T
    assert bool(((got - a.to(F64) @ w.to(F64).T).abs() <= (K + 2) * ULP * size).all())
    near = C.linear_fp32(a.to(DEV), w.to(DEV)).cpu().to(F64)
    assert torch.equal(got, near)  # the same tiles: the same sums in the same order


# gathered rows count from the first token: tokens that 32 bits reach, and do not
@pytest.mark.parametrize("step", [(1 << 30) // 70 // 4 * 4 - 4, 1 << 24])
def test_experts_of_tokens_far_apart(C, step):  # noqa: F811
    T, top, E, K, F = 70, 2, 3, 128, 48
    h, w, ws = rand(T, K, seed=1), rand(E, 2 * F, K, seed=2) * 0.1, rand(2 * F, K, seed=3) * 0.1
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int().to(DEV)
    perm, tiles = C.moe_group(ids, E, 64)
    room = torch.empty((T - 1) * step + K, device=DEV).as_strided((T, K), (step, 1))
    room.copy_(h)
    got = C.moe_up(room, perm, tiles, top, w.to(DEV), 0.0, 1.0, ws.to(DEV), 0.0, 64)
    near = C.moe_up(h.to(DEV), perm, tiles, top, w.to(DEV), 0.0, 1.0, ws.to(DEV), 0.0, 64)
    assert torch.equal(got[0], near[0]) and torch.equal(got[1], near[1])
    y = (h.to(F64) @ ws.to(F64).T).reshape(T, F // 16, 2, 16)
    gate, up = y[:, :, 0].reshape(T, F), y[:, :, 1].reshape(T, F)
    want = gate * torch.sigmoid(gate) * up
    assert float((got[1].cpu().to(F64) - want).abs().max()) < 1e-5 * float(want.abs().max())
