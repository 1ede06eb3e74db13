"""QKV projection on 256 x 256 tiles: heads that do and do not divide a tile's halves, part tiles."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


@pytest.mark.parametrize("M", [257, 300, 512])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("heads,kv,hd", [(4, 2, 64), (3, 1, 128), (5, 2, 96), (7, 5, 16), (2, 1, 256), (25, 25, 64)])
@pytest.mark.parametrize("kind", [4, 1])
def test_qkv(M, rope, heads, kv, hd, kind):
    """A sum of K products and a bias is off by K + 4 ulp of their sizes, its turn by two more, the result by
    half a bf16 step."""
    from llm_sharding_demo_amd import _C as C

    K, N, seq = 192, (heads + 2 * kv) * hd, 40
    g = torch.Generator().manual_seed(M + hd)
    a, w, b = (torch.randn(*s, generator=g).bfloat16() for s in ((M, K), (N, K), (N,)))
    kc, vc = (torch.zeros(M + 1, kv, seq, hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    slot, pos = torch.randperm(M, generator=g).int(), (torch.arange(M) * 7 % seq).int()
    table = torch.randn(seq, hd // 2, 2, generator=g)
    C.gemm_set_big_min(1)
    C.gemm_set_big_kind(kind)
    try:
        assert C.gemm_big_tiles(M, N, K, 1)
        q = C.linear_qkv(a.to(DEV), w.to(DEV), b.to(DEV), kc, vc, slot.to(DEV), pos.to(DEV), heads * hd, kv * hd, hd,
                         table.to(DEV) if rope else None, 1, 1, None)
    finally:
        C.gemm_set_big_kind(4)
        C.gemm_set_big_min(160)
    a, w, b, n = a.to(F64), w.to(F64), b.to(F64), (heads + kv) * hd

    def turn(y, sign, part):
        t = y[:, :n].reshape(M, heads + kv, hd // 2, 2)
        c, s = (part(table[pos.long()].to(F64)[:, None, :, i]) for i in (0, 1))
        t = torch.stack([t[..., 0] * c - sign * t[..., 1] * s, t[..., 1] * c + t[..., 0] * s], -1)
        return torch.cat([t.reshape(M, -1), y[:, n:]], 1)
    y, off = a @ w.T + b, (K + 6) * 2.0 ** -24 * (a.abs() @ w.abs().T + b.abs())
    if rope:
        y, off = turn(y, 1, lambda t: t), turn(off, -1, torch.abs)
    kc, vc = kc.cpu(), vc.cpu()
    got = torch.cat([q.cpu()] + [t[slot.long(), :, pos.long()].reshape(M, -1) for t in (kc, vc)], 1)
    assert bool(((got.to(F64) - y).abs() <= off + 2.0 ** -8 * y.abs()).all())
    for t in (kc, vc):  # nothing else is written
        t[slot.long(), :, pos.long()] = 0
        assert int(t.count_nonzero()) == 0


@pytest.mark.parametrize("M,kind,big", [(1000, 2, None), (1000, 3, None), (2000, 1, None), (2000, 1, 0), (2000, 1, 1), (2000, 1, 4)])
@pytest.mark.parametrize("heads,kv,hd", [(6, 2, 128), (3, 1, 256), (7, 2, 96)])
def test_turns_are_rounded_alike(M, kind, big, heads, kv, hd):
    """Sums of small whole numbers are exact, so a turned pair is a cos - (b sin), a sin + (b cos) to the bit, each
    bracket rounded by itself: the same from every kernel of tiles (kind 1: 256 x 256, 128 x 128 with big None)."""
    from llm_sharding_demo_amd import _C as C

    K, N, seq = 128, (heads + 2 * kv) * hd, 64
    g = torch.Generator(device=DEV).manual_seed(M + hd)
    a, w = (torch.randint(-9, 10, s, generator=g, device=DEV).bfloat16() for s in ((M, K), (N, K)))
    kc, vc = (torch.zeros(M, kv, seq, hd, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    slot, pos = torch.arange(M, device=DEV).int(), (torch.arange(M, device=DEV) * 7 % seq).int()
    angle = torch.rand(seq, hd // 2, generator=g, device=DEV) * 6.3
    table = torch.stack([angle.cos(), angle.sin()], -1).contiguous()
    C.gemm_set_big_min(1 << 30 if big is None else 1)
    C.gemm_set_big_kind(4 if big is None else big)
    try:
        assert kind != 1 or C.gemm_big_tiles(M, N, K, 1) == (big is not None)
        q = C.linear_qkv(a, w, None, kc, vc, slot, pos, heads * hd, kv * hd, hd, table, kind, 1,
                         torch.zeros(1 << 16, dtype=torch.int32, device=DEV))
    finally:
        C.gemm_set_big_kind(4)
        C.gemm_set_big_min(160)
    y = (a.cpu().to(F64) @ w.cpu().to(F64).T)[:, : (heads + kv) * hd].reshape(M, heads + kv, hd // 2, 2)
    c, s = (table.cpu()[pos.cpu().long()].to(F64)[:, None, :, i] for i in (0, 1))
    x, z = y[..., 0], y[..., 1]
    want = torch.stack([x * c - (z * s).float(), x * s + (z * c).float()], -1).float().bfloat16().reshape(M, -1)
    got = torch.cat([q.cpu(), kc.cpu()[slot.cpu().long(), :, pos.cpu().long()].reshape(M, -1)], 1)
    assert torch.equal(got, want)
