"""Recurrent decode steps where threads hold whole tiles of the state, against 64 bits and
against the general form, which takes portions of two tokens and rows off their vectors."""

import pytest
import torch

from .test_vizalix_gpu import BF, F32, C, DeltaCase, SsmCase, err, portions  # noqa: F401
from .test_vizalix_gpu import cuda, i32

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dt", [BF, F32])
T = 13


def check(case, V, dt):
    outs, states = [], []
    for sizes in ([1] * T, [2] * 6 + [1], [1, 1, 3, 1, 1, 4, 1, 1]):
        case.state.fill_(float("nan"))
        case.ring.fill_(float("nan"))
        outs.append(case.run(portions(T, sizes), False))
        states.append(case.state[1, ..., :V].clone())
        assert err(outs[-1], case.want) < (3e-2 if dt == BF else 3e-5)
        assert err(states[-1], case.S) < 2e-5
    for o, s in zip(outs[1:], states[1:]):  # two orders of rounding of the same sums
        assert err(o, outs[0].cpu()) < (8e-3 if dt == BF else 1e-5) and err(s, states[0].cpu()) < 1e-5


# (heads, key groups, D, V): tiles of 64 and 128 columns, several of them a head, and next to them
@DTYPES
@pytest.mark.parametrize("H,G,D,V", [(2, 1, 64, 64), (3, 3, 64, 128), (4, 2, 128, 64), (2, 1, 128, 128), (2, 2, 128, 256),
                                     (2, 1, 128, 192), (2, 2, 64, 60), (2, 1, 96, 64)])
def test_delta(C, H, G, D, V, dt):  # noqa: F811
    check(DeltaCase(C, H, G, D, V, 4, T, dt), V, dt)


@DTYPES
@pytest.mark.parametrize("H,V,N,G", [(4, 64, 128, 1), (6, 64, 64, 3), (2, 128, 64, 2), (2, 128, 128, 1), (2, 256, 128, 1),
                                     (4, 64, 96, 1), (4, 32, 128, 1), (2, 62, 128, 1)])
def test_ssm(C, H, V, N, G, dt):  # noqa: F811
    check(SsmCase(C, H, V, N, G, 1, 4, T, dt), V, dt)


@DTYPES
@pytest.mark.parametrize("c0", [64, 66, 67])
def test_delta_off_vectors(C, c0, dt):  # noqa: F811
    c = DeltaCase(C, 2, 1, 128, 128, 4, T, dt)
    cols, at = c.ch + 2, c0 - c.c0
    y = torch.zeros(T, -(-(c0 + cols) // 64) * 64, dtype=dt)
    y[:, c0: c0 + cols] = c.y[:, c.c0: c.c0 + cols]
    c.y, c.c0 = y, c.c0 + at
    check(c, 128, dt)


# 16 heads: one round of blocks of 512 threads (48 sequences), of 256 (49 .. 64), then two of 512
@DTYPES
@pytest.mark.parametrize("B", [1, 48, 49, 64, 65])
def test_forget_rounds(C, B, dt):  # noqa: F811
    H, D, V, eps = 16, 128, 128, 1e-5
    g = torch.Generator().manual_seed(B)
    y = torch.randn(B, H * (2 * D + V), generator=g).to(dt)
    bias, lower, norm = torch.randn(H * D, generator=g), torch.rand(H * D, generator=g), 1 + 0.2 * torch.randn(V, generator=g)
    S = torch.randn(B, H, D, V, generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    state, out = S.cuda(), torch.empty(B, H * V, dtype=dt, device="cuda")
    C.forget_seq(y.cuda(), torch.arange(B, **i32), torch.full((B,), 9, **i32), torch.arange(B + 1, **i32), H, D, V, bias.cuda(),
                 lower.cuda(), norm.cuda(), eps, state, out, False, 1)
    q, z, v = y.double().split([H * D, H * D, H * V], 1)
    write = ((1 - lower.double()) * torch.sigmoid(-z - bias.double())).reshape(B, H, D, 1)
    want = S.double() * (1 - write) + write * v.reshape(B, H, 1, V)
    assert err(state, want) < 2e-6  # three roundings a number, and expf in the gate
    q = q * torch.sigmoid(q)
    o = (want * q.reshape(B, H, D, 1)).sum(2)
    o = o / torch.sqrt(o.pow(2).mean(-1, keepdim=True) + eps) * norm.double()
    assert err(out.reshape(B, H, V), o) < (8e-3 if dt == BF else 1e-5)


# as many rows as sequences, but not one each: offsets 0, 2, 2, 3, ..
@DTYPES
@pytest.mark.parametrize("start", [0, 2, 9])
@pytest.mark.parametrize("sizes", [[2, 0, 1], [0, 3, 0], [1, 1, 1], [6, 0, 0, 0, 0, 0]])
def test_rows_in_order(C, sizes, start, dt):  # noqa: F811
    H, D, V = 2, 128, 128
    for vec in (0, 1):  # on its vectors and off them: the general form
        c = DeltaCase(C, H, H, D, V, 4, start + sum(sizes), dt)
        y = torch.zeros(c.y.shape[0], c.y.shape[1] + 64, dtype=dt)
        y[:, vec: vec + c.y.shape[1]] = c.y
        taps, A, dtb, norm = c.par
        n, last = len(sizes), sizes.index(max(sizes))
        ring, state = c.ring[:1].repeat(n, 1, 1), c.state[:1].repeat(n, 1, 1, 1)
        args = (H, H, D, V, taps, ring, state, A, dtb, norm, c.gain, c.eps)
        if start:
            C.delta_seq(cuda(y[:start]), c.c0 + vec, c.c0 + vec + c.ch, cuda(c.low[:start]), c.nl, i32([last]), i32([0]),
                        i32([0, start]), *args, torch.empty(start, H * V, dtype=dt, device="cuda"), False, False)
        starts, cu = [start if k == last else 0 for k in range(n)], torch.tensor([0] + sizes).cumsum(0).tolist()
        out = torch.full((sum(sizes), H * V), float("nan"), dtype=dt, device="cuda")
        rows = slice(start, start + sum(sizes))
        C.delta_seq(cuda(y[rows]), c.c0 + vec, c.c0 + vec + c.ch, cuda(c.low[rows]), c.nl, i32(list(range(n))), i32(starts), i32(cu),
                    *args, out, True, False)
        if sizes[last] > 1 and cu[last] == 0 and sizes[last] == sum(sizes):
            assert err(out, c.want[rows]) < (3e-2 if dt == BF else 3e-5)
            assert err(state[last], c.S) < 2e-5
        if vec == 0:
            tiles, held = (out, state.clone(), ring.clone()), [k for k, m in enumerate(sizes) if m]
    assert err(tiles[0], out.cpu()) < (8e-3 if dt == BF else 1e-5)
    assert err(tiles[1][held], state[held].cpu()) < 1e-5 and torch.equal(tiles[2][held].nan_to_num(), ring[held].nan_to_num())


# one sequence takes all rows: several V blocks (outputs normed behind them), Mamba-2 heads
@DTYPES
@pytest.mark.parametrize("case", [lambda C, T, dt: DeltaCase(C, 2, 2, 128, 256, 4, T, dt),
                                  lambda C, T, dt: DeltaCase(C, 2, 2, 64, 64, 4, T, dt),
                                  lambda C, T, dt: SsmCase(C, 2, 64, 128, 2, 1, 4, T, dt),
                                  lambda C, T, dt: SsmCase(C, 2, 128, 64, 2, 1, 4, T, dt)])
def test_all_rows_in_one(C, case, dt):  # noqa: F811
    from types import SimpleNamespace

    T = 5
    c = case(C, T, dt)
    calls = SimpleNamespace()

    def once(name):
        def call(*args):  # the case's own call, as one of T sequences of which the others have no row
            args = list(args)
            k = next(i for i, a in enumerate(args) if isinstance(a, torch.Tensor) and a.dtype == torch.int32)
            args[k: k + 3] = [i32([1] + [2] * (T - 1)), i32([0] * T), i32([0] + [T] * T)]
            flag = next(i for i, a in enumerate(args) if a is False)  # single
            args[flag] = True
            getattr(C, name)(*args)
        return call

    calls.delta_seq, calls.ssm_seq = once("delta_seq"), once("ssm_seq")
    c.C = calls
    assert err(c.run(portions(T, [T]), False), c.want) < (3e-2 if dt == BF else 3e-5)
    assert err(c.state[1, ..., : c.S.shape[-1]], c.S) < 2e-5
