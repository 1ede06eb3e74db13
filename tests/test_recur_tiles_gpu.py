"""Recurrent decode steps where threads hold whole tiles of the state, against 64 bits and
against the general form, which takes portions of two tokens and rows off their vectors."""

import pytest
import torch

from .test_vizalix_gpu import BF, F32, C, DeltaCase, SsmCase, err, portions  # noqa: F401

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
