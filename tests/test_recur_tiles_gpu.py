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
