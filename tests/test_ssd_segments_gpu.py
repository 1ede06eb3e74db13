"""Mamba-2 prompts in segments that run together, against 64 bits: the state of
each segment joined in fp32, so errors are those of one segment (bf16 factors).
Segments that are empty, of one token, and more than there are chunks.
"""

import pytest
import torch

from .test_vizalix_gpu import BF, C, SsmCase, cuda, err, i32, portions, up  # noqa: F401

pytestmark = pytest.mark.gpu


def run(c, parts, segs):
    H, V, N, G, NG = c.dims
    taps, bias, A, dtb, skip, norm = c.par
    c.state.fill_(float("nan"))
    outs = []
    for a, b in parts:
        out = torch.full((b - a, up(H * V, 64)), float("nan"), dtype=BF, device="cuda")
        c.C.ssm_seq(cuda(c.y[a:b]), i32([1]), i32([a]), i32([0, b - a]), H, G, N, V, NG, taps, bias, c.ring, c.state, A, dtb,
                    skip, norm, c.gain, c.eps, out, False, True, b - a, segs)
        outs.append(out[:, : H * V])
    return torch.cat(outs)


@pytest.mark.parametrize("H,V,N,G,NG", [(4, 64, 128, 1, 1), (3, 128, 64, 3, 3), (2, 12, 20, 2, 1), (2, 100, 36, 1, 2)])
@pytest.mark.parametrize("sizes", [[225], [129, 96], [33, 1, 191]])
@pytest.mark.parametrize("decay", [1.0, 0.01, 30.0])
def test_segments(C, H, V, N, G, NG, sizes, decay):  # noqa: F811
    c = SsmCase(C, H, V, N, G, NG, 4, 225, BF, decay=decay)
    one = run(c, portions(225, sizes), 1)
    base, base_state = err(one, c.want), err(c.state[1, ..., :V], c.S)
    for segs in (2, 3, 4, 8, 20):
        out = run(c, portions(225, sizes), segs)
        assert err(out, c.want) < 1.02 * base + 1e-5, segs
        assert err(c.state[1, ..., :V], c.S) < 1.02 * base_state + 1e-6, segs


def test_unequal_sequences(C):  # noqa: F811
    c = SsmCase(C, 4, 16, 32, 2, 2, 4, 300, BF)
    H, V, N, G, NG = c.dims
    taps, bias, A, dtb, skip, norm = c.par
    lens, slots = [300, 3, 33, 1, 128], [2, 0, 3, 1, 4]
    cu = [0, 300, 303, 336, 337, 465]
    ring = torch.full((5, 4, H * V + 2 * G * N), float("nan"), dtype=BF, device="cuda")
    outs = []
    for segs, longest in ((1, 300), (4, 300), (4, 0), (4, 128)):
        state = torch.full((5, H, N, V), float("nan"), device="cuda")
        out = torch.empty(465, H * V, dtype=BF, device="cuda")
        C.ssm_seq(cuda(torch.cat([c.y[:n] for n in lens])), i32(slots), i32([0] * 5), i32(cu), H, G, N, V, NG, taps, bias,
                  ring, state, A, dtb, skip, norm, c.gain, c.eps, out, False, True, longest, segs)
        for a, n in zip(cu, lens):
            assert err(out[a: a + n], c.want[:n]) < 6e-2
        assert err(state[2], c.S) < 3e-2
        outs.append(state)
    assert all(err(s, outs[0].cpu()) < 1e-5 for s in outs[1:])
