"""Chunked delta rule with factors of their own against the form that keeps a chunk in one
block (which tests/test_vizalix_gpu.py holds against the oracle): the same products of the same
operands, summed in another order, so outputs differ by a rounding of bf16 (2^-8 of the value
and of the row's root mean square, which the norm divides by) and states by fp32 sums."""
import pytest
import torch

from .test_vizalix_gpu import BF, DeltaCase, cuda, i32, portions, up

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def C():
    from llm_sharding_demo_amd import _C
    return _C


def run(C, split, lens, starts, H, G, D, V, n=4, strong=0.0, max_rows=0):
    g = torch.Generator(device=DEV).manual_seed(H * D + V + len(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    T, ch = sum(lens), 2 * G * D + H * V
    pad = lambda k, m: -(-k // m) * m  # noqa: E731
    y = torch.zeros(T, pad(ch + H, 64), device=DEV).bfloat16()
    y[:, : ch + H] = rnd(T, ch + H).bfloat16()
    nl = pad(max(H * D, H * V), 16)
    low = rnd(T, 2 * nl).bfloat16()
    dtb = rnd(H * D) - 2
    if strong:  # channels that outrun the range of a chunk's factors
        dtb += strong * (torch.rand(H * D, generator=g, device=DEV) < 0.2)
    ring = rnd(len(lens), n, ch).bfloat16()
    state = rnd(len(lens), H, D, pad(V, 4)) * 0.1
    cu = [0]
    for k in lens:
        cu.append(cu[-1] + k)
    out = torch.full((T, pad(H * V, 64)), float("nan"), device=DEV).bfloat16()
    C.delta_seq(y, 0, ch, low, nl, i32(list(range(len(lens)))), i32(starts), i32(cu), H, G, D, V, rnd(ch, n) / n ** 0.5, ring,
                state, -torch.exp(rnd(H)), dtb, 1 + 0.2 * rnd(V), 0.75, 1e-5, out, False, True, max_rows, split)
    return out.float(), state, ring


@pytest.mark.parametrize("H,G,D,V", [(2, 2, 8, 8), (4, 2, 24, 20), (3, 3, 64, 64), (2, 1, 128, 128), (4, 4, 32, 100), (5, 5, 96, 68)])
@pytest.mark.parametrize("lens,starts", [([1], [0]), ([16], [0]), ([17], [5]), ([160], [0]), ([33, 1, 100, 15], [0, 7, 0, 64])])
@pytest.mark.parametrize("strong", [0.0, 12.0])
def test_forms_agree(C, H, G, D, V, lens, starts, strong):
    a, b = (run(C, s, lens, starts, H, G, D, V, strong=strong, max_rows=m) for s, m in ((0, 0), (1, max(lens))))
    assert torch.equal(torch.isnan(a[0]), torch.zeros_like(a[0], dtype=torch.bool)) and not b[0].isnan().any()
    rms = a[0].pow(2).mean().sqrt()
    assert bool(((a[0] - b[0]).abs() <= 2.0 ** -7 * (a[0].abs() + rms)).all())
    scale = a[1].abs().amax()
    assert bool(((a[1][..., :V] - b[1][..., :V]).abs() <= 1e-4 * scale).all())
    assert torch.equal(a[2], b[2])


@pytest.mark.parametrize("H,D,V,lens", [(16, 128, 128, [20, 33]), (16, 128, 128, [20, 33, 1]), (43, 64, 100, [70]), (32, 24, 20, [17] * 5)])
def test_blocks_of_one_tile_and_of_two(C, H, D, V, lens):
    """Tiles of 16 columns on 256 CUs: as many, and more (two a block, odd numbers of them too)."""
    a, b = (run(C, s, lens, [0, 7, 0, 3, 0][: len(lens)], H, H, D, V, max_rows=max(lens)) for s in (0, 1))
    assert not b[0].isnan().any()
    assert bool(((a[0] - b[0]).abs() <= 2.0 ** -7 * (a[0].abs() + a[0].pow(2).mean().sqrt())).all())
    assert bool(((a[1][..., :V] - b[1][..., :V]).abs() <= 1e-4 * a[1].abs().amax()).all())


def test_long_sequences_in_portions(C):
    """256 (sequence, head) pairs: some chunks' factors fit the workspace at a time.  Sequences
    that end in the first, second and third portion, at its edge and behind cached tokens."""
    p = C.delta_portion_rows(128, 32, 8)
    lens = [2 * p + 5, 3, p, p + 1, 1, 16, p + 170, 17]
    assert max(lens) > 2 * p
    a, b = (run(C, s, lens, [0, 0, 5, 0, 9, 0, 130, 0], 32, 32, 128, 128, max_rows=max(lens)) for s in (0, 1))
    assert bool(((a[0] - b[0]).abs() <= 2.0 ** -7 * (a[0].abs() + a[0].pow(2).mean().sqrt())).all())
    assert bool(((a[1] - b[1]).abs() <= 1e-4 * a[1].abs().amax()).all())


@pytest.mark.parametrize("H,G,D,V", [(4, 2, 24, 20), (2, 1, 128, 128), (3, 3, 64, 100)])
@pytest.mark.parametrize("sizes", [[225], [129, 96], [33, 1, 191]])
@pytest.mark.parametrize("decay,strong", [(1.0, 0.0), (0.01, 0.0), (30.0, 0.0), (1.0, 12.0)])
def test_against_64_bits(C, H, G, D, V, sizes, decay, strong):
    """Factors of their own (decays from the chunk's beginning) are no further from 64 bits
    than those of the form that keeps a chunk in one block: root mean squares within 2 %."""
    c = DeltaCase(C, H, G, D, V, 4, 225, BF, decay=decay, strong=strong)
    taps, A, dtb, norm = c.par
    off = []
    for split in (0, 1):
        c.state.fill_(float("nan"))
        outs = []
        for a, b in portions(225, sizes):
            out = torch.full((b - a, up(H * V, 64)), float("nan"), dtype=BF, device=DEV)
            C.delta_seq(cuda(c.y[a:b]), c.c0, c.c0 + c.ch, cuda(c.low[a:b]), c.nl, i32([1]), i32([a]), i32([0, b - a]), H, G,
                        D, V, taps, c.ring, c.state, A, dtb, norm, c.gain, c.eps, out, False, True, b - a, split)
            outs.append(out[:, : H * V])
        off.append([float(((got.double().cpu() - want).pow(2).mean() / want.pow(2).mean()).sqrt())
                    for got, want in ((torch.cat(outs), c.want), (c.state[1, ..., :V], c.S))])
    (out0, state0), (out1, state1) = off
    assert out1 < 1.02 * out0 and state1 < 1.02 * state0, off


@pytest.mark.parametrize("lens,starts,hint", [([100, 37, 16], [0, 9, 0], 16), ([100, 37, 16], [0, 9, 0], 40),
                                              ([48, 33, 1], [4, 0, 0], 1), ([70], [0], 5)])
def test_longer_than_said(C, lens, starts, hint):
    """max_rows sizes launches: rows behind it are not left out, whatever it says."""
    a, b = (run(C, s, lens, starts, 2, 1, 128, 128, max_rows=m) for s, m in ((0, 0), (1, hint)))
    assert not b[0].isnan().any()
    assert bool(((a[0] - b[0]).abs() <= 2.0 ** -7 * (a[0].abs() + a[0].pow(2).mean().sqrt())).all())
    assert bool(((a[1] - b[1]).abs() <= 1e-4 * a[1].abs().amax()).all())
    assert torch.equal(a[2], b[2])
