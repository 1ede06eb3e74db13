"""The convolution in front of a chunked recurrence takes 4, 8, 16 or 32 rows in turn, by the
rows of the launch: a row's result is the same in all of them."""

import pytest
import torch

from .test_vizalix_gpu import C, i32  # noqa: F401

pytestmark = pytest.mark.gpu
H, V, N, TAPS = 2, 64, 64, 4
INNER, CH = H * V, H * V + 2 * N
LENGTHS = [33, 1, 7, 100, 64, 31, 8, 9, 57, 90]  # 400 rows: 4 in turn


@pytest.mark.parametrize("copies", [4, 26, 52])  # 1600 rows (8), 10400 (16), 20800 (32)
@pytest.mark.parametrize("starts", [0, 5])
@pytest.mark.parametrize("taps_n", [4, 3])
def test_rows_in_turn(C, copies, starts, taps_n):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(copies)
    R = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    lens = LENGTHS * copies
    cu = torch.tensor([0] + lens).cumsum(0).tolist()
    y = R(cu[-1], INNER + CH + 64).bfloat16()
    par = (R(CH, taps_n) * 0.5, R(CH) * 0.3)
    rest = (-torch.rand(H, generator=g, device="cuda"), R(H) - 1, R(H), torch.ones(INNER, device="cuda"))
    ring, state = R(len(lens), taps_n, CH).bfloat16(), R(len(lens), H, N, V)

    def run(a, b):  # sequences a .. b - 1 in a launch
        rows = slice(cu[a], cu[b])
        out = torch.empty(cu[b] - cu[a], INNER, dtype=torch.bfloat16, device="cuda")
        C.ssm_seq(y[rows], i32(list(range(a, b))), i32([starts] * (b - a)), i32([x - cu[a] for x in cu[a: b + 1]]), H, 1, N, V, 1,
                  *par, ring.clone(), state.clone(), *rest, 0.75, 1e-5, out, False, True, 0, 1)
        return out

    n = len(LENGTHS)
    want = torch.cat([run(k * n, (k + 1) * n) for k in range(copies)])
    assert torch.equal(run(0, len(lens)), want)
