"""Decode attention of 64-dim ungrouped heads: 2, 4 or 8 keys in flight by the longest context, whose
rounds end at 64, 128 and 256 keys, against float64 on the CPU."""

import pytest
import torch

from .test_gemv_gpu import C, bf  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


# few items, 512 and 2048 of them: the lines between two and four, four and eight keys
@pytest.mark.parametrize("B,nh,splits", [(3, 5, 1), (3, 5, 3), (64, 8, 1), (128, 16, 1)])
@pytest.mark.parametrize("longest", [1, 63, 64, 65, 128, 129, 256, 257, 400])
def test_contexts(C, B, nh, splits, longest):  # noqa: F811
    S = longest + 3
    kc, vc, q = bf(B + 1, nh, S, 64, seed=1), bf(B + 1, nh, S, 64, seed=2), bf(B, nh * 64, seed=3)
    slots = torch.arange(B, 0, -1, dtype=torch.int32, device=DEV)
    pos = torch.tensor([longest - 1 - (i * 5) % longest for i in range(B)], dtype=torch.int32, device=DEV)
    out = C.attn_decode(q, kc, vc, slots, pos, nh, splits, longest)
    qd, kd, vd = (t.double().cpu() for t in (q.view(B, nh, 64), kc[slots.long()], vc[slots.long()]))
    s = (kd @ qd[..., None])[..., 0] / 8
    s = s.masked_fill(torch.arange(S) > pos.cpu()[:, None, None], float("-inf"))
    want = (torch.softmax(s, -1)[:, :, None] @ vd)[:, :, 0].flatten(1)
    # fp32 sums and a result rounded to bf16: half a step of 2^-8 of the value, and of a value near zero what its terms round to
    err = (out.double().cpu() - want).abs()
    assert bool((err <= want.abs() * 2.0**-8 + 1e-4).all()), float(err.max())
