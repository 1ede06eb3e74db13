"""Prompt attention with mixed heads, its keys in parts as long as the longest tile's: parts without keys, and what
stands where their outputs would."""

import pytest
import torch

from .paged_helpers import BF, Batch, err
from .test_vizalix_gpu import C, attention_case, frag, unpad, up  # noqa: F401



def test_rule():
    from llm_sharding_demo_amd.ops.routing import Routing

    r = Routing()
    for qlens, starts, window, want in [([1000], [0], 1024, 11), ([500], [0], 1024, 16), ([250] * 4, [0] * 4, 1024, 8), ([100], [0], 1024, 4),
                                        ([1500], [0], 1024, 7), ([4000], [0], 1024, 2), ([20000], [0], 1024, 1), ([16], [7000], 1 << 30, 16),
                                        ([0, 5], [3, 0], 64, 1), ([0], [0], 64, 1)]:
        assert r.talk_prefill_parts(qlens, starts, window, 16) == want, (qlens, starts)
    # partial outputs of every token and split: as many as equal prompts have, not more where one is longer than the others
    for qlens, starts, window, want in [([16] * 800 + [16], [0] * 800 + [30000], 1 << 30, 1), ([16] * 500 + [16], [0] * 500 + [8000], 1024, 1),
                                        ([16] * 100 + [1000], [0] * 101, 1024, 6), ([1] * 300 + [16], [0] * 300 + [8000], 1024, 16)]:
        got = r.talk_prefill_parts(qlens, starts, window, 16)
        assert got == want and (got == 1 or got * sum(qlens) <= 2 * 490 * 16), (len(qlens), got)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V", [(16, 4, 64, 64), (6, 2, 24, 20), (32, 8, 128, 128)])
@pytest.mark.parametrize("window,splits,keys", [(1 << 30, 3, 130), (1 << 30, 5, 163), (1 << 30, 16, 163), (1 << 30, 2, 64), (67, 4, 67),
                                                (67, 4, 163), (5, 3, 163), (1 << 30, 3, 4096)])
def test_parts(C, H, G, D, V, window, splits, keys):  # noqa: F811
    b = Batch((1, 0, 75), (2, 70, 2), (0, 130, 33))
    q, K, Vp, table, talk, want, out, scale, cap = attention_case(H, G, D, V, BF, b, window)
    hp = C.talk_heads(H, G, up(D, 32), up(V, 16), cap)
    torch.full((1 << 22,), float("nan"), device="cuda")  # (given back: the partial outputs begin as this)
    C.talk_prefill(q, K, Vp, table, frag(talk, hp), b.tiles(C.talk_tile(hp)), b.slots, b.start, b.cu, window, scale, cap,
                   splits, out, keys)
    assert err(unpad(out, H, V), want) < 3e-2
