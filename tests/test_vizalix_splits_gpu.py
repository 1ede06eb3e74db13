"""Prompt attention with mixed heads, its keys in parts as long as the longest tile's: parts without keys, and what
stands where their outputs would."""

from types import SimpleNamespace

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


def layer(meta, calls, heads=16):
    """The arguments (splits, keys) that a layer's launch over this batch takes."""
    from llm_sharding_demo_amd.ops.hip import HipBackend

    b = HipBackend.__new__(HipBackend)
    b.C = SimpleNamespace(talk_tile=lambda hp: 16, talk_prefill=lambda *a: calls.append((a[12], a[14])))
    b.fp32 = False
    weights = {"mixer.talk_prefill": torch.zeros(heads, heads)}
    m = SimpleNamespace(heads=heads, window=1024, softcap=6.0, keep_first=0, talking=True, talk_weights=False, scale=1.0)
    cache = torch.zeros(1, 4, 64, 128)
    b._attention(torch.zeros(meta.num_tokens, heads * 128), lambda n, *d: weights.get(n), m, cache, cache,
                 SimpleNamespace(table=None), meta, None, None)


def test_splits_are_reckoned_once_a_batch(monkeypatch):
    from llm_sharding_demo_amd.ops.hip import HipBackend
    from llm_sharding_demo_amd.runtime.batch import BatchMeta

    asked, calls, rule = [], [], HipBackend.R.talk_prefill_parts
    monkeypatch.setattr(type(HipBackend.R), "talk_prefill_parts", lambda self, *a: asked.append(a) or rule(*a))
    for first in (0, 400):
        meta = BatchMeta.build([0, 1], [0, first], [500, 100], "cpu")
        for _ in range(3):
            layer(meta, calls)
    assert len(asked) == 2 and len(set(calls)) == 1 and len(calls) == 6


def test_splits_of_a_captured_chunk():
    """Its replays start elsewhere: splits by tiles, each as long as its tile's keys over them, not as the captured context's."""
    from llm_sharding_demo_amd.runtime.batch import BatchMeta

    calls = []
    layer(BatchMeta.build([0], [0], [1000], "cpu"), calls)
    meta = BatchMeta.build([0], [3000], [200], "cpu")
    meta.host_starts = None
    layer(meta, calls)
    assert calls == [(11, 1000), (8, 0)]


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


@pytest.mark.gpu
@pytest.mark.parametrize("splits,keys", [(5, 0), (3, 0), (4, 163)])
def test_replays_at_other_starts(C, splits, keys):  # noqa: F811
    H, G, D, V, window = 16, 4, 64, 64, 1 << 30
    batches = [Batch((1, 0, 75), (2, 70, 2), (0, 130, 33)), Batch((0, 88, 75), (1, 73, 2), (2, 39, 33))]
    cases = [attention_case(H, G, D, V, BF, b, window, seed=i) for i, b in enumerate(batches)]
    own = [[*c[:4], b.slots, b.start] for c, b in zip(cases, batches)]
    held = [t.clone() for t in own[0]]
    hp = C.talk_heads(H, G, D, V, cases[0][8])
    f, tiles, cu, out = [frag(c[4], hp) for c in cases], batches[0].tiles(C.talk_tile(hp)), batches[0].cu, cases[0][6]
    mix = f[0].clone()

    def call():
        C.talk_prefill(held[0], held[1], held[2], held[3], mix, tiles, held[4], held[5], cu, window, cases[0][7], cases[0][8], splits, out, keys)
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for i in (0, 1, 0, 1):
        for t, new in zip(held + [mix], own[i] + [f[i]]):
            t.copy_(new)
        out.fill_(float("nan"))
        graph.replay()
        assert err(unpad(out, H, V), cases[i][5]) < 3e-2
