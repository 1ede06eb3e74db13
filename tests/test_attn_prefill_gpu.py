"""Prompt attention in query tiles of 64 and 128 against 64 bits: edges of the
query and key tiles, cached keys in front, groups of heads, sequences whose
scores grow late, and a cache whose rows behind the last key are not numbers.

Weights and values are rounded to bf16 once each (2^-9 each way), and so is the
result; errors of the keys' terms are independent.
"""

import pytest
import torch

from llm_sharding_demo_amd.ops.hip import latent_tiles
from llm_sharding_demo_amd.runtime.batch import BatchMeta

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def attend(q, k, v, start):
    """[T, H, D] queries behind `start` cached keys, [K, G, D] keys, in 64 bits."""
    q, k, v = q.double(), k.double(), v.double()
    G = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    s = (q.transpose(0, 1) @ k.permute(1, 2, 0)) * q.shape[2] ** -0.5
    hide = torch.arange(k.shape[0])[None] > start + torch.arange(q.shape[0])[:, None]
    return (torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ v.transpose(0, 1)).transpose(0, 1)


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("hd,nh,n_kv", [(64, 3, 3), (64, 16, 2), (128, 8, 2), (128, 5, 1)])
@pytest.mark.parametrize("late", [False, True])
def test_edges(hd, nh, n_kv, rows, late):
    from llm_sharding_demo_amd import _C as C

    starts = [0, 0, 0, 0, 0, 5, 63, 64, 65, 200, 130]
    lens = [1, 16, 63, 64, 65, 129, 1, 31, 127, 128, 193]
    B, S = len(lens), 400
    gen = torch.Generator().manual_seed(hd + nh)
    kc, vc = (torch.randn(B + 1, n_kv, S, hd, generator=gen).bfloat16() for _ in range(2))
    q = torch.randn(sum(lens), nh * hd, generator=gen).bfloat16()
    if late:  # weights of later keys leave the earlier ones behind, in steps
        kc *= (1 + 4 * (torch.arange(S) // 50)[:, None] / 8).bfloat16()
        q *= 3
    slots = torch.randperm(B + 1, generator=gen)[:B].tolist()
    for s, st, n in zip(slots, starts, lens):
        kc[s, :, st + n:], vc[s, :, st + n:] = float("nan"), float("nan")
    meta = BatchMeta.build(slots, starts, lens, DEV)
    got = C.attn_prefill(q.to(DEV), kc.to(DEV), vc.to(DEV), latent_tiles(meta, 1, rows).to(DEV), meta.seq_slots,
                         meta.q_start, meta.cu_q, nh, rows).cpu().reshape(-1, nh, hd)
    at = 0
    for s, st, n in zip(slots, starts, lens):
        want = attend(q[at:at + n].reshape(n, nh, hd), kc[s, :, :st + n].transpose(0, 1),
                      vc[s, :, :st + n].transpose(0, 1), st)
        d = (got[at:at + n].double() - want).pow(2).mean().sqrt()
        assert float(d) < 3 * 2 ** -9 * float(want.pow(2).mean().sqrt()), (st, n)
        at += n
