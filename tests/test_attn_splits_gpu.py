"""Decode attention whose contexts are taken in more splits than the caller asks for: the rule, and
contexts that end in, on and before a split's last tile."""

import pytest


def test_rule():
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")
    for B, splits, keys, want in [(40, 3, 1490, 4), (40, 2, 780, 4), (40, 1, 257, 3), (40, 1, 256, 1), (40, 3, 0, 3),
                                  (64, 1, 400, 1), (63, 1, 400, 3), (16, 4, 2000, 12), (5, 8, 4000, 16), (32, 1, 260, 3),
                                  (24, 64, 2000, 64), (31, 1, 1000, 2), (0, 1, 1000, 4)]:
        assert _C.attn_decode_total(B, 8, 4, 128, splits, keys) == want, (B, splits, keys)
    assert _C.attn_decode_total(40, 8, 3, 128, 2, 900) == 2 and _C.attn_decode_total(40, 8, 4, 64, 2, 900) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("nh", [16, 32, 64])
@pytest.mark.parametrize("B,splits,last,keys", [(32, 1, 256, 257), (40, 1, 383, 384), (63, 2, 300, 912), (36, 2, 911, 912),
                                                (150, 1, 911, 912), (255, 1, 320, 912), (256, 1, 320, 912)])
def test_more_splits(nh, B, splits, last, keys):
    from .test_attn_few_gpu import test_few_sequences as check

    check(B, nh, 8, splits, last, keys)
