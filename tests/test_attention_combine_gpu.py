"""Partial outputs of decode attention combined: by one wave up to eight splits, by four from nine on, some of them with
few splits or none, and splits without keys."""

import pytest

from .paged_helpers import BF, Batch
from .test_kedasun_gpu import AttentionCase, C  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V", [(6, 2, 40, 24), (16, 4, 128, 128), (1, 1, 64, 16), (20, 5, 128, 48)])
@pytest.mark.parametrize("window,keep", [(None, 0), (67, 5)])
def test_splits(C, H, G, D, V, window, keep):  # noqa: F811
    c = AttentionCase(C, H, G, D, V, BF, Batch((1, 0, 1), (2, 63, 1), (0, 1300, 1)), window, keep, False)
    for splits in (2, 8, 9, 10, 13, 33, 64, 65, 200, 256):
        assert c.err(c.decode(splits)) < 3e-2, splits  # whole rows' bound: the same terms, summed in fp32
