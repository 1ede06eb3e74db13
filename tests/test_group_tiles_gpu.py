"""The order of expert tiles: row tiles in groups whose last one is full or ends early, of few and of
many tokens."""

import pytest
import torch

from .test_timisun_gpu import C, test_experts_grouped as check_experts  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [513, 577, 2048, 2049, 2200])
def test_shared_tiles(C, dtype, T):  # noqa: F811
    check_experts(C, dtype, T, 64, 5, 2, 32, 48)
