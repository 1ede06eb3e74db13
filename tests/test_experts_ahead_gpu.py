"""Captured decode steps whose experts run beside the attention: the tokens of eager steps, replay after replay."""

import pytest

from . import timisun_oracle as orc
from .test_timisun_gpu import MODELS, ids_of, make_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(MODELS))
@pytest.mark.parametrize("seqs", [5, 17])
def test_graphs_match_eager(name, seqs, tmp_path):
    from llm_sharding_demo_amd.config import SamplingParams

    make, kw = MODELS[name]
    cfg = orc.config(make(), **kw)
    path = str(tmp_path)
    orc.save(path, cfg, orc.random_weights(cfg, 3))
    room = dict(max_batch=seqs, max_seq_len=192, kv_tokens=192 * seqs)
    prompts = [ids_of(5 + 3 * i, cfg["vocab"], i) for i in range(seqs)]
    sp = SamplingParams(temperature=0.8, top_k=20, seed=5, max_new_tokens=40)
    eager = make_engine(path, "bf16", use_graphs=False, **room)
    want = eager.generate_ids(prompts, sp)
    assert not eager.stages[0].backend._sides
    eng = make_engine(path, "bf16", **room)
    for _ in range(3):
        assert eng.generate_ids(prompts, sp) == want
    assert bool(eng.stages[0].backend._sides) == any(layer.get("mlp") for layer in cfg["layers"])
