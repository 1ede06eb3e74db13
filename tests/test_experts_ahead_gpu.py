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


class Spy:
    """The kernels, with the parts of every latent attention and the rows of slabs that an out-projection leaves."""

    def __init__(self, C):
        self.C, self.parts, self.slabs = C, [], 0

    def __getattr__(self, name):
        return getattr(self.C, name)

    def latent_decode(self, q, *args):
        self.parts.append((q.shape[0], args[7]))
        return self.C.latent_decode(q, *args)

    def linear_residual(self, *args):
        self.slabs += len(args) > 8 and args[8] is not None
        return self.C.linear_residual(*args)


def wide_model(path, heads=16, rank=512):
    """Contexts that decode attention takes in parts, and an out-projection that leaves slabs."""
    cfg = orc.config([orc.layer(heads=heads, dim=64, vdim=64, rank=rank, window=None, experts=8, ff=128, shared_ff=64),
                      orc.layer(heads=heads, dim=64, vdim=64, rank=rank, window=None, kv_from=0, experts=8, ff=128, shared_ff=64)],
                     vocab=200, width=256)
    orc.save(path, cfg, orc.random_weights(cfg, 3))
    return cfg


@pytest.mark.parametrize("seqs", [5, 17])
def test_parts_are_those_of_eager_steps(seqs, tmp_path):
    """How many parts a step's attention takes hangs on its rows and contexts, not on whether it is captured, so an
    engine's first use of a bucket and the later ones draw the same tokens."""
    from llm_sharding_demo_amd.config import SamplingParams

    path = str(tmp_path)
    cfg = wide_model(path)
    room = dict(max_batch=seqs, max_seq_len=768, kv_tokens=768 * seqs)
    prompts = [ids_of(250 + 23 * i, cfg["vocab"], i) for i in range(seqs)]
    sp = SamplingParams(temperature=0.8, top_k=20, seed=5, max_new_tokens=24)
    eager, eng = make_engine(path, "bf16", use_graphs=False, **room), make_engine(path, "bf16", **room)
    spies = []
    for e in (eager, eng):
        be = e.stages[0].backend
        be.C = Spy(be.C)
        spies.append(be.C)
    want = eager.generate_ids(prompts, sp)
    for _ in range(2):
        assert eng.generate_ids(prompts, sp) == want
    assert eng.stages[0].backend._sides and bool(spies[1].slabs) == (seqs > 8)  # (up to 8 rows are added by a GEMV)
    parts = [set(s.parts) for s in spies]
    assert parts[0] == parts[1] and max(p for _, p in parts[0]) > 1


def test_graphs_of_two_lanes(tmp_path):
    """Steps with the chip to themselves and steps beside another lane have graphs of their own, also of one size."""
    from llm_sharding_demo_amd.config import SamplingParams

    path = str(tmp_path)
    cfg = wide_model(path, heads=4, rank=192)
    room = dict(max_batch=16, max_seq_len=192, kv_tokens=192 * 16, num_microbatches=2)
    prompts = [ids_of(20 + i, cfg["vocab"], i) for i in range(16)]
    sps = [SamplingParams(temperature=0.8, top_k=20, seed=5, max_new_tokens=n) for n in (60, 20)]
    eager, eng = make_engine(path, "bf16", use_graphs=False, **room), make_engine(path, "bf16", **room)
    for order in ([0] * 8 + [1] * 8, [0, 1] * 8):
        args = prompts, [sps[i] for i in order]
        want = eager.generate_ids(*args)
        for _ in range(2):
            assert eng.generate_ids(*args) == want
    keys = [k for gs in eng.workers[0].groups.values() for k in gs.graphs]
    alone = {k[:3] for k in keys if k[3]}
    assert alone & {k[:3] for k in keys if not k[3]}


def test_side_stream_is_not_the_capturing_one(tmp_path, monkeypatch):
    """Streams come from a pool, which hands the side stream out again after 32 others."""
    import torch

    from llm_sharding_demo_amd.config import SamplingParams

    path = str(tmp_path)
    cfg = wide_model(path, heads=4, rank=192)
    room = dict(max_batch=8, max_seq_len=192, kv_tokens=192 * 8)
    prompts = [ids_of(20 + i, cfg["vocab"], i) for i in range(8)]
    sp = SamplingParams(temperature=0.8, top_k=20, seed=5, max_new_tokens=20)
    eng = make_engine(path, "bf16", **room)
    want = eng.generate_ids(prompts, sp)
    be, w = eng.stages[0].backend, eng.workers[0]
    side, new, made = be._sides[0], torch.cuda.Stream, []

    def stream(*args, **kw):
        if "stream_id" in kw:  # one that exists
            return new(*args, **kw)
        made.append(side if not made else new(*args, **kw))
        return made[-1]
    for gs in w.groups.values():
        gs.drop_graphs(w)
    monkeypatch.setattr(torch.cuda, "Stream", stream)
    for _ in range(2):
        assert eng.generate_ids(prompts, sp) == want
    assert made and be._sides[0] != side
