"""Workloads of the framework: one forward of a pipeline stage over the shapes it is served at.

Prompts and decode steps go through StageModel.forward, what every stage process runs; a
decode step is captured in a hipGraph once and replayed, as the stage worker does.  Replays
of given texts go through a TraceSession, as the trace command does.  Weights are the random
ones of the architecture.  A model and its cache are kept from one state to the next; a state
owns cache slots of its own.

A prompt writes the cache that it attends to and a decode step attends to the rows it writes,
so the logits show what the caches got; a recurrence shows its state in the next pass.
"""
from __future__ import annotations

import math
from functools import partial

import torch
import torch.nn.functional as F

from llm_sharding_demo_amd.config import (AttentionSpec, ChannelDeltaSpec, EngineConfig, ForgetSpec, LatentAttentionSpec,
                                          SSMSpec, get_model_config)
from llm_sharding_demo_amd.models.stage import StageModel
from llm_sharding_demo_amd.models.weights import init_stage_weights
from llm_sharding_demo_amd.runtime.batch import BatchMeta
from llm_sharding_demo_amd.runtime.engine import Engine
from llm_sharding_demo_amd.runtime.trace import TraceSession

DEV = "cuda"
STATES = 4           # states alive at once
FILL = 16384         # tokens a launch of a preparation brings
WEIGHT_SEED = 0


def _case(name, model, kind, seqs, shortest, longest, dtype="bf16"):
    return {"name": name, "model": model, "kind": kind, "seqs": seqs, "shortest": shortest, "longest": longest, "dtype": dtype}


def listed():
    """kind prompt: sequences of shortest .. longest tokens, logits of the last ones.
    kind decode: one token per sequence behind as many cached ones.  kind replay: given
    texts in one step of a trace."""
    return [
        # one user at a terminal, the smallest model: a chain of small launches
        _case("gpt2-decode-1", "gpt2", "decode", 1, 203, 203),
        # one group of the headline's decode step, mid-way through its 128 new tokens
        _case("gpt2-xl-decode-256", "gpt2-xl", "decode", 256, 129, 255),
        # prompts of a full batch join at once, none longer than the headline's 128
        _case("gpt2-xl-prompt-200", "gpt2-xl", "prompt", 200, 33, 128),
        # one user, the largest model: weights stream at the rate of the memory
        _case("llama-3-8b-decode-1", "llama-3-8b", "decode", 1, 911, 911),
        # a serving batch in mid-flight, contexts of all lengths
        _case("llama-3-8b-decode-40", "llama-3-8b", "decode", 40, 70, 1490),
        # one long document, near the context limit
        _case("llama-3-8b-prompt-1-long", "llama-3-8b", "prompt", 1, 7937, 7937),
        # experts and latents, a serving batch
        _case("timisun-2b-decode-64", "timisun-2b", "decode", 64, 100, 1300),
        # one prompt: recurrences whose steps follow one another
        _case("vizalix-2b-prompt-1", "vizalix-2b", "prompt", 1, 1000, 1000),
        # recurrent state of a batch, read and written every step
        _case("vizalix-2b-decode-96", "vizalix-2b", "decode", 96, 60, 420),
        # prompts of mixed lengths join together, weights mixed over the heads
        _case("kedasun-2b-prompt-12", "kedasun-2b", "prompt", 12, 150, 1850),
        # a small batch of a model with many small launches per layer
        _case("fagunex-2b-decode-24", "fagunex-2b", "decode", 24, 90, 700),
        # given texts scored in full precision
        _case("timisun-2b-replay-fp32", "timisun-2b", "replay", 4, 61, 222, "fp32"),
    ]


# largest batch and prompt tokens that a drawn case brings
_LIMITS = {"gpt2": (512, 32768), "gpt2-medium": (384, 32768), "gpt2-xl": (256, 24576), "llama-3-8b": (64, 7936),
           "timisun-2b": (192, 16384), "vizalix-2b": (160, 16384), "kedasun-2b": (160, 16384), "fagunex-2b": (160, 16384)}


def _spread(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    model = rng.choice(sorted(_LIMITS))
    kind = rng.choice(["prompt", "decode", "prompt", "decode", "decode", "replay"])
    batch, tokens = _LIMITS[model]
    cap = min(get_model_config(model).max_positions - 1, 8000)
    few = 1
    if model.startswith("timisun"):  # the logits of few rows hang on single close calls of a router
        few = 32
    if kind == "replay":
        dtype = rng.choice(["bf16", "fp32"]) if model.endswith("-2b") and few == 1 else "fp32" if few > 1 else "bf16"
        seqs, longest = rng.randint(1, 6), _spread(rng, 8, 250)
        return _pure(model, kind, seqs, _spread(rng, 2, longest), longest, dtype)
    if kind == "decode":
        seqs = _spread(rng, few, batch)
        longest = _spread(rng, 16, max(16, min(cap, 2 * 30000 // seqs)))
    else:
        seqs = _spread(rng, few, 128)
        longest = _spread(rng, 16, max(16, min(cap, tokens // seqs)))
    return _pure(model, kind, seqs, _spread(rng, max(1, longest // 16), longest), longest)


def _pure(*a):
    c = _case("", *a)
    del c["name"]
    return c


def _lengths(case):
    """Tokens of every sequence: evenly from the shortest to the longest, in mixed order."""
    n, lo, hi = case["seqs"], case["shortest"], case["longest"]
    return [hi] if n == 1 else [lo + (i * 7919 % n) * (hi - lo) // (n - 1) for i in range(n)]


def _tokens(case, seed):
    """Token ids, host: the prompts one behind the other, and one more per sequence."""
    g = torch.Generator().manual_seed(seed)
    V = get_model_config(case["model"]).vocab_size
    total = sum(_lengths(case))
    ids = torch.randint(0, V, (total + case["seqs"],), generator=g, dtype=torch.int32)
    return ids[:total], ids[total:]


# ---------------------------------------------------------------------------
# The model, kept; the states
# ---------------------------------------------------------------------------

class _Kept:
    """The model of the last case, its cache slots in groups."""

    key, stage, groups = None, None, []

    @classmethod
    def of(cls, case):
        kind = case["kind"]
        key = (case["model"], case["dtype"], kind == "replay", case["seqs"], case["longest"])
        if cls.key != key:
            cls.key = cls.stage = None
            cls.groups = []
            torch.cuda.empty_cache()
            mc, n = get_model_config(case["model"]), case["seqs"]
            room = case["longest"] + 1
            if kind == "replay":
                cls.stage = Engine(EngineConfig(model_id=case["model"], dtype=case["dtype"], device=DEV, max_batch=n,
                                                max_seq_len=-(-room // 64) * 64, use_graphs=False, seed=WEIGHT_SEED))
            else:
                cls.stage = StageModel(mc, 0, mc.n_layers, True, True, device=DEV, dtype=torch.bfloat16, seed=WEIGHT_SEED,
                                       max_slots=STATES * n, max_seq=room)
            cls.groups = [list(range(k * n, (k + 1) * n)) for k in range(STATES)]
            cls.key = key
        return cls.stage


class _State:
    """Slots of the kept model's cache, given back with the state."""

    def __init__(self, case):
        self.kind, self.stage = case["kind"], _Kept.of(case)
        self._key, self.slots = _Kept.key, _Kept.groups.pop()

    def __del__(self):
        self.graph = self.logits = None
        if _Kept is not None and _Kept.key == self._key:  # (None: the interpreter ends)
            _Kept.groups.append(self.slots)


def prepare(case, seed):
    s = _State(case)
    lengths, (prompts, last) = _lengths(case), _tokens(case, seed)
    if s.kind == "replay":
        s.session = TraceSession(s.stage)
        s.entries = [{"id": str(i), "tokens": p.tolist(), "want": [len(p) - 1]} for i, p in enumerate(prompts.split(lengths))]
        s.ends = [e["id"] for e in s.entries]
        return s
    s.vocab = s.stage.cfg.vocab_size
    if s.kind == "prompt":
        s.ids = prompts.to(DEV)
        s.meta = BatchMeta.build(s.slots, [0] * len(lengths), lengths, DEV)
        return s
    with torch.no_grad():
        i = at = 0
        while i < len(lengths):  # the contexts
            j, n = i, 0
            while j < len(lengths) and (j == i or n + lengths[j] <= FILL):
                n, j = n + lengths[j], j + 1
            s.stage.forward(BatchMeta.build(s.slots[i:j], [0] * (j - i), lengths[i:j], DEV), prompts[at: at + n].to(DEV), head=False)
            i, at = j, at + n
        s.ids = last.to(DEV)
        s.meta = BatchMeta.decode(s.slots, lengths, DEV, max(lengths) + 1)
        saved = _recurrent(s)
        s.stage.forward(s.meta, s.ids)  # allocates what the step keeps
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            s.logits = s.stage.forward(s.meta, s.ids)[:, : s.vocab]
        for t, before in saved:
            t[s.slots[0]: s.slots[-1] + 1] = before
    return s


def _recurrent(s):
    """(tensor, the state's part) of everything per slot that a step moves on."""
    if not s.stage.cfg.layers:
        return []
    per_slot = [t for e in s.stage.kv.entries for t in e if t.shape[0] == s.stage.kv.slots]
    return [(t, t[s.slots[0]: s.slots[-1] + 1].clone()) for t in per_slot]


def run(s):
    if s.kind == "replay":
        return s.session.step(s.entries, s.ends)
    if s.kind == "decode":
        s.graph.replay()
        return s.logits
    with torch.no_grad():
        m = s.meta  # a batch of its own per pass, as a step makes one
        meta = BatchMeta(m.token_slots, m.token_pos, m.seq_slots, m.q_start, m.cu_q, m.last_idx, m.num_tokens, m.num_seqs,
                         m.max_q, m.max_ctx, m.is_decode, m.host_qlens, m.host_starts)
        return s.stage.forward(meta, s.ids)[:, : s.vocab]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _mlp_params(mc, i, tokens):
    """(parameters read, parameters a token meets) of layer i's feed-forward."""
    f = mc.layers[i].mlp
    if not hasattr(f, "experts"):
        return f.params(mc.hidden), f.params(mc.hidden)
    one = 3 * mc.hidden * f.expert.ff
    rest = f.params(mc.hidden) - f.experts * one
    hit = f.experts * (1 - (1 - f.top / f.experts) ** tokens)
    return hit * one + rest, f.top * one + rest


def work(case):
    mc, n = get_model_config(case["model"]), _lengths(case)
    elt = 4 if case["dtype"] == "fp32" else 2
    decode = case["kind"] == "decode"
    B = len(n)
    T = B if decode else sum(n)
    read = mc.lm_head_params() + min(T, mc.vocab_size) * mc.hidden * (1 + mc.token_side * mc.n_layers / mc.hidden)
    flops = 2.0 * B * mc.lm_head_params()
    state = 0.0
    seen = set()
    for i in range(mc.n_layers):
        if mc.layers:
            m = mc.layers[i].mixer
            mr, ma = m.params(mc.hidden), m.params(mc.hidden)
            fr, fa = _mlp_params(mc, i, T)
            if mc.weight_layer(i) in seen:
                mr = fr = 0
            seen.add(mc.weight_layer(i))
            per_key = 2 * m.heads * (getattr(m, "q_dim", 0) + m.vdim if isinstance(m, LatentAttentionSpec) else
                                     m.dim + m.vdim if isinstance(m, AttentionSpec) else 0)
            cached, window = m.cached_per_token, getattr(m, "window", None) or 1 << 30
            if isinstance(m, (ChannelDeltaSpec, SSMSpec, ForgetSpec)):
                size = m.heads * m.vdim * (m.state if isinstance(m, SSMSpec) else m.dim)
                state += B * size * 4 * (2 if decode else 1)
                flops += 6.0 * T * size
        else:
            mr = ma = mc.block_params()
            fr = fa = 0
            per_key, cached, window = 4 * mc.q_size, 2 * mc.kv_size, 1 << 30
        read += mr + fr
        flops += 2.0 * T * (ma + fa)
        if decode:
            keys = sum(min(x + 1, window) for x in n)
            state += elt * cached * (keys + B)
        else:
            keys = sum(x * (x + 1) // 2 if x <= window else window * (window + 1) // 2 + (x - window) * window for x in n)
            state += elt * cached * T
        flops += per_key * keys
    return {"bytes": elt * read + state + 4 * B * mc.vocab_size, "flops": flops}


def tolerance(case):
    """Against 64 bits the forwards are 0.003 - 0.0065 off in bf16 and 1.2e-6 in fp32.  Where a
    router picks experts by sigmoids that lie close together, one pick in some dozens is
    another one in bf16: 0.028."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["model"].startswith("timisun"):
        return {"rel": 0.03, "max": 0.8}
    return {"rel": 0.025, "max": 0.3}


# ---------------------------------------------------------------------------
# The models in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    if work(dict(case, kind="prompt"))["flops"] > 7e14 or sum(_lengths(case)) > 60000:
        return None  # more than about 20 seconds
    _Kept.key = _Kept.stage = None
    torch.cuda.empty_cache()
    mc = get_model_config(case["model"])
    dt = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
    w = init_stage_weights(mc, range(mc.n_layers), True, True, WEIGHT_SEED, torch.device(DEV), dt)
    lengths, (prompts, last) = _lengths(case), _tokens(case, seed)
    texts = list(prompts.split(lengths))
    if case["kind"] == "decode":
        texts = [torch.cat([p, last[i: i + 1]]) for i, p in enumerate(texts)]
    with torch.no_grad():
        out = _Plain(mc, w, [len(t) for t in texts]).forward(torch.cat(texts).to(DEV).long())
    return out.cpu() if case["kind"] == "replay" else out


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


class _Plain:
    """Whole sequences, packed one behind the other, float64, no cache."""

    def __init__(self, mc, w, lengths):
        self.mc, self.raw, self.n = mc, w, lengths
        ends = torch.tensor(lengths).cumsum(0)
        self.parts = [slice(int(e) - n, int(e)) for e, n in zip(ends, lengths)]
        self.last = (ends - 1).to(DEV)
        self.pos = torch.cat([torch.arange(n) for n in lengths]).to(DEV)
        rows = torch.arange(max(lengths), device=DEV)
        first = (ends - torch.tensor(lengths)).to(DEV)
        self.real = rows[None] < torch.tensor(lengths, device=DEV)[:, None]
        self.padded = (first[:, None] + torch.minimum(rows[None], torch.tensor(lengths, device=DEV)[:, None] - 1))

    def w(self, name):
        return self.raw[name].to(torch.float64)

    def lin(self, x, name):
        return x @ self.w(name).T

    def forward(self, ids):
        mc = self.mc
        table = self.raw["wte" if mc.arch == "gpt2" else "embed_tokens"]
        x = table[ids].double() * mc.embed_scale
        if mc.arch == "gpt2":
            x = x + self.raw["wpe"][self.pos].double()
        self.ids, self.x0, self.values = ids, x, None
        layer = getattr(self, "_" + mc.arch)
        for i in range(mc.n_layers):
            x = layer(x, i, partial(self._name, i))
        x = x[self.last]
        if mc.arch == "gpt2":
            x = F.layer_norm(x, (mc.hidden,), self.w("ln_f.weight"), self.w("ln_f.bias"), mc.norm_eps)
        elif mc.arch == "kedasun":
            x = self.group_norm(x, "norm.weight")
        elif mc.arch == "fagunex":
            x = self.tanh_norm(x, "norm")
        else:
            x = _rms(x, mc.norm_eps) * (self.w("norm.weight") + (mc.arch == "timisun"))
        return self.lin(x, {"gpt2": "wte", "timisun": "embed_tokens"}.get(mc.arch, "lm_head"))

    def _name(self, i, leaf):
        return f"{'h' if self.mc.arch == 'gpt2' else 'layers'}.{self.mc.weight_layer(i)}.{leaf}"

    # -- attention: q [T, H, D], k, v [T, G, .] ------------------------------
    def attend(self, q, k, v, scale, window=None, keep=0, slopes=None, cap=None, mix_scores=None, mix_weights=None, sink=None):
        H, G = q.shape[1], k.shape[1]
        out = torch.empty(q.shape[0], H, v.shape[2], dtype=q.dtype, device=q.device)
        for p in self.parts:
            n = p.stop - p.start
            kk = k[p].permute(1, 2, 0).repeat_interleave(H // G, 0).contiguous()
            vv = v[p].transpose(0, 1).repeat_interleave(H // G, 0).contiguous()
            step = max(64, min(n, (1 << 27) // (H * n)))
            for a in range(0, n, step):
                b = min(n, a + step)
                s = torch.bmm(q[p.start + a: p.start + b].transpose(0, 1).contiguous(), kk[..., :b].contiguous()) * scale
                if cap:
                    s = cap * torch.tanh(s / cap)
                far = torch.arange(a, b, device=DEV)[:, None] - torch.arange(b, device=DEV)[None]
                if slopes is not None:
                    s = s - slopes[:, None, None] * far
                if mix_scores is not None:
                    s = (mix_scores @ s.reshape(H, -1)).reshape(s.shape)
                dark = far < 0
                if window is not None:
                    dark = dark | ((far >= window) & (torch.arange(b, device=DEV)[None] >= keep))
                s = s.masked_fill(dark, -math.inf)
                if sink is not None:
                    s = torch.softmax(torch.cat([s, sink[:, None, None].expand(H, b - a, 1)], -1), -1)[..., :-1]
                else:
                    s = torch.softmax(s, -1)
                if mix_weights is not None:
                    s = (mix_weights @ s.reshape(H, -1)).reshape(s.shape)
                out[p.start + a: p.start + b] = torch.bmm(s.contiguous(), vv[:, :b].contiguous()).transpose(0, 1)
        return out

    def turn(self, x, freq, interleaved=False):
        """x [T, heads, dims]: all of it rotated."""
        a = self.pos.double()[:, None, None] * torch.tensor(freq, dtype=torch.float64, device=DEV)
        half = x.shape[-1] // 2
        u, v = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., :half], x[..., half:])
        u, v = u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()
        return torch.stack([u, v], -1).flatten(-2) if interleaved else torch.cat([u, v], -1)

    def rope(self, x, rope):
        if rope is None or not rope.dims:
            return x
        d = rope.dims
        return torch.cat([self.turn(x[..., :d], rope.frequencies(), rope.interleaved), x[..., d:]], -1)

    def conv(self, x, taps):
        """Short convolution over time; the last tap weighs the current token."""
        y = torch.zeros_like(x)
        for back in range(taps.shape[1]):
            moved = torch.cat([torch.zeros_like(x[:back]), x[: x.shape[0] - back]])
            y += taps[:, taps.shape[1] - 1 - back] * torch.where((self.pos >= back)[:, None], moved, 0.0)
        return y

    def over_time(self, step, *rows):
        """step(t-th rows of all sequences) -> outputs, one token after the other."""
        rows = [r[self.padded] for r in rows]
        out = torch.stack([step(*(r[:, t] for r in rows)) for t in range(self.padded.shape[1])], 1)
        return out[self.real]

    def experts(self, h, name, f, ids, weights, act):
        y = torch.zeros_like(h)
        gu, dn = self.raw[name("mlp.experts.gate_up.weight")], self.raw[name("mlp.experts.down.weight")]
        for e in range(f.experts):
            t, c = (ids == e).nonzero(as_tuple=True)
            if len(t):
                y.index_add_(0, t, weights[t, c][:, None] * self.glu(h[t], gu[e].double(), dn[e].double(), act, f.expert.limit))
        return y

    def glu(self, h, gate_up, down, act, limit=None):
        g, u = (h @ gate_up.T).chunk(2, -1)
        if limit is not None:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return (act(g) * (u + (1 if limit is not None else 0))) @ down.T

    @staticmethod
    def swish(g):
        return g * torch.sigmoid(1.702 * g)

    # -- GPT-2 and Llama ------------------------------------------------------
    def _gpt2(self, x, i, name):
        mc, w, T = self.mc, self.w, x.shape[0]
        norm = lambda t, n: F.layer_norm(t, (mc.hidden,), w(name(n + ".weight")), w(name(n + ".bias")), mc.norm_eps)  # noqa: E731
        lin = lambda t, n: self.lin(t, name(n + ".weight")) + w(name(n + ".bias"))  # noqa: E731
        q, k, v = (t.reshape(T, mc.n_heads, -1) for t in lin(norm(x, "ln_1"), "attn.c_attn").chunk(3, -1))
        x = x + lin(self.attend(q, k, v, mc.head_dim ** -0.5).flatten(1), "attn.c_proj")
        return x + lin(F.gelu(lin(norm(x, "ln_2"), "mlp.c_fc"), approximate="tanh"), "mlp.c_proj")

    def _llama(self, x, i, name):
        mc, w, T, D = self.mc, self.w, x.shape[0], self.mc.head_dim
        h = _rms(x, mc.norm_eps) * w(name("input_layernorm.weight"))
        q, k, v = self.lin(h, name("self_attn.qkv.weight")).split([mc.q_size, mc.kv_size, mc.kv_size], -1)
        freq = [mc.rope_theta ** (-2.0 * j / D) for j in range(D // 2)]
        q, k = (self.turn(t.reshape(T, -1, D), freq) for t in (q, k))
        o = self.attend(q, k, v.reshape(T, -1, D), D ** -0.5)
        x = x + self.lin(o.flatten(1), name("self_attn.o_proj.weight"))
        h = _rms(x, mc.norm_eps) * w(name("post_attention_layernorm.weight"))
        return x + self.glu(h, w(name("mlp.gate_up.weight")), w(name("mlp.down_proj.weight")), F.silu)

    # -- Timisun ----------------------------------------------------------------
    def _timisun(self, x, i, name):
        mc, w, T = self.mc, self.w, x.shape[0]
        m, f = mc.layers[i].mixer, mc.layers[i].mlp
        if i == 0:
            self.latents = {}
        h = _rms(x, mc.norm_eps) * (1 + w(name("input_layernorm.weight")))
        if m.kv_from is None:
            self.latents[i] = _rms(self.lin(h, name("attn.dkv.weight")), mc.norm_eps) * w(name("attn.dkv_norm.weight"))
        c = self.latents[i if m.kv_from is None else m.kv_from]
        q, k, v = (self.lin(a, name(f"attn.{n}.weight")).reshape(T, m.heads, -1) for a, n in ((h, "q"), (c, "uk"), (c, "uv")))
        y = self.lin(self.attend(q, k, v, m.scale, m.window).flatten(1), name("attn.o.weight"))
        s = torch.sigmoid(self.lin(h, name("mlp.router.weight")))
        ids = (s + w(name("mlp.correction"))).topk(f.top, -1).indices
        ws = s.gather(1, ids)
        y = y + self.experts(h, name, f, ids, ws / (ws.sum(-1, keepdim=True) + 1e-20), self.swish)
        sh = self.glu(h, w(name("mlp.shared.gate_up.weight")), w(name("mlp.shared.down.weight")), self.swish, f.shared.limit)
        return x + y + sh

    # -- Vizalix ----------------------------------------------------------------
    def _vizalix(self, x, i, name):
        mc, w, spec = self.mc, self.w, self.mc.layers[i]
        if spec.enter is not None:
            x = self.lin(torch.cat([x, self.x0], -1), "loop.in") + w("loop.step")[spec.enter]
        r = _rms(x, mc.norm_eps)
        m, h, wm = spec.mixer, r * w(name("input_layernorm.weight")), lambda n: w(name("mixer." + n))  # noqa: E731
        if isinstance(m, ChannelDeltaSpec):
            y = self.delta(h, m, wm)
        elif isinstance(m, SSMSpec):
            y = self.mamba(h, m, wm)
        else:
            q, k, v = (h @ wm(n).T for n in "qkv")
            q, k = (self.rope(t.reshape(len(t), -1, m.dim), m.rope) for t in (q, k))
            y = self.attend(q, k, v.reshape(len(v), m.kv_heads, -1), m.scale, m.window, cap=m.softcap, mix_scores=wm("talk"))
            y = y.flatten(1)
        y = y @ wm("o").T
        h = r * w(name("post_attention_layernorm.weight"))
        gelu = partial(F.gelu, approximate="tanh")
        return x + y + self.glu(h, w(name("mlp.gate_up.weight")), w(name("mlp.down_proj.weight")), gelu)

    def delta(self, h, m, w):
        T, H, G, D = h.shape[0], m.heads, m.kv_heads, m.dim
        q, k, v = (F.silu(self.conv(h @ w(n).T, w(n + ".conv"))) for n in "qkv")
        q, k = (t.reshape(T, G, D).repeat_interleave(H // G, 1) for t in (q, k))
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        dt = F.softplus(h @ w("a1").T @ w("a2").T + w("dt_bias")).reshape(T, H, D)
        decay = torch.exp(-torch.exp(w("A_log"))[None, :, None] * dt)
        beta = torch.sigmoid(h @ w("b").T)
        S = torch.zeros(len(self.n), H, D, m.vdim, dtype=h.dtype, device=DEV)

        def step(q, k, v, g, b):
            S.mul_(g[..., None])
            u = b[..., None] * (v - (k[:, :, None] @ S)[:, :, 0])
            S.add_(k[..., None] * u[:, :, None])
            return (q[:, :, None] @ S)[:, :, 0]

        o = self.over_time(step, q * D ** -0.5, k, v.reshape(T, H, -1), decay, beta)
        return (_rms(o, self.mc.norm_eps) * w("norm") * torch.sigmoid(h @ w("g1").T @ w("g2").T).reshape(T, H, -1)).flatten(1)

    def mamba(self, h, m, w):
        T, H, G, N = h.shape[0], m.heads, m.groups, m.state
        z, xbc, dt = (h @ w("in").T).split([m.inner, m.conv_channels, H], -1)
        xbc = F.silu(self.conv(xbc, w("conv")) + w("conv.b"))
        x, B, C = xbc.split([m.inner, G * N, G * N], -1)
        x = x.reshape(T, H, -1)
        B, C = (t.reshape(T, G, N).repeat_interleave(H // G, 1) for t in (B, C))
        dt = F.softplus(dt + w("dt_bias"))
        S = torch.zeros(len(self.n), H, N, m.vdim, dtype=h.dtype, device=DEV)

        def step(x, B, C, g, dt):
            S.mul_(g[..., None, None]).add_((dt[..., None] * B)[..., None] * x[:, :, None])
            return (C[:, :, None] @ S)[:, :, 0]

        y = self.over_time(step, x, B, C, torch.exp(-torch.exp(w("A_log")) * dt), dt) + w("D")[:, None] * x
        y = (y.flatten(1) * F.silu(z)).reshape(T, m.norm_groups, -1)
        return _rms(y, self.mc.norm_eps).flatten(1) * w("norm")

    # -- Kedasun ----------------------------------------------------------------
    def group_norm(self, x, name):
        return _rms(x.reshape(len(x), self.mc.norm_groups, -1), self.mc.norm_eps).flatten(1) * self.w(name)

    def _kedasun(self, x, i, name):
        mc, w, T = self.mc, self.w, x.shape[0]
        m, f, wm = mc.layers[i].mixer, mc.layers[i].mlp, lambda n: w(name("mixer." + n))  # noqa: E731
        h = self.group_norm(x, name("input_layernorm.weight"))
        q, k, v = (h @ wm(n).T + (wm(n + ".b") if m.bias else 0) for n in "qkv")
        if m.conv:
            q, k, v = (self.conv(t, wm(n + ".conv")) for t, n in ((q, "q"), (k, "k"), (v, "v")))
        q, k, v = (t.reshape(T, -1, d) for t, d in ((q, m.dim), (k, m.dim), (v, m.vdim)))
        if m.qk_norm:
            q, k = _rms(q, mc.norm_eps), _rms(k, mc.norm_eps)
        q, k = self.rope(q, m.rope), self.rope(k, m.rope)
        if m.mix_values == i:
            self.values = v
        elif m.mix_values is not None:
            v = (1 - wm("vmix")) * v + wm("vmix") * self.values
        slopes = torch.tensor(m.slopes(), dtype=h.dtype, device=DEV) if m.distance_bias else None
        o = self.attend(q, k, v, m.scale, m.window, m.keep_first, slopes, mix_weights=wm("talk") if m.talking else None)
        if m.head_gate:
            o = o * torch.sigmoid(h @ wm("g").T)[:, :, None]
        y = o.flatten(1) @ wm("o").T + (wm("o.b") if m.bias else 0)
        x = x + self.group_norm(y, name("mixer.out_norm.weight"))
        h = self.group_norm(x, name("post_attention_layernorm.weight"))
        y = self.glu(h, w(name("mlp.gate_up.weight")), w(name("mlp.down_proj.weight")), self.swish, f.limit)
        return x + self.group_norm(y, name("mlp.out_norm.weight"))

    # -- Fagunex ----------------------------------------------------------------
    def tanh_norm(self, x, name):
        return torch.tanh(self.w(name + ".alpha") * x) * self.w(name + ".weight") + self.w(name + ".bias")

    def _fagunex(self, x, i, name):
        mc, w, T = self.mc, self.w, x.shape[0]
        m, f = mc.layers[i].mixer, mc.layers[i].mlp
        h = self.tanh_norm(x, name("norm1"))
        before = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
        h = h + (torch.where((self.pos > 0)[:, None], before, 0.0) - h) * w(name("shift"))
        if isinstance(m, ForgetSpec):
            y = self.forget(h, m, lambda n: w(name("mixer." + n)))
        else:
            y = self.latent(h, m, lambda n: w(name("attn." + n)))
        x = x + self.tanh_norm(y, name("norm1b"))
        h = self.tanh_norm(x, name("norm2"))
        z = self.lin(h, name("mlp.router.weight"))
        top = z.topk(f.top, -1)
        y = self.experts(h, name, f, top.indices, torch.softmax(top.values, -1), F.silu)
        sh = self.glu(h, w(name("mlp.shared.gate_up.weight")), w(name("mlp.shared.down.weight")), F.silu)
        x = x + self.tanh_norm(y + torch.sigmoid(self.lin(h, name("mlp.shared.sg"))) * sh, name("norm2b"))
        e = self.raw[name("side.embed")][self.ids].double()
        g = F.gelu(self.lin(x, name("side.gate")), approximate="tanh") * e
        return x + _rms(self.lin(g, name("side.proj")), mc.norm_eps) * w(name("side.norm"))

    def forget(self, h, m, w):
        T, H, D = h.shape[0], m.heads, m.dim
        low = w("lower")
        f = (low + (1 - low) * torch.sigmoid(h @ w("f").T + w("f.b"))).reshape(T, H, D)
        S = torch.zeros(len(self.n), H, D, m.vdim, dtype=h.dtype, device=DEV)

        def step(q, f, v):
            S.mul_(f[..., None]).add_((1 - f)[..., None] * v[:, :, None])
            return (q[:, :, None] @ S)[:, :, 0]

        o = self.over_time(step, F.silu(h @ w("q").T).reshape(T, H, D), f, (h @ w("v").T).reshape(T, H, -1))
        return (_rms(o, self.mc.norm_eps) * w("norm")).flatten(1) @ w("o").T

    def latent(self, h, m, w):
        T, H, eps = h.shape[0], m.heads, self.mc.norm_eps
        if m.q_rank is not None:
            q = (_rms(h @ w("dq.weight").T, eps) * w("dq_norm.weight")) @ w("uq.weight").T
        else:
            q = h @ w("q.weight").T
        q = q.reshape(T, H, m.q_dim)
        c, kr = (h @ w("dkv.weight").T).split([m.kv_rank, m.rot_dim], -1)
        c = _rms(c, eps) * w("dkv_norm.weight")
        q = torch.cat([q[..., : m.dim], self.rope(q[..., m.dim:], m.rope)], -1)
        kr = self.rope(kr[:, None], m.rope).expand(T, H, m.rot_dim)
        k = torch.cat([(c @ w("uk.weight").T).reshape(T, H, m.dim), kr], -1)
        o = self.attend(q, k, (c @ w("uv.weight").T).reshape(T, H, m.vdim), m.scale, m.window,
                        sink=w("sink") if m.sink else None).flatten(1)
        return (o * torch.sigmoid(h @ w("g.weight").T) if m.gate else o) @ w("o.weight").T
