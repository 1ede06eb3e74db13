"""Kernel routing of the HIP backend: which hand-written kernel (and how many
K splits) every GEMM / norm / attention launch of a forward takes.

One frozen table (`Routing`) holds every tunable with its measured default
and the profile that set it; the decisions are pure functions of the launch
shape and the forward's phase (decode vs prefill, concurrent microbatch
lanes), so `tests/test_routing.py` pins the whole table per (model, GEMM,
rows) on CPU.  Defaults are the production configuration; an A/B run
overrides fields with ONE variable:

    LSD_ROUTING="ring8=0,sk_target=256"      (field=value, comma-separated)

hipBLASLt (csrc/blaslt.cpp) is not on the default hot path: every GEMM runs
on the gfx950 kernels of csrc/kernels.  `blaslt=1` turns the library routes
on for A/B comparisons (the library as an oracle for the hand-written
prefill GEMMs); its thresholds are the `blaslt_*` fields.

Reference: the block's projections these route are `/root/reference/server.py:84-85,99-100`
(GPT2Block c_attn / c_proj / c_fc / c_proj) and the head `server.py:102`.
"""
from __future__ import annotations

import dataclasses
import math
import os
from dataclasses import dataclass


@dataclass(frozen=True)
class Routing:
    # -- single stream / small batches ------------------------------------
    # decode GEMMs of <= gemv_max_m rows on the weight-streaming GEMV
    # (gemv.hip, fused epilogues); <= gemv_norm_max_m rows also fold the
    # preceding LayerNorm / RMSNorm into its prologue (0 disables)
    gemv_max_m: int = 8
    gemv_norm_max_m: int = 2
    gemv_nt: int = 0  # non-temporal weight loads in gemv_kernel (A/B; gemv_stream_kernel's always are)
    # -- decode attention --------------------------------------------------
    target_blocks: int = 512  # >> 256 CUs: VALU decode attention splits the context up to this
    split_keys: int = 256      # ... with at least this many keys per split (64 / 128 lose at 1-16
    #                            sequences: the combine launch costs more, r6_split_keys.log)
    # grouped-query decode attention on MFMA (attn_decode_mfma_kernel) at >=
    # attn_mfma_min waves; fewer than attn_mfma_split_below items split the
    # context towards attn_mfma_waves waves, >= 512 keys per split (Llama-3
    # 8B, 2K-8K contexts: 1.3-1.45x the VALU kernel; profiles/r2_long_context.log)
    attn_mfma_min: int = 256
    attn_mfma_split_below: int = 1024
    attn_mfma_waves: int = 1024
    # waves per small-batch VALU attention block; 0: 4 waves, whose keys in flight follow from the
    # context (64-dim ungrouped heads; decode_keys in attention.hip), 8 for others
    attn_small_waves: int = 0
    # ... for 128-dim heads: 88 = 8 waves with 8 keys per wave in flight (a 256-key
    # context in one round of loads; Llama-3 8B single stream -0.6 %, r6_attn_u8.log)
    attn_small_waves128: int = 88
    # full-batch block: 4 waves (64-dim ungrouped heads: keys in flight by the context, as above); 8
    # waves 10 % slower (r4_attn_large_waves.log); 42 = 4 waves with 2 keys per wave in flight, 2 = 2-wave
    # blocks
    attn_large_waves: int = 4
    attn_max_wg: int = 0       # cap the attention grid (A/B; 0 = none)
    # -- decode GEMMs ------------------------------------------------------
    # Of up to 256 rows most run on the deep ring whatever family is chosen here (on_deep);
    # the fields below then matter for what it leaves: K off 64, wide outputs, the 256-row
    # kernel, more rows.  Their figures compare the kernels behind it.
    # split-K (last-arriver) kernel up to sk_max_m rows; tiled above
    # tiled_all_m rows at any width, above tiled_min_m rows when >=
    # tiled_min_n wide (GPT-2 XL 2 x 256: split-K 41.2k, all tiled 46.3k tok/s;
    # profiles/r1_ab_tiled_min_n.log, r1_ab_ring_n64.log)
    sk_max_m: int = 256
    tiled_all_m: int = 128
    tiled_min_m: int = 64
    tiled_min_n: int = 4000
    # short-K GEMMs (GPT-2 small K = 768) tiled at any row count above the
    # GEMV: QKV 9.9-15.7 -> 7.6-8.0 us at 8-128 rows (profiles/r5_small_k_routing.log)
    tiled_short_k: int = 1024
    # split-K workgroup target (0: 384 / concurrent lanes) and the k-steps
    # per split; row blocks of sk_rows when the grid is under-filled
    sk_target: int = 0
    sk_min_steps: int = 2
    sk_rows: int = 64
    defer_resid: int = 1  # residual split-K partials as slabs folded by the next norm
    # LDS ring kernels: grids of <= tiled3_max 128x64 tiles (QKV at 256 rows
    # 25.8 -> 20.4 us; profiles/r1_ab_ring_n64.log), ring depth, tile columns
    # (0 = auto: 32-wide below ring_fill 64-wide workgroups; r2_ring_tn32.log)
    tiled3_max: int = 512
    ring_slots: int = 3
    ring_tn: int = 0
    ring_fill: int = 128
    # 8-wave 128x64 ring (2 = 8 computing waves): QKV 16.7 -> 15.2 us at 256
    # rows, bench 48.9k -> 49.7k tok/s (profiles/r3_ring8_ab.log)
    ring8: int = 2
    # residual projections: ring K-split target, 257-1024-row 128x128-tile
    # target (Llama-3 8B down at 512 rows 119.7 -> 81.5 us; r2_resid512_splits.log),
    # 8 splits for K >= 8192 above resid_longk_min_m rows (down at 256 rows 71.9 -> 55.3 us)
    ring_resid_target: int = 256
    resid_wg_target: int = 1024
    resid_longk: int = 1
    resid_longk_min_m: int = 128
    # K per split of a short-K (<= tiled_short_k) residual projection on the
    # ring: GPT-2 small out-proj (K 768) runs unsplit on 24 workgroups at 512
    resid_short_k_per_split: int = 384
    # 129-256-row long-K GEMMs on the 8-wave all-rows kernel (gemm_d256):
    # Llama-3 8B gate/up at 256 rows 84.6 -> 69.0 us (profiles/r3_d256_ab.log)
    d256: int = 1
    d256_min_k: int = 4096
    d256_slots: int = 3
    d256_target: int = 192
    # ... and over 256-row blocks up to d256_rb_max_m rows for long-K GEMMs at
    # most d256_rb_max_n wide: Llama-3 8B QKV at 512 rows 54.6 (8-wave ring)
    # -> 45.2 us (128-wide tiles, 2 K splits; the 28672-wide gate_up stays on
    # the 256x256 kernel: 120 vs 145 us; profiles/r6_llama512_gemm.log)
    d256_rb_max_m: int = 512
    d256_rb_max_n: int = 8192
    # the 256x256 pipelined kernel (gemm_p8) where the 128x128 tiles take more than a round of
    # two a CU (big_tiles in gemm.hip), or once a tiled launch has this
    # many 256x256 tiles; the 128x128 kernels below (launch_tiled in gemm.hip)
    big_min_blocks: int = 160
    # -- grouped GEMMs (experts, per-head latent projections) ----------------
    # row-tile rows by the mean rows of a group: 32 up to group_tm32, 64 up to
    # group_tm64, else 128
    group_tm32: int = 24
    group_tm64: int = 96
    # row tiles that walk an expert's columns together in a long prompt (8: down
    # projection 702 -> 787 TF/s over 4)
    moe_group_rows: int = 8
    # up to this many tokens, narrow projections (routers, token-side gates) take 16
    # rows a block; a router's K in splits of at least router_k, towards router_target blocks
    rows_few_t: int = 1024
    router_k: int = 256
    router_target: int = 256
    # up to this many tokens, experts stream their weights per (token, choice)
    moe_few_t: int = 4
    # prompts of at least latent_expand_t tokens attend over expanded keys and
    # values where that saves multiply-adds (latent_expand; 0 disables)
    latent_expand_t: int = 256
    # recurrent layers: prompts of more than chunk_min tokens per sequence on
    # average run in chunks, shorter ones token by token
    chunk_min: int = 4
    # recurrences with forget gates: blocks a prompt launch aims for, segments of a
    # sequence at least forget_tokens long
    forget_target: int = 512
    forget_tokens: int = 64
    # decode attention with mixed heads: 64-key tiles that a launch takes one a block, as
    # many blocks with two and more each beyond (a step of 96 sequences of 300 keys: 1 / 3 / 5 splits 977 / 932 / 919
    # us, of 600, 5 / 10 splits 951 / 957; 48 of 900, 8 / 15 splits 673 / 673; 24 of 500, 4 / 8 522 / 504)
    talk_target: int = 768
    # ... and prompt attention with few query tiles
    talk_prefill_target: int = 512
    # prompt attention: query tiles of 128 (else 64) from attn_tile_min blocks (32 heads
    # of 128: 2000 tokens, 512 blocks, 58 against 62 us; 500 tokens, 128 blocks, 16 against 12)
    attn_tile_min: int = 512
    # attention over paged heads without mixing: query tiles of 128 (else 64) from
    # paged_tile_min blocks; decode waves a launch aims for, at least paged_split_keys
    # keys each
    paged_tile_min: int = 512
    paged_waves: int = 2048
    paged_split_keys: int = 64
    # decode attention with mixed weights: blocks a launch aims for
    mix_target: int = 256
    # -- norms / head ------------------------------------------------------
    # one wave per row from norm_wave_min rows (prefill 32 K x 1600 97.7 ->
    # 53.7 us; r5_normwave.log) and from norm_wave_narrow_min rows when H <=
    # 1024 (GPT-2 small decode +0.9 %; r5_normwave_decode.log)
    norm_wave_min: int = 4096
    norm_wave_narrow_min: int = 256
    segmax: int = 1  # lm_head epilogue writes 8-logit segment maxima for the sampler
    # -- hipBLASLt A/B oracle (off: hand-written kernels only) ---------------
    blaslt: int = 0
    blaslt_min_m: int = 4096             # prefill routes at >= this many rows
    blaslt_resid_min_k: int = 4096       # residual projections with K >= this
    blaslt_gelu_min_m: int = 65536       # prefill MLP-up bias + GELU
    blaslt_decode_gelu_min_m: int = 384  # decode MLP-up bias + GELU
    blaslt_silu_min_m: int = 64          # decode gate_up + SiLU*up pass
    blaslt_silu_max_m: int = 128
    blaslt_qkv_min_m: int = 512          # decode QKV (fp32) + RoPE / cache-append pass
    blaslt_qkv_min_k: int = 4096

    @classmethod
    def from_env(cls, spec: str | None = None) -> "Routing":
        spec = os.environ.get("LSD_ROUTING", "") if spec is None else spec
        kw = {}
        names = {f.name for f in dataclasses.fields(cls)}
        for item in filter(None, (s.strip() for s in spec.split(","))):
            k, _, v = item.partition("=")
            k = k.strip()
            if k not in names:
                raise ValueError(f"LSD_ROUTING: unknown field {k!r}")
            kw[k] = int(v, 0)
        return cls(**kw)

    def replace(self, **kw) -> "Routing":
        return dataclasses.replace(self, **kw)

    # ------------------------------------------------------------------
    # decode GEMM decisions (decode: the forward is a decode step; lanes:
    # microbatch lanes running concurrently)
    # ------------------------------------------------------------------
    def tiled(self, M: int, N: int = 0) -> bool:
        return (M > self.sk_max_m or M > self.tiled_all_m
                or (M > self.tiled_min_m and N >= self.tiled_min_n))

    def d256_bn(self, M: int, N: int, K: int) -> int:
        """Tile columns when this GEMM runs on gemm_d256_kernel, else 0
        (mirrors d256_bn() in gemm.hip)."""
        if not self.d256 or K % 64 or N > 32768 or not self.tiled(M, N):
            return 0
        if 256 < M <= self.d256_rb_max_m:  # several 256-row blocks (auto only)
            if self.d256 != 1 or K < self.d256_min_k or N > self.d256_rb_max_n:
                return 0
            return 128 if N % 128 == 0 else 64
        if not (128 < M <= 256):
            return 0
        if self.d256 == 1:  # auto: long-K GEMMs; 128-wide tiles when they alone fill the chip
            if K < self.d256_min_k:
                return 0
            return 128 if N % 128 == 0 and N // 128 >= 128 else 64
        return 128 if self.d256 == 128 and N % 128 == 0 else 64

    @staticmethod
    def d256_kind(bn: int) -> int:  # lsd_gemm launch kind of gemm_d256
        return 3 if bn == 128 else 2

    @staticmethod
    def d256_splits(N: int, K: int, bn: int, target: int, M: int = 256) -> int:
        tiles = math.ceil(N / bn) * math.ceil(M / 256)  # column tiles x 256-row blocks
        return max(1, min(round(target / tiles), K // 64 // 2 or 1, 16))

    def sk_splits(self, M: int, N: int, K: int, lanes: int = 1, nw: int = 1) -> int:
        """nw: 64-column tiles per workgroup (2 for SiLU*up: sk_nw() in gemm.hip)."""
        tiles = math.ceil(N / (64 * nw))  # >= the target: never row-blocked
        target = self.sk_target or max(128, 384 // max(1, lanes))
        return max(1, min(math.ceil(target / tiles), K // 32 // self.sk_min_steps or 1))

    def gemm_kw(self, M: int, N: int, K: int, lanes: int = 1, nw: int = 1):
        """(tiled kind, K splits) of a non-residual GEMM (QKV, MLP-up,
        gate_up, lm_head below vocab width)."""
        bn = self.d256_bn(M, N, K)
        if bn:
            return self.d256_kind(bn), self.d256_splits(N, K, bn, self.d256_target, M)
        if self.tiled(M, N) or (K <= self.tiled_short_k and M <= self.sk_max_m and K % 64 == 0):
            return True, 1
        return False, self.sk_splits(M, N, K, lanes, nw)

    def resid_splits(self, M: int, N: int, K: int, decode: bool = True, lanes: int = 1) -> int:
        """K splits of a residual projection (x += a w^T + b)."""
        if self.tiled(M, N):
            if M <= self.sk_max_m and self.tiled3_max and self.ring_tn in (0, 32, 64):
                # decode rows on the 128x64 ring: as many splits as keep the
                # grid on the ring kernel, at most one per 512 of K (GPT-2 XL
                # out-proj: 3 splits 11.8 us vs 5 splits 12.6 at 256 rows)
                if M > self.resid_longk_min_m and K >= 8192 and self.resid_longk:
                    return min(8, K // 1024)  # leaves the ring for the 128x128 kernel
                tiles = math.ceil(M / 128) * math.ceil(N / 64)
                target = min(self.tiled3_max, self.ring_resid_target or self.tiled3_max)
                kps = self.resid_short_k_per_split if K <= self.tiled_short_k else 512
                return max(1, min(target // tiles, K // kps or 1))
            tiles = math.ceil(M / 128) * math.ceil(N / 128)
            if M <= 1024 and self.resid_wg_target and decode:
                # decode groups of 257-1024 rows: ~resid_wg_target 128x128
                # tiles, at most one split per 1024 of K (at least 2)
                return max(1, min(math.ceil(self.resid_wg_target / tiles), max(2, K // 1024),
                                  K // 64 // 2 or 1))
            return max(1, min(math.ceil(256 / tiles), K // 64 // 2 or 1))
        if self.defer_resid:
            # deferred slabs cost S x M x N x 4 B of writes + norm reads:
            # ~800 k per split, 4..8 splits (tools/microbench.py resid)
            return max(1, min(8, max(4, K // 800), K // 64))
        return self.sk_splits(M, N, K, lanes)

    def residual_splits(self, M: int, N: int, K: int, decode: bool = True, lanes: int = 1) -> int:
        """K splits a residual projection is launched with: the rule above, and
        what the kernels behind it make of slabs.  Prompts' slabs of more than 256
        rows are reckoned once more at their launch (launch_slabs)."""
        S = self.resid_splits(M, N, K, decode, lanes)
        if not decode:
            S = self.prompt_slabs(M, N, K, S)
        if self.tiled(M, N) or self.defer_resid:
            S = self.slab_splits(M, N, K, S)
        return S

    # gemm_wave4.hip's tiles in rows and columns of 64, blocks a CU, and what a launch takes in 1/1000 us: fixed, a
    # round, a round's K-tile with one block a CU, with two; the last one is the 256 x 256 kernel
    _WAVE4 = ((2, 2, 2, 4850, 2580, 496, 835), (3, 2, 2, 5890, 3770, 544, 1089), (3, 3, 1, 6640, 7540, 705, 0),
              (4, 2, 2, 6400, 4390, 791, 1358), (4, 3, 1, 7500, 10750, 849, 0), (3, 4, 1, 7460, 10050, 867, 0),
              (4, 4, 1, 6320, 11770, 1072, 0))

    @classmethod
    def launch_slabs(cls, M: int, N: int, K: int, S: int) -> int:
        """Slabs that a prompt's residual projection is launched with where the rule leaves S
        (mirrors lsd_gemm_prompt_slabs() in gemm_wave4.hip)."""
        if S <= 1 or M <= 256 or K % 64 or K < 256:
            return S

        def cost(s):
            if -(-M // 128) * -(-N // 64) * s <= 256:
                least = 5500 + 570 * (K // 64) // s
            else:
                least = None
                for mi, nj, bpc, fixed, a_round, one, two in cls._WAVE4:
                    tiles, cap = -(-M // (64 * mi)) * -(-N // (64 * nj)) * s, 256 * bpc
                    rounds = -(-tiles // cap)
                    last = tiles - cap * (rounds - 1)
                    k = (rounds - 1) * (two if bpc == 2 else one) + (two if bpc == 2 and last > 256 else one)
                    c = fixed + a_round * (rounds - 1) + K // 64 * k // s
                    least = c if least is None else min(least, c)
            return least + s * (150 + M * N * 11 // 10000)

        best = min(range(2, min(8, K // 128) + 1), key=cost)
        return best if S <= 8 or cost(S) >= cost(best) else S

    @staticmethod
    def on_deep(M: int, N: int, K: int, splits: int = 1, pairs: bool = False) -> bool:
        """Whether a split-K or tiled launch runs on the deep ring (mirrors
        lsd_gemm_deep_ok() in gemm_deep.hip).  splits: slabs (other sums run
        unsplit); pairs: gate / up rows."""
        if not 1 <= M <= 256 or K < 64 or K % 64 or N % (32 if pairs else 16) or splits > K // 64:
            return False
        if M <= 48:
            return True
        rows = 128 if M > 192 else 96 if M > 128 else 128 if M > 96 else 96 if M > 64 else 64
        two = math.ceil(M / rows)
        best = least = 0
        for bn in (64, 32, 16):
            if bn == 16 and (M > 64 or pairs or K % 128 or K // 128 < splits):
                break
            blocks = math.ceil(N / bn) * splits * two
            cost = math.ceil(blocks / 256) * (bn + rows)
            if not best or cost < least:
                best, least = blocks, cost
        return best <= (512 if M > 64 else 640)

    @staticmethod
    def slab_splits(M: int, N: int, K: int, S: int) -> int:
        """K splits of a residual projection of 9 .. 128 rows that leaves slabs,
        near the S of resid_splits: on the deep ring (gemm_deep.hip) a CU takes in
        about 50 KB a us, so the blocks' share per CU counts, and a slab costs the
        next norm 0.25 us (4096 x 4096 at 40 rows: 5 slabs on 320 blocks 10.9 us, 4
        on 256 8.7; 4096 x 14336: 8 slabs 21.9, 4 21.3, and the norm 5.7 -> 4.9).
        A split has at least four k-steps of 64: below, its launch is all latency, and
        an unsplit sum goes to the residual in fp32."""
        if S <= 1 or not 8 < M <= 128 or K % 64:
            return S
        rows = 128 if M > 96 else 96 if M > 64 else math.ceil(M / 16) * 16

        def us(s: int) -> float:
            share = min(math.ceil(math.ceil(N / bn) * s / 256) * (bn + rows) for bn in (64, 32))
            return share * K / s * 2 / 50e3 + 0.25 * s

        most = max(1, K // 256)
        return min((min(s, most) for s in (S, 4, 6, 8)), key=us)

    @staticmethod
    def prompt_slabs(M: int, N: int, K: int, S: int) -> int:
        """K splits of a prompt's residual projection whose rule leaves S > 1
        slabs: as many as let the 256 x 256 kernel (from 160 blocks on) fill one
        round of the CUs, where that beats S on the 128-row rings, slabs written
        and read included.  1000 rows with their norm: 2048 x 5632 2 splits 42.5 us,
        8 34.6; 2048 x 2048 2 21.0 (kept), 8 23.9; 1600 x 6400 3 39.0, 8 32.5; 500 rows
        have too few tiles.  Each slab is rounded to bf16, and is as much smaller as there
        are more: their sum is 1.66e-3 off 64 bits (2048 x 5632, 1600 x 6400) with 1, 2, 3, 5
        and 8 of them alike."""
        if S <= 1 or M < 256 or K % 64:
            return S
        big, ring = math.ceil(M / 256) * math.ceil(N / 256), math.ceil(M / 128) * math.ceil(N / 128)
        if big * S >= 160:
            return S
        slab = M * N * 4 / 5.2e6

        def us(s: int) -> float:
            if big * s >= 160:
                return math.ceil(big * s / 256) * (K / s * 0.021 + 10) + s * slab
            return max(1.0, ring * s / 256) * K / s * 0.0115 + 4 + s * slab

        return min([S] + [s for s in range(S + 1, 9) if 160 <= big * s <= 256 and K >= 512 * s], key=us)

    def logits_kw(self, M: int, N: int, K: int, lanes: int = 1):
        """lm_head: the 128x128 LDS-tiled kernel at vocab width (fills the
        chip without split-K; 41.8 vs 64.2 us at 128 rows, GPT-2 XL)."""
        if N >= 16384 and K % 64 == 0:
            return True, 1
        return self.gemm_kw(M, N, K, lanes)

    # ------------------------------------------------------------------
    # hipBLASLt A/B routes (never taken unless blaslt=1)
    # ------------------------------------------------------------------
    def blaslt_prefill(self, M: int, decode: bool) -> bool:
        return bool(self.blaslt and self.blaslt_min_m) and M >= self.blaslt_min_m and not decode

    def blaslt_gelu(self, M: int, decode: bool) -> bool:
        if not self.blaslt:
            return False
        if decode:
            return bool(self.blaslt_decode_gelu_min_m) and M >= self.blaslt_decode_gelu_min_m
        return self.blaslt_prefill(M, decode) and M >= self.blaslt_gelu_min_m

    def blaslt_silu(self, M: int, N: int, decode: bool) -> bool:
        return (bool(self.blaslt and self.blaslt_silu_min_m) and decode
                and self.blaslt_silu_min_m <= M <= self.blaslt_silu_max_m and N % 32 == 0)

    def blaslt_qkv(self, M: int, K: int, decode: bool) -> bool:
        return (bool(self.blaslt and self.blaslt_qkv_min_m) and decode and M >= self.blaslt_qkv_min_m
                and K >= self.blaslt_qkv_min_k)

    def blaslt_resid(self, M: int, K: int, decode: bool) -> bool:
        return self.blaslt_prefill(M, decode) and K >= self.blaslt_resid_min_k

    # ------------------------------------------------------------------
    def group_tm(self, rows: float) -> int:
        return 32 if rows <= self.group_tm32 else 64 if rows <= self.group_tm64 else 128

    def batch_tm(self, M: int, groups: int, N: int) -> int:
        """Row tile of a per-head GEMM: the largest that still fills the chip."""
        for tm in (128, 64):
            if M > tm // 2 and groups * math.ceil(M / tm) * math.ceil(N / 128) >= 512:
                return tm
        return 32

    def latent_expand(self, T: int, keys: float, rows: int, dim: int, vdim: int, rank: int) -> bool:
        """Multiply-adds per (token, head): scores and weighted sum in the
        latent space plus the way in and out, against per-head scores plus the
        expansion of `rows` latents."""
        if not self.latent_expand_t or T < self.latent_expand_t:
            return False
        latent = keys * 2 * rank + rank * (dim + vdim)
        expanded = keys * (dim + vdim) + rank * (dim + vdim) * rows / T
        return expanded * 1.25 < latent

    def latent_splits(self, B: int, heads: int, keys: int, rank: int, beside: bool = False) -> int:
        """Context splits of a latent decode launch: the least of what a block's steps
        take, more where others share its CU, and the merge of the parts.  rank 512, us, for
        splits 1 / 2 / 4 / 8: 64 sequences of 300 keys 16.0 / 15.8 / 15.4 / 19.3, 24 of 470 22 / 17 / 13.1 /
        12.7, 96 of 250 13.8 / 15.4 / 17.6 / 24, 160 of 250 13.9 / 21 / 24 / 31.  Blocks of ranks below 320 are smaller:
        more of them share a CU, and a round that is partly full costs what it holds (160 sequences of 500 to 2000 keys,
        splits 1 / 2 / 3 / 4: rank 64, 64 heads 19.7 / 23.4 / 22.7 / 23.1, rank 192, 64 heads 38.1 / 43.0 / 46.8 / 50.9, 32 heads
        30.2 / 31.3 / 29.9 / 31.9).  Of 475 launches of ranks 64 to 576 the splits taken are 0.9 % behind the best on
        average, 5 % at most behind as many as give 256 blocks but for one sequence of 64 heads.  beside: experts run at the
        same time, so a merge and its bytes weigh twice (a timisun-2b step, splits 1 / 2 / 4 / 8: 64 sequences of
        300 keys 994 / 1006 / 1023 / 1048, 24 of 1024 1011 / 942 / 921 / 925, 64 of 1000 1071 / 1041 / 1053 / 1071)."""
        items, wide = B * -(-heads // 16), rank >= 320
        steps = max(1, -(-keys // (64 if wide else 128)))  # keys a block takes at a time
        best, least = 1, 0.0
        for k in (steps, 32, 16, 12, 8, 6, 5, 4, 3, 2, 1):  # steps a block
            if k > steps:
                continue
            s = min(-(-steps // k), 64)
            share = max(1.0, items * s / 256)  # blocks a CU
            if wide:
                cost, merge = (0.4 + 0.0035 * rank) * (0.45 + 0.55 * math.ceil(share)), 2.5
            else:
                cost, merge = (0.6 + 0.0025 * rank) * (0.2 + 0.4 * (share + math.ceil(share))), 1.5
            cost *= -(-steps // s)
            if s > 1:
                cost += (merge + 2e-6 * B * heads * rank * s) * (2 if beside else 1)
            if k == steps or cost < least:
                best, least = s, cost
        return best

    def forget_segments(self, items: int, tokens: int) -> int:
        """Segments of every sequence in a chunked recurrence (items: sequences x
        heads): two launches over all of them where that fills the chip."""
        n = min(self.forget_target // max(1, items), math.ceil(tokens / self.forget_tokens), 16)
        return n if n > 2 else 1

    def router_splits(self, T: int, K: int) -> int:
        return max(1, min(self.router_target // math.ceil(T / 16), K // self.router_k, 16))

    def talk_splits(self, B: int, keys: int, windowed: bool) -> int:
        """Context splits of a decode attention launch with mixed heads (one
        block holds all heads of a token, 64 keys a step)."""
        tiles = math.ceil(keys / 64) + windowed  # a window may begin inside one
        return max(1, min(math.ceil(tiles / max(1, math.ceil(B * tiles / self.talk_target))), 64))

    def talk_prefill_splits(self, tiles: int, keys: int) -> int:
        """Key splits of a prompt attention launch with mixed heads: few query
        tiles over long contexts, at least four 32-key tiles each."""
        return max(1, min(self.talk_prefill_target // max(1, tiles), keys // 128, 16))

    def talk_prefill_parts(self, qlens, starts, window: int, rows: int, blocks: int = 490) -> int:
        """Key splits of a prompt attention launch with capped mixed scores, in which a tile of
        `rows` queries takes as many of them as it has keys for (attention_talk.hip): as
        short as leave `blocks` blocks, a little less than two a CU.  us with the combine, 16
        heads of 128, splits by tiles alone -> here: 1000 tokens 73 -> 58, 500 61 -> 37, 4 x 250 67 -> 37, 100
        31 -> 19, 1500 97 -> 80, 1000 and 400 86 -> 72; a split more or less than two a CU
        takes 1000 72, 1500 102.
        Every token has partial outputs in every split: no more of them than prompts of one length
        come to, twice `rows` a block (128 MB with 16 heads of 128; without this bound 800 tokens'
        prompts of 16 and one such chunk at position 30000 took 1.7 GB a layer)."""
        most = int(2 * blocks * rows / max(1, sum(qlens)))
        if most <= 1:
            return 1
        tiles, keys, longest = 0, 0.0, 0
        for n, first in zip(qlens, starts):
            t, lo, hi = math.ceil(n / rows), first + min(n, rows), first + n
            if hi <= window:
                mean = (lo + hi) / 2
            elif lo >= window:
                mean = window
            else:
                mean = ((window - lo) * (window + lo) / 2 + (hi - window) * window) / (hi - lo)
            tiles, keys, longest = tiles + t, keys + t * (mean / 32 + 0.5), max(longest, min(hi, window + rows + 31))
        room = blocks - tiles / 2  # (a tile's last split is half full on average)
        if room <= 0 or longest == 0:
            return 1
        return max(1, min(math.ceil(math.ceil(longest / 32) / max(1, math.ceil(keys / room))), 16, most))

    def paged_splits(self, items: int, keys: int) -> int:
        """Context splits of decode attention, a wave per (token, K / V head)."""
        return max(1, min(math.ceil(self.paged_waves / items), math.ceil(keys / self.paged_split_keys), 64))

    def mix_splits(self, B: int, keys: int, heads: int, kv_heads: int) -> int:
        """Context splits of decode attention with mixed weights (one block per
        token, 64-key tiles).  A split leaves partial sums of every head and K /
        V head: heads kv_heads rows against the 64 a tile holds per K / V head."""
        tiles = math.ceil((keys + 63) / 64) + 1
        per = 1 if B * tiles <= self.mix_target else max(1, min(4, heads // 16 * 2))
        return max(1, min(math.ceil(self.mix_target / B), math.ceil(tiles / per), 64))

    def attn_splits(self, B: int, nh: int, n_kv: int, hd: int, max_ctx: int) -> int:
        """Context splits of a decode attention launch (a graph-captured
        property: max_ctx is the captured context bucket)."""
        G, items = nh // n_kv, B * n_kv
        if hd == 128 and G in (2, 4, 8):
            ms = 1
            if items < self.attn_mfma_split_below:
                ms = max(1, min(math.ceil(self.attn_mfma_waves / items), math.ceil(max_ctx / 512), 256))
            if items * ms >= self.attn_mfma_min:
                return ms
        if hd == 64 and max_ctx <= 2 * self.split_keys:
            # two rounds of a block's loads cost less than a merge of its own (12 heads, 300 keys 5.4 us,
            # in two splits 6.0; 450 5.7 and 6.1; three rounds and splits: 700 7.3 and 6.1; up to 400 items, 280 to
            # 512 keys 0.3 to 2 us less, and grouped heads likewise or within 2 %: 32 over 8, one sequence of
            # 280 7.3 and 8.5, 512 8.55 and 8.40, 16 over 8 5.8 and 6.6; behind by up to a tenth where 256
            # blocks and more have over 350: 32 sequences, 12 heads, 450 8.7 and 8.0, 16 over 8, 400 9.2 and 8.3)
            return 1
        if items < self.target_blocks:
            return min(math.ceil(self.target_blocks / items), max(1, math.ceil(max_ctx / self.split_keys)))
        return 1


def route_table(model: str, rows, routing: Routing | None = None) -> dict:
    """{(gemm, rows, phase): route} of one model's projections: what
    `tests/test_routing.py` pins and `python -m llm_sharding_demo_amd.ops.routing`
    prints.  route = kernel family + K splits, no extension calls.  "deep": the deep ring,
    which takes split-K and tiled launches of up to 256 rows (on_deep) and sums what is
    not left as slabs unsplit."""
    from ..config import get_model_config

    r = routing or Routing.from_env("")
    mc = get_model_config(model)
    H, F = mc.hidden, mc.ffn
    up_n = (2 if mc.arch == "llama" else 1) * F
    shapes = {"qkv": (mc.qkv_size, H, "gemm"), "o": (H, mc.q_size, "resid"),
              "up": (up_n, H, "gemm"), "down": (H, F, "resid"), "lm_head": (mc.vocab_padded, H, "logits")}
    out = {}
    for M in rows:
        for decode in ((True, False) if M >= 256 else (True,)):
            lanes = 2 if decode else 1
            for g, (N, K, kind) in shapes.items():
                if M <= r.gemv_max_m and decode:
                    route = "gemv"
                elif kind == "resid":
                    s = r.residual_splits(M, N, K, decode, lanes)
                    if not decode:
                        s = r.launch_slabs(M, N, K, s)
                    t = r.tiled(M, N)
                    slabs = s if t or r.defer_resid else 1
                    route = f"{'tiled' if t else 'splitk-slab' if r.defer_resid and s > 1 else 'splitk'}/s{s}"
                    if r.on_deep(M, N, K, slabs):
                        route = f"deep/s{slabs}"
                else:
                    if kind == "logits":
                        t, s = r.logits_kw(M, N, K, lanes)
                    else:
                        t, s = r.gemm_kw(M, N, K, lanes, 2 if (g == "up" and mc.arch == "llama") else 1)
                    route = {False: "splitk", True: "tiled", 2: "d256-64", 3: "d256-128"}[t] + f"/s{s}"
                    if t in (False, True) and r.on_deep(M, N, K, 1, g == "up" and mc.arch == "llama"):
                        route = "deep/s1"
                if r.blaslt and ((g == "up" and (r.blaslt_gelu(M, decode) and mc.arch == "gpt2"
                                                 or mc.arch == "llama" and r.blaslt_silu(M, N, decode)))
                                 or (g == "qkv" and r.blaslt_qkv(M, K, decode))
                                 or (kind == "resid" and r.blaslt_resid(M, K, decode))):
                    route = "hipblaslt"
                out[(g, M, "decode" if decode else "prefill")] = route
    return out


if __name__ == "__main__":
    import sys

    model = sys.argv[1] if len(sys.argv) > 1 else "gpt2-xl"
    rows = [1, 8, 64, 128, 256, 512, 32768, 65536]
    for (g, M, ph), route in sorted(route_table(model, rows).items(), key=lambda x: (x[0][1], x[0][2], x[0][0])):
        print(f"{model:12s} {ph:8s} {M:6d} {g:8s} {route}")
