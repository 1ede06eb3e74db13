"""Decode GEMM routing rule for residual projections (CPU: the rule only,
no extension calls).  The kernels it routes to are checked on the GPU by
tests/test_kernels_gpu.py::test_resid_splits_above_256_rows."""


def test_resid_split_rule_above_256_rows():
    from llm_sharding_demo_amd.ops.hip import HipBackend
    b = HipBackend.__new__(HipBackend)  # routing rule only: no extension calls
    assert b._resid_splits(512, 4096, 14336) == 8   # Llama-3 8B down
    assert b._resid_splits(512, 4096, 4096) == 4    # Llama-3 8B o-proj
    assert b._resid_splits(512, 1600, 6400) == 6    # GPT-2 XL MLP-down
    assert b._resid_splits(512, 1600, 1600) == 2    # GPT-2 XL out-proj
    assert b._resid_splits(65536, 1600, 6400) == 1  # prefill keeps the old rule


def test_resid_split_rule_long_k_256_rows():
    from llm_sharding_demo_amd.ops.hip import HipBackend
    b = HipBackend.__new__(HipBackend)
    assert b._resid_splits(256, 4096, 14336) == 8   # Llama-3 8B down: off the ring
    assert b._resid_splits(256, 4096, 4096) == 2    # o-proj stays on the ring rule
    assert b._resid_splits(256, 1600, 6400) == 5    # GPT-2 XL MLP-down unchanged
    assert b._resid_splits(256, 1600, 1600) == 3    # GPT-2 XL out-proj unchanged
    assert b._resid_splits(128, 4096, 14336) == 4   # 128 rows unchanged


def test_resid_rule_prefill_chunks_keep_prefill_rule():
    """the 257-1024-row decode target must not re-route prefill
    chunks of that size (the backend learns decode vs prefill per forward)."""
    from llm_sharding_demo_amd.ops.hip import HipBackend
    b = HipBackend.__new__(HipBackend)
    b.decode = True
    dec = b._resid_splits(512, 1600, 6400)
    b.decode = False
    pre = b._resid_splits(512, 1600, 6400)
    assert dec == 6 and pre == max(1, min(-(-256 // 52), 6400 // 64 // 2))


def test_prompt_slabs():
    """More slabs only for prompts that leave some anyway and have tiles enough."""
    from llm_sharding_demo_amd.ops.routing import Routing

    for M, N, K, S, want in [(1000, 2048, 5632, 2, 8), (1000, 2048, 2048, 2, 2), (1000, 1600, 6400, 3, 8),
                             (500, 2048, 5632, 4, 4), (512, 1600, 6400, 5, 5), (3000, 2048, 5632, 1, 1),
                             (200, 2048, 5632, 8, 8), (1000, 2048, 96, 2, 2), (700, 4096, 14336, 2, 5)]:
        assert Routing.prompt_slabs(M, N, K, S) == want, (M, N, K)


def test_gemv_ok_matches_dispatch():
    """lsd_gemv_ok must accept exactly the (epilogue, norm) pairs lsd_gemv
    instantiates: BF16+LN etc. read 'not ok' so the caller
    materialises the norm instead of failing at launch."""
    import pytest
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")
    dispatched = {(0, 0), (1, 0), (1, 1), (2, 0), (2, 2), (3, 0), (3, 1), (3, 2), (4, 0),
                  (6, 0), (6, 1), (6, 2)}
    for epi in (0, 1, 2, 3, 4, 5, 6):
        for norm in (0, 1, 2):
            ok = bool(_C.gemv_ok(1, 1600, epi, norm))
            assert ok == ((epi, norm) in dispatched), (epi, norm)


def test_deep_ring_leaves_wide_outputs_to_the_tiles():
    """The deep ring (gemm_deep.hip) holds all rows of a block: with more than 48 rows, outputs
    of more blocks than run together (vocabularies) are faster on the 128 x 128 tiles."""
    import pytest
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")
    EPI_F32, EPI_SLAB = 3, 5

    for M, N, K, epi, splits, want in [
            (9, 50304, 1600, EPI_F32, 1, True), (48, 128256, 4096, EPI_F32, 1, True), (49, 50304, 1600, EPI_F32, 1, False),
            (64, 40960, 1600, EPI_F32, 1, True), (64, 128256, 4096, EPI_F32, 1, False), (65, 32768, 2048, EPI_F32, 1, True),
            (65, 32832, 2048, EPI_F32, 1, False), (128, 50304, 768, EPI_F32, 1, False), (256, 50304, 768, EPI_F32, 1, False),
            (40, 1600, 1632, EPI_F32, 1, False), (128, 4096, 14336, EPI_SLAB, 8, True), (257, 1600, 1600, EPI_F32, 1, False)]:
        assert _C.gemm_on_deep(M, N, K, epi, 1, splits) == want, (M, N, K)
    assert not _C.gemm_on_deep(40, 4096, 4096, EPI_F32, 2, 1)  # the all-rows kernel


def test_decode_attention_parts_by_context():
    """Few waves take their ranges of keys in parts, unless the merge costs more than
    they save: one unsplit launch for short contexts, no parts of less than a tile."""
    import pytest
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")

    for B, n_kv, splits, keys, want in [(32, 8, 1, 20, 1), (32, 8, 1, 130, 1), (32, 8, 1, 260, 2), (16, 8, 1, 60, 1),
                                        (1, 8, 1, 20, 1), (1, 8, 1, 60, 1), (1, 8, 1, 100, 4), (1, 8, 4, 912, 4),
                                        (1, 8, 4, 100, 1), (40, 8, 2, 780, 1), (1, 8, 200, 8000, 1), (1, 8, 4, 0, 1),
                                        (1, 1, 100, 8000, 2), (0, 8, 1, 100, 4)]:
        assert _C.attn_decode_split(B, n_kv, 4, 128, splits, keys) == want, (B, splits, keys)
    assert _C.attn_decode_split(1, 8, 3, 128, 1, 900) == 1 and _C.attn_decode_split(1, 8, 4, 64, 1, 900) == 1


def test_delta_rule_splits_by_length():
    """Factors of their own only where the longest sequence has chunks enough for them."""
    import pytest
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")

    for heads, seqs, rows, want in [(16, 1, 16, False), (16, 1, 17, True), (4, 40, 5, False), (16, 4, 20, True),
                                    (16, 8, 20, False), (16, 8, 64, True), (16, 12, 64, False), (16, 12, 100, True),
                                    (16, 13, 4000, False), (16, 1, 0, False)]:
        assert _C.delta_split(heads, seqs, rows) == want, (heads, seqs, rows)


def test_slabs_of_prompts_at_their_launch():
    """By what tiles and norm take: 2 to 8 where the rule leaves some, and nothing else is changed."""
    import pytest
    try:
        from llm_sharding_demo_amd import _C
    except Exception as e:  # pragma: no cover - extension not built here
        pytest.skip(f"_C not importable: {e}")
    from llm_sharding_demo_amd.ops.hip import HipBackend

    for M, N, K, S, want in [(1000, 2048, 5632, 8, 2), (1000, 2048, 2048, 2, 2), (500, 2048, 2048, 4, 4), (260, 1600, 1600, 7, 5), (700, 768, 1024, 8, 4),
                             (257, 768, 256, 4, 2), (260, 768, 4096, 15, 8), (3000, 2048, 5632, 1, 1), (256, 2048, 5632, 8, 8),
                             (1000, 2048, 96, 2, 2), (1000, 2048, 5600, 3, 3), (257, 768, 192, 3, 3)]:
        assert _C.gemm_prompt_slabs(M, N, K, S) == want, (M, N, K)
    for M in (257, 300, 700, 2000, 20000):
        for N in (16, 768, 2048, 4096):
            for K in (256, 768, 2048, 14336):
                assert 2 <= _C.gemm_prompt_slabs(M, N, K, 5) <= min(8, K // 128)
    b = HipBackend.__new__(HipBackend)
    b.C = _C
    b.decode = False
    assert b._launch_splits(1000, 2048, 5632) == 2 and b._resid_splits(1000, 2048, 5632) == 8
    assert b._launch_splits(65536, 1600, 6400) == 1
    b.decode = True
    assert b._launch_splits(512, 4096, 14336) == b._resid_splits(512, 4096, 14336) == 8
