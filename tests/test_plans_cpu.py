"""Launch-plan heuristics that need no GPU (host code of libdashinfer_hip.so): the split plan of the decode attention.

The numbers are the ones the round-3 measurements settled on (profiles/r03_attn_timeline.txt, r03ab_*): 17 splits at batch 1,
4 at BASELINE configs[2] (batch 32, uint4 cache), 16 -- not 32 -- for one TP = 8 rank of Qwen2-72B, 4 -- not 8 -- for the 57B MoE
step; and the invariants behind them."""
import ctypes as C
import importlib

import pytest

capi = importlib.import_module("dash-infer_amd.capi")


def plan(batch, n_heads, n_groups, max_len, kv="none", dtype=None, cus=256):
    lib = capi.lib()
    ns, mf = C.c_int(), C.c_int()
    rc = lib.dihip_debug_attn_plan(batch, n_heads, n_groups, max_len, capi.KV[kv],
                                   capi.BF16 if dtype is None else dtype, cus, C.byref(ns), C.byref(mf))
    assert rc == 0
    return ns.value, bool(mf.value)


@pytest.mark.parametrize("shape,expect", [
    ((1, 28, 4, 2049, "none"), 17),      # headline: 17 x 4 workgroups of 128 tokens
    ((32, 28, 4, 2049, "u4"), 4),        # configs[2]: two workgroups per CU, 512 tokens per split
    ((16, 8, 1, 4097, "none"), 16),      # configs[3] rank: one workgroup per CU (32 splits of 128 tokens measured 3 us slower)
    ((16, 28, 4, 1025, "none"), 4),      # configs[4] step
])
def test_measured_shapes_keep_their_split_counts(shape, expect):
    b, n, g, L, kv = shape
    ns, mfma = plan(b, n, g, L, kv)
    assert mfma and ns == expect


@pytest.mark.parametrize("batch", [1, 2, 3, 8, 16, 32, 64, 200])
@pytest.mark.parametrize("n,g", [(28, 4), (8, 1), (64, 8), (32, 32)])
@pytest.mark.parametrize("L", [1, 100, 129, 1024, 2049, 4097, 32768])
def test_split_plan_invariants(batch, n, g, L):
    ns, _ = plan(batch, n, g, L)
    assert 1 <= ns <= 256
    assert ns == 1 or (L + ns - 1) // ns >= 64           # a split never falls under half the 128-token floor's rounding
    assert ns <= max(1, (L + 127) // 128)                # >= 128 tokens per split before rounding
    if batch * g * ns > 256 + batch * g:                 # clearly more than one workgroup per CU (past the rounding of the split
        assert ns == 1 or (L + ns - 1) // ns >= 256      # count) only while a split keeps >= 256 tokens


def test_plan_rejects_bad_shapes():
    lib = capi.lib()
    assert lib.dihip_debug_attn_plan(1, 28, 5, 128, 0, capi.BF16, 256, None, None) != 0
    assert lib.dihip_debug_attn_plan(0, 28, 4, 128, 0, capi.BF16, 256, None, None) != 0


@pytest.mark.parametrize("lens,rows,top_k,want", [
    ([64, 64, 64], 4096, 0, [[0, 1, 2]]), ([64, 63, 64, 70], 4096, 0, [[0], [1], [2, 3]]), ([3, 2, 64], 4096, 0, [[0], [1], [2]]),
    ([100, 100, 100], 200, 0, [[0, 1], [2]]), ([5000, 64], 4096, 0, [[0], [1]]), ([64], 4096, 0, [[0]]),
    ([200, 200], 4096, 8, [[0], [1]]), ([128, 128, 64], 4096, 8, [[0, 1], [2]]), ([300, 64], 4096, 8, [[0], [1]]), ([64] * 5, 4096, 16, [[0, 1], [2, 3], [4]])])
def test_prompts_that_share_products(lens, rows, top_k, want):
    """Neighbours of 64 rows and more, up to the row limit; with experts up to the 2048 slots of the grouped launches."""
    decoder = importlib.import_module("dash-infer_amd.decoder")
    assert decoder.prompt_groups(lens, rows, top_k) == want


@pytest.mark.parametrize("T,N,K", [(129, 3050, 5760), (193, 2050, 4096), (65, 1001, 2048), (65, 1003, 2048), (65, 1000, 2048), (129, 3051, 5760), (70, 66, 4096), (513, 2045, 8192)])
def test_gated_products_workspace_holds_both_halves_of_every_part(T, N, K):
    """A K part's slab is [row][two matrices][columns padded to whole four] f32: the workspace is a whole number (two and more) of them, whatever N % 4 is."""
    seq_capi = importlib.import_module("dash-infer_amd.seq_capi")
    need = C.c_size_t(0)
    assert seq_capi.lib().dihip_linear_gated_query(T, N, K, K, C.byref(need)) == 1
    part = T * 2 * (N + 3 & ~3) * 4
    assert need.value % part == 0 and need.value // part >= 2, (need.value, part)


@pytest.mark.parametrize("H,counts", [(32, [700] + [1] * 24), (32, [2048]), (16, [500] + [1] * 13), (8, [300, 1, 129, 128, 65]), (2, [17] * 40), (128, [40, 17])])
def test_gated_linear_attention_workspace_counts_the_chunks_there_are(H, counts):
    """One record (64 x 128 state and 64 decays, f32) and head for every chunk that the portions can make, whatever their chunks' length, and at most one a portion more."""
    seq_capi = importlib.import_module("dash-infer_amd.seq_capi")
    T, E, size = sum(counts), len(counts), H * (64 * 128 + 64) * 4
    need = seq_capi.lib().dihip_gla_gated_workspace_bytes(T, E, max(counts), H, 64, 128)
    assert need % size == 0
    fits = [rows for rows in (16, 32, 64) if sum(-(-c // rows) for c in counts) <= need // size <= T // rows + E]
    assert fits, (need // size, counts)
    if counts == [700] + [1] * 24:
        assert need < 60e6
