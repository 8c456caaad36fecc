"""Launch-plan heuristics that need no GPU (host code of libdashinfer_hip.so): the split plan of the decode attention.

The numbers are measured ones (profiles/r03_attn_timeline.txt, r03ab_*; the uint4 rule's stand at attn_plan): 17 splits at batch 1,
2 of eight waves for batch 32 of 2048 tokens on the uint4 cache, 16 -- not 32 -- for one TP = 8 rank of Qwen2-72B, 4 -- not 8 -- for the 57B MoE
step; and the invariants behind them."""
import ctypes as C
import importlib
import os
import subprocess
import sys
import types

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
    ((32, 28, 4, 2049, "u4"), 2),        # one workgroup of eight waves per CU, 1024 tokens per split
    ((16, 8, 1, 4097, "none"), 16),      # one workgroup per CU (32 splits of 128 tokens measured 3 us slower)
    ((16, 28, 4, 1025, "none"), 4),
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


def launch_plan(batch, n_heads, n_groups, max_len, kv="u4"):
    ns, mf, waves, part = C.c_int(), C.c_int(), C.c_int(), C.c_size_t()
    assert capi.lib().dihip_debug_attn_launch_plan(batch, n_heads, n_groups, max_len, capi.KV[kv], capi.BF16, 0, C.byref(ns), C.byref(mf), C.byref(waves), C.byref(part)) == 0
    return ns.value, waves.value, part.value


# uint4 cache, 256 CUs: eight waves where nine tenths of the CUs and more get one long split (448 tokens and more), or where four waves would leave more than 32 records
@pytest.mark.parametrize("shape,expect", [
    ((32, 28, 4, 2049), (2, 8)), ((32, 28, 4, 896), (2, 8)), ((32, 28, 4, 895), (2, 4)),       # 448 tokens a split, one less
    ((16, 28, 4, 2048), (4, 8)), ((20, 28, 4, 1400), (3, 8)), ((29, 28, 4, 3000), (2, 8)),     # 256, 240 and 232 of 256 CUs have a split
    ((20, 28, 4, 1000), (4, 4)),                                                               # 240, but 334 tokens a split
    ((25, 28, 4, 2000), (6, 4)), ((28, 28, 4, 2000), (5, 4)), ((40, 28, 4, 2000), (4, 4)),     # 200, 224, 160
    ((4, 28, 4, 8000), (16, 8)), ((4, 28, 4, 4096), (16, 4)), ((1, 28, 4, 4096), (32, 4)), ((1, 28, 4, 4097), (17, 8)), ((1, 28, 4, 8000), (32, 8)),
    ((64, 28, 4, 8000), (1, 8)), ((65, 28, 4, 8000), (2, 4)),                                  # 256 CUs with one split each; more requests than that
    ((32, 64, 4, 2049), (4, 4)),                                                               # 16 heads a group: four waves only
])
def test_uint4_splits_of_four_and_eight_waves(shape, expect):
    assert launch_plan(*shape)[:2] == expect


CHECK_PARTS = """
import ctypes as C, importlib
capi = importlib.import_module("dash-infer_amd.capi")
l, seen = capi.lib(), set()
for batch in (1, 2, 3, 5, 8, 16, 20, 25, 32, 33, 64, 65, 200):
    for n, g in ((28, 4), (8, 1), (8, 2), (64, 8), (32, 32), (7, 7), (64, 4), (4, 1)):
        for L in (1, 100, 257, 447, 448, 600, 895, 897, 1000, 1793, 2049, 4097, 8000, 8193, 32768):
            for kv in ("none", "i8", "u4"):
                ns, mf, waves, part = C.c_int(), C.c_int(), C.c_int(), C.c_size_t()
                assert l.dihip_debug_attn_launch_plan(batch, n, g, L, capi.KV[kv], capi.BF16, 0, C.byref(ns), C.byref(mf), C.byref(waves), C.byref(part)) == 0
                seen.add((kv, waves.value))
                room = min(l.dihip_span_attn_decode_workspace_bytes(batch, n, 128, L, 0), l.dihip_span_attn_fused_workspace_bytes(batch, n, g, 128, L))
                assert part.value <= room, (batch, n, g, L, kv, ns.value, waves.value, part.value, room)
                # (buffers are sized for the longest length a request may have, plans made for shorter ones)
                assert part.value <= l.dihip_span_attn_decode_workspace_bytes(batch, n, 128, 32768, 0)
print("uint4, eight waves:", ("u4", 8) in seen)
"""


@pytest.mark.parametrize("tokens", [None, 32, 256, 512, 2000])
def test_launched_splits_fit_the_workspace_queries(tokens):
    """The records of the plan that is launched never need more than the queries answer, whatever DIHIP_ATTN_SPLIT_TOKENS is (read once: a process each)."""
    env = dict(os.environ)
    env.pop("DIHIP_ATTN_SPLIT_TOKENS", None)
    if tokens:
        env["DIHIP_ATTN_SPLIT_TOKENS"] = str(tokens)
    r = subprocess.run([sys.executable, "-c", CHECK_PARTS], env=env, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-1500:]
    assert "True" in r.stdout


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


@pytest.mark.parametrize("H,G,D,E,keys,one", [
    (32, 8, 128, 32, 12000, True), (32, 32, 128, 8, 10, True), (32, 32, 128, 10, 500, True), (32, 32, 128, 10, 900, False), (32, 32, 128, 13, 2000, True), (32, 32, 128, 13, 6000, False), (32, 8, 128, 48, 6000, False), (32, 32, 128, 16, 6000, True),
    (16, 16, 64, 24, 2000, True), (16, 16, 64, 24, 2100, False), (16, 16, 64, 28, 3000, True), (16, 16, 64, 28, 4000, False), (16, 16, 64, 32, 12000, False), (32, 32, 64, 20, 12000, True), (32, 32, 64, 64, 100, True), (32, 32, 128, 24, 100, True),
    (32, 32, 128, 28, 100, False), (32, 32, 128, 64, 400, False), (32, 32, 128, 64, 1000, True), (32, 32, 128, 2047, 100, False), (32, 32, 128, 2048, 100, True)])
def test_decoding_step_of_attention_in_one_launch_only_where_it_is_no_slower(monkeypatch, H, G, D, E, keys, one):
    """More (request, key head) pairs than units, with long walks or in many short rounds: the two launches, which these measured faster (and which take 65535 pairs)."""
    mixers, so = importlib.import_module("dash-infer_amd.mixers"), importlib.import_module("dash-infer_amd.seq_ops")
    taken = []
    for name in ("gqa_decode_step", "gqa_attn_mc"):
        monkeypatch.setattr(so, name, lambda *a, _n=name, **k: taken.append(_n))
    m = mixers.GroupedQueryAttention.__new__(mixers.GroupedQueryAttention)
    m.__dict__.update(H=H, G=G, D=D, V=D, k_lo=H * D, v_lo=(H + G) * D, ktables=[None], vtables=[None], head_gate=False, elem_gate=False, out_gain=None, step=True, mc=True, taps=0, talk=None,
                      differential=None, value_mix=None, maps=1, window=0, keep_first=0, q_norm=None, k_norm=None, freq=None, rot_dims=0, layout=0, mag=1.0, scale=1.0, sink=None, sink_mode=0,
                      softcap=0.0, _prep=lambda *a: taken.append("prep"))
    ctx = types.SimpleNamespace(E=E, T=E, math=so.MATH_BF16, max_count=1, max_pos=(keys + 511) // 512 * 512 - 1, eps=1e-6, tok_pos=None, ent_slot=None, ent_row0=None, ent_count=None,
                                act_buffer=lambda n: None)
    m.mix(ctx, None)
    assert taken == (["gqa_decode_step"] if one else ["prep", "gqa_attn_mc"])


@pytest.mark.parametrize("units,D,DV,keys,want", [(96, 64, 64, 12000, 5), (160, 64, 64, 12000, 3), (192, 64, 64, 12000, 1), (96, 64, 128, 12000, 2), (96, 64, 64, 1000, 1), (8, 128, 128, 12000, 32),
                                                  (48, 64, 64, 12000, 5), (1, 128, 128, 1025, 6), (300, 128, 128, 12000, 1)])
def test_splits_of_the_decoding_steps_attention(units, D, DV, keys, want):
    so = importlib.import_module("dash-infer_amd.seq_ops")
    assert so.gqa_decode_step_splits(units, D, DV, (keys + 511) // 512 * 512 - 1) == want


@pytest.mark.parametrize("T,N,K,one", [(64, 2048, 1000, True), (65, 2048, 1000, False), (330, 2048, 1000, False), (700, 2048, 1000, True), (65, 2048, 1024, True), (1025, 1024, 200, True),
                                       (1024, 1024, 200, False)])
@pytest.mark.parametrize("left", [True, False])
def test_products_with_the_residual_step_take_it_along_only_where_that_is_no_slower(monkeypatch, T, N, K, one, left):
    """K no whole number of 64 and few tiles: the product, then the step (the sums in the same order)"""
    so = importlib.import_module("dash-infer_amd.seq_ops")
    torch = so.torch
    taken = []
    real, lib = so.lib(), types.SimpleNamespace(dihip_linear_residual_dyt=lambda *a: taken.append("one") or 0)
    lib.dihip_linear_workspace_bytes = real.dihip_linear_workspace_bytes
    monkeypatch.setattr(so, "lib", lambda: lib)
    monkeypatch.setattr(so, "stream", lambda: 0)
    monkeypatch.setattr(so, "linear", lambda *a, **k: taken.append("linear") or "y")
    monkeypatch.setattr(so, "add_dyt", lambda x, a, b, norm, x_out, want16: taken.append((a is not None, b is not None, x is x_out, want16)) or (None, "h16"))
    x, w, s, bf = torch.empty(T, K, dtype=torch.bfloat16), torch.empty(N, K, dtype=torch.bfloat16), torch.empty(T, N), torch.empty(N, dtype=torch.bfloat16)
    h = so.linear_residual_dyt(x, w, s, torch.empty(T, N) if left else None, (0.5, bf, bf))
    assert taken == (["one"] if one else ["linear", (True, left, True, True)])
    assert h.shape == (T, N) if one else h == "h16"
