"""The mechanisms of the Vogusun design, each alone, against the float64 restatement in oracle/vogusun.py: the norm without
statistics and the parallel residual step, grouped-query attention in both of its forms (norm, rotation layouts, sink, cap, gate,
value mixing, pages), gated linear attention (state, portions, chunks), the gated and the routed feed-forward."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from oracle import vogusun as ov
from tests.conftest import load_pkg
from tests.seq_helpers import MixerRig, dev_weights, rel_err

pytestmark = pytest.mark.gpu
bf = ov.bf16_values


@pytest.fixture(scope="module")
def so():
    load_pkg()
    from dash_infer_amd import seq_ops
    return seq_ops


def dev(a, dt=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dt).cuda()


def i32(a):
    return torch.tensor(a, dtype=torch.int32, device="cuda")


# ---------------------------------------------------------------------------------------------------------------- norm + residual
def test_add_dyt_residual_norm_and_row_index(so):
    rng = np.random.default_rng(0)
    T, K = 37, 100
    x, a, b = (rng.normal(0, 1.5, (T, K)).astype(np.float32) for _ in range(3))
    w, bias, alpha = bf(1 + 0.2 * rng.normal(size=K)), bf(0.2 * rng.normal(size=K)), 0.71875
    xs = x.astype(np.float64) + (a.astype(np.float64) + b)
    want = ov.dyt_norm(xs, alpha, w, bias)
    xd = dev(x)
    wide = dev(np.concatenate([a, b], 1))                    # sublayer outputs as column slices of a wider buffer
    h, h16 = so.add_dyt(xd, wide[:, :K], wide[:, K:], norm=(alpha, dev(w, torch.bfloat16), dev(bias, torch.bfloat16)), x_out=xd)
    assert h16 is None and rel_err(xd.cpu().numpy(), xs) < 1e-6 and rel_err(h.cpu().numpy(), want) < 2e-6
    _, h16 = so.add_dyt(xd, norm=(alpha, dev(w, torch.bfloat16), dev(bias, torch.bfloat16)), want16=True)
    assert torch.equal(h16.cpu(), h.cpu().to(torch.bfloat16))
    rows = [5, 0, 36, 5]
    hr, _ = so.add_dyt(xd, norm=(alpha, dev(w, torch.bfloat16), dev(bias, torch.bfloat16)), row_idx=i32(rows))
    assert torch.equal(hr.cpu(), h.cpu()[rows])
    only, _ = so.add_dyt(dev(x), dev(a), None, norm=(alpha, dev(w), dev(bias)))      # one sublayer, f32 weights, no stream written
    assert rel_err(only.cpu().numpy(), ov.dyt_norm(x.astype(np.float64) + a, alpha, w, bias)) < 2e-6


# one row (whole and part pieces of K, more columns than a workgroup has threads for, the short-row kernel), rows streamed through LDS and past it, tiles whole and in K parts;
# columns that do not come in fours
@pytest.mark.parametrize("T,N,K", [(1, 4096, 14336), (1, 700, 2056), (1, 140000, 2048), (1, 40, 512), (3, 33, 200), (2, 130, 1024), (24, 2048, 8192), (33, 2050, 1088), (64, 100, 72), (65, 2048, 8192),
                                   (300, 514, 192), (513, 1001, 1024), (70, 40, 72)])
@pytest.mark.parametrize("left,normed", [(True, True), (False, True), (True, False)])
def test_product_that_ends_in_the_residual_step_and_the_norm(so, T, N, K, left, normed):
    """the same bits as the product, then add_dyt"""
    g = torch.Generator("cuda").manual_seed(T + N + K)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, w = rand(T, K + 8).bfloat16()[:, 8:], (rand(N, K) * K ** -0.5).bfloat16()
    stream, a = rand(T, N), rand(T, N + 4)[:, 4:] if left else None
    norm = (0.75, rand(N).bfloat16(), rand(N).bfloat16()) if normed else None
    want, got = stream.clone(), stream.clone()
    y = so.linear(x, w, math=so.MATH_BF16)
    _, h16 = so.add_dyt(want, a if left else y, y if left else None, norm=norm, x_out=want, want16=True)
    out = so.linear_residual_dyt(x, w, got, a, norm)
    assert torch.equal(got, want)
    assert torch.equal(out, h16) if normed else out is None


# K no whole number of 64: 56 and 64 tiles (the two launches), 72 (one)
@pytest.mark.parametrize("T,N,K", [(1000, 896, 200), (1024, 897, 200), (1100, 1001, 76), (1100, 1004, 1000)])
@pytest.mark.parametrize("left,normed", [(True, True), (False, True), (True, False)])
def test_product_of_an_uneven_k_that_ends_in_the_residual_step(so, T, N, K, left, normed):
    test_product_that_ends_in_the_residual_step_and_the_norm(so, T, N, K, left, normed)


def test_embedding_and_its_norm(so):
    g = torch.Generator("cuda").manual_seed(5)
    table, w, b = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((50, 1100), (1100,), (1100,)))
    ids = i32([3, 49, 0, 3, 17])
    x, h16 = so.embed_dyt(ids, table, (0.7, w, b))
    want = so.embed_sum(ids, table)
    assert torch.equal(x, want) and torch.equal(h16, so.add_dyt(want, norm=(0.7, w, b), want16=True)[1])


# heads that do not fill a wave or the workgroups, one batch of heads per wave and several, each rotary layout over none, a part and all of the head, two maps, mixed values
@pytest.mark.parametrize("D,V,H,G,maps", [(128, 128, 16, 4, 1), (64, 64, 4, 4, 1), (128, 36, 6, 2, 2), (64, 100, 70, 35, 1), (128, 128, 64, 8, 1)])
@pytest.mark.parametrize("T", [1, 5, 300])
@pytest.mark.parametrize("layout,part", [(0, 1.0), (0, 0.25), (1, 1.0), (1, 0.625), (0, 0.0)])
def test_prep_in_whole_pieces(so, D, V, H, G, maps, T, layout, part):
    """the kernel of rows in 16-byte pieces against the one of any rows (columns off by two): sums of squares in another order, everything else the same"""
    from dash_infer_amd.seq_state import SequenceStateManager
    rot = int(D * part)
    freq = torch.rand(max(rot // 2, 1), device="cuda") if rot else None
    nq, nk, nv = H * maps * D, G * maps * D, G * V
    g = torch.Generator("cuda").manual_seed(D + T + H)
    src = torch.randn(T, nq + nk + nv, generator=g, device="cuda")
    norms = [torch.randn(D, generator=g, device="cuda").bfloat16() if T != 5 else None for _ in range(2)]
    first = torch.randn(T, nv, generator=g, device="cuda") if T != 1 else None
    outs = []
    for off in (0, 2):
        st = SequenceStateManager(512, 2, 64, "cuda")
        kt, vt = st.add_span_cache("k", G * maps * D, torch.bfloat16), st.add_span_cache("v", nv, torch.bfloat16)
        st.admit("a")
        st.reserve("a", T)
        st.upload()
        rows = torch.zeros(T, nq + nk + nv + 4, device="cuda")
        rows[:, off:off + src.shape[1]] = src
        keep = torch.zeros(T, nv, device="cuda") if T == 1 else None
        so.qkv_prep_append(rows, off, off + nq, off + nq + nk, H, G, D, V, norms[0], norms[1], 1e-5, freq, rot, layout, 1.1, 0.3 if T != 1 else 0.0, first, keep, kt, vt,
                           i32([st.live["a"].index] * T), i32(list(range(T))), maps=maps)
        outs.append((rows[:, off:off + src.shape[1]].clone(), kt.pool.pool.view(torch.bfloat16).float().clone(), vt.pool.pool.view(torch.bfloat16).float().clone(), keep))
    (r0, k0, v0, f0), (r1, k1, v1, f1) = outs
    assert rel_err(r0.cpu().numpy(), r1.cpu().numpy()) < 2e-6
    assert rel_err(k0.cpu().numpy(), k1.cpu().numpy()) < 2.0 ** -8 and float(k0.abs().max()) > 0      # a rounding to bf16 that goes the other way
    assert torch.equal(v0, v1) and (f0 is None or torch.equal(f0, f1))


# ---------------------------------------------------------------------------------------------------------------- attention
def attention_weights(rng, kind, width, H, G, D, V):
    r = lambda *s, sd=None: bf(rng.normal(0, sd if sd is not None else 1.0 / math.sqrt(s[-1]), s))
    w = {"q": r(H * D, width), "k": r(G * D, width), "v": r(G * V, width), "o": r(width, H * V), "vmix": bf(np.float32(0.375))}
    if kind == "attention":
        w.update({"q.norm": bf(1 + 0.2 * rng.normal(size=D)), "k.norm": bf(1 + 0.2 * rng.normal(size=D)), "g": r(H, width)})
    else:
        w.update({"q.b": bf(0.2 * rng.normal(size=H * D)), "k.b": bf(0.2 * rng.normal(size=G * D)), "v.b": bf(0.2 * rng.normal(size=G * V))})
    return w


def attention_rig(kind, w, m, dtype, value_mix=None, **kw):
    load_pkg()
    from dash_infer_amd import mixers
    rot = m["rot"]
    extra = dict(rot_layout="pairs", qk_norm=True, sink="zero", head_gate=True) if kind == "attention" else \
        dict(rot_layout="halves", softcap=m.get("softcap"))
    build = lambda state, dt: mixers.GroupedQueryAttention("t", m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["scale"], dev_weights(w), state,
                                                           dt, rot_dims=rot["dims"], rot_base=rot["base"], rot_scaling=rot.get("scaling"),
                                                           value_mix=value_mix, **extra)
    return MixerRig(build, dtype, **kw)


SHAPES = [  # width, heads, kv heads, dim, vdim, rotated dims
    (72, 6, 2, 24, 16, 24),      # head sizes that are no multiple of 32 / 16
    (64, 4, 4, 32, 32, 16),      # as many key/value heads as query heads, half of the head rotated
    (80, 5, 1, 40, 8, 40),       # one key/value head, an odd number of query heads
    (64, 2, 1, 128, 64, 64),     # wide heads
    (48, 3, 3, 20, 12, 8),       # head sizes the matrix-core kernel does not serve
    (64, 2, 1, 160, 128, 32),    # the widest tiles of the matrix-core kernel
]


@pytest.mark.parametrize("kind", ["attention", "attention_2"])
@pytest.mark.parametrize("shape", SHAPES)
def test_attention_whole_decoded_and_in_portions(kind, shape):
    width, H, G, D, V, rd = shape
    rng = np.random.default_rng(H * 100 + D)
    m = {"heads": H, "kv_heads": G, "dim": D, "vdim": V, "scale": 1.7 / math.sqrt(D), "rot": {"base": 3000.0, "dims": rd}}
    if kind == "attention_2":
        m["softcap"] = 4.0     # low enough to bend many scores
        m["rot"]["scaling"] = {"factor": 4.0, "original": 48, "fast": 8.0, "slow": 1.0}
    w = attention_weights(rng, kind, width, H, G, D, V)
    n = 150
    h = rng.normal(0, 1, (n, width)).astype(np.float32)
    want, _ = ov.attention(h, w, m, 1e-5, kind)
    rig = attention_rig(kind, w, m, torch.float32)
    whole = rig.step([("w", h)])[0]
    assert rel_err(whole, want) < 2e-5
    dec = np.concatenate([rig.step([("d", h[i:i + 1])])[0] for i in range(n)])
    assert rel_err(dec, whole) < 1e-6
    parts, at = [], 0
    for size in [2, 61, 3, 1, 64, 2, 17]:                       # ends inside a page, at its border, one row into the next
        parts.append(rig.step([("p", h[at:at + size])])[0])
        at += size
    assert at == n and rel_err(np.concatenate(parts), whole) < 1e-6
    rig16 = attention_rig(kind, w, m, torch.bfloat16)
    h16 = bf(h)
    want16, _ = ov.attention(h16, w, m, 1e-5, kind)
    whole16 = rig16.step([("w", h16)])[0]
    assert rel_err(whole16, want16) < 0.03
    dec16 = np.concatenate([rig16.step([("d", h16[:100])])[0]] + [rig16.step([("d", h16[i:i + 1])])[0] for i in range(100, n)])
    assert rel_err(dec16, want16) < 0.03


def test_attention_value_mixing_between_layers():
    rng = np.random.default_rng(3)
    width, H, G, D, V = 64, 4, 2, 16, 24
    m = {"heads": H, "kv_heads": G, "dim": D, "vdim": V, "scale": 0.25, "rot": {"base": 100.0, "dims": D}, "v_mix": True}
    w1, w2 = attention_weights(rng, "attention", width, H, G, D, V), attention_weights(rng, "attention_2", width, H, G, D, V)
    h1, h2 = rng.normal(0, 1, (70, width)).astype(np.float32), rng.normal(0, 1, (70, width)).astype(np.float32)
    want1, v1 = ov.attention(h1, w1, m, 1e-5, "attention", None)
    want2, _ = ov.attention(h2, w2, m, 1e-5, "attention_2", v1)
    plain2, _ = ov.attention(h2, w2, m, 1e-5, "attention_2", None)
    assert rel_err(plain2, want2) > 0.05                         # the comparison below sees whether the values were mixed
    load_pkg()
    from dash_infer_amd import mixers

    def build(state, dt):      # both layers in one step: the second reads the values the first one left for it
        mk = lambda key, w, vm, **kw: mixers.GroupedQueryAttention(key, H, G, D, V, 0.25, dev_weights(w), state, dt, rot_dims=D, rot_base=100.0,
                                                                   value_mix=vm, **kw)
        first = mk("a", w1, ("source", "v"), rot_layout="pairs", qk_norm=True, sink="zero", head_gate=True)
        second = mk("b", w2, ("mix", "v", 0.375), rot_layout="halves")
        return lambda ctx, h, h16=None: torch.cat([first(ctx, h[:, :width].contiguous()), second(ctx, h[:, width:].contiguous())], 1)
    rig = MixerRig(build)
    both = np.concatenate([h1, h2], 1)
    for lo, hi in ((0, 33), (33, 34), (34, 70)):
        o = rig.step([("s", both[lo:hi])])[0]
        assert rel_err(o[:, :width], want1[lo:hi]) < 2e-5 and rel_err(o[:, width:], want2[lo:hi]) < 2e-5


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sink_one", [True, False])
def test_attention_far_keys_page_borders_and_the_sink(so, cdt, sink_one):
    """keys and values are written by hand: one key far back stands out for some queries; for others every score is low, so that
    the sink's share of the softmax decides the result"""
    load_pkg()
    from dash_infer_amd.seq_state import SequenceStateManager
    rng = np.random.default_rng(11)
    H, G, D, V, n = 4, 2, 32, 16, 200
    q = rng.normal(0, 0.3, (n, H, D))
    k = rng.normal(0, 0.3, (n, G, D))
    v = rng.normal(0, 1, (n, G, V))
    far = {199: 3, 130: 63, 129: 64, 128: 127, 70: 0}            # query position -> the key it must find (page borders at 64, 128)
    for qp, kp in far.items():
        k[kp] = rng.normal(0, 0.3, (G, D))
        q[qp] = np.repeat(k[kp], H // G, 0) * 60.0               # a score far above all others
    low = [5, 66, 150]
    for qp in low:
        q[qp] = -np.repeat(k[:qp + 1].mean(0), H // G, 0) * 30 - 3.0 * np.sign(np.repeat(k[:qp + 1].mean(0), H // G, 0))
    q, k, v = bf(q), bf(k), bf(v)
    want = ov.causal_attention_rows(q.astype(np.float64), k, v, 0.5, sink_one=sink_one).reshape(n, H * V)
    other = ov.causal_attention_rows(q.astype(np.float64), k, v, 0.5, sink_one=not sink_one).reshape(n, H * V)
    assert max(rel_err(other[p], want[p]) for p in low) > 0.2    # a sink left out (or put in) shows
    for qp, kp in far.items():
        assert rel_err(want[qp].reshape(H, V), np.repeat(v[kp], H // G, 0)) < (0.6 if sink_one else 1e-3)
    st = SequenceStateManager(512, 2, 64, "cuda")
    kt, vt = st.add_span_cache("k", G * D, cdt), st.add_span_cache("v", G * V, cdt)
    st.admit("a")
    st.reserve("a", n)
    st.upload()
    slot = st.live["a"].index
    rows = dev(np.concatenate([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], 1))
    so.qkv_prep_append(rows, 0, H * D, (H + G) * D, H, G, D, V, None, None, 1e-5, None, 0, 0, 1.0, 0.0, None, None, kt, vt,
                       i32([slot] * n), i32(list(range(n))))
    mode = so.SINK_ZERO if sink_one else so.SINK_NONE
    got = so.gqa_attn(rows, kt, vt, i32([slot] * n), i32(list(range(n))), H, G, D, V, 0.5, sink_mode=mode).cpu().numpy()
    assert rel_err(got, want) < (2e-5 if cdt == torch.float32 else 2e-5)
    one = so.gqa_attn(rows[199:200], kt, vt, i32([slot]), i32([199]), H, G, D, V, 0.5, sink_mode=mode).cpu().numpy()   # decoded alone
    assert np.array_equal(one[0], got[199])
    if cdt == torch.bfloat16:
        for nsplit in (1, 3):
            mc = so.gqa_attn_mc(rows, kt, vt, i32(list(range(n))), i32([slot]), i32([0]), i32([n]), n, n - 1, H, G, D, V, 0.5, sink_mode=mode,
                                nsplit=nsplit).cpu().numpy()
            assert rel_err(mc, want) < 0.01
            for p in low + list(far):
                assert rel_err(mc[p], want[p]) < 0.02, (p, nsplit)
        for p in (199, 129, 66):                                  # decoded alone: one row, the key walk split
            mc1 = so.gqa_attn_mc(rows[p:p + 1], kt, vt, i32([p]), i32([slot]), i32([0]), i32([1]), 1, p, H, G, D, V, 0.5, sink_mode=mode).cpu().numpy()
            assert rel_err(mc1[0], want[p]) < 0.02


# ---------------------------------------------------------------------------------------------------------------- gated linear attention
def gla_weights(rng, width, H, D, V, rank, decay_bias=1.0):
    r = lambda *s, sd=None: bf(rng.normal(0, sd if sd is not None else 1.0 / math.sqrt(s[-1]), s))
    return {"q": r(H * D, width), "k": r(H * D, width), "v": r(H * V, width), "g": r(H * V, width), "o": r(width, H * V),
            "norm": bf(1 + 0.2 * rng.normal(size=V)), "a1": r(rank, width), "a2": r(H * D, rank, sd=1.0),
            "a2.b": bf(rng.normal(decay_bias, 1.0, H * D))}


def gla_rig(w, m, dtype, **kw):
    load_pkg()
    from dash_infer_amd import mixers
    return MixerRig(lambda state, dt: mixers.GatedLinearAttention("t", m["heads"], m["dim"], m["vdim"], m["tau"], dev_weights(w), state), dtype, **kw)


@pytest.mark.parametrize("shape", [(72, 3, 20, 24, 8, 8.0), (64, 1, 64, 64, 4, 1.0), (96, 2, 72, 130, 16, 12.0), (64, 2, 8, 200, 1, 2.0),
                                   (64, 1, 136, 40, 4, 4.0)])
def test_gla_whole_decoded_portions_and_chunks(shape):
    width, H, D, V, rank, tau = shape
    rng = np.random.default_rng(D + V)
    m = {"heads": H, "dim": D, "vdim": V, "tau": tau}
    w = gla_weights(rng, width, H, D, V, rank, decay_bias=3.0 if tau < 4 else 0.0)
    n = 330
    h = rng.normal(0, 1, (n, width)).astype(np.float32)
    want = ov.gla(h, w, m, 1e-5)
    rig = gla_rig(w, m, torch.float32)
    whole = rig.step([("w", h)])[0]                              # long enough for the chunks that run side by side
    assert rel_err(whole, want) < 3e-5
    dec = np.concatenate([rig.step([("d", h[i:i + 1])])[0] for i in range(n)])     # long decoding through the state
    assert rel_err(dec, want) < 3e-5
    parts, at = [], 0
    for size in [2, 100, 1, 129, 64, 3, 31]:
        parts.append(rig.step([("p", h[at:at + size])])[0])
        at += size
    assert at == n and rel_err(np.concatenate(parts), want) < 3e-5
    rig.release("w")
    again = rig.step([("w2", h[:40])])[0]                         # a slot that held a state starts from zero again
    assert rel_err(again, want[:40]) < 3e-5
    rig16 = gla_rig(w, m, torch.bfloat16)
    h16 = bf(h)
    assert rel_err(rig16.step([("w", h16)])[0], ov.gla(h16, w, m, 1e-5)) < 0.03


def test_gla_sequences_side_by_side():
    rng = np.random.default_rng(21)
    m = {"heads": 2, "dim": 24, "vdim": 40, "tau": 4.0}
    w = gla_weights(rng, 64, 2, 24, 40, 8)
    hs = [rng.normal(0, 1, (n, 64)).astype(np.float32) for n in (140, 9, 1)]
    want = [ov.gla(h, w, m, 1e-5) for h in hs]
    rig = gla_rig(w, m, torch.float32)
    a = rig.step([("a", hs[0][:130]), ("b", hs[1][:2]), ("c", hs[2])])     # a chunked portion beside short ones
    b = rig.step([("b", hs[1][2:]), ("a", hs[0][130:])])
    assert rel_err(np.concatenate([a[0], b[1]]), want[0]) < 3e-5
    assert rel_err(np.concatenate([a[1], b[0]]), want[1]) < 3e-5 and rel_err(a[2], want[2]) < 3e-5


# portions below, at and past the 16 rows of a staged batch and the 16, 32 and 64 of a chunk (by the number of heads); channels that fill a wave's quarter or not, one and two columns per lane
@pytest.mark.parametrize("H,D,DV,rank", [(3, 64, 128, 64), (2, 16, 4, 32), (1, 48, 100, 96), (2, 128, 128, 128), (4, 80, 64, 32), (32, 32, 8, 32), (128, 16, 4, 32)])
@pytest.mark.parametrize("counts", [[1], [1, 1, 1], [16, 3], [17, 1, 16], [33, 64, 1, 2], [300, 1, 129, 128, 65]])
def test_gla_in_one_kernel(H, D, DV, rank, counts):
    """z, recurrence, norm and gate against 64 bits (the rank's rows rounded to bf16, as the product rounds them), and the states left in their slots: f32 sums"""
    load_pkg()
    from dash_infer_amd import seq_ops as so
    rng = np.random.default_rng(D + DV + sum(counts))
    T, E, tau, eps, sc = sum(counts), len(counts), 4.0, 1e-5, D ** -0.5
    hd, hv = H * D, H * DV
    rows = rng.normal(0, 1, (T, 2 * hd + 2 * hv + rank)).astype(np.float32)
    a2, b2, norm = bf(rng.normal(0, rank ** -0.5, (hd, rank))), bf(rng.normal(1, 1, hd)), bf(1 + 0.2 * rng.normal(size=DV))
    state = rng.normal(0, 1, (E + 2, H, D, DV)).astype(np.float32)
    slots = rng.permutation(E + 2)[:E]
    row0 = np.cumsum([0] + counts[:-1])
    S_dev, y = dev(state), torch.full((T, hv + 4), 7.0, device="cuda")
    wdev = lambda a: torch.tensor(a).cuda().to(torch.bfloat16)
    assert so.gla_gated_supported(wdev(a2), wdev(b2), wdev(norm), H, D, DV)
    lo = (hd, 2 * hd, 2 * hd + hv, 2 * hd + 2 * hv)
    so.gla_gated(dev(rows), *lo, wdev(a2), wdev(b2), wdev(norm), sc, tau, eps, S_dev, i32(slots), i32(row0), i32(counts), max(counts), H, D, DV, out=y[:, :hv])
    r = rows.astype(np.float64)
    a1 = torch.tensor(rows[:, lo[3]:]).to(torch.bfloat16).double().numpy()
    al = ((1 / (1 + np.exp(-(a1 @ a2.T.astype(np.float64) + b2)))) ** (1 / tau)).reshape(T, H, D)
    q, k, v, g = (r[:, b:b + n].reshape(T, H, -1) for b, n in ((0, hd), (lo[0], hd), (lo[1], hv), (lo[2], hv)))
    want, S_want = np.zeros((T, H, DV)), state.astype(np.float64)
    for e in range(E):
        S = S_want[slots[e]]
        for t in range(row0[e], row0[e] + counts[e]):
            S = al[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None]
            want[t] = (S * (q[t] * sc)[:, :, None]).sum(1)
        S_want[slots[e]] = S
    want = want / np.sqrt((want ** 2).mean(-1, keepdims=True) + eps) * norm * g
    assert rel_err(y[:, :hv].cpu().numpy(), want.reshape(T, hv)) < 3e-5 and bool((y[:, hv:] == 7).all())
    assert rel_err(S_dev.cpu().numpy(), S_want) < 3e-5


@pytest.mark.parametrize("H,counts", [(32, [200] + [1] * 24), (2, [17, 300, 1, 16, 33]), (3, [130] * 5)])
def test_gla_in_one_kernel_stays_in_its_workspace(H, counts):
    """long and short portions in any order with a workspace of exactly the queried size: the bytes behind it are left alone, and every portion comes out as it does by itself"""
    load_pkg()
    from dash_infer_amd import seq_ops as so
    D, DV, rank, T, E = 64, 128, 64, sum(counts), len(counts)
    g = torch.Generator("cuda").manual_seed(T)
    hd, hv = H * D, H * DV
    rows = torch.randn(T, 2 * hd + 2 * hv + rank, generator=g, device="cuda")
    a2, b2, gamma = ((torch.randn(*s, generator=g, device="cuda") * 0.125).to(torch.bfloat16) for s in ((hd, rank), (hd,), (DV,)))
    state, row0 = torch.randn(E, H, D, DV, generator=g, device="cuda"), np.cumsum([0] + counts[:-1])
    need = int(so.lib().dihip_gla_gated_workspace_bytes(T, E, max(counts), H, D, DV))
    ws = torch.full((need + (1 << 20),), 0x5A, dtype=torch.uint8, device="cuda")
    col = lambda c: C.c_void_p(rows.data_ptr() + 4 * c)
    S, y, slots, first, count = state.clone(), torch.empty(T, hv, device="cuda"), i32(list(range(E))), i32(row0), i32(counts)
    so.check(so.lib().dihip_gla_gated(so.stream(), so.ptr(y), so.dt(y), hv, col(0), col(hd), col(2 * hd), col(2 * hd + hv), col(2 * hd + 2 * hv), rows.shape[1], so.ptr(a2), so.ptr(b2),
                                      so.ptr(gamma), rank, 0.125, 4.0, 1e-5, so.ptr(S), so.ptr(slots), so.ptr(first), so.ptr(count), T, E, max(counts), H, D, DV,
                                      so.ptr(ws), need), "gla_gated")
    assert bool((ws[need:] == 0x5A).all())
    for e, n in enumerate(counts):
        S1, y1 = state[e:e + 1].clone(), torch.empty(n, hv, device="cuda")
        part = rows[row0[e]:row0[e] + n].contiguous()
        so.gla_gated(part, hd, 2 * hd, 2 * hd + hv, 2 * hd + 2 * hv, a2, b2, gamma, 0.125, 4.0, 1e-5, S1, i32([0]), i32([0]), i32([n]), n, H, D, DV, out=y1)
        assert rel_err(y[row0[e]:row0[e] + n].cpu().numpy(), y1.cpu().numpy()) < 3e-5 and rel_err(S[e:e + 1].cpu().numpy(), S1.cpu().numpy()) < 3e-5


# ---------------------------------------------------------------------------------------------------------------- feed-forward
def test_gated_mlp():
    load_pkg()
    from dash_infer_amd import mixers
    rng = np.random.default_rng(31)
    width, ff = 72, 100
    w = {"gate": bf(rng.normal(0, 0.2, (ff, width))), "up": bf(rng.normal(0, 0.2, (ff, width))), "down": bf(rng.normal(0, 0.1, (width, ff)))}
    h = rng.normal(0, 1, (70, width)).astype(np.float32)
    dw = dev_weights(w)
    rig = MixerRig(lambda state, dt: mixers.GatedMlp(dw["gate"], dw["up"], dw["down"], "gelu_tanh"))
    assert rel_err(rig.step([("a", h)])[0], ov.dense_ff(h, w)) < 1e-5


@pytest.mark.parametrize("experts,top,T", [(5, 2, 1), (5, 2, 70), (10, 3, 300), (4, 4, 9), (3, 1, 40), (40, 6, 130)])
def test_routed_experts(so, experts, top, T):
    load_pkg()
    from dash_infer_amd import mixers
    rng = np.random.default_rng(experts * 10 + top)
    width, ff, limit = 64, 24, 0.75                                # a limit that clips many units
    w = {"router": bf(rng.normal(0, 0.5, (experts, width))), "router.b": bf(rng.normal(0, 0.5, experts))}
    for e in range(experts):
        w[f"e{e}.gate"], w[f"e{e}.up"] = bf(rng.normal(0, 0.25, (ff, width))), bf(rng.normal(0, 0.25, (ff, width)))
        w[f"e{e}.down"] = bf(rng.normal(0, 0.2, (width, ff)))
    h = bf(rng.normal(0, 1, (T, width)))
    chosen = []
    want = ov.moe_ff(h, w, experts, top, limit, chosen)
    dw = dev_weights(w)
    build = lambda state, dt: mixers.ExpertMlp(dw["router"], dw["router.b"], [dw[f"e{e}.gate"] for e in range(experts)],
                                               [dw[f"e{e}.up"] for e in range(experts)], [dw[f"e{e}.down"] for e in range(experts)], top, limit)
    rig = MixerRig(build)
    got = rig.step([("a", h)])[0]
    z = dev(h.astype(np.float64) @ w["router"].astype(np.float64).T + w["router.b"])
    ids, wts, seg, src, dst = so.moe_route(z, top)
    assert ids.cpu().tolist() == chosen and abs(float(wts.sum()) - T) < 1e-4
    seg = seg.cpu().tolist()
    assert seg[0] == 0 and seg[-1] == T * top and all(a <= b for a, b in zip(seg, seg[1:]))
    assert rel_err(got, want) < 1e-5
    rig16 = MixerRig(build, torch.bfloat16)
    assert rel_err(rig16.step([("a", h)])[0], want) < 0.03
    if T > 1:                                                     # a token's result does not depend on the others of the batch
        assert rel_err(rig.step([("b", h[T // 2:T // 2 + 1])])[0], got[T // 2:T // 2 + 1]) < 1e-6


@pytest.mark.parametrize("T,N,K", [(100, 12, 192), (300, 5, 64), (40, 64, 1000), (17, 1, 8)])
def test_router_logits_many_rows_few_columns(so, T, N, K):
    """the f32 product of many rows with few output columns: unrounded operands, the same bits for a row whatever the batch"""
    rng = np.random.default_rng(T + N)
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    w, b = bf(rng.normal(0, 0.3, (N, K))), bf(rng.normal(0, 0.3, N))
    want = x.astype(np.float64) @ w.astype(np.float64).T + b
    got = so.linear(dev(x), dev(w, torch.bfloat16), dev(b, torch.bfloat16), math=so.MATH_F32_STREAM)
    assert rel_err(got.cpu().numpy(), want) < 2e-6
    part = so.linear(dev(x[T // 2:T // 2 + 20]), dev(w, torch.bfloat16), dev(b, torch.bfloat16), math=so.MATH_F32_STREAM)
    assert torch.equal(part.cpu(), got.cpu()[T // 2:T // 2 + 20])
    x16 = dev(x, torch.bfloat16)
    got16 = so.linear(x16, dev(w, torch.bfloat16), dev(b, torch.bfloat16), math=so.MATH_F32_STREAM)
    assert rel_err(got16.cpu().numpy(), x16.double().cpu().numpy() @ w.astype(np.float64).T + b) < 2e-6


# ---- the 64-key tile form (head sizes of exactly 64 / 128) -------------------------------------------------------------------------
def attention_f64(q, k, v, pos, scale, sink=None, softcap=0.0, gate=None, window=0, keep_first=0):
    """q [n, H, maps, D] at positions pos, k [m, G, maps, D], v [m, G, V], all float64 on the device -> [n, H, maps, V]"""
    n, H, M, _ = q.shape
    hpg = H // k.shape[1]
    kk, vv = k.repeat_interleave(hpg, 1), v.repeat_interleave(hpg, 1)
    s = torch.einsum("nhmd,khmd->nhmk", q, kk) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    key = torch.arange(k.shape[0], device=q.device)
    p = pos[:, None]
    seen = (key <= p) & ((p - key < window) | (key < keep_first) if window else True)
    s = s.masked_fill(~seen[:, None, None], -torch.inf)
    if sink is not None:
        s = torch.cat([s, sink.double()[None, :, None, None].expand(n, H, M, 1)], -1)
    w = torch.softmax(s, -1)[..., :k.shape[0]]
    o = torch.einsum("nhmk,khv->nhmv", w, vv)
    return o * gate.double()[:, :, None, None] if gate is not None else o


@pytest.mark.parametrize("H,G,D,V,maps,span,kw", [
    (8, 2, 128, 128, 1, 64, dict()),
    (8, 2, 128, 128, 1, 128, dict(sink=True, gate=True)),
    (6, 6, 64, 64, 1, 64, dict(softcap=8.0)),
    (3, 1, 64, 128, 1, 64, dict(window=70, keep_first=5)),
    (4, 2, 128, 64, 2, 64, dict(window=64, sink=True)),
    (64, 8, 128, 128, 1, 64, dict(softcap=30.0, window=130, gate=True)),
    (64, 64, 64, 64, 1, 64, dict(gate=True, window=70)),          # (enough key heads for two operands per wave without a split)
    (96, 48, 128, 128, 1, 64, dict(sink=True)),
])
@pytest.mark.parametrize("nsplit", [1, 4, 40])                    # (40: two operands per wave at any number of key heads)
def test_attention_in_64_key_tiles(so, H, G, D, V, maps, span, kw, nsplit):
    """Portions that end at, before and behind the borders of 64 keys, of 64 and 128 (row, head) pairs and of pages, from the start and from the
    middle of a sequence, one row alone; pages whose unwritten rows hold infinities (what another request may have left)."""
    from dash_infer_amd.seq_state import SequenceStateManager
    torch.manual_seed(H * 1000 + D + V + span)
    past, counts = [0, 0, 63, 128, 300, 191, 700], [1, 130, 65, 64, 33, 1, 1]
    st = SequenceStateManager(8192, len(past), span, "cuda")
    kt, vt = st.add_span_cache("k", G * maps * D, torch.bfloat16), st.add_span_cache("v", G * V, torch.bfloat16)
    for t in (kt, vt):
        t.pool.pool.view(torch.bfloat16).fill_(float("inf"))
    want, qs, poss, slots, row0 = [], [], [], [], []
    T = sum(counts)
    sink = torch.randn(H, device="cuda") if kw.get("sink") else None
    gate = torch.rand(T, H, device="cuda") if kw.get("gate") else None
    scale, at = D ** -0.5, 0
    for r, (p0, n) in enumerate(zip(past, counts)):
        st.admit(r)
        st.reserve(r, p0 + n)
        st.upload()
        slot = st.live[r].index
        m = p0 + n
        rows = torch.randn(m, (H + G) * maps * D + G * V, device="cuda")
        nq, nk = H * maps * D, G * maps * D
        rows[:, :nq] *= 2.0
        so.qkv_prep_append(rows, 0, nq, nq + nk, H, G, D, V, None, None, 1e-5, None, 0, 0, 1.0, 0.0, None, None, kt, vt, i32([slot] * m), i32(list(range(m))),
                           maps=maps)
        q = rows[p0:, :nq].contiguous()
        r16 = rows.to(torch.bfloat16).double()
        want.append(attention_f64(r16[p0:, :nq].view(n, H, maps, D), r16[:, nq:nq + nk].view(m, G, maps, D), r16[:, nq + nk:].view(m, G, V),
                                  torch.arange(p0, m, device="cuda"), scale, sink, kw.get("softcap", 0.0), gate[at:at + n] if gate is not None else None,
                                  kw.get("window", 0), kw.get("keep_first", 0)).reshape(n, -1))
        qs.append(q)
        poss += list(range(p0, m))
        slots.append(slot)
        row0.append(at)
        at += n
    got = so.gqa_attn_mc(torch.cat(qs), kt, vt, i32(poss), i32(slots), i32(row0), i32(counts), max(counts), max(poss), H, G, D, V, scale, sink,
                         so.SINK_PER_HEAD if sink is not None else so.SINK_NONE, kw.get("softcap", 0.0), gate, nsplit=nsplit, maps=maps,
                         window=kw.get("window", 0), keep_first=kw.get("keep_first", 0))
    for r in range(len(past)):       # weights rounded to bf16 (2^-9 each, independent) against sums of as many
        g, w = got[row0[r]:row0[r] + counts[r]].cpu().numpy(), want[r].cpu().numpy()
        assert rel_err(g, w) < 2.0 ** -8, (r, nsplit)


@pytest.mark.parametrize("H,G,D,V,span,kw", [
    (8, 2, 128, 128, 64, dict(norm=True, layout=1, rot=True)),
    (16, 1, 128, 64, 128, dict(sink=True, gate=True, layout=0, rot=True)),
    (6, 6, 64, 64, 64, dict(softcap=8.0, norm=True, layout=0, rot=True)),
    (9, 3, 64, 128, 256, dict(layout=1, rot=True, sink_zero=True)),
    (64, 8, 128, 128, 64, dict(norm=True, softcap=30.0, gate=True)),
    (1, 1, 64, 64, 64, dict(norm=True, layout=1, rot=True, far=True)),       # (more than 64 tiles to a wave)
])
@pytest.mark.parametrize("nsplit", [1, 3, 40])
def test_decoding_step_of_attention_in_one_launch(so, H, G, D, V, span, kw, nsplit):
    """Preparation, append and attention of one token per request against the launches one by one: the first row, both sides of the borders of tiles and of pages, a wave
    without a tile, splits without one; what other requests left in the pages are infinities."""
    from dash_infer_amd.seq_state import SequenceStateManager
    torch.manual_seed(H * 1000 + D + V + span)
    pos = [0, 1, 63, 64, 255, 256, 300, 1087] + ([17000] if kw.get("far") else [])
    E = len(pos)
    st = SequenceStateManager(sum(pos) + 256 * E, E, span, "cuda")
    kt, vt = st.add_span_cache("k", G * D, torch.bfloat16), st.add_span_cache("v", G * V, torch.bfloat16)
    for t in (kt, vt):
        t.pool.pool.view(torch.bfloat16).fill_(float("inf"))
    nq, nk = H * D, G * D
    rot = D if kw.get("rot") else 0
    freq = torch.tensor([10000.0 ** (-2.0 * i / D) for i in range(D // 2)], dtype=torch.float32, device="cuda") if rot else None
    qn, kn = (torch.rand(D, device="cuda") + 0.5, torch.rand(D, device="cuda") + 0.5) if kw.get("norm") else (None, None)
    args = (H, G, D, V, qn, kn, 1e-5, freq, rot, kw.get("layout", 0), 1.25)
    slots = []
    for r, p in enumerate(pos):
        st.admit(r)
        st.reserve(r, p + 1)
        st.upload()
        slots.append(st.live[r].index)
        if p:
            old = torch.randn(p, nq + nk + G * V, device="cuda")
            so.qkv_prep_append(old, 0, nq, nq + nk, *args, 0.0, None, None, kt, vt, i32([slots[r]] * p), i32(list(range(p))))
    order = list(reversed(range(E)))                 # (entries in another order than their rows)
    rows = torch.randn(E, nq + nk + G * V, device="cuda")
    rows[:, :nq] *= 2.0
    sink = torch.randn(H, device="cuda") if kw.get("sink") else None
    mode = so.SINK_PER_HEAD if sink is not None else so.SINK_ZERO if kw.get("sink_zero") else so.SINK_NONE
    gate = torch.rand(E, H, device="cuda") if kw.get("gate") else None
    before = rows.clone()
    pools = [t.pool.pool.clone() for t in (kt, vt)]
    entry = (i32(pos), i32([slots[r] for r in order]), i32(order))
    got = so.gqa_decode_step(rows, 0, nq, nq + nk, *args, kt, vt, *entry, max(pos), D ** -0.5, sink, mode, kw.get("softcap", 0.0), gate, nsplit=nsplit)
    assert torch.equal(rows, before)
    new = [t.pool.pool.clone() for t in (kt, vt)]
    for t, p in zip((kt, vt), pools):
        t.pool.pool.copy_(p)
    so.qkv_prep_append(rows, 0, nq, nq + nk, *args, 0.0, None, None, kt, vt, i32(slots), i32(pos))
    want = so.gqa_attn_mc(rows, kt, vt, *entry, i32([1] * E), 1, max(pos), H, G, D, V, D ** -0.5, sink, mode, kw.get("softcap", 0.0), gate, nsplit=1)
    assert torch.equal(new[1], vt.pool.pool)
    a, b = new[0].view(torch.bfloat16).float(), kt.pool.pool.view(torch.bfloat16).float()
    assert torch.equal(a.isinf(), b.isinf())
    a, b = a[~a.isinf()], b[~b.isinf()]
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -20).all())       # (the sum under a norm's root in another order: at most the neighbouring bf16, and rotation's cancelled last bits)
    for r in range(E):               # weights rounded to bf16 (2^-9 each, independent) on both sides
        assert rel_err(got[r].cpu().numpy(), want[r].cpu().numpy()) < 2.0 ** -7, (r, nsplit)


@pytest.mark.parametrize("nsplit", [1, 3])
def test_decoding_step_of_attention_leaves_other_rows_alone(so, nsplit):
    """fewer requests than rows, in any order: the rows that no request names keep what they held, the others are those of a call with their rows alone"""
    from dash_infer_amd.seq_state import SequenceStateManager
    H, G, D, T, order = 8, 2, 128, 6, [4, 0, 3]
    st = SequenceStateManager(64 * 12, T, 64, "cuda")
    kt, vt = st.add_span_cache("k", G * D, torch.bfloat16), st.add_span_cache("v", G * D, torch.bfloat16)
    for r in range(T):
        st.admit(r)
        st.reserve(r, 90)
    st.upload()
    for t in (kt, vt):
        t.pool.pool.view(torch.bfloat16).normal_()
    slot = [st.live[r].index for r in range(T)]
    rows, pos = torch.randn(T, (H + 2 * G) * D, device="cuda"), [70 + r for r in range(T)]
    pools = [t.pool.pool.clone() for t in (kt, vt)]
    call = lambda x, p, s, r0, out: so.gqa_decode_step(x, 0, H * D, (H + G) * D, H, G, D, D, None, None, 1e-5, None, 0, 0, 1.0, kt, vt, i32(p), i32(s), i32(r0), max(pos), D ** -0.5,
                                                       out=out, nsplit=nsplit)
    out = call(rows, pos, [slot[r] for r in order], order, torch.full((T, H * D), 7.0, device="cuda"))
    for t, p in zip((kt, vt), pools):
        t.pool.pool.copy_(p)
    alone = call(rows[order].contiguous(), [pos[r] for r in order], [slot[r] for r in order], [0, 1, 2], torch.empty(3, H * D, device="cuda"))
    assert torch.equal(out[order], alone) and bool((out[[r for r in range(T) if r not in order]] == 7.0).all())
