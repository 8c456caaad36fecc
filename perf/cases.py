"""The passes whose time counts: what programs built on this framework have it do, through the classes they use.

Two engines are measured over the range of calls that serving makes:
  "qdecode" / "qprefill"  decoder.DecodeSession: weight-only quantised models (int4 in groups of 128, int8 per channel), one decode step
                          of a batch as the captured graph that a server replays, or the context phase of a few prompts;
  "seqdecode" / "seqprefill" / "seqmixed"  engine.SeqEngine with bf16 weights: one token of every live request, a whole prompt, and the
                          mixed steps of continuous batching (a portion of a prompt beside decoded tokens).
Layer counts are cut (all layers of a model do the same work) so that inputs are quickly made; every step ends with the logits.
Weights are drawn with the spread that keeps activations near unit size; the output matrix leans on the embedding, so that the most
likely token stands out as a trained model's does.  Everything is made on the GPU from the seed."""
import math

import torch

from __graft_entry__ import _load_pkg

_load_pkg()
from dash_infer_amd import decoder, models, ops, tp  # noqa: E402
from dash_infer_amd.engine import SeqEngine  # noqa: E402

DEV = "cuda"
SPAN = 128

# width, heads, kv heads (of 128), feed-forward, vocabulary: those of this repository's benchmark and a small model
QMODELS = {
    "7b": dict(hidden=3584, n_heads=28, n_kv=4, inter=18944, vocab=152064),
    "small": dict(hidden=1024, n_heads=8, n_kv=2, inter=4096, vocab=32000),
    # 64 routed experts of 2560, 8 per token, and a shared one
    "moe": dict(hidden=3584, n_heads=28, n_kv=4, inter=20480, vocab=151936, experts=64, top=8, expert_inter=2560),
}
# the layer sizes of the sequence engine's benchmarks and a small model
SMODELS = {
    "4k": dict(width=4096, heads=32, kv_heads=8, gla_heads=32, gla_dim=64, gla_vdim=128, rank=64, ff=14336, vocab=32000),
    "2k": dict(width=2048, heads=16, kv_heads=4, gla_heads=16, gla_dim=64, gla_vdim=128, rank=64, ff=8192, vocab=32000),
    "small": dict(width=512, heads=4, kv_heads=2, gla_heads=4, gla_dim=64, gla_vdim=128, rank=32, ff=2048, vocab=8192),
}
SPATTERN = ("attention", "gla", "attention_2")


def listed():
    return [
        # one user's chat on a large model, the configuration the benchmark quotes
        dict(name="chat_int4_b1_2048", kind="qdecode", model="7b", layers=8, wbits=4, ft="bf16", kv="none", batch=1, ctx=2048, ragged=False),
        # the same user on 8-bit weights with an 8-bit cache, a short odd context
        dict(name="chat_int8_b1_777", kind="qdecode", model="7b", layers=6, wbits=8, ft="bf16", kv="i8", batch=1, ctx=777, ragged=False),
        # a small model (a draft model, an embedded assistant): latency and launches
        dict(name="chat_small_b1_300", kind="qdecode", model="small", layers=4, wbits=4, ft="bf16", kv="none", batch=1, ctx=300, ragged=False),
        # a busy server with the 4-bit cache
        dict(name="serve_int4_b32_u4kv_2048", kind="qdecode", model="7b", layers=8, wbits=4, ft="bf16", kv="u4", batch=32, ctx=2048, ragged=False),
        # a few users whose contexts differ widely, the longest a long document
        dict(name="serve_int4_b7_ragged_8100", kind="qdecode", model="7b", layers=6, wbits=4, ft="bf16", kv="none", batch=7, ctx=8100, ragged=True),
        # a mixture of experts under a medium batch
        dict(name="serve_moe_int8_b16_1024", kind="qdecode", model="moe", layers=2, wbits=8, ft="bf16", kv="none", batch=16, ctx=1024, ragged=False),
        # a long prompt; two short ones of odd lengths
        dict(name="prompt_int4_2048", kind="qprefill", model="7b", layers=4, wbits=4, ft="bf16", kv="none", batch=1, ctx=2048, ragged=False),
        dict(name="prompts_int8_217", kind="qprefill", model="7b", layers=4, wbits=8, ft="bf16", kv="none", batch=2, ctx=217, ragged=True),
        # the sequence engine: one user, a small server, a long prompt, continuous batching
        dict(name="seq_chat_b1_1500", kind="seqdecode", model="4k", layers=3, batch=1, ctx=1500, ragged=False),
        dict(name="seq_serve_b24_700", kind="seqdecode", model="2k", layers=3, batch=24, ctx=700, ragged=True),
        dict(name="seq_prompt_2048", kind="seqprefill", model="4k", layers=3, batch=1, ctx=2048, ragged=False),
        dict(name="seq_mixed_500_and_13", kind="seqmixed", model="2k", layers=3, batch=13, ctx=600, ragged=True, portion=500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["qdecode", "qdecode", "qprefill", "seqdecode", "seqprefill", "seqmixed"])
    if kind == "qdecode":
        model = rng.choice(["7b", "7b", "small"])
        batch = _log(rng, 1, 32)
        ctx = _log(rng, 256, min(8192, 65536 // batch))
        return dict(kind=kind, model=model, layers=rng.randint(2, 6), wbits=rng.choice([4, 4, 8]), ft=rng.choice(["bf16"] * 5 + ["f16"]),
                    kv=rng.choice(["none", "none", "i8", "u4"]), batch=batch, ctx=ctx, ragged=rng.random() < 0.5)
    if kind == "qprefill":
        return dict(kind=kind, model=rng.choice(["7b", "7b", "small"]), layers=rng.randint(2, 3), wbits=rng.choice([4, 4, 8]),
                    ft=rng.choice(["bf16"] * 5 + ["f16"]), kv="none", batch=rng.randint(1, 2), ctx=_log(rng, 24, 1024), ragged=True)
    model = rng.choice(["4k", "2k", "small"])
    if kind == "seqdecode":
        return dict(kind=kind, model=model, layers=rng.randint(2, 3), batch=_log(rng, 1, 32), ctx=_log(rng, 64, 2048), ragged=rng.random() < 0.5)
    if kind == "seqprefill":
        return dict(kind=kind, model=model, layers=rng.randint(2, 3), batch=rng.randint(1, 3), ctx=_log(rng, 24, 680), ragged=True)
    return dict(kind=kind, model=model, layers=rng.randint(2, 3), batch=_log(rng, 2, 24), ctx=_log(rng, 64, 1500), ragged=True,
                portion=_log(rng, 32, 700))


# ------------------------------------------------------------------------------------------------------------ common
def _gen(seed, *more):
    v = int(seed) & 0xFFFFFFFF
    for m in more:
        v = (v * 1000003 + int(m) + 17) & 0x7FFFFFFF
    return torch.Generator(device=DEV).manual_seed(v)


def _lengths(c):
    """the requests' lengths: all the same, or from the longest down to a fifth of it in uneven steps"""
    B, L = c["batch"], c["ctx"]
    if not c["ragged"]:
        return [L] * B
    return [max(1, int(L * (1.0 - 0.8 * (0.618034 * b % 1.0)))) for b in range(B)]


def _tokens(c, seed, vocab, n, which):
    return torch.randint(0, vocab, (n,), generator=_gen(seed, 3, which), device=DEV).tolist()


# ----------------------------------------------------------------------------------------- quantised decoder: weights
def _ft(c):
    return torch.bfloat16 if c["ft"] == "bf16" else torch.float16


def _group(c):
    return 128 if c["wbits"] == 4 else -1


def _qmat(c, g, K, N):
    """one quantised matrix as a checkpoint holds it: (q, scales, zeros)"""
    w4 = c["wbits"] == 4
    mid, sdq = (7.5, 2.7) if w4 else (0.0, 36.0)
    lo, hi = (0, 15) if w4 else (-128, 127)
    q = torch.randn(K, N, generator=g, device=DEV).mul_(sdq).add_(mid).round_().clamp_(lo, hi)
    G = K // 128 if w4 else 1
    s = (1.0 / math.sqrt(K) / sdq * (1 + 0.1 * torch.randn(G, N, generator=g, device=DEV))).to(_ft(c))
    z = (mid + 0.1 * sdq * torch.randn(G, N, generator=g, device=DEV)).to(_ft(c))
    if w4:
        q = q.to(torch.uint8)
        return (q[:, 1::2] << 4) | q[:, 0::2], s, z
    return q.to(torch.int8), s, z


def _dequantised(c, m):
    q, s, z = m
    if c["wbits"] == 4:
        q = torch.stack([q & 0xF, q >> 4], -1).reshape(q.shape[0], -1)
    K, N = q.shape
    per = K // s.shape[0]
    return ((q.double().view(-1, per, N) - z.double()[:, None]) * s.double()[:, None]).view(K, N)


def _qlayer(c, seed, i):
    d, g, ft = QMODELS[c["model"]], _gen(seed, 1, i), _ft(c)
    n, kv, W, F = d["n_heads"] * 128, d["n_kv"] * 128, d["hidden"], d["inter"]
    vec = lambda k, at, sd: (at + sd * torch.randn(k, generator=g, device=DEV)).to(ft)  # noqa: E731
    w = dict(qkv=_qmat(c, g, W, n + 2 * kv), o=_qmat(c, g, n, W), gate=_qmat(c, g, W, F), up=_qmat(c, g, W, F), down=_qmat(c, g, F, W),
             qkv_bias=vec(n + 2 * kv, 0.0, 0.1), ln1=vec(W, 1.0, 0.1), ln2=vec(W, 1.0, 0.1))
    if "experts" in d:
        E, P = d["experts"], d["expert_inter"]
        w["router"] = (2.0 / math.sqrt(W) * torch.randn(W, E, generator=g, device=DEV)).to(ft)
        w["sig"] = (1.0 / math.sqrt(W) * torch.randn(W, 1, generator=g, device=DEV)).to(ft)
        w["experts"] = [(_qmat(c, g, W, P), _qmat(c, g, W, P), _qmat(c, g, P, W)) for _ in range(E)]
    return w


def _qends(c, seed):
    """embedding, final norm, output matrix [hidden, vocab]"""
    d, g, ft = QMODELS[c["model"]], _gen(seed, 2), _ft(c)
    embed = torch.randn(d["vocab"], d["hidden"], generator=g, device=DEV).to(ft)
    norm = (1 + 0.1 * torch.randn(d["hidden"], generator=g, device=DEV)).to(ft)
    follows = torch.randperm(d["vocab"], generator=g, device=DEV)   # the token that comes before each
    head = (embed[follows].float() / math.sqrt(d["hidden"])).to(ft).t().contiguous()
    return embed, norm, head


def _context(c, seed, layer, b, L):
    """the cached keys and values of one request in one layer, [L, kv heads * 128] each"""
    g, kv = _gen(seed, 4, layer, b), QMODELS[c["model"]]["n_kv"] * 128
    return [torch.randn(L, kv, generator=g, device=DEV).to(_ft(c)) for _ in range(2)]


def _qmodel(c, seed):
    d = QMODELS[c["model"]]
    moe = decoder.MoEConfig(d["experts"], d["top"], d["expert_inter"]) if "experts" in d else None
    cfg = decoder.ModelConfig(c["model"], d["hidden"], c["layers"], d["n_heads"], d["n_kv"], 128, d["inter"], d["vocab"], moe=moe)
    G, bits = _group(c), c["wbits"]
    layers = []
    for i in range(c["layers"]):
        w = _qlayer(c, seed, i)
        p = {k: ops.pack_lowp(*w[k], G, bits) for k in ("qkv", "o", "gate", "up", "down")}
        lw = decoder.LayerWeights(ln1=w["ln1"], qkv=p["qkv"], qkv_bias=w["qkv_bias"], o=p["o"], ln2=w["ln2"], gate=p["gate"], up=p["up"], down=p["down"])
        if moe is not None:
            lw.router, lw.shared_sig, lw.ep = ops.pack_dense(w["router"]), ops.pack_dense(w["sig"]), (0, d["experts"])
            stack = [ops.pack_experts([e[j][0] for e in w["experts"]], [e[j][1] for e in w["experts"]], [e[j][2] for e in w["experts"]], G, bits)
                     for j in range(3)]
            lw.exp_gate, lw.exp_up, lw.exp_down = stack
        layers.append(lw)
        del w
    embed, norm, head = _qends(c, seed)
    heads = tp.shard_heads(d["n_heads"], d["n_kv"], 1)[0]
    return decoder.ModelWeights(cfg, decoder.QuantSpec(bits, G), 0, 1, heads, embed, layers, norm, ops.pack_dense(head), 0, d["vocab"])


def _prepare_q(c, seed):
    model, lens, d = _qmodel(c, seed), _lengths(c), QMODELS[c["model"]]
    room = max(lens) + (64 if c["kind"] == "qdecode" else 0)
    s = decoder.DecodeSession(model, c["batch"], room, span_len=SPAN, kv_mode=c["kv"])
    if c["kind"] == "qprefill":
        return {"session": s, "prompts": [_tokens(c, seed, d["vocab"], n, b) for b, n in enumerate(lens)]}
    for i in range(c["layers"]):
        for b, n in enumerate(lens):
            k, v = _context(c, seed, i, b, n)
            for rows, x in ((s.kv[i].k_ptrs[b], k), (s.kv[i].v_ptrs[b], v)):
                ops.kv_context_copy(rows, x, x.shape[1], n, 0, d["n_kv"], 128, SPAN, c["kv"])
    ids = torch.tensor(_tokens(c, seed, d["vocab"], c["batch"], 99), dtype=torch.int64, device=DEV)
    at = torch.tensor(lens, dtype=torch.int32, device=DEV)
    s.set_state(ids, at)
    s.capture()
    return {"session": s, "ids": ids, "lens": at}


# -------------------------------------------------------------------------------------------- sequence engine: weights
def _smodel(c, seed):
    d, g = SMODELS[c["model"]], _gen(seed, 5)
    W, H, G, F = d["width"], d["heads"], d["kv_heads"], d["ff"]

    def mat(*shape, sd=None):
        sd = 1.0 / math.sqrt(shape[-1]) if sd is None else sd
        return (torch.randn(*shape, generator=g, device=DEV) * sd).to(torch.bfloat16)

    def ones(n):
        return (1 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16)

    cfg = {"architecture": "Vogusun", "width": W, "vocab": d["vocab"], "norm": {"eps": 1e-6}, "layers": []}
    t = {"embed": mat(d["vocab"], W, sd=1.0), "head": mat(d["vocab"], W)}
    for name in ["final.norm"] + ["l%d.norm1" % i for i in range(c["layers"])]:
        t[name], t[name + ".b"], t[name + ".alpha"] = ones(W), mat(W, sd=0.1), torch.tensor(0.75, dtype=torch.bfloat16, device=DEV)
    for i in range(c["layers"]):
        kind, p = SPATTERN[i % 3], "l%d." % i
        if kind == "gla":
            h, a, v, r = d["gla_heads"], d["gla_dim"], d["gla_vdim"], d["rank"]
            m = {"heads": h, "dim": a, "vdim": v, "tau": 8.0}
            t.update({p + "mix.q": mat(h * a, W), p + "mix.k": mat(h * a, W), p + "mix.v": mat(h * v, W), p + "mix.g": mat(h * v, W),
                      p + "mix.o": mat(W, h * v), p + "mix.norm": ones(v), p + "mix.a1": mat(r, W), p + "mix.a2": mat(h * a, r),
                      p + "mix.a2.b": mat(h * a, sd=1.0)})
        else:
            m = {"heads": H, "kv_heads": G, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 1000000.0, "dims": 128}}
            t.update({p + "mix.q": mat(H * 128, W), p + "mix.k": mat(G * 128, W), p + "mix.v": mat(G * 128, W), p + "mix.o": mat(W, H * 128)})
            if kind == "attention":
                t.update({p + "mix.q.norm": ones(128), p + "mix.k.norm": ones(128), p + "mix.g": mat(H, W)})
            else:
                t.update({p + "mix.q.b": mat(H * 128, sd=0.1), p + "mix.k.b": mat(G * 128, sd=0.1), p + "mix.v.b": mat(G * 128, sd=0.1)})
                m["softcap"] = 50.0
        t.update({p + "mlp.gate": mat(F, W), p + "mlp.up": mat(F, W), p + "mlp.down": mat(W, F)})
        cfg["layers"].append({"type": kind, "mixer": m, "mlp": {"kind": "dense", "ff": F}})
    return cfg, t


def _prepare_s(c, seed):
    cfg, t = _smodel(c, seed)
    lens, V = _lengths(c), SMODELS[c["model"]]["vocab"]
    new = c.get("portion", 0)
    pages = sum(n // 64 + 2 for n in lens) + new // 64 + 2
    eng = SeqEngine(models.resolve(cfg), cfg, t, max_tokens=64 * pages, max_slots=c["batch"] + 1)
    prompts = [_tokens(c, seed, V, n + 2, b) for b, n in enumerate(lens)]
    state = {"engine": eng, "prompts": prompts}
    if c["kind"] == "seqprefill":
        state["entries"] = [(b, p[:n], [n - 1]) for b, (p, n) in enumerate(zip(prompts, lens))]
        return state
    for b, (p, n) in enumerate(zip(prompts, lens)):
        eng.step([(b, p[:n], [])])
    eng.step([(b, p[n:n + 1], [0]) for b, (p, n) in enumerate(zip(prompts, lens))])   # the first decoded token: the graph is there
    state["lens"] = [n + 1 for n in lens]
    state["entries"] = [(b, p[n + 1:n + 2], [0]) for b, (p, n) in enumerate(zip(prompts, lens))]
    if new:
        state["entries"].append(("new", _tokens(c, seed, V, new, 1000), [new - 1]))
    return state


# ------------------------------------------------------------------------------------------------------------- the passes
def prepare(case, seed):
    return (_prepare_q if case["kind"].startswith("q") else _prepare_s)(case, seed)


def run(state):
    if "session" in state:
        s = state["session"]
        if "prompts" in state:
            logits = s.prefill(state["prompts"])
        else:
            s.set_state(state["ids"], state["lens"])
            s.replay()
            logits = s.logits
        pool = s.pool.pool
        return {"logits": logits, "next": s.ids, "cache": pool.view(s.model.embed.dtype) if s.kv_mode == "none" else pool}
    eng = state["engine"]
    live = eng.state.live
    for rid, tokens, _ in state["entries"]:
        if rid == "new" or "lens" not in state:
            eng.release(rid)                          # a request that begins with this pass
        else:
            live[rid].length = state["lens"][rid]     # the token before was a rejected draft: its position is taken again
    logits = eng.step(state["entries"])
    return {"logits": logits, "caches": [t.pool.pool.view(t.dtype) for t in eng.state.tables.values()], "states": list(eng.state.states.values())}


def work(case):
    c, lens = case, _lengths(case)
    B, D = c["batch"], 128
    if c["kind"].startswith("q"):
        d = QMODELS[c["model"]]
        W, n, kv, F, V = d["hidden"], d["n_heads"] * D, d["n_kv"] * D, d["inter"], d["vocab"]
        size = lambda K, N: K * N * c["wbits"] / 8 + (K // 128 if c["wbits"] == 4 else 1) * N * 4  # noqa: E731
        mats = [(W, n + 2 * kv), (n, W), (W, F), (W, F), (F, W)]
        rows = B if c["kind"] == "qdecode" else sum(lens)
        by, fl = sum(size(*m) for m in mats), 2.0 * rows * sum(k * m for k, m in mats)
        if "experts" in d:
            P, E = d["expert_inter"], d["experts"]
            met = E * (1 - (1 - d["top"] / E) ** rows)          # experts that some row meets
            by += met * (2 * size(W, P) + size(P, W)) + 2 * W * (E + 1)
            fl += 2.0 * rows * d["top"] * 3 * W * P
        per = {"none": 2 * D, "i8": D + 8, "u4": D // 2 + 8}[c["kv"]] * d["n_kv"] * 2
        if c["kind"] == "qdecode":
            by += per * (sum(lens) + B)
            fl += 4.0 * n * (sum(lens) + B)
        else:
            by += per * rows
            fl += sum(2.0 * n * x * (x + 1) for x in lens)
        head_rows = B
        return {"bytes": c["layers"] * by + 2.0 * W * V + 4.0 * head_rows * V + 2.0 * rows * W, "flops": c["layers"] * fl + 2.0 * head_rows * W * V}
    d = SMODELS[c["model"]]
    W, H, G, F, V = d["width"], d["heads"] * D, d["kv_heads"] * D, d["ff"], d["vocab"]
    new = c.get("portion", 0)
    fresh = lens if c["kind"] == "seqprefill" else ([1] * B + ([new] if new else []))
    past = [0] * B if c["kind"] == "seqprefill" else [n + 1 for n in lens] + ([0] if new else [])
    rows, by, fl = sum(fresh), 0.0, 0.0
    for i in range(c["layers"]):
        p = 3 * W * F
        if SPATTERN[i % 3] == "gla":
            h, a, v, r = d["gla_heads"], d["gla_dim"], d["gla_vdim"], d["rank"]
            p += W * (2 * h * a + 3 * h * v + r) + r * h * a
            by += 8.0 * h * a * v * len(fresh)
            fl += 4.0 * rows * h * a * v
        else:
            p += W * (2 * H + 2 * G)
            by += 4.0 * G * (sum(past) + rows)
            fl += sum(4.0 * H * (f * q + f * (f + 1) / 2) for f, q in zip(fresh, past))
        by += 2.0 * p
        fl += 2.0 * rows * p
    return {"bytes": by + 2.0 * W * V + 4.0 * len(fresh) * V + 2.0 * rows * W, "flops": fl + 2.0 * len(fresh) * W * V}


def tolerance(case):
    # four times what the logits were measured to be off the 64-bit ones: 0.0034 .. 0.006 for bf16 activations through the quantised layers, 0.0004
    # for f16 ones, 0.002 .. 0.003 for the sequence engine's f32 residual rows between bf16 products.  Whole values: cache bytes of the new token,
    # whose quantiser may round the other way.
    if case["kind"].startswith("q"):
        return {"rel": 2e-2 if case["ft"] == "bf16" else 2e-3, "max": 0.15, "differ": 0.01}
    return {"rel": 1e-2, "max": 0.15}


# --------------------------------------------------------------------------------------------------- the same in 64 bits
def _rms(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _sig(x):
    return torch.sigmoid(x)


def _angles(pos, dims, base):
    f = (1.0 / (base ** (torch.arange(0, dims, 2, dtype=torch.float64) / dims))).float().to(DEV)
    a = (pos.float()[:, None] * f).double()       # the angle is a 32-bit product
    return torch.cos(a), torch.sin(a)


def _turn(x, pos, base, pairs):
    """x [rows, heads, 128]"""
    co, si = (t[:, None] for t in _angles(pos, x.shape[-1], base))
    if pairs:
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * co - v * si, v * co + u * si], -1).reshape(x.shape)
    u, v = x[..., : x.shape[-1] // 2], x[..., x.shape[-1] // 2:]
    return torch.cat([u * co - v * si, v * co + u * si], -1)


def _attend(q, k, v, first, scale, cap=0.0, sink=False):
    """q [n, H, D] at positions first .., k / v [m, G, D] -> [n, H * D]"""
    n, H, D = q.shape
    G = k.shape[1]
    s = torch.matmul(q.view(n, G, H // G, D).permute(1, 2, 0, 3).reshape(G, -1, D), k.permute(1, 2, 0).contiguous()) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    s = s.view(G, H // G, n, -1)
    late = torch.arange(k.shape[0], device=DEV)[None] > torch.arange(first, first + n, device=DEV)[:, None]
    s = s.masked_fill(late, -math.inf)
    if sink:
        s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
    p = torch.softmax(s, -1)
    if sink:
        p = p[..., :-1]
    o = torch.matmul(p.reshape(G, -1, p.shape[-1]), v.permute(1, 0, 2).contiguous())
    return o.view(G, H // G, n, D).permute(2, 0, 1, 3).reshape(n, H * D)


def _through_cache(c, x):
    """[L, kv heads, 128] as the cache gives it back"""
    if c["kv"] == "none":
        return x.double()
    lo, hi = (-128.0, 127.0) if c["kv"] == "i8" else (0.0, 15.0)
    x = x.float()
    mx, mn = x.amax(-1, keepdim=True), x.amin(-1, keepdim=True)
    s = ((mx - mn) / (hi - lo)).clamp_min(1e-5)
    z = (lo - mn / s).clamp(max=hi)
    z = (z.clamp(min=lo) if c["kv"] == "i8" else z).round()
    return ((z + x / s).clamp(lo, hi).round() - z).double() * s.double()


def _exact_q(c, seed):
    d, lens = QMODELS[c["model"]], _lengths(c)
    n, g, W = d["n_heads"], d["n_kv"], d["hidden"]
    embed, norm, head = _qends(c, seed)
    if c["kind"] == "qdecode":
        seqs = [[t] for t in _tokens(c, seed, d["vocab"], c["batch"], 99)]
        start = lens
    else:
        seqs = [_tokens(c, seed, d["vocab"], x, b) for b, x in enumerate(lens)]
        start = [0] * len(lens)
    cut = [len(s) for s in seqs]
    h = embed[torch.tensor(sum(seqs, []), device=DEV)].double()
    pos = torch.cat([torch.arange(a, a + m, device=DEV) for a, m in zip(start, cut)])
    for i in range(c["layers"]):
        w = _qlayer(c, seed, i)
        x = _rms(h, w["ln1"]) @ _dequantised(c, w["qkv"]) + w["qkv_bias"].double()
        q = _turn(x[:, :n * 128].view(-1, n, 128), pos, 1000000.0, False)
        k = _turn(x[:, n * 128:(n + g) * 128].view(-1, g, 128), pos, 1000000.0, False)
        v = x[:, (n + g) * 128:].view(-1, g, 128)
        outs, at = [], 0
        for b, m in enumerate(cut):
            kk, vv = k[at:at + m], v[at:at + m]
            if start[b]:
                ck, cv = (_through_cache(c, t.view(-1, g, 128)) for t in _context(c, seed, i, b, start[b]))
                kk, vv = torch.cat([ck, kk]), torch.cat([cv, vv])
            outs.append(_attend(q[at:at + m], kk, vv, start[b], 128 ** -0.5))
            at += m
        h = h + torch.cat(outs) @ _dequantised(c, w["o"])
        x = _rms(h, w["ln2"])
        a = x @ _dequantised(c, w["gate"])
        f = (a * _sig(a) * (x @ _dequantised(c, w["up"]))) @ _dequantised(c, w["down"])
        if "experts" in d:
            p, e = torch.softmax(x @ w["router"].double(), -1).topk(d["top"], -1)
            y = f * _sig(x @ w["sig"].double())
            for j in e.unique().tolist():
                r, slot = (e == j).nonzero(as_tuple=True)
                wg, wu, wd = (_dequantised(c, m) for m in w["experts"][j])
                a = x[r] @ wg
                y[r] += p[r, slot, None] * ((a * _sig(a) * (x[r] @ wu)) @ wd)
            f = y
        h = h + f
        del w
    last = torch.tensor(cut, device=DEV).cumsum(0) - 1
    logits = _rms(h[last], norm) @ head.double()
    return {"logits": logits, "next": logits.argmax(-1), "cache": None}


def _exact_s(c, seed):
    cfg, t = _smodel(c, seed)
    lens, V = _lengths(c), SMODELS[c["model"]]["vocab"]
    new = c.get("portion", 0)
    more = 0 if c["kind"] == "seqprefill" else 2
    seqs = [_tokens(c, seed, V, n + 2, b)[:n + more] for b, n in enumerate(lens)]
    if new:
        seqs.append(_tokens(c, seed, V, new, 1000))
    dyt = lambda x, name: torch.tanh(t[name + ".alpha"].double() * x) * t[name].double() + t[name + ".b"].double()  # noqa: E731
    out = []
    for toks in seqs:
        x = t["embed"][torch.tensor(toks, device=DEV)].double()
        n = x.shape[0]
        pos = torch.arange(n, device=DEV)
        for i, lc in enumerate(cfg["layers"]):
            w = {k[len("l%d." % i):]: v.double() for k, v in t.items() if k.startswith("l%d." % i)}
            h, m, kind = dyt(x, "l%d.norm1" % i), lc["mixer"], lc["type"]
            if kind == "gla":
                H, D, E = m["heads"], m["dim"], m["vdim"]
                q, k = (h @ w["mix.q"].t() * D ** -0.5).view(n, H, D), (h @ w["mix.k"].t()).view(n, H, D)
                v = (h @ w["mix.v"].t()).view(n, H, E)
                a = (_sig((h @ w["mix.a1"].t()) @ w["mix.a2"].t() + w["mix.a2.b"]) ** (1.0 / m["tau"])).view(n, H, D)
                S, o = torch.zeros(H, D, E, dtype=torch.float64, device=DEV), []
                for r in range(n):
                    S = a[r][:, :, None] * S + k[r][:, :, None] * v[r][:, None]
                    o.append((S * q[r][:, :, None]).sum(1))
                z = h @ w["mix.g"].t()
                mo = (_rms(torch.stack(o), t["l%d.mix.norm" % i]).reshape(n, H * E) * z * _sig(z)) @ w["mix.o"].t()
            else:
                H, G, D = m["heads"], m["kv_heads"], m["dim"]
                q, k, v = ((h @ w["mix." + s].t() + w.get("mix.%s.b" % s, 0.0)).view(n, -1, D) for s in "qkv")
                first = kind == "attention"
                if first:
                    q, k = _rms(q, w["mix.q.norm"]), _rms(k, w["mix.k.norm"])
                q, k = (_turn(y, pos, m["rot"]["base"], first) for y in (q, k))
                o = _attend(q, k, v, 0, m["scale"], m.get("softcap", 0.0), first)
                if first:
                    o = (o.view(n, H, D) * _sig(h @ w["mix.g"].t())[:, :, None]).reshape(n, H * D)
                mo = o @ w["mix.o"].t()
            a = h @ w["mlp.gate"].t()
            gelu = 0.5 * a * (1 + torch.tanh(math.sqrt(2 / math.pi) * (a + 0.044715 * a ** 3)))
            x = x + mo + (gelu * (h @ w["mlp.up"].t())) @ w["mlp.down"].t()
            del w
        out.append(dyt(x[-1:], "final.norm") @ t["head"].double().t())
    return {"logits": torch.cat(out), "caches": None, "states": None}


def exact(case, seed):
    return (_exact_q if case["kind"].startswith("q") else _exact_s)(case, seed)
