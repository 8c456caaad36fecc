"""End-to-end greedy decode against the oracle (north star: "bit-exact token IDs under greedy decode, logits within
1e-2 for bf16").

A small random model of the Qwen2 architecture (same graph as python/pyhie/allspark/model/qwen_v15.py:210-388: RMSNorm ->
qkv GEMM + bias -> Rotary -> span attention over the paged cache -> o GEMM + residual -> RMSNorm -> SiLU(gate) * up -> down
GEMM + residual; final norm -> bf16 lm_head -> greedy) is decoded from an empty cache by the product path
(decoder.DecodeSession: every fused HIP entry point the bench uses, eager and through a captured hipGraph) and, token by
token, by the numpy decoder of oracle/model.py (quantised linear of gemm_ref, cache codec of kv_codec, attention / glue;
itself checked on CPU in test_oracle_model.py).  The oracle is fed the tokens the GPU chose, so one near-tie cannot derail the comparison; token IDs
must agree wherever the oracle's top-2 margin exceeds the logit tolerance.
"""
import numpy as np
import pytest
import torch

from oracle import glue, model as omodel

pytestmark = pytest.mark.gpu

# north star: logits within 1e-2 for bf16 -- taken relative to the logit scale (absolute below 1): one bf16 ulp of a logit
# of magnitude 3 is already 1.6e-2, and the int4 models here reach |logit| ~ 3 with errors of 1.0e-2 ... 1.8e-2 on every
# kernel family alike (GEMV at batch 4, small-batch GEMMs at batch 32).  The uint4 cache is outside that statement (parity unpinned): a
# 16-level code turns a one-ulp difference of a K / V element that sits on a rounding boundary (or of the row's min / max,
# which moves every boundary) into a step of range / 15, so the end-to-end bound there is twice as wide (measured up to 4.6e-2 at |logit| 3); the codec and the
# attention over identical cache bytes are pinned bit-exactly / to 1e-2 in test_gpu_kv_attn.py.
LOGIT_TOL = {"none": 1e-2, "i8": 1e-2, "u4": 2e-2}   # x max(1, max |logit|)


def oracle_of(model, kv_mode):
    """The numpy decoder (oracle/model.py) over the product model's own quantised weights (build_random_model(keep_fp=True))."""
    cfg = model.cfg
    f = lambda t: t.float().cpu().numpy()
    layers = []
    for li in range(len(model.layers)):
        p = model.fp[li]
        lw = {k: tuple((x.cpu().numpy() if x.dtype in (torch.uint8, torch.int8) else f(x)) for x in p[k])
              for k in ("qkv", "o", "gate", "up", "down")}
        lw.update(qkv_bias=f(p["qkv_bias"]), ln1=f(p["ln1"]), ln2=f(p["ln2"]))
        if "moe" in p:
            conv = lambda q: tuple((x.cpu().numpy() if x.dtype in (torch.uint8, torch.int8) else f(x)) for x in q)
            mo = p["moe"]
            lw["moe"] = {"router": f(mo["router"]), "shared_gate_w": f(mo["shared_gate_w"]), "top_k": mo["top_k"],
                         "experts_gate": [conv(q) for q in mo["experts_gate"]], "experts_up": [conv(q) for q in mo["experts_up"]],
                         "experts_down": [conv(q) for q in mo["experts_down"]]}
        layers.append(lw)
    ft = "f16" if model.embed.dtype == torch.float16 else "bf16"
    return omodel.DecoderOracle(layers, f(model.fp["embed"]), f(model.fp["final_norm"]), f(model.fp["lm_head"]), cfg.n_heads,
                                cfg.n_kv, cfg.head_dim, model.quant.wbits, model.quant.group, eps=cfg.eps,
                                rope_theta=cfg.rope_theta, kv_mode=kv_mode, ft=ft)


SMALL = dict(hidden=512, layers=2, n_heads=4, n_kv=2, head_dim=128, inter=1024, vocab=2048)
WIDE = dict(hidden=1024, layers=2, n_heads=8, n_kv=4, head_dim=128, inter=2048, vocab=4096)


@pytest.mark.parametrize("shape,wbits,group,kv_mode,batch,graph,gptq", [
    (SMALL, 4, 128, "none", 1, False, False),   # int4 g128, batch 1 (GEMV kernels, fused MFMA attention)
    (SMALL, 4, 128, "none", 1, True, False),    # the same through a captured hipGraph (what bench.py times)
    (SMALL, 8, -1, "none", 3, False, False),    # configs[1]: int8 per-channel
    (SMALL, 4, 128, "i8", 2, False, False),     # quantised caches: decode-step kernel
    (SMALL, 4, 128, "u4", 3, True, False),
    (SMALL, 4, 128, "i8", 2, True, False),
    (WIDE, 4, 128, "u4", 32, False, False),     # configs[2]: batch 32, uint4 cache (MFMA attention at the op boundary, small-batch GEMMs)
    (WIDE, 8, 128, "none", 17, False, False),   # odd batch, int8 sub-channel, 16-bit cache
    (SMALL, 4, 128, "none", 2, False, True),   # GPTQ-style integer zero points in [1, 16] (configs[2] weights)
    (WIDE, 4, 128, "i8", 32, True, True),      # batch 32 through the captured graph: fused norm path, int8 cache
    (WIDE, 4, 128, "none", 32, False, False),  # batch 32, 16-bit cache
    (WIDE, 4, 128, "none", 4, False, False),   # the same model on the GEMV kernels
])
def test_greedy_decode_matches_oracle(pkg, shape, wbits, group, kv_mode, batch, graph, gptq):
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("test", **shape)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group, gptq_like_zeros=gptq), seed=4321, keep_fp=True)
    steps = 6
    sess = decoder.DecodeSession(model, batch, max_len=32, span_len=16, kv_mode=kv_mode)
    rng = np.random.default_rng(batch * 17 + wbits)
    ids = rng.integers(0, cfg.vocab, batch)
    sess.set_state(ids, [0] * batch)
    gpu_logits, gpu_ids = [], []
    if graph:
        # capture replays the step on the live state: warm up on a scratch state first, then restart from the empty cache
        sess.capture(warmup=1)
        sess.set_state(ids, [0] * batch)
    for _ in range(steps):
        if graph:
            sess.replay()
        else:
            sess.step()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    ref = oracle_of(model, kv_mode)
    cur, decided, worst = ids, 0, 0.0
    for t in range(steps):
        lo = ref.step(cur)
        tol = LOGIT_TOL[kv_mode] * max(1.0, float(np.abs(lo).max()))
        err = np.abs(gpu_logits[t] - lo).max()
        worst = max(worst, float(err))
        assert err <= tol, f"step {t}: logits differ by {err:.3e} (max |logit| {np.abs(lo).max():.2f})"
        top2 = np.sort(lo, axis=-1)[:, -2:]
        sure = (top2[:, 1] - top2[:, 0]) > 2 * tol
        assert np.array_equal(gpu_ids[t][sure], glue.greedy(lo)[sure]), f"step {t}: greedy token IDs differ"
        decided += int(sure.sum())
        cur = gpu_ids[t]  # follow the product path's choice: a near-tie must not derail the later steps
    assert decided >= steps * batch // 4, "too few decisive steps for the token-ID check to mean anything"
    print(f"worst logit error {worst:.2e}; {decided}/{steps * batch} decisive greedy choices")


# ------------------------------------------------------------------------------------------------------------------
# Mixture-of-experts decoder (BASELINE configs[4] architecture, python/pyhie/allspark/model/qwen_v20_moe.py:318-382): every
# layer's feed-forward block is router -> top-k of the routed experts -> combine, + the shared expert behind its sigmoid
# gate.  Same comparison as above against oracle/model.py::_moe_mlp (router / experts of oracle/moe.py).
MOE_SMALL = dict(hidden=512, layers=2, n_heads=4, n_kv=2, head_dim=128, inter=512, vocab=2048)


@pytest.mark.parametrize("wbits,group,batch,experts,top_k", [(8, -1, 1, 8, 2), (4, 128, 3, 8, 2), (8, -1, 4, 16, 4)])
def test_moe_greedy_decode_matches_oracle(pkg, wbits, group, batch, experts, top_k):
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("moe-test", **MOE_SMALL, moe=decoder.MoEConfig(experts, top_k, 256))
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group), seed=2468, keep_fp=True)
    steps = 5
    sess = decoder.DecodeSession(model, batch, max_len=32, span_len=16, kv_mode="none")
    rng = np.random.default_rng(batch * 5 + wbits)
    ids = rng.integers(0, cfg.vocab, batch)
    sess.set_state(ids, [0] * batch)
    gpu_logits, gpu_ids = [], []
    for _ in range(steps):
        sess.step()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    ref = oracle_of(model, "none")
    cur, decided, worst = ids, 0, 0.0
    for t in range(steps):
        lo = ref.step(cur)
        tol = 1e-2 * max(1.0, float(np.abs(lo).max()))
        err = float(np.abs(gpu_logits[t] - lo).max())
        worst = max(worst, err)
        assert err <= tol, f"step {t}: logits differ by {err:.3e} (max |logit| {np.abs(lo).max():.2f})"
        top2 = np.sort(lo, axis=-1)[:, -2:]
        sure = (top2[:, 1] - top2[:, 0]) > 2 * tol
        assert np.array_equal(gpu_ids[t][sure], glue.greedy(lo)[sure]), f"step {t}: greedy token IDs differ"
        decided += int(sure.sum())
        cur = gpu_ids[t]
    assert decided >= steps * batch // 4
    print(f"MoE: worst logit error {worst:.2e}; {decided}/{steps * batch} decisive greedy choices")


# ------------------------------------------------------------------------------------------------------------------
# The same comparison at Qwen2-7B WIDTHS (hidden 3584, 28 / 4 heads, intermediate 18944, vocabulary 152064; 2 of the 28
# layers) with a 2048-token history produced by the product's own context phase (DecodeSession.prefill: qkv GEMM, Rotary,
# ContextSpanCopy, MFMA prefill attention, ...), then greedy decode steps on the kernels bench.py times (GEMV family,
# decode-step MFMA attention at 2048+ tokens, 17 splits).  The oracle is independent of the GPU: it runs its own prefill of
# the same prompt (numpy, f64 accumulation) and is only fed the tokens the GPU chose.
#
# The north star's bar is "logits within 1e-2 for bf16, bit-exact greedy ids".  The test asserts a bound it can hold on
# every box and PRINTS the measured numbers (no margin filter on the ids): they go to DESIGN.md section 0.
WIDTH7B = dict(hidden=3584, layers=2, n_heads=28, n_kv=4, head_dim=128, inter=18944, vocab=152064)


@pytest.mark.parametrize("wbits,group,gptq", [(4, 128, True)])   # (int8 per-channel and int4 IQ zeros: the full-depth test below)
def test_qwen7b_width_prefill_then_decode_vs_oracle(pkg, wbits, group, gptq):
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("qwen2-7b-width", **WIDTH7B)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group, gptq_like_zeros=gptq), seed=77, keep_fp=True)
    L, steps = 2048, 4
    sess = decoder.DecodeSession(model, 1, max_len=L + steps + 8, span_len=128, kv_mode="none")
    rng = np.random.default_rng(2048 + wbits)
    prompt = [int(t) for t in rng.integers(0, cfg.vocab, L)]
    lo_gpu0 = sess.prefill([prompt]).cpu().numpy()
    gpu_logits, gpu_ids = [], [sess.ids.cpu().numpy().copy()]
    sess.capture(warmup=0)  # the captured hipGraph is what bench.py replays
    for _ in range(steps):
        sess.replay()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    report = {}
    for rounding in ("x86", "ft_graph"):
        ref = oracle_of(model, "none")
        ref.rounding = rounding
        ref._wcache = {}  # dequantise each matrix once (2 layers of 7B-width weights)
        ref.acc, ref.threads = np.float32, 16
        lo0 = ref.prefill([prompt])
        errs = [float(np.abs(lo_gpu0 - lo0).max())]
        mism = [int((glue.greedy(lo0) != gpu_ids[0]).sum())]
        margins = [float(np.sort(lo0, axis=-1)[0, -1] - np.sort(lo0, axis=-1)[0, -2])]
        scale = float(np.abs(lo0).max())
        cur = gpu_ids[0]
        for t in range(steps):
            lo = ref.step(cur)
            errs.append(float(np.abs(gpu_logits[t] - lo).max()))
            mism.append(int((glue.greedy(lo) != gpu_ids[t + 1]).sum()))
            top = np.sort(lo, axis=-1)[0]
            margins.append(float(top[-1] - top[-2]))
            scale = max(scale, float(np.abs(lo).max()))
            cur = gpu_ids[t + 1]
        report[rounding] = (errs, mism, margins, scale)
        print(f"[7B-width int{wbits} g{group}] oracle rounding={rounding}: max |logit err| per step (prefill last token, then "
              f"{steps} decode steps) = {['%.2e' % e for e in errs]}; max |logit| {scale:.2f}; greedy id mismatches (no margin "
              f"filter) = {sum(mism)}/{len(mism)}; oracle top-2 margins {['%.3f' % m for m in margins]}")
    errs, mism, margins, scale = report["x86"]
    # what holds on every box: the absolute error stays below 1e-2 x max(1, max |logit|), and an id can only differ where the
    # oracle's own top-2 margin is smaller than twice the measured logit error (a genuine near-tie)
    assert max(errs) <= 1e-2 * max(1.0, scale), f"logits differ by {max(errs):.3e} at max |logit| {scale:.2f}"
    for e, m, g in zip(errs, mism, margins):
        assert m == 0 or g <= 2 * e, f"greedy id differs although the oracle's margin {g:.3e} exceeds twice the logit error {e:.3e}"


# ------------------------------------------------------------------------------------------------------------------
# FULL DEPTH at the BASELINE configuration: all 28 layers of Qwen2-7B widths, a 2048-token history from the
# product's own context phase, then 8 greedy steps through the captured hipGraph (the launches bench.py times), compared with
# the numpy oracle under FIVE sets of rounding points (oracle/model.py: ft_graph, x86 = the hybrid with an FT cache,
# x86_pure_bf16 = the reference x86 path under medium_bf16 -- f32 qkv / cache / attention output, bf16 weight reorder --,
# x86_pure_f32, and the exact-weight ablation).  The oracle is fed the tokens the GPU chose and evaluates all positions in one
# teacher-forced pass (oracle.model.teacher_forced_logits: every layer dequantised once, all roundings in lockstep, f32
# accumulation as cblas_sgemm / oneDNN carry it) -- the same function as prefill + step() (tests/test_oracle_model.py).
# Printed per rounding and step: max |logit error| ABSOLUTE, greedy-id mismatches with NO margin filter, the oracle's top-2
# margins.  Asserted: what holds on every box (error relative to the logit scale against the `x86` rounding, an id may differ
# only inside a genuine near-tie); the measured numbers go to DESIGN.md section 0.
class _LazyOracleLayers:
    """layer li's oracle dict built from the product model's GPU tensors on access (28 layers of 7B-width matrices stay on the GPU)."""

    def __init__(self, model):
        self.model = model

    def __len__(self):
        return len(self.model.layers)

    def __getitem__(self, li):
        f = lambda t: t.float().cpu().numpy()
        p = self.model.fp[li]
        lw = {k: tuple((x.cpu().numpy() if x.dtype in (torch.uint8, torch.int8) else f(x)) for x in p[k])
              for k in ("qkv", "o", "gate", "up", "down")}
        lw.update(qkv_bias=f(p["qkv_bias"]), ln1=f(p["ln1"]), ln2=f(p["ln2"]))
        return lw


def _teacher_forced_report(model, prompt, gpu_prefill_logits, gpu_step_logits, gpu_ids, roundings, tag, f64_twin=False):
    """gpu_ids[0] = the token after the prompt, gpu_ids[t + 1] = the token step t chose.  Returns {rounding: (errs, mism, margins, scale)}
    and the oracle-to-oracle distances.  f64_twin: one more pass of roundings[0] with float64 accumulation -- the same
    rounding points, another summation precision: the noise floor every bf16-graph comparison at this depth sits on."""
    import os
    cfg = model.cfg
    f = lambda t: t.float().cpu().numpy()
    steps = len(gpu_step_logits)
    layers = _LazyOracleLayers(model)
    embed, fn, lm = f(model.fp["embed"]), f(model.fp["final_norm"]), f(model.fp["lm_head"])
    oracles, names = [], list(roundings) + ([roundings[0] + "@f64"] if f64_twin else [])
    for r in names:
        o = omodel.DecoderOracle(layers, embed, fn, lm, cfg.n_heads, cfg.n_kv, cfg.head_dim, model.quant.wbits, model.quant.group,
                                 eps=cfg.eps, rope_theta=cfg.rope_theta, kv_mode="none", rounding=r.split("@")[0])
        o.acc = np.float64 if r.endswith("@f64") else np.float32
        oracles.append(o)
    seq = list(prompt) + [int(gpu_ids[t][0]) for t in range(steps)]   # the step-t input is the id chosen before it
    los = omodel.teacher_forced_logits(oracles, layers, seq, steps + 1, threads=min(16, os.cpu_count() or 1))
    gpu = np.concatenate([gpu_prefill_logits.reshape(1, -1)] + [l.reshape(1, -1) for l in gpu_step_logits])
    report = {}
    for r, lo in zip(names, los):
        errs = [float(np.abs(gpu[t] - lo[t]).max()) for t in range(steps + 1)]
        mism = [int(glue.greedy(lo[t:t + 1])[0] != int(gpu_ids[t][0])) for t in range(steps + 1)]
        srt = np.sort(lo, axis=-1)
        margins = [float(srt[t, -1] - srt[t, -2]) for t in range(steps + 1)]
        scale = float(np.abs(lo).max())
        report[r] = (errs, mism, margins, scale)
        print(f"[{tag}] product vs oracle rounding={r}: max |logit err| (prefill last token, then {steps} decode steps) = "
              f"{['%.2e' % e for e in errs]}; worst {max(errs):.2e} at max |logit| {scale:.2f}; greedy id mismatches (no margin "
              f"filter) = {sum(mism)}/{len(mism)}; oracle top-2 margins {['%.3f' % m for m in margins]}")
    dist = {}
    for i in range(len(names)):
        for j in range(i + 1, len(names)):
            dist[(names[i], names[j])] = float(np.abs(los[i] - los[j]).max())
            ids_differ = int((glue.greedy(los[i]) != glue.greedy(los[j])).sum())
            print(f"[{tag}] oracle vs oracle: {names[i]} <-> {names[j]}: max |logit diff| {dist[(names[i], names[j])]:.2e}, greedy ids differ at "
                  f"{ids_differ}/{steps + 1} positions")
    return report, dist


# Modes of the always-on test: the hybrid the product's rounding points were designed against, and the two literal x86 paths.
# DIHIP_FULL_DEPTH_ABLATION=1 (tools/gpu_round_end.sh; output committed under profiles/) adds the CUDA bf16 graph, the
# exact-weight ablation and the float64 twin of `x86` (the summation-precision noise floor).
@pytest.mark.parametrize("wbits,group,gptq,roundings", [
    (4, 128, False, ("x86", "x86_pure_bf16", "x86_pure_f32")),   # the BASELINE headline configuration
    (8, -1, False, ("x86",)),                                    # configs[1]
])
def test_qwen7b_full_depth_decode_vs_oracle(pkg, wbits, group, gptq, roundings):
    import os
    from dash_infer_amd import decoder
    ablation = os.environ.get("DIHIP_FULL_DEPTH_ABLATION", "0") == "1"
    if ablation and wbits == 4:
        roundings = roundings + ("ft_graph", "x86_pure_bf16_exactw")
    cfg = decoder.QWEN2_7B
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group, gptq_like_zeros=gptq), seed=77, keep_fp=True)
    L, steps = 2048, 8
    sess = decoder.DecodeSession(model, 1, max_len=L + steps + 8, span_len=128, kv_mode="none")
    rng = np.random.default_rng(4096 + wbits)
    prompt = [int(t) for t in rng.integers(0, cfg.vocab, L)]
    lo_gpu0 = sess.prefill([prompt]).cpu().numpy()
    gpu_logits, gpu_ids = [], [sess.ids.cpu().numpy().copy()]
    sess.capture(warmup=0)  # the captured hipGraph is what bench.py replays
    for _ in range(steps):
        sess.replay()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    del sess
    rep, dist = _teacher_forced_report(model, prompt, lo_gpu0, gpu_logits, gpu_ids, roundings, f"7B FULL DEPTH int{wbits} g{group}",
                                       f64_twin=ablation and wbits == 4)
    errs, mism, margins, scale = rep["x86"]
    # What holds on every box.  The literal "1e-2 absolute" of the north star does not exist at this depth for ANY pair of
    # evaluations of the graph: two oracles that differ in nothing but the summation precision are already further apart
    # (the @f64 twin of the ablation run; DESIGN.md section 0 has the measured table).  Asserted: the product stays within
    # 3e-2 of the logit scale of the hybrid rounding (measured 2.2e-2; the clause itself is asserted on a DECISIVE model and per
    # layer in tests/test_gpu_parity_depth.py -- this random N(0, 0.02) model is kept as the explanation of why it has to be), is
    # closer to it than the reference's own x86 variants are to each other,
    # and a greedy id differs from an oracle's only inside that oracle's genuine near-tie.
    assert max(errs) <= 3e-2 * max(1.0, scale), f"logits differ by {max(errs):.3e} at max |logit| {scale:.2f}"
    if ("x86_pure_bf16", "x86_pure_f32") in dist:
        assert max(errs) <= dist[("x86_pure_bf16", "x86_pure_f32")], "further from the hybrid oracle than the two x86 precisions are from each other"
    for r in rep:
        for e, m, g in zip(*rep[r][:3]):
            assert m == 0 or g <= 2 * e, f"[{r}] greedy id differs although the oracle's margin {g:.3e} exceeds twice the logit error {e:.3e}"


# configs[2] (batch 32, uint4 KV cache, GPTQ-style integer zero points) and the per-rank shapes of configs[3] (one rank of
# Qwen2-72B at TP = 8: 8 query / 1 KV head, 8192 -> 1280 / 1024 -> 8192 / 8192 -> 3712 / 3712 -> 8192, batch 16) at 2 layers of their REAL
# widths: ragged histories from the product's context phase, then greedy steps on the small-batch GEMM family / the quantised-cache
# attention kernels, against oracle.step() (the oracle's own prefill + per-step cache codec).
@pytest.mark.parametrize("name,shape,kv_mode,batch,gptq,hist", [
    ("configs[2] widths", dict(hidden=3584, layers=2, n_heads=28, n_kv=4, head_dim=128, inter=18944, vocab=8192), "u4", 32, True, (40, 200)),
    ("configs[3] rank widths", dict(hidden=8192, layers=2, n_heads=8, n_kv=1, head_dim=128, inter=3712, vocab=19008), "none", 16, False, (100, 300)),
])
def test_real_width_batched_decode_vs_oracle(pkg, name, shape, kv_mode, batch, gptq, hist):
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig(name, **shape)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(4, 128, gptq_like_zeros=gptq), seed=99, keep_fp=True)
    steps = 4
    rng = np.random.default_rng(batch)
    lens = [int(x) for x in rng.integers(hist[0], hist[1], batch)]
    prompts = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in lens]
    sess = decoder.DecodeSession(model, batch, max_len=max(lens) + steps + 8, span_len=32, kv_mode=kv_mode)
    lo_gpu0 = sess.prefill(prompts).cpu().numpy()
    gpu_logits, gpu_ids = [], [sess.ids.cpu().numpy().copy()]
    sess.capture(warmup=0)
    for _ in range(steps):
        sess.replay()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    ref = oracle_of(model, kv_mode)
    ref._wcache = {}
    ref.acc = np.float32
    lo = ref.prefill(prompts)
    # real widths: the uint4 cache's code steps (range / 15 per element, the row's min / max moving every boundary) weigh
    # more than at the toy widths above -- measured 3.8e-2 (context) ... 1.1e-1 (4th step, each step appending rows quantised
    # from slightly different bf16 values) at |logit| ~ 4; the codec bytes themselves are pinned bit-exactly elsewhere
    tol_unit = {"none": 1e-2, "i8": 1e-2, "u4": 5e-2}[kv_mode]
    errs, mism, n_ids, scale_all = [], 0, 0, 0.0
    cur = gpu_ids[0]
    for t in range(steps + 1):
        g = lo_gpu0 if t == 0 else gpu_logits[t - 1]
        e = float(np.abs(g - lo).max())
        errs.append(e)
        tol = tol_unit * max(1.0, float(np.abs(lo).max()))
        scale_all = max(scale_all, float(np.abs(lo).max()))
        assert e <= tol, f"{name} step {t}: logits differ by {e:.3e} (max |logit| {np.abs(lo).max():.2f})"
        top2 = np.sort(lo, axis=-1)[:, -2:]
        margin = top2[:, 1] - top2[:, 0]
        differ = glue.greedy(lo) != gpu_ids[t]
        mism += int(differ.sum())
        n_ids += batch
        assert not (differ & (margin > 2 * e)).any(), f"{name} step {t}: a greedy id differs outside a near-tie"
        if t < steps:
            lo = ref.step(gpu_ids[t])
    print(f"[{name}, batch {batch}, kv {kv_mode}] max |logit err| per step {['%.2e' % e for e in errs]} at max |logit| {scale_all:.2f}; greedy id "
          f"mismatches (no margin filter) {mism}/{n_ids}")


# ------------------------------------------------------------------------------------------------------------------
# f16 activations through the FUSED decode-step forms (the reference's span-attention and GEMMs serve
# FT in {f32, f16, bf16} on every path; until round 3 f16 had the op-boundary kernels only).  Same comparison as
# test_greedy_decode_matches_oracle with FT = f16 in the product (embedding, weights' scales / zeros, qkv, cache, attention output)
# and in the oracle (DecoderOracle(ft="f16")): context phase through the fused entries at M = prompt length (general kernel),
# decode steps on the GEMV kernels (M <= 4) and, at batch 17, the general kernel.  f16 carries 11 bits against bf16's 8: the bound
# is the north star's 1e-2 of the logit scale with room to spare (measured: ~1e-3).
@pytest.mark.parametrize("shape,wbits,group,kv_mode,batch,graph", [
    (SMALL, 4, 128, "none", 1, True),      # GEMV kernels, Rotary + append + attention in one launch, hipGraph
    (SMALL, 8, -1, "none", 3, False),      # int8 per-channel
    (SMALL, 4, 128, "i8", 2, False),       # quantising append + the int8-cache attention kernels
    (WIDE, 8, 128, "none", 4, False),      # int8 sub-channel at M = 4
    (WIDE, 4, 128, "u4", 17, False),       # M > 4: small-batch kernels (f16 since round 5) with the fused norm, f16 + uint4 cache (VALU attention kernel)
    (WIDE, 4, 128, "i8", 32, True),        # batch 32, int8 cache, captured graph: FRAG32 chain in f16
    (WIDE, 8, -1, "none", 9, False),       # int8 per-channel, 16-bit cache
])
def test_f16_greedy_decode_matches_oracle(pkg, shape, wbits, group, kv_mode, batch, graph):
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("test-f16", **shape)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group), seed=1357, keep_fp=True, dtype=torch.float16)
    steps = 5
    rng = np.random.default_rng(batch * 3 + wbits)
    prompts = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in rng.integers(1, 12, batch)]
    sess = decoder.DecodeSession(model, batch, max_len=40, span_len=16, kv_mode=kv_mode)
    assert sess.logits.dtype == torch.float32 and sess.qkv.dtype == torch.float16
    lo0 = sess.prefill(prompts).cpu().numpy()
    gpu_ids = [sess.ids.cpu().numpy().copy()]
    gpu_logits = []
    if graph:
        sess.capture(warmup=0)
    for _ in range(steps):
        if graph:
            sess.replay()
        else:
            sess.step()
        torch.cuda.synchronize()
        gpu_logits.append(sess.logits.cpu().numpy().copy())
        gpu_ids.append(sess.ids.cpu().numpy().copy())
    ref = oracle_of(model, kv_mode)
    assert ref.ft == "f16"
    lo = ref.prefill(prompts)
    worst, decided = 0.0, 0
    tol_unit = 2e-2 if kv_mode == "u4" else 1e-2
    for t in range(steps + 1):
        g = lo0 if t == 0 else gpu_logits[t - 1]
        tol = tol_unit * max(1.0, float(np.abs(lo).max()))
        err = float(np.abs(g - lo).max())
        worst = max(worst, err)
        assert err <= tol, f"step {t}: logits differ by {err:.3e} (max |logit| {np.abs(lo).max():.2f})"
        top2 = np.sort(lo, axis=-1)[:, -2:]
        sure = (top2[:, 1] - top2[:, 0]) > 2 * max(err, 1e-4)
        assert np.array_equal(gpu_ids[t][sure], glue.greedy(lo)[sure]), f"step {t}: greedy token IDs differ"
        decided += int(sure.sum())
        if t < steps:
            lo = ref.step(gpu_ids[t])
    assert decided >= (steps + 1) * batch // 2
    print(f"f16 int{wbits} kv {kv_mode} batch {batch}: worst logit error {worst:.2e}; {decided}/{(steps + 1) * batch} decisive greedy choices")


@pytest.mark.parametrize("lens", [[70, 64, 3, 130, 200], [63, 90, 64]])
@pytest.mark.parametrize("wbits,group,kv_mode", [(4, 128, "none"), (8, -1, "u4")])
def test_prompts_that_share_products_equal_prompts_alone(pkg, wbits, group, kv_mode, lens):
    """Prompts of 64 rows and more share the products (f32 sums in another order: logits within the tolerance of this file, at the same tokens wherever the margin
    exceeds it); one below runs alone, to the bit."""
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("prompts-test", **SMALL)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group), seed=77, keep_fp=True)
    rng = np.random.default_rng(len(lens))
    prompts = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in lens]
    both = decoder.DecodeSession(model, len(lens), max_len=256, span_len=16, kv_mode=kv_mode)
    got, ids = both.prefill(prompts).clone(), both.ids.cpu().tolist()
    both.step()
    torch.cuda.synchronize()
    for b, p in enumerate(prompts):
        one = decoder.DecodeSession(model, 1, max_len=256, span_len=16, kv_mode=kv_mode)
        want = one.prefill([p])[0].clone()
        if len(p) < 64:
            assert torch.equal(got[b], want)
        tol = LOGIT_TOL[kv_mode] * max(1.0, float(want.abs().max()))
        assert float((got[b] - want).abs().max()) <= tol
        top = torch.topk(want, 2).values
        if float(top[0] - top[1]) > 2 * tol:
            assert ids[b] == int(want.argmax())
            one.step()                             # reads what the prompt left in the spans
            torch.cuda.synchronize()
            assert float((both.logits[b] - one.logits[0]).abs().max()) <= 2 * tol


@pytest.mark.parametrize("first", ["side", "default"])
@pytest.mark.parametrize("how", ["step", "replay", "replay_steps", "set_state", "prefill"])
def test_steps_on_another_stream_wait_for_the_prompt(pkg, how, first):
    """prefill returns before the device has run it; what the session does next on another stream comes behind it all the same"""
    from dash_infer_amd import decoder
    cfg = decoder.ModelConfig("streams-test", **SMALL)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(4, 128), seed=81)
    prompt, other = [5, 6, 7, 8] * 10, [9, 3] * 20

    def run(busy):
        s = decoder.DecodeSession(model, 1, max_len=64, span_len=16)
        if how.startswith("replay"):
            s.set_state([0], [0])
            s.capture()
        s.prefill([other])
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(), torch.cuda.default_stream()]
        a, b = streams if first == "side" else streams[::-1]
        ids, lens = torch.tensor([3], device="cuda"), torch.tensor([17], dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            if busy:
                torch.cuda._sleep(200_000_000)      # (the prompt's launches stand behind this)
            s.prefill([prompt])
        if not busy:
            torch.cuda.synchronize()
        with torch.cuda.stream(b):
            if how == "prefill":
                s.prefill([other[:30]])
            elif how == "set_state":
                s.set_state(ids, lens)
                s.step()
            else:
                {"step": s.step, "replay": s.replay, "replay_steps": lambda: s.replay_steps(1)}[how]()
        torch.cuda.synchronize()
        return s.ids.tolist(), s.old_lens.tolist(), s.pool.pool.clone()
    want, got = run(False), run(True)
    assert got[:2] == want[:2] and torch.equal(got[2], want[2])


def test_next_token_of_a_prompt_whose_logits_hold_a_nan(pkg, monkeypatch):
    """torch.argmax's answer: the NaN's column, in one of two rows"""
    from dash_infer_amd import decoder, ops
    cfg = decoder.ModelConfig("nan-test", **SMALL)
    s = decoder.DecodeSession(decoder.build_random_model(cfg, decoder.QuantSpec(4, 128), seed=80), 2, max_len=64, span_len=16)
    head = ops.lm_head

    def with_nan(h, *a, out, **kw):
        head(h, *a, out=out, **kw)
        if out.data_ptr() == rows[0]:
            out[0, 77] = float("nan")
    real, rows = torch.empty, []

    def empty(*size, **kw):                     # (the first row of the logits that prefill makes)
        t = real(*size, **kw)
        if size[:2] == (2, cfg.vocab):
            rows.append(t.data_ptr())
        return t
    monkeypatch.setattr(ops, "lm_head", with_nan)
    monkeypatch.setattr(torch, "empty", empty)
    logits = s.prefill([[1, 2, 3], [4, 5]])
    assert len(rows) == 1 and s.ids.tolist() == [77, int(logits[1].argmax())]


@pytest.mark.parametrize("lens,rows", [([64] * 40, 4096),                     # one group of 40 prompts: more last rows than a streaming kernel takes
                                       ([100, 64, 92, 65, 191, 64, 300, 70], 256)])   # groups that end at, before and beyond the row limit; one prompt above it
def test_groups_of_prompts_at_the_row_limit(pkg, monkeypatch, lens, rows):
    from dash_infer_amd import decoder
    monkeypatch.setattr(decoder.DecodeSession, "PREFILL_ROWS", rows)
    cfg = decoder.ModelConfig("prompt-groups-test", **SMALL)
    model = decoder.build_random_model(cfg, decoder.QuantSpec(4, 128), seed=79)
    rng = np.random.default_rng(rows)
    prompts = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in lens]
    both = decoder.DecodeSession(model, len(lens), max_len=320, span_len=16)
    got = both.prefill(prompts).clone()
    both.step()
    for b in range(0, len(lens), 1 if len(lens) < 10 else 7):
        one = decoder.DecodeSession(model, 1, max_len=320, span_len=16)
        want = one.prefill([prompts[b]])[0].clone()
        tol = LOGIT_TOL["none"] * max(1.0, float(want.abs().max()))
        assert float((got[b] - want).abs().max()) <= tol
        top = torch.topk(want, 2).values
        if float(top[0] - top[1]) > 2 * tol:
            one.step()                                 # reads what the prompt left in the spans
            torch.cuda.synchronize()
            assert float((both.logits[b] - one.logits[0]).abs().max()) <= 2 * tol


@pytest.mark.parametrize("lens,experts,top_k", [([200, 100, 56, 200, 70], 16, 8),    # 256 rows fill the grouped launches: three prompts, then two
                                                ([64] * 64, 16, 16)])                # together 65536 slots, more than one launch takes
def test_expert_prompts_share_products_within_the_grouped_launches(pkg, lens, experts, top_k):
    """Prompts whose (row, choice) slots fit the grouped expert launches alone but not together: served, and equal to the prompts alone within this file's tolerance."""
    from dash_infer_amd import decoder, ops
    cfg = decoder.ModelConfig("moe-prompts-test", **MOE_SMALL, moe=decoder.MoEConfig(experts, top_k, 256))
    model = decoder.build_random_model(cfg, decoder.QuantSpec(8, -1), seed=78)
    for grp in decoder.prompt_groups(lens, decoder.DecodeSession.PREFILL_ROWS, top_k):
        assert sum(lens[b] for b in grp) * top_k <= ops.MOE_GROUP_MAX_SLOTS
    rng = np.random.default_rng(len(lens))
    prompts = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in lens]
    got = decoder.DecodeSession(model, len(lens), max_len=256, span_len=16).prefill(prompts)
    for b in (0, 1, len(lens) // 2, len(lens) - 1):
        want = decoder.DecodeSession(model, 1, max_len=256, span_len=16).prefill([prompts[b]])[0]
        assert float((got[b] - want).abs().max()) <= LOGIT_TOL["none"] * max(1.0, float(want.abs().max()))
