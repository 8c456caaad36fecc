"""Library of the tensor-parallel loop-back tests (tests/test_gpu_tp_loopback.py, tests/p2p_worker.py): the ranks of a TP
group as threads of one process on one GPU.  See test_gpu_tp_loopback.py."""
import os
import threading

import numpy as np
import torch



SETUP_LOCK = threading.Lock()


class LoopbackComm:
    """Collectives between threads of one process on one device.  All ranks enqueue on the same (default) stream, so a
    host-side barrier between "producers enqueued" and "consumers enqueued" is all the ordering the data needs."""

    class Shared:
        def __init__(self, n):
            self.slots = [None] * n
            self.bar = threading.Barrier(n)

    def __init__(self, shared, rank, nranks):
        self.sh, self.rank, self.nranks = shared, rank, nranks

    def allreduce_(self, t):
        self.sh.slots[self.rank] = t
        self.sh.bar.wait()
        total = torch.stack([self.sh.slots[r] for r in range(self.nranks)]).sum(0)  # fixed rank order on every rank
        self.sh.bar.wait()      # every rank has enqueued its sum before any rank enqueues the overwrite below
        t.copy_(total)
        return t

    def allgather(self, src, dst):
        self.sh.slots[self.rank] = src
        self.sh.bar.wait()
        gathered = torch.cat([self.sh.slots[r].reshape(-1) for r in range(self.nranks)])
        self.sh.bar.wait()
        dst.view(-1).copy_(gathered)
        return dst


class LoopbackP2PComm:
    """The product's one-shot peer-to-peer all-reduce (dihip_p2p_allreduce_sum) between rank THREADS: every rank owns a
    receive buffer and a stream, the "peers' IPC pointers" are the plain device pointers of the other threads' buffers.
    The kernels of the ranks run concurrently and really wait for one another's flags.  All-gather stays a host loop-back."""
    backend = "p2p-oneshot(loop-back)"

    class Shared:
        def __init__(self, n):
            import ctypes as C
            from dash_infer_amd.capi import check, lib
            self.n = n
            self.bufs = []
            for _ in range(n):
                p = C.c_void_p()
                check(lib().dihip_p2p_ar_alloc(C.byref(p)), "p2p alloc")
                self.bufs.append(p)
            self.slots = [None] * n
            self.bar = threading.Barrier(n)

        def close(self):
            from dash_infer_amd.capi import lib
            for p in self.bufs:
                lib().dihip_p2p_ar_free(p)

    def __init__(self, shared, rank, nranks):
        import ctypes as C
        from dash_infer_amd.capi import check, lib
        self.sh, self.rank, self.nranks = shared, rank, nranks
        ptrs = (C.c_void_p * nranks)(*[b.value for b in shared.bufs])
        self.handle = C.c_void_p()
        check(lib().dihip_p2p_ar_create(C.byref(self.handle), rank, nranks, ptrs), "p2p create")

    def allreduce_(self, t):
        from dash_infer_amd import ops
        from dash_infer_amd.capi import check, lib
        check(lib().dihip_p2p_allreduce_sum(self.handle, ops.cur_stream(), ops.ptr(t), ops.ptr(t), t.numel(), ops.dt_code(t)), "p2p ar")
        return t

    def allgather(self, src, dst):
        torch.cuda.current_stream().synchronize()
        self.sh.slots[self.rank] = src
        self.sh.bar.wait()
        gathered = torch.cat([self.sh.slots[r].reshape(-1) for r in range(self.nranks)])
        dst.view(-1).copy_(gathered)
        torch.cuda.current_stream().synchronize()
        self.sh.bar.wait()
        return dst


def run_p2p_allreduce(nranks):
    """dihip_p2p_allreduce_sum: sums of bf16 / f16 / f32 rows of decode sizes (one 7 KB row ... the slot limit), in place and
    out of place, many back-to-back calls (the two slot sets alternate; the epoch lives on the device), identical bits on
    every rank; over-long and misaligned messages are refused."""
    import ctypes as C
    from dash_infer_amd import ops
    from dash_infer_amd.capi import DihipError, check, lib
    shared = LoopbackP2PComm.Shared(nranks)
    results, errors = [None] * nranks, []
    cases = [(torch.bfloat16, 3584), (torch.float32, 3584), (torch.float16, 4 * 3584), (torch.bfloat16, 32 * 3584), (torch.float32, 8),
             (torch.bfloat16, 4), (torch.float32, 65536)]

    def worker(rank):
        try:
            torch.cuda.set_device(0)
            comm = LoopbackP2PComm(shared, rank, nranks)
            st = torch.cuda.Stream()
            outs = []
            with torch.cuda.stream(st):
                for rep in range(3):
                    for ci, (dt, n) in enumerate(cases):
                        g = torch.Generator(device="cuda").manual_seed(1000 * rep + 10 * ci + rank)
                        x = torch.randn(n, generator=g, device="cuda", dtype=torch.float32).to(dt)
                        y = x.clone()
                        comm.allreduce_(y)
                        outs.append((rep, ci, x, y))
                st.synchronize()
                too_big = torch.zeros(int(lib().dihip_p2p_ar_max_bytes()) // 2 + 4, dtype=torch.bfloat16, device="cuda")
                for bad in (too_big, torch.zeros(6, dtype=torch.bfloat16, device="cuda")):  # too long; 12 bytes: not whole words
                    try:
                        comm.allreduce_(bad)
                    except DihipError:
                        continue
                    raise AssertionError("an over-long / misaligned message was accepted")
            results[rank] = [(rep, ci, x.float().cpu(), y.cpu()) for rep, ci, x, y in outs]
        except Exception as e:  # noqa: BLE001
            errors.append((rank, repr(e)))
            shared.bar.abort()

    threads = [threading.Thread(target=worker, args=(r,)) for r in range(nranks)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=120)
    shared.close()
    assert not errors, errors
    for k in range(len(results[0])):
        rep, ci, _, y0 = results[0][k]
        want = sum(results[r][k][2] for r in range(nranks))  # f32 sum in rank order, as the kernel does
        dt = cases[ci][0]
        assert torch.equal(y0.float(), want.to(dt).float()), (rep, ci)
        for r in range(1, nranks):
            assert torch.equal(results[r][k][3], y0), f"rank {r} differs (case {ci}, repetition {rep})"


def run_tp_decode(nranks, kv_mode, batch, wbits, group, comm_kind, overlap, moe=False, lm_head_split=None):
    import os
    from dash_infer_amd import decoder
    os.environ["DIHIP_TP_OVERLAP"] = "1" if overlap else "0"
    # inter = 8 groups of 128 -> 2 per rank at TP = 4; n = 8, g = 2: TP = 4 puts every KV head on two ranks (2 + 2 query heads)
    cfg = decoder.ModelConfig("tp-test", hidden=1024, layers=2, n_heads=8, n_kv=2, head_dim=128, inter=1024, vocab=4096)
    if nranks == 8:  # 28 query / 4 KV heads: every KV head on two ranks with 4 + 3 query heads (tp.shard_heads)
        cfg = decoder.ModelConfig("tp8-test", hidden=1024, layers=2, n_heads=28, n_kv=4, head_dim=128, inter=1024, vocab=4096)
    if moe:  # mixture-of-experts layers, expert parallel: 8 routed experts (top-2) over the ranks + the shared expert's slices
        cfg = decoder.ModelConfig("tp-moe-test", hidden=1024, layers=2, n_heads=8, n_kv=2, head_dim=128, inter=1024, vocab=4096,
                                  moe=decoder.MoEConfig(8, 2, 256))
    spec = decoder.QuantSpec(wbits, group)
    steps = 5
    rng = np.random.default_rng(nranks * 31 + batch)
    ids0 = rng.integers(0, cfg.vocab, batch)

    def run_single():
        model = decoder.build_random_model(cfg, spec, seed=99)
        sess = decoder.DecodeSession(model, batch, max_len=32, span_len=16, kv_mode=kv_mode)
        sess.set_state(ids0, [0] * batch)
        out = []
        for _ in range(steps):
            sess.step()
            torch.cuda.synchronize()
            out.append((sess.logits.cpu().numpy().copy(), sess.ids.cpu().numpy().copy()))
        return out

    ref = run_single()
    p2p = comm_kind == "p2p"
    shared = (LoopbackP2PComm if p2p else LoopbackComm).Shared(nranks)
    results = [None] * nranks
    errors = []

    def worker(rank):
        try:
            torch.cuda.set_device(0)
            model = decoder.build_random_model(cfg, spec, seed=99, rank=rank, nranks=nranks, lm_head_split=lm_head_split)
            comm = (LoopbackP2PComm if p2p else LoopbackComm)(shared, rank, nranks)
            # P2P: the ranks' kernels wait for one another, so every rank needs a stream of its own
            st = torch.cuda.Stream() if p2p else torch.cuda.current_stream()
            with torch.cuda.stream(st):
                # Session set-up is serialised between the rank threads: eight threads issuing small pageable host-to-device
                # copies on one device at once corrupted the first element of a copy now and then (row 0 of step 0 only --
                # a property of this many-ranks-in-one-process harness, not of the product: a rank is a process)
                with SETUP_LOCK:
                    sess = decoder.DecodeSession(model, batch, max_len=32, span_len=16, kv_mode=kv_mode, comm=comm)
                    assert sess.ar_overlap == overlap
                    sess.set_state(ids0, [0] * batch)
                    torch.cuda.synchronize()
                    assert sess.ids.cpu().tolist() == [int(i) for i in ids0] and sess.old_lens.cpu().tolist() == [0] * batch
                shared.bar.wait()
                out = []
                for _ in range(steps):
                    sess.step()
                    torch.cuda.synchronize()
                    out.append((sess.logits.cpu().numpy().copy(), sess.ids.cpu().numpy().copy()))
                    shared.bar.wait()  # keep the ranks in step (a rank may not start the next step's collectives early)
            results[rank] = out
        except Exception as e:  # noqa: BLE001
            errors.append((rank, repr(e)))
            shared.bar.abort()

    threads = [threading.Thread(target=worker, args=(r,)) for r in range(nranks)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=300)
    if p2p:
        shared.close()
    assert not errors, errors
    assert all(r is not None for r in results)
    tol = 6e-2 if kv_mode == "u4" else 1e-2
    if moe:
        # the ranks' partial MoE outputs and partial shared-expert outputs are FT tensors (the operators' outputs, as in the
        # reference, which all-reduces exactly those): two / four bf16 roundings of partial sums where the single rank has
        # one of the whole sum.  Measured 0.6e-2 ... 1.3e-2 on logits of magnitude ~3.
        tol = 2.5e-2
    for t in range(steps):
        if lm_head_split == "k":
            # the reference's K-split lm_head + logits all-reduce (model_base.py:690-703): EVERY rank holds the full logits row
            logits = results[0][t][0]
            assert logits.shape[1] == cfg.vocab
            for r in range(1, nranks):
                assert np.array_equal(results[r][t][0], logits), f"rank {r}: the all-reduced logits row differs from rank 0's"
        else:
            logits = np.concatenate([results[r][t][0] for r in range(nranks)], axis=1)  # vocabulary-parallel slices
        ids_tp = results[0][t][1]
        for r in range(1, nranks):
            assert np.array_equal(results[r][t][1], ids_tp)            # every rank holds the same next token
        ref_logits, ref_ids = ref[t]
        if os.environ.get("DIHIP_TP_TEST_VERBOSE"):
            print("step", t, "row max err", np.abs(logits - ref_logits).max(axis=1), "ids", ids_tp, ref_ids, flush=True)
        np.testing.assert_allclose(logits, ref_logits, rtol=0, atol=tol)
        top2 = np.sort(ref_logits, axis=-1)[:, -2:]
        sure = (top2[:, 1] - top2[:, 0]) > 2 * tol
        assert np.array_equal(ids_tp[sure], ref_ids[sure])
        if not np.array_equal(ids_tp, ref_ids):
            break  # a near-tie resolved differently: the sequences part here, nothing further to compare


def write_model_asparam(path, model, n_heads, n_kv, head_dim, group, tp_lm_head=True):
    """The WHOLE model (decoder.build_random_model(keep_fp=True), one rank) as a serialized weight file the way the reference's converter
    exports it for tensor parallelism -- names of ref_graph.register_weights, SplitModes and group_lists of qwen_v15.py:130-165, 540-569 /
    model_base.py:690-703 -- written by the REFERENCE'S OWN writer (oracle/_ref/libdashinfer_ref_asparam.so, tests/golden/make_asparam_golden.py)."""
    import importlib.util
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    spec = importlib.util.spec_from_file_location("make_asparam_golden", os.path.join(root, "tests", "golden", "make_asparam_golden.py"))
    mk = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mk)
    NOSPLIT, VSPLIT, HSPLIT, GROUP_VSPLIT = 0, 1, 2, 6
    fp = model.fp
    w4 = model.quant.wbits == 4
    recs = []

    def host(t):
        t = t.detach().cpu().contiguous()
        if t.dtype == torch.bfloat16:
            return t.view(torch.int16).numpy().view(np.uint16), True
        return t.numpy(), False

    def put(name, t, mode, groups=()):
        a, bf = host(t)
        recs.append((name, a, mode, bf, list(groups)))

    def lowp(name, qsz, mode, groups=()):
        q, s, z = qsz
        put(name + ".weight", q, mode, [x // 2 for x in groups] if w4 else groups)
        # parameters of a row-split weight: sub-channel -> split along the groups, per-channel -> whole on every rank (qwen_v15.py:556-569)
        pmode = mode if (mode != HSPLIT or group > 0) else NOSPLIT
        put(name + ".weight.scale", s, pmode, groups)
        put(name + ".weight.zero_point", z, pmode, groups)

    qkv = [n_heads * head_dim, n_kv * head_dim, n_kv * head_dim]
    put("embedding.word_embeddings", fp["embed"], NOSPLIT)
    for li in range(len(model.layers)):
        p = f"decoder.layer.{li}."
        put(p + "attention.layernorm.gamma", fp[li]["ln1"], NOSPLIT)
        put(p + "ffn.layernorm.gamma", fp[li]["ln2"], NOSPLIT)
        lowp(p + "attention.self", fp[li]["qkv"], GROUP_VSPLIT, qkv)
        put(p + "attention.self.bias", fp[li]["qkv_bias"], GROUP_VSPLIT, qkv)
        lowp(p + "attention.output.dense", fp[li]["o"], HSPLIT)
        lowp(p + "ffn.intermediate.dense", fp[li]["gate"], VSPLIT)
        lowp(p + "ffn.linear.dense", fp[li]["up"], VSPLIT)
        lowp(p + "ffn.output.dense", fp[li]["down"], HSPLIT)
    put("final.layernorm.gamma", fp["final_norm"], NOSPLIT)
    put("lm_head.weight", fp["lm_head"], HSPLIT if tp_lm_head else VSPLIT)
    mk.write(path, recs)
    return len(recs)


def run_tp_decode_host(nranks, kv_mode, batch, wbits, group, weight_file=None, n_kv=2, return_results=False, graph=False):
    """Tensor-parallel decode through the C++ OPERATOR LAYER: one hostapi.Model (HIPContext with rank / nranks, the rank's one-shot
    P2P communicator) per rank THREAD, the reference's operator list with its AllReduce operators and the K-split lm_head
    (ref_graph.qwen2_graph(tp_allreduce=True, tp_lm_head=True): qwen_v15.py:187-388, model_base.py:690-703) -> fusion pass ->
    OpFactory(HIP) -> model runner, each rank over its own slices of the quantised weights (decoder.build_random_model(rank, nranks,
    keep_fp=True): GROUP_VSPLIT / HSPLIT / VSPLIT as the reference's splitters cut them) and its own share of the KV heads.  Every rank
    must hold the SAME all-reduced logits row and the same next token; both must match the single-rank DecodeSession (the row-parallel
    layers only change the f32 summation order; the TP tail's logits are FT: tolerance 2^-7 of the logit scale).  The reference runs a
    thread per rank in one process as well (as_engine.cpp:243-286)."""
    from dash_infer_amd import decoder, hostapi, ops, ref_graph, tp
    cfg = decoder.ModelConfig("tp-host-test", hidden=1024, layers=2, n_heads=8, n_kv=n_kv, head_dim=128, inter=1024, vocab=4096)
    if nranks == 8:
        cfg = decoder.ModelConfig("tp8-host-test", hidden=1024, layers=2, n_heads=28, n_kv=4, head_dim=128, inter=1024, vocab=4096)
    spec = decoder.QuantSpec(wbits, group)
    steps, span, max_len = 5, 16, 32
    rng = np.random.default_rng(nranks * 37 + batch)
    ids0 = [int(t) for t in rng.integers(0, cfg.vocab, batch)]
    model1 = decoder.build_random_model(cfg, spec, seed=99)
    sess = decoder.DecodeSession(model1, batch, max_len=max_len, span_len=span, kv_mode=kv_mode)
    sess.set_state(ids0, [0] * batch)
    ref = []
    for _ in range(steps):
        sess.step()
        torch.cuda.synchronize()
        ref.append((sess.logits.cpu().numpy().copy(), sess.ids.cpu().numpy().copy()))
    del sess, model1
    shared = LoopbackP2PComm.Shared(nranks)
    results, errors, reports = [None] * nranks, [], [None] * nranks
    KV = {"none": 0, "i8": 1, "u4": 2}
    nl, spr = cfg.layers, (max_len + span - 1) // span

    def worker(rank):
        try:
            torch.cuda.set_device(0)
            # weight_file: the rank's tensors come from ONE export of the whole model, split at load by the C++ layer (dihost_weights_load_file:
            # the reference's WeightSplitter rules); else from decoder.build_random_model's own tp.py slices, bound as tensors
            model = None if weight_file else decoder.build_random_model(cfg, spec, seed=99, rank=rank, nranks=nranks, keep_fp=True, lm_head_split="k")
            comm = LoopbackP2PComm(shared, rank, nranks)
            g_loc = len(tp.shard_heads(cfg.n_heads, cfg.n_kv, nranks)[rank].kv_heads)
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                with SETUP_LOCK:
                    pool = ops.SpanPool(2 * batch * nl * spr + 4, g_loc, span, cfg.head_dim, kv_mode, torch.bfloat16)
                    m = hostapi.Model(ops.cur_stream(), cfg.n_heads, cfg.n_kv, cfg.head_dim, span, KV[kv_mode], max_batch=batch, max_len=max_len,
                                      rank=rank, nranks=nranks)
                    m.set_p2p_comm(comm.handle)
                    if weight_file:
                        assert m.load_weight_file(weight_file) > 0
                    else:
                        ref_graph.register_weights(m, model)
                    ref_graph.add_graph(m, ref_graph.qwen2_graph(nl, wbits, group, cfg.eps, cfg.n_heads, cfg.n_kv, cfg.rope_theta,
                                                                 tp_allreduce=True, tp_lm_head=True))
                    reports[rank] = m.graph_build(fuse=True)
                    for b in range(batch):
                        ks = [[pool.alloc()[0] for _ in range(spr)] for _ in range(nl)]
                        vs = [[pool.alloc()[0] for _ in range(spr)] for _ in range(nl)]
                        m.request_adopt(0, ids0[b], ks, vs)
                    torch.cuda.synchronize()
                shared.bar.wait()
                # operators reshaped and the step captured BEFORE any rank launches one: growing a tensor frees the old one, and hipFree waits for everything on
                # the device, so also for the all-reduce of a peer that is waiting for this rank.  One rank at a time, when no other synchronises the device: a
                # capture in progress does not survive that
                with SETUP_LOCK:
                    m.decode_prepare(graph=graph)
                    st.synchronize()
                shared.bar.wait()
                out = []
                for _ in range(steps):
                    m.decode_steps(1, graph=graph)   # graph: every rank thread captures its step once (its all-reduce launches inside) and replays it
                    ids = m.sync_ids()
                    _, shp, ptr = m.get_tensor("logits")
                    st.synchronize()
                    out.append((_view_bf16(ptr, shp).float().cpu().numpy().reshape(-1, shp[-1]).copy(), np.array(ids)))
                    shared.bar.wait()
                m.close()
            results[rank] = out
        except Exception as e:  # noqa: BLE001
            import traceback
            errors.append((rank, repr(e), traceback.format_exc()[-1500:]))
            shared.bar.abort()

    threads = [threading.Thread(target=worker, args=(r,)) for r in range(nranks)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=300)
    shared.close()
    assert not errors, errors
    assert all(r is not None for r in results)
    assert all(rep["fused"] and rep["device_resident"] for rep in reports), [rep["why"] for rep in reports]
    for t in range(steps):
        logits, ids_tp = results[0][t]
        assert logits.shape[1] == cfg.vocab
        for r in range(1, nranks):
            assert np.array_equal(results[r][t][0], logits), f"step {t}: rank {r} holds another logits row than rank 0"
            assert np.array_equal(results[r][t][1], ids_tp), f"step {t}: rank {r} chose another token"
        ref_logits, ref_ids = ref[t]
        scale = max(1.0, float(np.abs(ref_logits).max()))
        tol = (6e-2 if kv_mode == "u4" else 1e-2) + 2.0 ** -7 * scale
        np.testing.assert_allclose(logits, ref_logits, rtol=0, atol=tol, err_msg=f"step {t}")
        top2 = np.sort(ref_logits, axis=-1)[:, -2:]
        sure = (top2[:, 1] - top2[:, 0]) > 2 * tol
        assert np.array_equal(ids_tp[sure], ref_ids[sure]), f"step {t}: greedy ids"
        if not np.array_equal(ids_tp, ref_ids):
            break
    print(f"[host TP loop-back] nranks {nranks}, batch {batch}, kv {kv_mode}{', hipGraph replay' if graph else ''}{', weights split at load from ' + weight_file if weight_file else ''}: "
          f"{reports[0]['ops']} operators, logits within tolerance, ids equal", flush=True)
    if return_results:
        return results


def run_tp_decode_host_from_file(nranks, kv_mode, batch, wbits, group, n_kv, which, out_path):
    """ONE serialized export of the whole model (written by the reference's own writer with the
    converter's SplitModes and group_lists) feeds every rank of a TP group -- each rank's C++ model splits the records for itself at load
    (dihost_weights_load_file: host/weight_file.h SliceForRank = the reference's WeightSplitter rules).  The decode must be BIT-IDENTICAL
    to the same ranks bound to dash-infer_amd/tp.py's slices as tensors, logits row and tokens, every step, every rank.
    which = "file" | "bound": ONE variant per process (rank threads of two runs in one process can end up sharing a hardware queue,
    and a rank that waits for a peer queued behind it never returns); every rank's (logits, ids) of every step -> out_path (.npz)."""
    import os
    import tempfile
    from dash_infer_amd import decoder
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    if which == "file" and not os.path.exists(os.path.join(root, "oracle", "_ref", "libdashinfer_ref_asparam.so")):
        print("[host TP from file] oracle/_ref/libdashinfer_ref_asparam.so not built: skipped", flush=True)
        return
    with tempfile.TemporaryDirectory() as d:
        path = None
        if which == "file":
            cfg = decoder.ModelConfig("tp-host-test", hidden=1024, layers=2, n_heads=8, n_kv=n_kv, head_dim=128, inter=1024, vocab=4096)
            whole = decoder.build_random_model(cfg, decoder.QuantSpec(wbits, group), seed=99, keep_fp=True)
            path = os.path.join(d, "whole_model.asparam")
            n = write_model_asparam(path, whole, cfg.n_heads, cfg.n_kv, cfg.head_dim, group)
            del whole
            print(f"[host TP from file] {n} records written by the reference's writer", flush=True)
        res = run_tp_decode_host(nranks, kv_mode, batch, wbits, group, weight_file=path, n_kv=n_kv, return_results=True)
    np.savez(out_path, **{f"r{r}_t{t}_{k}": v for r in range(nranks) for t, (lo, ids) in enumerate(res[r]) for k, v in (("logits", lo), ("ids", ids))})


def _view_bf16(ptr, shape):
    """a torch view of device memory the C++ layer owns (tests/test_gpu_host_runner.py: view_of)"""
    from tests.test_gpu_host_graph import view_of
    return view_of(ptr, shape, torch.bfloat16)
