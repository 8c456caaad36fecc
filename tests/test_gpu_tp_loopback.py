"""Tensor-parallel decode on ONE GPU: the ranks of a TP group run as threads of this process, each with its own
DecodeSession over its tp.py shard (real packed weights, real kernels at the odd per-rank shapes), and a loop-back
communicator stands in for RCCL (sum all-reduce of the hidden rows after the o and down projections, all-gather of the
per-rank arg-max pairs; the RCCL wrappers themselves need more than one GPU).
The greedy tokens and the vocabulary-parallel logits must match the single-rank session: the row-parallel layers only
change the f32 summation order.  Covers whole KV heads per rank (TP = 2) and a KV head replicated on two ranks with its
query heads split (TP = 4 at g = 2: the case the reference refuses, head_gqa.h:29-49) -- what `bench.py --gpus N` runs.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_worker(*args, timeout=600, env_extra=None):
    """The peer-to-peer scenarios run in a process of their own: the ranks' kernels WAIT for one another, so every rank's
    stream needs its own hardware queue -- GPU_MAX_HW_QUEUES (default 4, read when HIP initialises) is raised for that
    process only.  (On a node every rank has a GPU to itself.)  A worker that fails is not started again."""
    env = dict(os.environ, GPU_MAX_HW_QUEUES="32", HSA_ENABLE_IPC_MODE_LEGACY="0", **(env_extra or {}))
    r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "p2p_worker.py")] + [str(a) for a in args], env=env, cwd=ROOT,
                       capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0 and "P2P_WORKER_OK" in r.stdout, (r.stdout[-2000:], r.stderr[-3000:])


@pytest.mark.parametrize("nranks", [2, 4, 8])
def test_p2p_allreduce_between_rank_threads(pkg, nranks):
    """dihip_p2p_allreduce_sum: sums of bf16 / f16 / f32 rows of decode sizes (one 7 KB row ... the slot limit), in place,
    many back-to-back calls (the two slot sets alternate; the epoch lives on the device), identical bits on every rank;
    over-long and misaligned messages are refused."""
    run_worker("allreduce", nranks)


@pytest.mark.parametrize("nranks,kv_mode,batch,wbits,group,comm_kind,overlap", [
    (2, "none", 1, 4, 128, "host", False), (4, "none", 2, 4, 128, "host", False), (4, "u4", 5, 8, -1, "host", False),
    (2, "i8", 32, 4, 128, "host", False),
    (8, "none", 1, 4, 128, "host", False),    # Qwen2-7B head geometry at TP = 8: 28 / 4 heads -> 4 + 3 query heads per KV-head replica
    (8, "none", 2, 4, 128, "p2p", False),     # the same through the product's one-shot P2P all-reduce (rank threads, own streams)
    (4, "none", 1, 4, 128, "p2p", True),      # all-reduce on a side stream between events, weight prefetch beside it
    (2, "i8", 3, 8, -1, "host", True),
    (2, "none", 2, 8, -1, "host-moe", False),  # mixture-of-experts layers under expert parallelism (4 of 8 experts per rank)
    (4, "none", 1, 4, 128, "host-moe", False),
    # the reference-shaped lm_head under TP: K-split Gemm + all-reduce of the partial logits (model_base.py:690-703,
    # gemm_op.cpp:95-98) -- every rank holds the FULL f32 logits row, equal to the single rank's
    (2, "none", 2, 4, 128, "host-ksplit", False),
    (4, "i8", 1, 8, -1, "host-ksplit", False),
])
def test_tp_decode_matches_single_rank(pkg, monkeypatch, nranks, kv_mode, batch, wbits, group, comm_kind, overlap):
    if comm_kind == "p2p":
        run_worker("decode", nranks, kv_mode, batch, wbits, group, int(overlap))
        return
    from tests import tp_loopback_lib
    monkeypatch.setenv("DIHIP_TP_OVERLAP", "1" if overlap else "0")
    moe = comm_kind.endswith("-moe")
    tp_loopback_lib.run_tp_decode(nranks, kv_mode, batch, wbits, group, comm_kind.split("-")[0], overlap, moe=moe,
                                  lm_head_split="k" if comm_kind.endswith("-ksplit") else None)


@pytest.mark.parametrize("nranks,kv_mode,batch,wbits,group,graph", [
    (2, "none", 1, 4, 128, False), (4, "none", 2, 4, 128, False), (8, "none", 1, 4, 128, False), (2, "i8", 3, 8, -1, False),
    # the step state is device-resident under TP too (DihipGreedy behind the K-split tail) -> every rank thread captures its step,
    # all-reduce launches included, and replays it; batch 1 (GEMV kernels) and batch 16 (small-batch GEMMs, the norm its own launch behind
    # the all-reduce), TP 2 / 4 / 8
    (2, "none", 1, 4, 128, True), (2, "none", 16, 4, 128, True), (4, "none", 1, 4, 128, True), (4, "none", 16, 4, 128, True),
    (8, "none", 1, 4, 128, True), (8, "none", 16, 4, 128, True), (2, "u4", 16, 8, -1, True)])
def test_tp_decode_through_the_cpp_operator_layer(pkg, nranks, kv_mode, batch, wbits, group, graph):
    """The C++ operator layer under tensor parallelism -- one model runner per rank THREAD in one process (as the
    reference's engine runs its ranks, as_engine.cpp:243-286), the reference's operator list with its AllReduce operators and the K-split
    lm_head, each rank on its own weight slices and KV heads, the product's one-shot P2P all-reduce between the threads' streams: every
    rank ends each step with the same all-reduced logits row and token, equal to the single-rank DecodeSession within the FT tail's
    tolerance (tests/tp_loopback_lib.py::run_tp_decode_host).  TP = 2 / 4 / 8 incl. the 4 + 3 query-head split of a replicated KV head."""
    run_worker("hostdecode", nranks, kv_mode, batch, wbits, group, "graph" if graph else "eager")


@pytest.mark.parametrize("nranks,kv_mode,batch,wbits,group,n_kv", [(2, "none", 1, 4, 128, 2), (4, "none", 2, 4, 128, 4), (2, "i8", 3, 8, -1, 2)])
def test_tp_ranks_split_one_serialized_export_at_load(pkg, tmp_path, nranks, kv_mode, batch, wbits, group, n_kv):
    """A whole-model .asparam written by the reference's writer (the converter's SplitModes + group_lists) ->
    dihost_weights_load_file on every rank of a TP 2 / 4 group splits it for that rank -> logits and tokens BIT-IDENTICAL to the ranks bound
    to tp.py's slices as tensors; int4 sub-channel (parameters split along the groups) and int8 per-channel (parameters whole).  One
    variant per worker process (tests/tp_loopback_lib.py run_tp_decode_host_from_file)."""
    import numpy as np
    if not os.path.exists(os.path.join(ROOT, "oracle", "_ref", "libdashinfer_ref_asparam.so")):
        pytest.skip("oracle/_ref/libdashinfer_ref_asparam.so not built (needs /root/reference: oracle/Makefile refasparam)")
    out = {}
    for which in ("bound", "file"):
        path = str(tmp_path / f"{which}.npz")
        run_worker("hostfile", nranks, kv_mode, batch, wbits, group, n_kv, which, path)
        out[which] = np.load(path)
    assert sorted(out["bound"].files) == sorted(out["file"].files) and len(out["file"].files) == nranks * 5 * 2
    for k in out["bound"].files:
        assert np.array_equal(out["bound"][k], out["file"][k]), f"{k}: split-at-load differs from the tensor-bound slices"


@pytest.mark.parametrize("nranks,batch,graph", [(2, 1, False), (2, 1, True), (4, 16, True)])
def test_allreduce_beside_the_next_weights_in_the_cpp_layer(pkg, nranks, batch, graph):
    """The all-reduce beside the next GEMM's weights, on a side HIP stream, in the C++ operator layer:
    with DIHIP_TP_OVERLAP=1 AllReduceOpHIP runs its collective on the context's side stream between two events while the main stream pulls
    the packed weights of the operator that reads the reduced rows on-die (HIPContext::ConsumerWeights + dihip_prefetch), then joins; under
    capture the events are a fork / join of the step's graph.  Same logits and tokens as without (the same sums in the same order)."""
    run_worker("hostdecode", nranks, "none", batch, 4, 128, "graph" if graph else "eager", env_extra={"DIHIP_TP_OVERLAP": "1"})
