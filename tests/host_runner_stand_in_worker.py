"""One scenario of tests/test_host_runner_cpu.py: a rank of the C++ operator layer over the stand-in of the HIP runtime (tests/host_runtime_stand_in.cpp), in a process that
never loads another one.  usage: host_runner_stand_in_worker.py <stand-in library> <scenario> <rank> <nranks> <batch> <wbits> <graph>; prints one JSON object."""
import ctypes as C
import json
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.modules["torch"] = None          # torch brings a HIP runtime of its own
FAKE = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
FAKE.stand_in_log.restype = C.c_size_t
FAKE.stand_in_block.restype = C.c_void_p
FAKE.stand_in_block.argtypes = [C.c_size_t]
from __graft_entry__ import _load_pkg  # noqa: E402

_load_pkg()
from dash_infer_amd import capi, hostapi, ref_graph  # noqa: E402

scenario, rank, nranks, batch, wbits, graph = sys.argv[2], *(int(a) for a in sys.argv[3:8])
HIDDEN, LAYERS, HEAD, INTER, VOCAB, SPAN, MAX = 1024, 2, 128, 1024, 4096, 16, 32
HEADS, KV = (28, 4) if nranks == 8 else (8, 2)


class Array:
    """a numpy array with the three calls by which hostapi.Model takes a tensor"""

    def __init__(self, *shape, dtype=np.uint16):
        self.a = np.zeros(shape, dtype)
        self.shape = self.a.shape

    def dim(self):
        return self.a.ndim

    def data_ptr(self):
        return self.a.ctypes.data


def log():
    n = FAKE.stand_in_log(None, C.c_size_t(0))
    buf = C.create_string_buffer(n + 1)
    FAKE.stand_in_log(buf, C.c_size_t(n + 1))
    return [x for x in buf.value.decode().split("\n") if x]


def heads_of(rank):
    """query heads and KV heads of a rank; more ranks than KV heads: every KV head on several, its query heads shared out"""
    if nranks <= KV:
        return HEADS // nranks, KV // nranks
    rep, hpg = nranks // KV, HEADS // KV
    return hpg // rep + (1 if rank % rep < hpg % rep else 0), 1


n, g = heads_of(rank)
m = hostapi.Model(C.c_void_p(1), HEADS, KV, HEAD, SPAN, 0, max_batch=batch, max_len=MAX, rank=rank, nranks=nranks)
bufs = (C.c_void_p * nranks)()
for r in range(nranks):
    p = C.c_void_p()
    capi.check(capi.lib().dihip_p2p_ar_alloc(C.byref(p)), "alloc")
    bufs[r] = p.value
comm = C.c_void_p()
capi.check(capi.lib().dihip_p2p_ar_create(C.byref(comm), rank, nranks, bufs), "create")
ar_state = (C.c_uint * 3).from_address(FAKE.stand_in_block(12))     # its {epoch, done, error}
if nranks > 1:
    m.set_p2p_comm(comm)


def lowp(name, k, cols):
    m.set_weight(name + ".weight", Array(k, cols // 2 if wbits == 4 else cols, dtype=np.uint8 if wbits == 4 else np.int8), "u8" if wbits == 4 else "i8")
    for part in (".weight.scale", ".weight.zero_point"):
        m.set_weight(name + part, Array(k // 128 if wbits == 4 else 1, cols), "bf16")


m.set_weight("embedding.word_embeddings", Array(VOCAB, HIDDEN), "bf16")
for li in range(LAYERS):
    p = f"decoder.layer.{li}."
    m.set_weight(p + "attention.layernorm.gamma", Array(HIDDEN), "bf16")
    m.set_weight(p + "ffn.layernorm.gamma", Array(HIDDEN), "bf16")
    lowp(p + "attention.self", HIDDEN, (n + 2 * g) * HEAD)
    m.set_weight(p + "attention.self.bias", Array((n + 2 * g) * HEAD), "bf16")
    lowp(p + "attention.output.dense", n * HEAD, HIDDEN)
    lowp(p + "ffn.intermediate.dense", HIDDEN, INTER // nranks)
    lowp(p + "ffn.linear.dense", HIDDEN, INTER // nranks)
    lowp(p + "ffn.output.dense", INTER // nranks, HIDDEN)
m.set_weight("final.layernorm.gamma", Array(HIDDEN), "bf16")
m.set_weight("lm_head.weight", Array(HIDDEN // nranks, VOCAB), "bf16")
ref_graph.add_graph(m, ref_graph.qwen2_graph(LAYERS, wbits, 128 if wbits == 4 else -1, 1e-6, HEADS, KV, 1e6, tp_allreduce=nranks > 1, tp_lm_head=nranks > 1))
rep = m.graph_build(fuse=True)
assert rep["fused"] and rep["device_resident"], rep["why"]
spr = MAX // SPAN
page = [Array(SPAN * g * HEAD) for _ in range(2 * batch * LAYERS * spr)]
at = iter(page)
for b in range(batch):
    ks, vs = ([[next(at).data_ptr() for _ in range(spr)] for _ in range(LAYERS)] for _ in range(2))
    m.request_adopt(3, 5, ks, vs)

if scenario == "prepare":
    m.decode_prepare(graph=bool(graph))
    FAKE.stand_in_clear()
    m.decode_steps(1, graph=bool(graph))
    first = log()
    FAKE.stand_in_clear()
    m.decode_prepare(graph=bool(graph))      # (nothing left to prepare)
    again = log()
    m.decode_steps(2, graph=bool(graph))
    ids = m.sync_ids()
    print(json.dumps({"first": first, "again": again, "ids": len(ids)}))
elif scenario == "unprepared":
    FAKE.stand_in_clear()
    m.decode_steps(1, graph=bool(graph))
    print(json.dumps({"first": log()}))
elif scenario == "lost":
    m.decode_steps(2, graph=bool(graph))
    m.sync_ids()
    m.decode_steps(2, graph=bool(graph))
    ar_state[2] = 1
    try:
        m.sync_ids()
        err = ""
    except hostapi.HostError as e:
        err = str(e)
    e = C.c_int(0)
    capi.check(capi.lib().dihip_p2p_ar_error(comm, C.byref(e)), "error")
    ar_state[2] = 0
    m.decode_steps(1, graph=bool(graph))     # the lengths are back where the last good synchronise left them
    print(json.dumps({"err": err, "word": e.value, "after": len(m.sync_ids())}))
sys.stdout.flush()
os._exit(0)      # (no destructors: the stand-in keeps every block)
