"""GPU parity of the glue ops (RMSNorm, RoPE, Binary ADD, SiLU*MUL, embedding, step counter)
against oracle/glue.py (which restates csrc/core/kernel/cpu/layernorm.cpp:110-157 and
rotary.cpp:22-106)."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import glue
from oracle.numerics import bf16_round

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(pkg):
    from dash_infer_amd import ops as _ops
    assert torch.cuda.is_available()
    return _ops


def dev(a, dtype=torch.bfloat16):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dtype).cuda()


@pytest.mark.parametrize("rows,cols", [(1, 3584), (5, 896), (32, 1000)])
def test_rmsnorm(ops, rows, cols):
    rng = np.random.default_rng(rows)
    x = bf16_round(rng.normal(0, 2, (rows, cols)).astype(np.float32))
    gamma = bf16_round(rng.normal(1, 0.2, cols).astype(np.float32))
    y = ops.rmsnorm(dev(x), dev(gamma), 1e-6).float().cpu().numpy()
    ref = bf16_round(glue.rmsnorm(x, gamma, 1e-6))
    np.testing.assert_allclose(y, ref, rtol=2 ** -7, atol=1e-6)
    xf = rng.normal(0, 2, (rows, cols)).astype(np.float32)
    yf = ops.rmsnorm(dev(xf, torch.float32), dev(gamma, torch.float32), 1e-6).cpu().numpy()
    np.testing.assert_allclose(yf, glue.rmsnorm(xf, gamma, 1e-6), rtol=1e-5, atol=1e-6)


def test_rope_qk(ops):
    rng = np.random.default_rng(2)
    n, g, H, rows = 14, 2, 128, 6
    inv = glue.rope_inv_freq(H, 1000000.0)
    pos = np.array([0, 1, 17, 2047, 4095, 33], np.int32)
    qkv = rng.normal(0, 1, (rows, (n + 2 * g) * H)).astype(np.float32)
    t = dev(qkv, torch.float32)
    ops.rope_qk_(t, torch.from_numpy(pos).cuda(), torch.from_numpy(inv).cuda(), n, g, H)
    out = t.cpu().numpy()
    ref = qkv.copy()
    heads = qkv[:, : (n + g) * H].reshape(rows, n + g, H)
    ref[:, : (n + g) * H] = glue.rope(heads, pos, inv).reshape(rows, -1)
    np.testing.assert_allclose(out, ref, rtol=1e-4, atol=2e-4)  # sincosf of angles up to 4095 rad
    np.testing.assert_array_equal(out[:, (n + g) * H:], qkv[:, (n + g) * H:])  # V untouched


def test_binary_ops_and_embedding(ops):
    rng = np.random.default_rng(3)
    a = bf16_round(rng.normal(0, 2, 100003).astype(np.float32))
    b = bf16_round(rng.normal(0, 2, 100003).astype(np.float32))
    np.testing.assert_array_equal(ops.binary_add(dev(a), dev(b)).float().cpu().numpy(), bf16_round(a + b))
    sm = ops.silu_mul(dev(a), dev(b)).float().cpu().numpy()
    ref = bf16_round(bf16_round(glue.silu(a)) * b)
    np.testing.assert_allclose(sm, ref, rtol=2 ** -6, atol=1e-6)
    table = bf16_round(rng.normal(0, 1, (50, 96)).astype(np.float32))
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int64, device="cuda")
    np.testing.assert_array_equal(ops.embedding(ids, dev(table)).cpu().numpy(), table[[3, 49, 0, 3]])
    v = torch.tensor([0, 5, 2047], dtype=torch.int32, device="cuda")
    assert ops.increment_u32_(v).tolist() == [1, 6, 2048]


def test_nan_logits_and_wild_ids_stay_in_range(ops):
    """an all-NaN logits row must give a valid token id (0), not the 2^31 - 1 sentinel, and an id out of
    range must not make the embedding read outside its table."""
    logits = torch.randn(3, 5000, device="cuda")
    logits[1] = float("nan")
    ids = ops.argmax(logits)
    torch.cuda.synchronize()
    assert ids.tolist()[0] == int(torch.argmax(logits[0])) and ids.tolist()[1] == 0 and ids.tolist()[2] == int(torch.argmax(logits[2]))
    table = torch.randn(10, 64, device="cuda").to(torch.bfloat16)
    wild = torch.tensor([3, 2 ** 31 - 1, -5, 9], dtype=torch.int64, device="cuda")
    h = ops.embedding(wild, table)
    torch.cuda.synchronize()
    assert torch.equal(h[0], table[3].float()) and torch.equal(h[1], table[9].float()) and torch.equal(h[2], table[0].float())


# row lengths that come in fours and not, fewer columns than threads, one batch of loads per thread and more; ties go to the first column
@pytest.mark.parametrize("M,N", [(1, 4), (3, 1003), (2, 65536), (5, 65540), (33, 152064), (2, 300004), (2, 300001)])
def test_argmax_at_the_edges_of_its_loads(M, N):
    from dash_infer_amd import ops
    g = torch.Generator("cuda").manual_seed(N)
    logits = torch.randn(M, N, generator=g, device="cuda")
    at = [0, N - 1, N // 2, 65535 % N, (N // 3) | 3]
    for m in range(M):
        logits[m, min(at[m % 5], N - 1)] = 9.0
    assert torch.equal(ops.argmax(logits), torch.argmax(logits, -1))
    logits[:, N - 1] = logits[:, N // 2] = 12.0
    assert ops.argmax(logits).tolist() == [N // 2] * M
    logits[0] = float("-inf")
    assert int(ops.argmax(logits)[0]) == 0


@pytest.mark.parametrize("M,N", [(1, 4), (3, 1003), (5, 65540), (33, 152064), (2, 300001)])
def test_argmax_with_nan(M, N):
    """NaN first is torch.argmax, whatever else the row holds (infinities, NaN of either sign, nothing but NaN, the first of several); without it a NaN is passed over"""
    from dash_infer_amd import ops
    g = torch.Generator("cuda").manual_seed(N)
    logits = torch.randn(M, N, generator=g, device="cuda")
    assert torch.equal(ops.argmax(logits, nan_first=True), torch.argmax(logits, -1))
    logits[:, N // 2] = float("inf")
    logits[:, 1] = float("-inf")
    assert torch.equal(ops.argmax(logits, nan_first=True), torch.argmax(logits, -1))
    for m in range(M):
        logits[m, (m * 7919 + N - 1) % N] = float("nan") if m % 2 else -float("nan")
        logits[m, N - 1] = float("nan")
    want = torch.argmax(logits, -1)
    assert torch.equal(ops.argmax(logits, nan_first=True), want) and bool(torch.isnan(logits[torch.arange(M), want]).all())
    plain = ops.argmax(logits)
    assert torch.equal(plain, torch.argmax(torch.where(torch.isnan(logits), float("-inf"), logits), -1))
    logits[0] = float("nan")
    assert ops.argmax(logits, nan_first=True)[0] == 0 and ops.argmax(logits)[0] == 0


@pytest.mark.parametrize("B", [1, 64, 65])
def test_decode_state_from_device_tensors(B):
    """set_state of a session: the same state from device tensors (one launch) as from host values"""
    from types import SimpleNamespace
    from dash_infer_amd import decoder
    ids, lens = torch.randint(0, 1 << 40, (B,), device="cuda"), torch.randint(0, 1 << 20, (B,), device="cuda", dtype=torch.int32)
    got = []
    for a, b in ((ids, lens), (ids.cpu(), lens.tolist())):
        s = SimpleNamespace(B=B, ids=torch.zeros(B, dtype=torch.int64, device="cuda"), **{k: torch.zeros(B, dtype=torch.int32, device="cuda") for k in ("old_lens", "new_lens")})
        decoder.DecodeSession.set_state(s, a, b)
        got.append((s.ids.tolist(), s.old_lens.tolist(), s.new_lens.tolist()))
    assert got[0] == got[1] == (ids.tolist(), lens.tolist(), (lens + 1).tolist())


def test_decode_state_while_another_device_is_current(monkeypatch):
    """no launch on another device's stream: the copies find the session's device by themselves"""
    from types import SimpleNamespace
    from dash_infer_amd import decoder
    s = SimpleNamespace(B=2, ids=torch.zeros(2, dtype=torch.int64, device="cuda"), **{k: torch.zeros(2, dtype=torch.int32, device="cuda") for k in ("old_lens", "new_lens")})
    ids, lens = torch.tensor([5, 9], device="cuda"), torch.tensor([3, 4], dtype=torch.int32, device="cuda")
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    monkeypatch.setattr(decoder, "lib", lambda: pytest.fail("launched on the current device's stream"))
    decoder.DecodeSession.set_state(s, ids, lens)
    assert (s.ids.tolist(), s.old_lens.tolist(), s.new_lens.tolist()) == ([5, 9], [3, 4], [4, 5])


@pytest.mark.parametrize("dtype,n", [(torch.float32, 3584), (torch.bfloat16, 4), (torch.float16, 32 * 3584)])
def test_p2p_allreduce_gives_up_without_its_peer(pkg, dtype, n):
    """The bounded wait of a rank whose peer never calls (a short limit from the host): the kernel ends, the error word is set, the sums are NaN -- also of
    the next call, which does not wait.  A rank alone is not affected."""
    from dash_infer_amd import ops
    from dash_infer_amd.capi import check, lib
    bufs = [torch.zeros(int(lib().dihip_p2p_ar_buffer_bytes()), dtype=torch.uint8, device="cuda") for _ in range(2)]
    for ranks in (1, 2):
        comm = C.c_void_p()
        check(lib().dihip_p2p_ar_create(C.byref(comm), 0, ranks, (C.c_void_p * ranks)(*[b.data_ptr() for b in bufs[:ranks]])), "create")
        check(lib().dihip_p2p_ar_set_timeout(comm, 64, 0), "limit")
        word = torch.full((1,), 7, dtype=torch.int32).pin_memory()
        for _ in range(2):
            x = torch.randn(n, device="cuda").to(dtype)
            y = torch.zeros_like(x)
            check(lib().dihip_p2p_allreduce_sum(comm, ops.cur_stream(), ops.ptr(x), ops.ptr(y), n, ops.dt_code(x)), "sum")
            check(lib().dihip_p2p_ar_error_async(comm, ops.cur_stream(), word.data_ptr()), "word")
            torch.cuda.synchronize()
            e = C.c_int(9)
            check(lib().dihip_p2p_ar_error(comm, C.byref(e)), "error")
            assert int(word[0]) == e.value == ranks - 1
            assert torch.equal(y, x) if ranks == 1 else bool(torch.isnan(y).all())
        lib().dihip_p2p_ar_destroy(comm)
