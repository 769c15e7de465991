"""TopKCompressor.decompress (one launch for ascending payloads, the order-free kernels behind it)
against the oracle at the edges of its tiles (8192 elements) and of its 256 samples, for spread,
clustered, unordered and repeated indices, and for indices past the end."""
import ctypes as ct
import time

import numpy as np
import pytest
import torch
import torch.distributed  # noqa: F401

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_np, bits

pytestmark = pytest.mark.gpu


def _payload(idx, val):
    w = np.empty(1 + 2 * idx.size, np.uint32)
    w[0] = idx.size
    w[1::2] = idx
    w[2::2] = val.view(np.uint32)
    return w.view(np.uint8)


def _status(wire, n):
    from mccl_amd import _lib
    dense = torch.full((n,), 3.0, device=DEV)
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    rc = _lib.load().mccl_hip_topk_decompress_sorted(ct.c_void_p(wire.data_ptr()), wire.numel(), ct.c_void_p(dense.data_ptr()), n,
                                                    ct.c_void_p(st.data_ptr()), None)
    torch.cuda.synchronize()
    return rc, int(st), dense


@pytest.mark.parametrize("n,k", [(1, 1), (8191, 1), (8192, 8192), (8193, 255), (8193, 256), (16_385, 257),
                                 (70_001, 700), (1_000_003, 10_000), (3_000_001, 150_001)])
def test_ascending_payloads(n, k):
    from mccl_amd import _C
    rng = np.random.default_rng(n + k)
    comp = _C.TopKCompressor(min(1.0, (k + 0.5) / n))
    spread = np.sort(rng.choice(n, k, replace=False)).astype(np.uint32)
    for idx in (spread, np.arange(k, dtype=np.uint32), np.arange(n - k, n, dtype=np.uint32)):
        w = _payload(idx, rng.standard_normal(k).astype(np.float32))
        want, rc = oracle.topk_decompress(w, n)
        assert rc == 0
        dw = torch.from_numpy(w).to(DEV)
        rc, st, dense = _status(dw, n)
        assert (rc, st) == (0, 0) and np.array_equal(bits(to_np(dense, F32)), bits(want))
        assert np.array_equal(bits(to_np(comp.decompress(dw, n), F32)), bits(want))


@pytest.mark.parametrize("k", [2, 300, 20_000])
def test_unordered_payloads_take_the_other_kernels(k):
    from mccl_amd import _C
    n = 100_003
    rng = np.random.default_rng(k)
    comp = _C.TopKCompressor(min(1.0, (k + 0.5) / n))
    idx = np.sort(rng.choice(n, k, replace=False)).astype(np.uint32)
    val = rng.standard_normal(k).astype(np.float32)
    for at in {0, (k - 1) // 2, k - 2}:
        sw = idx.copy()
        sw[at], sw[at + 1] = idx[at + 1], idx[at]     # one pair of neighbours exchanged
        rep = idx.copy()
        rep[at + 1] = idx[at]                         # one index twice, with the same value
        same = val.copy()
        same[at + 1] = val[at]
        for i, v in ((sw, val), (rep, same)):
            w = _payload(i, v)
            want, _ = oracle.topk_decompress(w, n)
            dw = torch.from_numpy(w).to(DEV)
            assert _status(dw, n)[1] == -11
            assert np.array_equal(bits(to_np(comp.decompress(dw, n), F32)), bits(want))
    w = torch.from_numpy(_payload(idx, val)).to(DEV)
    assert _status(w, int(idx[-1]))[1] == oracle.ERR_INDEX
    with pytest.raises(RuntimeError, match="index out of bounds"):
        comp.decompress(w, int(idx[-1]))
    w[:4] = 0
    assert _status(w, n)[1] == oracle.ERR_SIZE


@pytest.mark.parametrize("n", [8192, 64 * 8192, 64 * 8192 + 1, 97 * 8192 + 5])  # one block, and both ways of arriving
def test_calls_that_report_before_their_launch_ends(n):
    """Good payloads between ones that break a rule, on two streams in turn and behind earlier work: every call sees its
    own report, and the counters are left as they were found."""
    from mccl_amd import _C
    rng = np.random.default_rng(n)
    k = n // 50
    comp = _C.TopKCompressor(0.02)
    other = torch.cuda.Stream()
    idx = np.sort(rng.choice(n - 1, k, replace=False)).astype(np.uint32)
    sw = idx.copy()
    sw[k // 2], sw[k // 2 + 1] = idx[k // 2 + 1], idx[k // 2]
    past = idx.copy()
    past[-1] = n
    for i in range(6):
        with torch.cuda.stream(other if i % 2 else torch.cuda.default_stream()):
            for ids in (idx, sw, past):
                w = _payload(ids, rng.standard_normal(k).astype(np.float32))
                dw = torch.from_numpy(w).to(DEV)
                if i >= 4:
                    torch.cuda._sleep(5_000_000)   # a few milliseconds
                if ids is past:
                    with pytest.raises(RuntimeError, match="index out of bounds"):
                        comp.decompress(dw, n)
                else:
                    want, _ = oracle.topk_decompress(w, n)
                    assert np.array_equal(bits(to_np(comp.decompress(dw, n), F32)), bits(want))


def test_reports_of_the_entry_point():
    from mccl_amd import _lib
    lib = _lib.load()
    n, k = 700_001, 7000
    rng = np.random.default_rng(5)
    counters = torch.zeros(8448 // 8, dtype=torch.int64, device=DEV)
    word = torch.zeros(1, dtype=torch.int64).pin_memory()
    flag = torch.zeros(1, dtype=torch.int32, device=DEV)
    idx = np.sort(rng.choice(n, k, replace=False)).astype(np.uint32)
    rep = idx.copy()
    rep[1] = rep[0]
    dense = torch.empty(n, device=DEV)
    for ticket, (ids, count, f, want) in enumerate([(idx, k, 0, 0), (idx, k, -10, -10), (rep, k, 0, -11), (idx, k - 1, 0, -11),
                                                    (idx, k, 0, 0)], 1):
        w = _payload(ids, np.ones(k, np.float32))
        w.view(np.uint32)[0] = count
        dw = torch.from_numpy(w).to(DEV)
        flag.fill_(f)
        dense.fill_(3.0)
        assert lib.mccl_hip_topk_decompress_sorted_done(
            ct.c_void_p(dw.data_ptr()), dw.numel(), ct.c_void_p(dense.data_ptr()), n, ct.c_void_p(flag.data_ptr()),
            ct.c_void_p(counters.data_ptr()), ct.c_void_p(word.data_ptr()), ticket, None) == 0
        torch.cuda.synchronize()
        v = int(word) & (2 ** 64 - 1)
        assert (v >> 32, v & 0xFFFFFFFF) == (ticket, want & 0xFFFFFFFF)
        assert not counters.any()
        if want != -11:
            assert int(dense.sum()) == k and int((dense == 0).sum()) == n - k
    many = torch.empty(4 + 8 * (2 ** 20 + 1), dtype=torch.uint8, device=DEV)   # more than 2^20 pairs: not launched
    assert lib.mccl_hip_topk_decompress_sorted_done(
        ct.c_void_p(many.data_ptr()), many.numel(), ct.c_void_p(dense.data_ptr()), n, None, ct.c_void_p(counters.data_ptr()),
        ct.c_void_p(word.data_ptr()), 99, None) == -3


@pytest.mark.parametrize("n", [2000, 65_537, 6_553_600])
def test_waiting_right_behind_a_call(n):
    """A program that waits for the GPU behind the call finds the marker of the launch's end on the stream: it waits for
    less than a launch and its marker take (measured 0.4 of that; 0.8 where the wait has to put a marker there)."""
    from mccl_amd import _C, hip_ops
    comp = _C.TopKCompressor(0.01)
    wire = comp.compress(torch.randn(n, device=DEV), stable_id=1)
    x = torch.zeros(64, device=DEV)

    def best(call, wait):
        times = []
        for _ in range(300):
            start = time.perf_counter()
            call()
            if wait:
                torch.cuda.synchronize()
            times.append(time.perf_counter() - start)
            torch.cuda.synchronize()
        return min(times)

    def back():
        return comp.decompress(wire, n)

    launch = best(lambda: hip_ops.fold2(x, x, hip_ops.SUM), True)
    returns, idle = best(back, False), best(back, True)
    print(f"{n}: launch {launch * 1e6:.1f} returns {returns * 1e6:.1f} idle {idle * 1e6:.1f}")
    assert idle - returns < 0.6 * launch, (launch, returns, idle)
