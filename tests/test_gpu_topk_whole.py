"""Lists that go in one launch: one bucket and as many as a list holds, groups of one tile and of several, groups whose
candidates do not fit LDS or whose tiles are dense, buckets that fall back beside others that don't, a wait that runs out; and
recorded ones, which go in two.  One launch leaves its windows published, two take them back: that tells the routes apart."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu
TILE = 4096


@pytest.fixture()
def ops():
    from mccl_amd import hip_ops
    hip_ops.set_tuning("topk_path", 2)
    yield hip_ops
    hip_ops.set_tuning("topk_path", 0)


def _misled(rng, n):
    """The sample misleads: every sampled run that meets one of the 5.0 blocks is all 5.0."""
    g = student_t(rng, n, ties=0.0) * np.float32(1e-6)
    step = n // 4 // 256 * 4
    for i in range(0, 256, 2):
        g[i * step: i * step + 32] = 5.0
    return g


STATE_WORDS, HIST_WORDS, S_READY = 32, 4096, 3   # per bucket, at the front of a workspace: histograms, then state


def _published(ws, count):
    return ws.view(torch.int32)[count * HIST_WORDS:count * (HIST_WORDS + STATE_WORDS)].view(count, STATE_WORDS)[:, S_READY].tolist()


def _check(ops, grads, ratio, single_pass=None, one_launch=True):
    longest, count = max(g.size for g in grads), len(grads)
    rng = np.random.default_rng(count)
    residuals = [(rng.standard_normal(g.size) * 1e-9).astype(np.float32) for g in grads]
    dres = [to_dev(r, F32, i % 4) for i, r in enumerate(residuals)]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = ops.topk_workspace(longest * count, longest, ratio, DEV)
    wires = ops.topk_compress_list([to_dev(g, F32, (i + 1) % 3) for i, g in enumerate(grads)], dres, ratio, workspace=ws, status=status)
    assert int(status) == 0
    assert [w != 0 for w in _published(ws, count)] == [one_launch] * count
    if single_pass is not None:
        assert ops.topk_path_report(ws, longest * count, longest, ratio) == (single_pass, count)
    for g, r, d, w in zip(grads, residuals, dres, wires):
        want, size = oracle.topk_compress(g, r, ratio)
        assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), g.size
        assert np.array_equal(bits(to_np(d, F32)), bits(r)), g.size


@pytest.mark.parametrize("ratio", [0.001, 0.01, 0.05])
@pytest.mark.parametrize("lengths", [
    [2_200_001], [8 * TILE], [8 * TILE + 1], [1], [2 * TILE - 1, 5],
    [7 * TILE, 8 * TILE + 3, 9 * TILE, 16 * TILE, 17 * TILE + 2, 3, 40_001],
    [900_001 - 37 * i for i in range(12)],
    [70_001 + i for i in range(64)]])
def test_lists(ops, lengths, ratio):
    rng = np.random.default_rng(len(lengths))
    # (a group of 8 tiles that may be all candidates, or of 12 at 5 %, has more than a block keeps)
    two = lengths == [1] or ratio == 0.05 and len(lengths) == 12
    _check(ops, [student_t(rng, n, ties=0.01) for n in lengths], ratio, one_launch=not two)


@pytest.mark.parametrize("ratio", [0.01, 0.05])
def test_candidates_that_lie_together(ops, ratio):
    """Nearly all picks in a few tiles: they run out of slots, or their group out of LDS."""
    rng = np.random.default_rng(5)
    grads = [student_t(rng, n, ties=0.0) * np.float32(1e-3) for n in (1_500_001, 600_000, 80_001)]
    for g in grads:
        at = g.size // 3
        g[at:at + int(g.size * ratio)] = student_t(rng, int(g.size * ratio), ties=0.0)      # dense tiles
        for lo in range(0, g.size // 4, 600):
            g[lo:lo + 20] *= np.float32(1e3)                                                # full ones
    _check(ops, grads, ratio)


def test_ties_zeros_and_nans(ops):
    rng = np.random.default_rng(6)
    a = np.zeros(500_001, np.float32)
    b = rng.choice(np.array([0.0, -0.0, 0.5, -0.5, 1.0], np.float32), 300_000)
    c = student_t(rng, 400_003, ties=0.3)
    d = student_t(rng, 700_001, ties=0.0)
    d[::1000] = np.nan
    d[1::5000] = -np.inf
    _check(ops, [a, b, c, d], 0.01)
    e = student_t(rng, 1_200_000, ties=0.0)
    e[rng.permutation(e.size)[:3000]] = np.sort(np.abs(e))[-12_000]      # the threshold, three thousand times
    _check(ops, [e, c], 0.01, single_pass=2)


@pytest.mark.parametrize("ratio", [0.01, 0.05])
def test_fallbacks_beside_others(ops, ratio):
    rng = np.random.default_rng(7)
    lengths = [1_500_001, 900_000, 1_200_007, 600_011, 65_537]
    grads = [(_misled if i in (0, 2) else student_t)(rng, n) for i, n in enumerate(lengths)]
    _check(ops, grads, ratio, single_pass=3)


def test_a_wait_that_runs_out(ops):
    rng = np.random.default_rng(8)
    grads = [to_dev(student_t(rng, n), F32) for n in (600_000, 300_001)]
    res = [torch.zeros_like(g) for g in grads]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = ops.topk_workspace(1_200_000, 600_000, 0.01, DEV)
    try:
        ops.set_tuning("topk_stall_test", 1)
        ops.set_tuning("topk_barrier_ms", 2)
        wires = ops.topk_compress_list(grads, res, 0.01, workspace=ws, status=status)
        torch.cuda.synchronize()
    finally:
        ops.set_tuning("topk_stall_test", 0)
        ops.set_tuning("topk_barrier_ms", 2000)
    assert int(status) == -9
    assert all(_published(ws, 2))
    assert all(int(w[:4].view(torch.int32)) == -1 for w in wires)
    status.zero_()
    for r in res:
        r.zero_()
    wires = ops.topk_compress_list(grads, res, 0.01, workspace=ws, status=status)
    assert int(status) == 0
    for g, w in zip(grads, wires):
        want, size = oracle.topk_compress(to_np(g, F32), np.zeros(g.numel(), np.float32), 0.01)
        assert w.cpu().numpy()[:size].tobytes() == want.tobytes()


def test_replays(ops):
    """A recorded list call, which takes two launches, replayed with other gradients: every replay carries the same number."""
    rng = np.random.default_rng(9)
    lengths = [700_001, 300_000, 5_000]
    grads = [torch.empty(n, device=DEV) for n in lengths]
    res = [torch.zeros(n, device=DEV) for n in lengths]
    want_res = [np.zeros(n, np.float32) for n in lengths]
    ws = ops.topk_workspace(max(lengths) * 3, max(lengths), 0.01, DEV)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    ops.topk_compress_list(grads, [r.clone() for r in res], 0.01, workspace=ws, status=status)
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        wires = ops.topk_compress_list(grads, res, 0.01, workspace=ws, status=status)
    torch.cuda.current_stream().wait_stream(side)
    for r in res:
        r.zero_()
    for _ in range(4):
        values = [student_t(rng, n) for n in lengths]
        for g, v in zip(grads, values):
            g.copy_(torch.from_numpy(v))
        graph.replay()
        torch.cuda.synchronize()
        assert int(status) == 0
        for v, r, want_r, w in zip(values, res, want_res, wires):
            want, size = oracle.topk_compress(v, want_r, 0.01)
            assert w.cpu().numpy()[:size].tobytes() == want.tobytes()
            assert np.array_equal(bits(to_np(r, F32)), bits(want_r))


def test_four_streams(ops):
    """Launches whose blocks wait for each other, on as many streams as there are hardware queues."""
    rng = np.random.default_rng(10)
    lengths = [800_001 - 1000 * i for i in range(6)]
    calls = []
    for s in range(4):
        values = [student_t(rng, n) for n in lengths]
        calls.append((torch.cuda.Stream(), values, [to_dev(v, F32) for v in values], [torch.zeros(n, device=DEV) for n in lengths],
                      ops.topk_workspace(lengths[0] * 6, lengths[0], 0.01, DEV), torch.zeros(1, dtype=torch.int32, device=DEV)))
    torch.cuda.synchronize()
    wires = []
    for rep in range(3):
        for stream, _, grads, res, ws, status in calls:
            with torch.cuda.stream(stream):
                wires.append(ops.topk_compress_list(grads, res, 0.01, workspace=ws, status=status))
    torch.cuda.synchronize()
    for s, (_, values, _, res, ws, status) in enumerate(calls):
        assert int(status) == 0 and all(_published(ws, len(lengths)))
        want_res = [np.zeros(n, np.float32) for n in lengths]
        for rep in range(3):
            for v, r, w in zip(values, want_res, wires[rep * 4 + s]):
                want, size = oracle.topk_compress(v, r, 0.01)
                assert w.cpu().numpy()[:size].tobytes() == want.tobytes()
        for r, d in zip(want_res, res):
            assert np.array_equal(bits(to_np(d, F32)), bits(r))


def test_a_recorded_list_takes_its_windows_back(ops):
    """One launch leaves the windows published under its number.  A replay carries the number of the replay before, so a
    recorded list has to end with them taken back, also when its blocks gave up."""
    rng = np.random.default_rng(12)
    lengths, ratio = [700_001, 300_000, 5_000], 0.01
    count, longest = len(lengths), max(lengths)
    grads = [to_dev(student_t(rng, n), F32) for n in lengths]
    res = [torch.zeros(n, device=DEV) for n in lengths]
    ws = ops.topk_workspace(longest * count, longest, ratio, DEV)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    call = lambda: ops.topk_compress_list(grads, res, ratio, workspace=ws, status=status)
    call()
    assert all(_published(ws, count))
    graphs, wires = [], []
    try:
        for stall in (1, 0):
            ops.set_tuning("topk_stall_test", stall)
            ops.set_tuning("topk_barrier_ms", 1 if stall else 2000)
            side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
                wires.append(call())
            torch.cuda.current_stream().wait_stream(side)
            graphs.append(graph)
    finally:
        ops.set_tuning("topk_stall_test", 0)
        ops.set_tuning("topk_barrier_ms", 2000)
    for step in range(3):
        status.zero_()
        graphs[0].replay()
        torch.cuda.synchronize()
        assert int(status) == -9
        assert _published(ws, count) == [0] * count
        values = [student_t(rng, n, scale=10.0 ** -step) for n in lengths]
        for g, r, v in zip(grads, res, values):
            g.copy_(torch.from_numpy(v))
            r.zero_()
        status.zero_()
        graphs[1].replay()
        torch.cuda.synchronize()
        assert int(status) == 0
        assert _published(ws, count) == [0] * count
        for v, r, w in zip(values, res, wires[1]):
            want_r = np.zeros(v.size, np.float32)
            want, size = oracle.topk_compress(v, want_r, ratio)
            assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), step
            assert np.array_equal(bits(to_np(r, F32)), bits(want_r)), step
