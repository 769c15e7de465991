"""The entry points only enqueue kernels on the caller's stream (no host
synchronisation, no allocation, no memset nodes), so a launch-bound sequence
such as the launches of a one-bucket top-k compress (two on the single-pass path, six on the
exact path) can be captured in a HIP
graph.  Every replay is checked against the eager result and the oracle, with
eager work and synchronisations in between."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_np, bits, student_t

pytestmark = pytest.mark.gpu


def test_topk_compress_and_fold_replay_from_a_graph():
    from mccl_amd import hip_ops as ops
    n, ratio = 1_000_003, 0.01
    rng = np.random.default_rng(5)
    grad = torch.empty(n, device=DEV)
    res = torch.zeros(n, device=DEV)
    other = torch.empty(n, device=DEV)
    ws = ops.topk_workspace(n, n, ratio, DEV)
    stride = ops.topk_wire_stride(n, ratio)
    wire = torch.zeros(stride, dtype=torch.uint8, device=DEV)
    # warm-up outside capture (library init, first-use paths)
    grad.copy_(torch.from_numpy(student_t(rng, n)))
    other.copy_(grad)
    ops.topk_compress(grad, res, ratio, wire=wire, workspace=ws)
    ops.fold2_scale(other, grad, 0.5)
    torch.cuda.synchronize()

    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            ops.topk_compress(grad, res, ratio, wire=wire, workspace=ws)
            ops.fold2_scale(other, grad, 0.5)
    torch.cuda.current_stream().wait_stream(side)

    res_o = np.zeros(n, np.float32)
    res.zero_()
    for step in range(4):
        gh = student_t(rng, n, ties=0.01)
        oh = (rng.standard_normal(n) * 1e-3).astype(np.float32)
        grad.copy_(torch.from_numpy(gh))
        other.copy_(torch.from_numpy(oh))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        w, rc = oracle.topk_compress(gh, res_o, ratio)
        assert wire.cpu().numpy()[:rc].tobytes() == w.tobytes(), step
        assert np.array_equal(bits(to_np(res, F32)), bits(res_o)), step
        want = oh.copy()
        oracle.fold2_scale(want, gh, F32, 0.5)
        assert np.array_equal(bits(to_np(other, F32)), bits(want)), step
        # eager work between replays
        assert float((other - torch.from_numpy(want).to(DEV)).abs().max()) == 0.0


STATE_WORDS, HIST_WORDS = 32, 4096   # per bucket, at the front of a top-k workspace: histograms, then state
S_LO, S_READY, S_TIMEOUT = 0, 3, 13


@pytest.mark.parametrize("path", [2, 3])
def test_replay_behind_a_run_that_was_given_up(path):
    """What an abandoned replay can leave in the workspace - the window published under the launch's
    own epoch number, barrier counters full, the give-up flag set - is planted before every replay of
    a captured compress; the replay must not take it for its own."""
    from mccl_amd import hip_ops as ops
    n, ratio = 300_001, 0.01
    rng = np.random.default_rng(path)
    grad, res = torch.empty(n, device=DEV), torch.zeros(n, device=DEV)
    ws = ops.topk_workspace(n, n, ratio, DEV)
    words = ws.view(torch.int32)
    state = words[HIST_WORDS:HIST_WORDS + STATE_WORDS]
    stride = ops.topk_wire_stride(n, ratio)
    wire = torch.zeros(stride, dtype=torch.uint8, device=DEV)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    grad.copy_(torch.from_numpy(student_t(rng, n)))
    call = lambda: ops.topk_compress(grad, res, ratio, wire=wire, workspace=ws, status=status)
    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    try:
        ops.set_tuning("topk_path", path)
        call()
        # A run whose waits all end at once publishes ~epoch; the next launch's epoch is one more.
        ops.set_tuning("topk_stall_test", 1)
        ops.set_tuning("topk_barrier_ms", 1)
        call()
        torch.cuda.synchronize()
        ops.set_tuning("topk_stall_test", 0)
        ops.set_tuning("topk_barrier_ms", 2000)
        assert int(status) == -9
        left = int(state[S_READY])
        epoch = ~left + 1 if left else None   # (path 2 leaves nothing published)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.cuda.graph(g, stream=side):
            call()
        torch.cuda.current_stream().wait_stream(side)
    finally:
        ops.set_tuning("topk_path", 0)
        ops.set_tuning("topk_stall_test", 0)
        ops.set_tuning("topk_barrier_ms", 2000)
    assert path == 2 and left == 0 or path == 3 and left != 0
    for step in range(3):
        gh = student_t(rng, n, ties=0.01)
        res_o = np.zeros(n, np.float32)
        grad.copy_(torch.from_numpy(gh))
        res.zero_()
        status.zero_()
        if epoch is not None:
            words.fill_(1000)
            state[S_LO:S_READY + 1] = torch.tensor([0, 0x7FFFFFFF, 0, epoch], dtype=torch.int32, device=DEV)
            state[S_TIMEOUT] = 1
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        w, rc = oracle.topk_compress(gh, res_o, ratio)
        assert int(status) == 0
        assert wire.cpu().numpy()[:rc].tobytes() == w.tobytes(), step
        assert np.array_equal(bits(to_np(res, F32)), bits(res_o)), step
        if path == 3:
            assert int(state[S_READY]) == 0
