"""Lists in two launches: the calls that go in one when they run at once, recorded and replayed, so that the list form of
k_topk_stream and k_topk_select meets dense tiles, full slots, many equal keys, zeros, short buckets and fallbacks as well."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_np, bits, student_t

pytestmark = pytest.mark.gpu
TILE = 4096
STATE_WORDS, HIST_WORDS, S_READY = 32, 4096, 3   # per bucket, at the front of a workspace: histograms, then state


def _misled(rng, n):
    """The sample misleads: every sampled run that meets one of the 5.0 blocks is all 5.0."""
    g = student_t(rng, n, ties=0.0) * np.float32(1e-6)
    step = n // 4 // 256 * 4
    for i in range(0, 256, 2):
        g[i * step: i * step + 32] = 5.0
    return g


def _dense(rng, n):
    """Tiles that run out of slots between ordinary ones."""
    g = student_t(rng, n, ties=0.0) * np.float32(1e-3)
    for lo in range(0, n - 2_000, 50_000):
        g[lo:lo + 2_000] = student_t(rng, 2_000, ties=0.0)
    return g


def _tied(rng, n):
    g = student_t(rng, n, ties=0.0) * np.float32(1e-3)
    g[::3] = 2.0
    return g


def _few(rng, n):
    g = student_t(rng, n)
    g[rng.random(n) < 0.995] = 0.0
    return g


CASES = {
    "ragged": ([student_t] * 7, [7 * TILE, 8 * TILE + 3, 9 * TILE, 16 * TILE, 17 * TILE + 2, 3, 40_001]),
    "groups": ([student_t] * 5, [900_001 - 37 * i for i in range(5)]),
    "most": ([student_t] * 64, [30_001 + i for i in range(64)]),
    "dense": ([_dense] * 5, [2_500_000, 300_007, 1_200_001, 65_541, 4099]),
    "dense, tied, misled": ([_dense, _misled, _tied, _dense, _dense], [2_500_000, 300_007, 1_200_001, 65_541, 4099]),
    "misled beside others": ([_misled, student_t, student_t, _misled, student_t, _misled], [1_500_001, 65_537, 4097, 2_200_001, 300_007, 1_000_003]),
    "zeros": ([_few, student_t, _few], [600_001, 300_000, 1_000_000]),
}


@pytest.mark.parametrize("ratio", [0.001, 0.01, 0.05])
@pytest.mark.parametrize("case", CASES)
def test_a_list_at_once_and_recorded(case, ratio):
    from mccl_amd import hip_ops as ops
    makes, lengths = CASES[case]
    count, longest = len(lengths), max(lengths)
    rng = np.random.default_rng(count)
    grads = [torch.empty(n, device=DEV) for n in lengths]
    res = [torch.zeros(n, device=DEV) for n in lengths]
    ws = ops.topk_workspace(longest * count, longest, ratio, DEV)
    published = ws.view(torch.int32)[count * HIST_WORDS:count * (HIST_WORDS + STATE_WORDS)].view(count, STATE_WORDS)[:, S_READY]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    wires = [torch.empty(ops.topk_wire_stride(n, ratio), dtype=torch.uint8, device=DEV) for n in lengths]
    call = lambda: ops.topk_compress_list(grads, res, ratio, wires=wires, workspace=ws, status=status)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    ops.set_tuning("topk_path", 2)
    try:
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            call()
        torch.cuda.current_stream().wait_stream(side)
        for run, one_launch in ((call, True), (graph.replay, False), (call, True), (graph.replay, False), (graph.replay, False)):
            values = [make(rng, n) for make, n in zip(makes, lengths)]
            for g, r, v in zip(grads, res, values):
                g.copy_(torch.from_numpy(v))
                r.zero_()
            run()
            torch.cuda.synchronize()
            assert int(status) == 0
            assert [w != 0 for w in published.tolist()] == [one_launch] * count
            for v, r, w in zip(values, res, wires):
                want_r = np.zeros(v.size, np.float32)
                want, size = oracle.topk_compress(v, want_r, ratio)
                assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), v.size
                assert np.array_equal(bits(to_np(r, F32)), bits(want_r)), v.size
    finally:
        ops.set_tuning("topk_path", 0)
