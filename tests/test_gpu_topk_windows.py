"""Sampled candidate windows whose ends lie in one digit of the key, in neighbouring ones, far apart, or nowhere, on the
streaming path and on the resident one."""
import numpy as np
import pytest
import torch

from oracle import F32
import oracle
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu


def _values(kind, n, ratio):
    rng = np.random.default_rng(n)
    if kind == "narrow":      # magnitudes of [1, 1.1): one digit
        return (1.0 + rng.random(n) * 0.1).astype(np.float32) * rng.choice(np.array([1, -1], np.float32), n)
    g = student_t(rng, n, ties=0.0)
    if kind == "cliff":       # half of the picks are far above everything else
        g[rng.random(n) < ratio / 2] *= np.float32(1e30)
    elif kind == "steps":     # magnitudes of many exponents, infinities on top
        g *= np.exp2(rng.integers(-60, 60, n)).astype(np.float32)
        g[rng.integers(0, n, 50)] = np.inf
    return g


@pytest.mark.parametrize("ratio", [0.0001, 0.01, 0.05])
@pytest.mark.parametrize("kind", ["spread", "narrow", "cliff", "steps"])
@pytest.mark.parametrize("n", [600_003, 2_200_001])
def test_windows(n, kind, ratio):
    from mccl_amd import hip_ops as ops
    g, res = _values(kind, n, ratio), np.zeros(n, np.float32)
    dres = to_dev(res, F32)
    ws = ops.topk_workspace(n, n, ratio, DEV)
    wire, _ = ops.topk_compress(to_dev(g, F32), dres, ratio, workspace=ws)
    want, size = oracle.topk_compress(g, res, ratio)
    # the window holds the threshold, and its bin few enough (with a few picks in the sample a window has no upper end)
    if kind == "spread" or kind == "narrow" and ratio > 0.001:
        assert ops.topk_path_report(ws, n, n, ratio) == (1, 1)
    assert wire.cpu().numpy()[:size].tobytes() == want.tobytes()
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))


def _with_zeros(n, share, seed):
    rng = np.random.default_rng(seed)
    g = rng.standard_normal(n).astype(np.float32)
    g[rng.random(n) < share] = 0.0
    return g


@pytest.mark.parametrize("share", [0.5, 0.985, 0.995, 0.9999, 1.0])   # of 1 % picks and the window's ends: none, one or all among the zeros
@pytest.mark.parametrize("n", [600_003, 2_200_001])
def test_windows_beside_zeros(n, share):
    from mccl_amd import hip_ops as ops
    g, res = _with_zeros(n, share, n), np.zeros(n, np.float32)
    dres = to_dev(res, F32)
    wire, _ = ops.topk_compress(to_dev(g, F32), dres, 0.01)
    want, size = oracle.topk_compress(g, res, 0.01)
    assert wire.cpu().numpy()[:size].tobytes() == want.tobytes()
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_a_window_down_to_zero_predicts_as_closely(seed):
    """The window's lower end lies among zeros, the other two ranks in one octave, 8 digits of 2^20 keys cut into 2048 cells: the
    predicted threshold is the middle of the sample's cell, of 4096 keys."""
    from mccl_amd import hip_ops as ops
    n, ratio, hist_words, s_that = 2_200_001, 0.01, 4096, 2
    rng = np.random.default_rng(seed)
    g = np.where(rng.random(n) < 0.987, 0.0, 1.0 + rng.random(n)).astype(np.float32)
    ws = ops.topk_workspace(n, n, ratio, DEV)
    ops.topk_compress(to_dev(g, F32), to_dev(np.zeros(n, np.float32), F32), ratio, workspace=ws)
    stride = n // 4 // 256 * 4                               # 256 sampled runs of 32 elements
    sample = np.sort(np.concatenate([np.abs(g[i * stride:i * stride + 32]) for i in range(256)]))[::-1]
    rank = int(np.float32(int(n * ratio)) * np.float32(8192) / np.float32(n))
    assert sample[rank - 1] > 0 and sample[rank + int(6 * rank**0.5) + 16] == 0
    predicted = int(ws.view(torch.int32)[hist_words + s_that])
    assert abs(predicted - int(sample[rank - 1].view(np.uint32))) <= 4096 // 2 + 1
