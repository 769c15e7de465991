"""Single-pass top-k of buckets around the sizes where the number of tile groups changes: 64 groups of up to
28 tiles (4096 elements each), then more groups, then, past 256 groups, more tiles in each."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu
TILE = 4096


@pytest.mark.parametrize("n", [64 * 28 * TILE, 64 * 28 * TILE + 1, 65 * 28 * TILE + 5, 256 * 28 * TILE + 4097])
def test_groups_of_tiles(n):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(n)
    grad = student_t(rng, n, ties=0.01)
    res = np.zeros(n, np.float32)
    dres = to_dev(res, F32)
    ws = ops.topk_workspace(n, n, 0.01, DEV)
    wire, _ = ops.topk_compress(to_dev(grad, F32), dres, 0.01, workspace=ws)
    want, size = oracle.topk_compress(grad, res, 0.01)
    assert ops.topk_path_report(ws, n, n, 0.01) == (1, 1)   # no fallback: the groups' counts are consistent
    assert wire.cpu().numpy()[:size].tobytes() == want.tobytes()
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))


def test_fallback_with_more_than_64_groups():
    """The sample misleads (every sampled run that meets one of the 5.0 blocks is all 5.0): the exact selection, by all
    groups of the bucket together."""
    from mccl_amd import hip_ops as ops
    n = 8_000_000
    rng = np.random.default_rng(3)
    grad = student_t(rng, n, ties=0.0) * np.float32(1e-6)
    stride = n // 4 // 256 * 4   # elements between two sampled runs of 32
    for i in range(0, 256, 2):
        grad[i * stride: i * stride + 32] = 5.0
    res = np.zeros(n, np.float32)
    dres = to_dev(res, F32)
    ws = ops.topk_workspace(n, n, 0.01, DEV)
    wire, _ = ops.topk_compress(to_dev(grad, F32), dres, 0.01, workspace=ws)
    want, size = oracle.topk_compress(grad, res, 0.01)
    assert ops.topk_path_report(ws, n, n, 0.01) == (0, 1)
    assert wire.cpu().numpy()[:size].tobytes() == want.tobytes()
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))


@pytest.mark.parametrize("n, bucket", [(3 * TILE, 3 * TILE), (TILE + 1, TILE + 1), (2_000_003, 500_001),
                                       (24_576_000 - 4096, 6_144_000), (24_576_001, 6_144_000)])
def test_blocks_of_one_or_two_tiles(n, bucket):
    """Odd numbers of tiles, and both sides of the number (6144) up to which a streaming block has two."""
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(n)
    grad = student_t(rng, n, ties=0.01)
    res = (rng.standard_normal(n) * 1e-4).astype(np.float32)
    dres = to_dev(res, F32)
    try:
        ops.set_tuning("topk_path", 2)
        wire, stride = ops.topk_compress(to_dev(grad, F32), dres, 0.01, bucket_elems=bucket)
    finally:
        ops.set_tuning("topk_path", 0)
    w = wire.cpu().numpy()
    for b, lo in enumerate(range(0, n, bucket)):
        part = res[lo:lo + bucket].copy()
        want, size = oracle.topk_compress(grad[lo:lo + bucket], part, 0.01)
        res[lo:lo + bucket] = part
        assert w[b * stride: b * stride + size].tobytes() == want.tobytes(), b
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))
