"""The threshold's bin in the streaming path: lists that are ranked at once, after one round of digits or after several, ties across
the cut on either side of what a wavefront ranks, and digits that lie in the index alone."""
import numpy as np
import pytest

from oracle import F32
import oracle
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu


def _check(g, ratio, bucket=None, path=None):
    from mccl_amd import hip_ops as ops
    n, bucket = g.size, bucket or g.size
    res = np.zeros(n, np.float32)
    dres = to_dev(res, F32)
    ws = ops.topk_workspace(n, bucket, ratio, DEV)
    wire, stride = ops.topk_compress(to_dev(g, F32), dres, ratio, bucket_elems=bucket, workspace=ws)
    if path is not None:
        assert ops.topk_path_report(ws, n, bucket, ratio) == path
    for b in range(-(-n // bucket)):
        at = slice(b * bucket, min(n, (b + 1) * bucket))
        r = res[at]
        want, size = oracle.topk_compress(g[at], r, ratio)
        assert wire.cpu().numpy()[b * stride: b * stride + size].tobytes() == want.tobytes(), b
        assert np.array_equal(bits(to_np(dres, F32))[at], bits(r)), b


@pytest.mark.parametrize("ties", [1, 2, 63, 64, 65, 500])
@pytest.mark.parametrize("n,ratio", [(2_097_153, 0.01), (2_200_001, 0.0001), (4_194_304, 0.001), (2_500_000, 0.05)])
def test_ties_across_the_cut(n, ratio, ties):
    rng = np.random.default_rng(ties)
    g = student_t(rng, n, ties=0.0)
    k = int(n * ratio)
    value = np.partition(np.abs(g), n - k)[n - k]
    at = rng.choice(n, ties, replace=False)
    g[at] = value * rng.choice(np.array([1, -1], np.float32), ties)
    _check(g, ratio, path=(1, 1) if ties < 500 else None)


def test_one_key_in_a_bin():
    """Values so few that every bin of the window holds one key: the digits lie in the index."""
    rng = np.random.default_rng(1)
    g = (rng.integers(0, 4000, 3_000_001) * np.float32(2.0**-12)).astype(np.float32)
    _check(g, 0.01)
    g = np.round(student_t(rng, 3_000_001, ties=0.0) * np.float32(64)) / np.float32(64)
    _check(g, 0.01)


def test_buckets_side_by_side():
    rng = np.random.default_rng(2)
    g = student_t(rng, 6_000_017, ties=0.001)
    _check(g, 0.01, bucket=1_000_000, path=(7, 7))
