"""Resident top-k: the threshold's bin around the sizes at which its elements are ranked, split first, or
split again (64 and 2048), spread or equal, in buckets of one block and of several."""
import numpy as np
import pytest

from tests.test_gpu_topk_resident import _check, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("equal", [0, 3, 5000])
@pytest.mark.parametrize("inside", [1, 64, 65, 2047, 2048, 2049, 4000])
@pytest.mark.parametrize("n", [8192, 8193, 70_001])
def test_elements_in_the_thresholds_bin(ops, n, inside, equal):  # noqa: F811
    """`inside` magnitudes of [1, 1.125), one bin of a histogram of eleven key bits, up to `equal` of them alike; 100 above."""
    rng = np.random.default_rng(n + inside)
    g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
    at = rng.permutation(n)[:inside + 100]
    g[at[:inside]] = 1.0 + rng.integers(0, 1 << 20, inside) / np.float32(1 << 23)
    g[at[:min(inside, equal)]] = 1.0625
    g[at[inside:]] = 2.0 + rng.random(100, dtype=np.float32)
    g[rng.random(n) < 0.5] *= -1
    for picked in {1, inside // 2, inside}:
        _check(ops, g, np.zeros(n, np.float32), (100 + picked + 0.5) / n)
