"""Single-pass top-k of buckets around the sizes where the number of tile groups (of 4096 elements a tile) changes.
A call whose select blocks fit one launch has up to 64 groups a bucket, 128 past 64 * 14 tiles, 256 past 128 * 16; another
more than 64 only past 64 * 28 tiles, more than 128 past 128 * 28.  tests/test_topk_route.py holds the groups and
launches of the sizes used here against the rule."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu
TILE = 4096


@pytest.mark.parametrize("n", [64 * 28 * TILE, 64 * 28 * TILE + 1, 65 * 28 * TILE + 5,   # 128 groups of 14 or 15 tiles
                               256 * 28 * TILE + 4097])                            # 248 of 29: more than a block keeps
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


@pytest.mark.parametrize("lengths", [
    [TILE + 1, 5, 3 * TILE + 7, 1_000_003, 4 * TILE, 16 * TILE + 1, 2_200_001, 257 * TILE, 256 * TILE],  # odd tiles, groups of four to nine
    [1_100_001 - 7 * i for i in range(20)] + [9],                         # 1341 groups: two select launches
    [100 + i for i in range(63)] + [2 * TILE],                            # as many buckets as a list holds
    [2_500_003] * 11 + [999],                                             # streaming blocks of one tile
])
def test_list_of_ragged_buckets(lengths):
    """Single-pass top-k of a list: its launches hold the blocks that its buckets have."""
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(len(lengths))
    grads = [student_t(rng, n, ties=0.01) for n in lengths]
    residuals = [(rng.standard_normal(n) * 1e-4).astype(np.float32) for n in lengths]
    dres = [to_dev(r, F32) for r in residuals]
    try:
        ops.set_tuning("topk_path", 2)
        wires = ops.topk_compress_list([to_dev(g, F32) for g in grads], dres, 0.01)
    finally:
        ops.set_tuning("topk_path", 0)
    for g, r, d, w in zip(grads, residuals, dres, wires):
        want, size = oracle.topk_compress(g, r, 0.01)
        assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), g.size
        assert np.array_equal(bits(to_np(d, F32)), bits(r)), g.size


def _misled(rng, n):
    """Values whose sample misleads (every sampled run that meets one of the 5.0 blocks is all 5.0), so that the selection
    falls back to the exact one."""
    grad = student_t(rng, n, ties=0.0) * np.float32(1e-6)
    stride = n // 4 // 256 * 4   # elements between two sampled runs of 32
    for i in range(0, 256, 2):
        grad[i * stride: i * stride + 32] = 5.0
    return grad


def _check(ops, grad, res, ratio, bucket):
    dres = to_dev(res, F32)
    n = grad.size
    ws = ops.topk_workspace(n, bucket, ratio, DEV)
    try:
        ops.set_tuning("topk_path", 2)
        wire, stride = ops.topk_compress(to_dev(grad, F32), dres, ratio, bucket_elems=bucket, workspace=ws)
    finally:
        ops.set_tuning("topk_path", 0)
    w = wire.cpu().numpy()
    for b, lo in enumerate(range(0, n, bucket)):
        part = res[lo:lo + bucket].copy()
        want, size = oracle.topk_compress(grad[lo:lo + bucket], part, ratio)
        res[lo:lo + bucket] = part
        assert w[b * stride: b * stride + size].tobytes() == want.tobytes(), b
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))
    return ops.topk_path_report(ws, n, bucket, ratio)


@pytest.mark.parametrize("n, bucket, ratio", [
    (65_536, 65_536, 0.0115), (65_541, 65_541, 0.05),          # the shortest buckets with 1024 slots a tile
    (3_000_001, 3_000_001, 0.05), (13_107_203, 6_553_600, 0.02),
    (3_000_000, 3_000_000, 0.1),                               # about 500 candidates a tile: more than are read ahead
    (40_000_000, 8_000_000, 0.05),                             # 128 groups a bucket, several tiles a wavefront
    (17 * 1_048_576 - 3, 1_048_576, 0.05),                     # 64 groups a bucket, two select launches
])
def test_many_candidates(n, bucket, ratio):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(n)
    buckets = -(-n // bucket)
    done = _check(ops, student_t(rng, n, ties=0.01), (rng.standard_normal(n) * 1e-4).astype(np.float32), ratio, bucket)
    assert done == (buckets, buckets)   # no fallback


def test_many_candidates_in_one_place():
    """A wavefront that runs out of its 256 staged candidates: dense tiles between ordinary ones, their zeros put back."""
    from mccl_amd import hip_ops as ops
    n = 2_500_000
    rng = np.random.default_rng(11)
    grad = student_t(rng, n, ties=0.0) * np.float32(1e-3)
    for lo in range(0, n, 50_000):
        grad[lo:lo + 2_000] = student_t(rng, 2_000, ties=0.0)
    _check(ops, grad, np.zeros(n, np.float32), 0.03, n)
    grad[::3] = 2.0                          # more equal keys than are picked
    _check(ops, grad, np.zeros(n, np.float32), 0.05, n)
    stride = n // 4 // 256 * 4               # the sample misleads: the exact selection, zeros put back first
    grad = student_t(rng, n, ties=0.0) * np.float32(1e-6)
    for i in range(0, 256, 2):
        grad[i * stride: i * stride + 32] = 5.0
    assert _check(ops, grad, np.zeros(n, np.float32), 0.05, n) == (0, 1)


@pytest.mark.parametrize("lengths", [[1_500_001, 65_537, 4097, 5, 3_000_003, 300_007], [1_300_001 - i for i in range(16)] + [3]])
def test_list_with_many_candidates(lengths):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(len(lengths))
    grads = [student_t(rng, n, ties=0.01) for n in lengths]
    residuals = [(rng.standard_normal(n) * 1e-4).astype(np.float32) for n in lengths]
    dres = [to_dev(r, F32) for r in residuals]
    try:
        ops.set_tuning("topk_path", 2)
        wires = ops.topk_compress_list([to_dev(g, F32) for g in grads], dres, 0.05)
    finally:
        ops.set_tuning("topk_path", 0)
    for g, r, d, w in zip(grads, residuals, dres, wires):
        want, size = oracle.topk_compress(g, r, 0.05)
        assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), g.size
        assert np.array_equal(bits(to_np(d, F32)), bits(r)), g.size


@pytest.mark.parametrize("n, bucket", [
    (64 * 14 * TILE, 64 * 14 * TILE), (64 * 14 * TILE + 1, 64 * 14 * TILE + 1), (128 * 16 * TILE, 128 * 16 * TILE),
    (128 * 16 * TILE + 3, 128 * 16 * TILE + 3),
    (9 * 900 * TILE, 900 * TILE), (8 * 900 * TILE, 900 * TILE)])   # 128 groups each would be more than 1024, and are not
def test_groups_of_few_buckets(n, bucket):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(n)
    buckets = n // bucket
    done = _check(ops, student_t(rng, n, ties=0.01), np.zeros(n, np.float32), 0.01, bucket)
    assert done == (buckets, buckets)


@pytest.mark.parametrize("tiles, last, ratio", [(520, 512, 0.01),     # 58 groups, the last bucket 64
                                                (1600, 1536, 0.01),   # 124 and 128
                                                (1600, 1536, 0.05)])  # 229 and 256, slots for many candidates
def test_last_bucket_with_more_groups(tiles, last, ratio):
    from mccl_amd import hip_ops as ops
    bucket, n = tiles * TILE, (tiles + last) * TILE
    rng = np.random.default_rng(tiles + last)
    grad = student_t(rng, n, ties=0.01)
    res = (rng.standard_normal(n) * 1e-4).astype(np.float32)
    dres = to_dev(res, F32)
    ws = ops.topk_workspace(n, bucket, ratio, DEV)
    wire, stride = ops.topk_compress(to_dev(grad, F32), dres, ratio, bucket_elems=bucket, workspace=ws)
    w = wire.cpu().numpy()
    assert ops.topk_path_report(ws, n, bucket, ratio) == (2, 2)
    for b, lo in enumerate(range(0, n, bucket)):
        part = res[lo:lo + bucket].copy()
        want, size = oracle.topk_compress(grad[lo:lo + bucket], part, ratio)
        res[lo:lo + bucket] = part
        assert w[b * stride: b * stride + size].tobytes() == want.tobytes(), b
    assert np.array_equal(bits(to_np(dres, F32)), bits(res))


@pytest.mark.parametrize("tiles, last, ratio", [(1600, 1536, 0.01), (1600, 1536, 0.05)])   # 124 and 128 groups, 229 and 256
@pytest.mark.parametrize("which", [(0,), (1,), (0, 1)])
def test_last_bucket_with_more_groups_falls_back(tiles, last, ratio, which):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(tiles + last)
    parts = [(_misled if b in which else student_t)(rng, n * TILE) for b, n in enumerate((tiles, last))]
    n = (tiles + last) * TILE
    done = _check(ops, np.concatenate(parts), (rng.standard_normal(n) * 1e-9).astype(np.float32), ratio, tiles * TILE)
    assert done == (2 - len(which), 2)


@pytest.mark.parametrize("ratio", [0.01, 0.05])
@pytest.mark.parametrize("lengths", [
    [1_500_001, 65_537, 4097, 2_200_001, 300_007, 1_000_003],
    [1_100_001 - 7 * i for i in range(20)] + [9]])         # two select launches, the second from the middle of the table
def test_list_whose_buckets_fall_back(lengths, ratio):
    """Every second bucket by length falls back, the others beside it don't."""
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(len(lengths))
    by_length = sorted(range(len(lengths)), key=lambda i: -lengths[i])
    misled = {i for at, i in enumerate(by_length) if at % 2 == 0 and lengths[i] > 500_000}
    grads = [(_misled if i in misled else student_t)(rng, n) for i, n in enumerate(lengths)]
    _check_list(ops, grads, ratio, len(lengths) - len(misled))


def test_list_with_dense_tiles():
    """Lists with slots for many candidates: tiles that run out of them between others, many equal keys, a fallback."""
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(17)
    lengths = [2_500_000, 300_007, 1_200_001, 65_541, 4099]
    grads = [student_t(rng, n, ties=0.0) * np.float32(1e-3) for n in lengths]
    for g in grads:
        for lo in range(0, g.size - 2_000, 50_000):
            g[lo:lo + 2_000] = student_t(rng, 2_000, ties=0.0)
    _check_list(ops, [g.copy() for g in grads], 0.03)
    grads[2][::3] = 2.0                                    # more equal keys than are picked
    grads[1] = _misled(rng, lengths[1])
    _check_list(ops, grads, 0.05)


def _check_list(ops, grads, ratio, single_pass=None):
    longest, count = max(g.size for g in grads), len(grads)
    residuals = [np.zeros(g.size, np.float32) for g in grads]
    dres = [to_dev(r, F32) for r in residuals]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = ops.topk_workspace(longest * count, longest, ratio, DEV)
    try:
        ops.set_tuning("topk_path", 2)
        wires = ops.topk_compress_list([to_dev(g, F32) for g in grads], dres, ratio, workspace=ws, status=status)
    finally:
        ops.set_tuning("topk_path", 0)
    assert int(status) == 0
    if single_pass is not None:
        assert ops.topk_path_report(ws, longest * count, longest, ratio) == (single_pass, count)
    for g, r, d, w in zip(grads, residuals, dres, wires):
        want, size = oracle.topk_compress(g, r, ratio)
        assert w.cpu().numpy()[:size].tobytes() == want.tobytes(), g.size
        assert np.array_equal(bits(to_np(d, F32)), bits(r)), g.size


@pytest.mark.parametrize("tiles, count, short", [(1850, 9, 0), (1850, 9, 3_000_001)])   # 128 groups at most, 124 in each
def test_many_large_buckets(tiles, count, short):
    """More select blocks than one launch holds, and more than 64 groups a bucket all the same; the second launch starts
    at bucket 8, the last of them, whole or shorter."""
    from mccl_amd import hip_ops as ops
    bucket = tiles * TILE
    rng = np.random.default_rng(tiles)
    base = student_t(rng, bucket, ties=0.01)
    grad = np.concatenate([np.roll(base, 1000 * b) * np.float32(1 + b) for b in range(count)])[:bucket * count - short]
    done = _check(ops, grad, np.zeros(grad.size, np.float32), 0.01, bucket)
    assert done == (count, count)
