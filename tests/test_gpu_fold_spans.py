"""The binary folds at the edges of their one-wavefront tiles (64 vectors of 16 bytes) and of the
scalar head and tail, for every element type, single and as a ragged list, with destinations and
sources that start at different offsets inside a vector."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32, F16, BF16, I32, I64, U8, OP_SUM, OP_MAX
from tests._gpu_util import DEV, to_dev, to_np, rand_vals, NP_DT

pytestmark = pytest.mark.gpu

SIZE = {F32: 4, F16: 2, BF16: 2, I32: 4, I64: 8, U8: 1}


def _rand(rng, n, dt):
    if dt in (F32, F16, BF16):
        return rand_vals(rng, n, dt, specials=False)
    info = np.iinfo(NP_DT[dt])
    return rng.integers(info.min, info.max, n, dtype=NP_DT[dt], endpoint=True)


@pytest.mark.parametrize("dt", [F32, F16, BF16, I32, I64, U8])
def test_edges_single_and_list(dt):
    from mccl_amd import hip_ops as ops
    rng = np.random.default_rng(dt)
    epv = 16 // SIZE[dt]
    tile = 64 * epv
    sizes = [1, epv - 1 or 1, epv, epv + 1, tile - 1, tile, tile + 1, 2 * tile + epv + 1, 9 * tile - 3, 70_001]
    for op in (OP_SUM, OP_MAX):
        dsts, srcs, wants = [], [], []
        for i, n in enumerate(sizes):
            a, b = _rand(rng, n, dt), _rand(rng, n, dt)
            want = a.copy()
            assert oracle.fold2(want, b, dt, op) == oracle.OK
            pad_d, pad_s = i % (epv + 1), (3 * i) % (epv + 1)
            d, s = to_dev(a, dt, pad_d), to_dev(b, dt, pad_s)
            guard = d.clone()
            ops.fold2(guard, s, op)
            assert np.array_equal(to_np(guard, dt), want), (n, op)
            dsts.append(d); srcs.append(s); wants.append(want)
        ops.fold2_batch(dsts * 1, srcs, op)     # ragged: the longest fold has a hundred times the others' blocks
        for d, s, want in zip(dsts, srcs, wants):
            assert np.array_equal(to_np(d, dt), want), (want.size, op)


def test_list_longer_than_one_launch_and_strided_grid():
    from mccl_amd import _lib, hip_ops as ops
    n = 2_000_000
    d = torch.arange(n, device=DEV, dtype=torch.float32)
    s = torch.ones(n, device=DEV)
    cuts = [0] + sorted(np.random.default_rng(1).choice(np.arange(1, n // 50), 299, replace=False).tolist()) + [n]
    dl = [d[a:b] for a, b in zip(cuts, cuts[1:])]      # 300 folds, three launches, the last one fifty times the rest
    ops.fold2_batch(dl, [s[a:b] for a, b in zip(cuts, cuts[1:])], ops.SUM)
    want = torch.arange(n, device=DEV, dtype=torch.float32) + 1
    assert torch.equal(d, want)
    shipped = _lib.load().mccl_hip_get_tuning(b"fold_blocks_per_cu")
    assert shipped == 4096                             # the folds above ran on the grid that is shipped
    try:
        ops.set_tuning("fold_blocks_per_cu", 1)        # the grid cap: blocks stride over the vectors
        ops.fold2(d, s, ops.SUM)
        ops.fold2_batch(dl, [s[a:b] for a, b in zip(cuts, cuts[1:])], ops.SUM)
    finally:
        ops.set_tuning("fold_blocks_per_cu", shipped)
    assert torch.equal(d, want + 2)
