"""Sparse accumulate of one bucket, where a block finds the starts of its runs itself: at the edges
of the run, the block and the sample count, against the oracle and against the position table.  The path "runs" takes
the runs at every size; which sizes take them by themselves is another rule's matter."""
import numpy as np
import pytest
import torch

import oracle
from mccl_amd import hip_ops
from tests._gpu_util import DEV
from tests.test_gpu_sparse_runs import RUNS, payload, run_case

pytestmark = pytest.mark.gpu


def ranks(rng, ws, n, k):
    out = []
    for r in range(ws):
        kr = max(1, k - r)
        idx = np.sort(rng.choice(n, kr, replace=False))
        out.append([(idx, rng.standard_normal(kr).astype(np.float32))])
    return out


@pytest.mark.parametrize("ws,n,k", [
    (1, 1, 1), (2, 2047, 20), (3, 2048, 80), (5, 2049, 81), (8, 16384, 160), (8, 16385, 161),
    (4, 131_071, 5119), (4, 131_073, 5121),            # 64 samples and one more: a lane's second one
    (7, 1_000_003, 10_000), (8, 700_001, 700),
    (8, 2_000_000, 20_480), (8, 2_000_000, 20_488),    # 2048 samples over all ranks; more takes the table
    (1, 4_194_304, 4000), (1, 4_194_305, 4000),        # one tile a run; two from one element more
    (2, 2_000_000, 81_920), (2, 2_000_000, 81_921),    # 1024 samples; one more takes the table
])
def test_one_bucket(ws, n, k):
    rng = np.random.default_rng(n + k)
    run_case(hip_ops, ranks(rng, ws, n, k), n, n, 1.0 / ws, paths=("runs", "table", "auto"))


@pytest.mark.parametrize("steps,ws,n,k", [
    (1, 5, 400_001, 6000), (2, 5, 400_001, 6000), (3, 5, 400_001, 6000), (7, 5, 400_001, 6000),
    (1, 1, 8_388_608, 9000), (1, 1, 8_388_609, 9000),  # 512 blocks; one more takes the table
])
def test_any_run_length(steps, ws, n, k):
    rng = np.random.default_rng(steps)
    hip_ops.set_tuning("sparse_run_steps", steps)
    try:
        run_case(hip_ops, ranks(rng, ws, n, k), n, n, 1.0 / ws, paths=("auto",))
    finally:
        hip_ops.set_tuning("sparse_run_steps", 0)


@pytest.mark.parametrize("at", [0, 79, 80, 5119, 5120, 5999])
def test_payloads_out_of_order_are_flagged(at):
    n, k = 300_000, 6001
    idx = np.sort(np.random.default_rng(at).choice(n, k, replace=False))
    idx[[at, at + 1]] = idx[[at + 1, at]]
    wires = [torch.from_numpy(payload(idx, np.ones(k, np.float32), k)).to(DEV)]
    for path in (0, 1, 2, 3):
        status = torch.zeros(1, dtype=torch.int32, device=DEV)
        hip_ops.set_tuning("sparse_path", path)
        try:
            hip_ops.sparse_accumulate(torch.empty(n, device=DEV), wires, 4 + 8 * k, bucket_elems=n, status=status)
        finally:
            hip_ops.set_tuning("sparse_path", 0)
        assert int(status) == oracle.ERR_INDEX, path


@pytest.mark.parametrize("ws,n,be,k", [
    (5, 2049, 2049, 81), (6, 16385, 16385, 161), (8, 1_000_001, 1_000_001, 10_000),   # a block finds its runs' starts
    (9, 2049, 2049, 20), (10, 300_001, 100_000, 1000), (11, 65_537, 65_537, 700), (12, 1_000_003, 400_000, 4000),
    (3, 16_900_001, 6_553_600, 131_072),                                              # runs of two dense tiles
    (12, 30_000, 30_000, 1400),                                                       # more pairs than the windows hold
    (3, 40_000_000, 6_553_600, 60_000), (6, 8_388_608, 8_388_608, 80_000),            # more than 8 M elements, not more
    (10, 16_777_217, 6_553_600, 65_536), (12, 16_777_216, 6_553_600, 65_536)])        # more than 16 M, not more
def test_runs_and_tiles(ws, n, be, k):
    """The runs for up to twelve ranks, forced and where the sizes choose them, and the tile kernels."""
    rng = np.random.default_rng(n + ws)
    buckets = [min(be, n - lo) for lo in range(0, n, be)]
    per_rank = []
    for r in range(ws):
        row = []
        for m in buckets:
            kr = max(1, min(m, k) - r)
            idx = np.unique(rng.integers(0, m, kr)) if m > 1_000_000 else np.sort(rng.choice(m, kr, replace=False))
            row.append((idx, rng.standard_normal(idx.size).astype(np.float32)))
        per_rank.append(row)
    run_case(hip_ops, per_rank, n, be, 1.0 / ws, paths=RUNS)
    hip_ops.set_tuning("sparse_run_steps", 2)   # (the runs, whatever the size)
    try:
        run_case(hip_ops, per_rank, n, be, 1.0 / ws, paths=("auto",))
    finally:
        hip_ops.set_tuning("sparse_run_steps", 0)


@pytest.mark.parametrize("ws", [6, 9, 12])
@pytest.mark.parametrize("at", [0, 63, 79, 80, 3000])
def test_many_ranks_flag_payloads_out_of_order(ws, at):
    n, k = 300_000, 3003
    rng = np.random.default_rng(at)
    wires = []
    for r in range(ws):
        idx = np.sort(rng.choice(n, k, replace=False))
        if r == ws - 1:
            idx[[at, at + 1]] = idx[[at + 1, at]]
        wires.append(torch.from_numpy(payload(idx, np.ones(k, np.float32), k)).to(DEV))
    for path in (0, 1, 2, 3):
        status = torch.zeros(1, dtype=torch.int32, device=DEV)
        hip_ops.set_tuning("sparse_path", path)
        try:
            hip_ops.sparse_accumulate(torch.empty(n, device=DEV), wires, 4 + 8 * k, bucket_elems=n, status=status)
        finally:
            hip_ops.set_tuning("sparse_path", 0)
        assert int(status) == oracle.ERR_INDEX, path
