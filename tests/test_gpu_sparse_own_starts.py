"""Sparse accumulate of one bucket, where a block finds the starts of its runs itself: at the edges
of the run, the block and the sample count, against the oracle and against the position table."""
import numpy as np
import pytest
import torch

import oracle
from mccl_amd import hip_ops
from tests._gpu_util import DEV
from tests.test_gpu_sparse_runs import payload, run_case

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
    run_case(hip_ops, ranks(rng, ws, n, k), n, n, 1.0 / ws, paths=("auto",))


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
    for path in (0, 2):
        status = torch.zeros(1, dtype=torch.int32, device=DEV)
        hip_ops.set_tuning("sparse_path", path)
        try:
            hip_ops.sparse_accumulate(torch.empty(n, device=DEV), wires, 4 + 8 * k, bucket_elems=n, status=status)
        finally:
            hip_ops.set_tuning("sparse_path", 0)
        assert int(status) == oracle.ERR_INDEX, path
