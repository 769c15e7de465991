"""The resident top-k path (one launch, the bucket kept on chip) against the oracle, bit for bit, at
the sizes where its block layout changes (4096 * 1 / 2 / 4 elements per block, one block against
several, a partial last vector) and on the inputs that steer its rounds: a sampled window that
holds, one that misleads, more equal keys than its list holds, ratios from one pick to all."""
import numpy as np
import pytest
import torch

import oracle
from oracle import F32
from tests._gpu_util import DEV, to_dev, to_np, bits, student_t

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 4095, 4096, 4097, 12_289, 262_143, 262_144, 262_145, 524_288, 524_289, 1_048_576, 1_048_577,
         2_097_151, 2_097_152]


@pytest.fixture()
def ops():
    from mccl_amd import hip_ops
    hip_ops.set_tuning("topk_path", 3)
    yield hip_ops
    hip_ops.set_tuning("topk_path", 0)


def _values(kind, n):
    rng = np.random.default_rng(n)
    if kind == "spread":
        return student_t(rng, n, ties=0.01), (rng.standard_normal(n) * 1e-4).astype(np.float32)
    if kind == "tied":        # a few values, signed zeros among them: the threshold is shared by thousands
        g = rng.choice(np.array([0.0, -0.0, 0.5, -0.5, 1.0, 2.0], np.float32), n)
    elif kind == "zero":      # nothing but ties
        g = np.zeros(n, np.float32)
    else:                     # "misled": every sampled run of 32 elements is large, nothing else is
        g = student_t(rng, n, ties=0.0) * np.float32(1e-6)
        step = max(n // 256 // 4 * 4, 32)
        for i in range(0, n, step):
            g[i:i + 32] = 5.0
    return g, np.zeros(n, np.float32)


def _check(ops, g, r, ratio):
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    dg, dr = to_dev(g, F32, g.size % 4), to_dev(r, F32, g.size % 3)
    wire, _ = ops.topk_compress(dg, dr, ratio, status=status)
    want = r.copy()
    w, rc = oracle.topk_compress(g, want, ratio)
    assert int(status) == 0
    assert wire.cpu().numpy()[:rc].tobytes() == w.tobytes()
    assert np.array_equal(bits(to_np(dr, F32)), bits(want))
    assert np.array_equal(bits(to_np(dg, F32)), bits(g))


@pytest.mark.parametrize("kind", ["spread", "tied", "zero", "misled"])
@pytest.mark.parametrize("n", SIZES)
def test_resident_equals_oracle(ops, n, kind):
    g, r = _values(kind, n)
    for ratio in (0.001, 0.01, 0.05) if n > 600_000 else (0.001, 0.01, 0.3, 1.0):
        _check(ops, g, r, ratio)


def test_resident_lists_and_uniform_buckets(ops):
    rng = np.random.default_rng(7)
    sizes = [1, 4096, 4097, 30_001, 262_145, 77]
    grads = [student_t(rng, n) for n in sizes]
    res = [(rng.standard_normal(n) * 1e-4).astype(np.float32) for n in sizes]
    dres = [to_dev(r, F32) for r in res]
    wires = ops.topk_compress_list([to_dev(x, F32) for x in grads], dres, 0.01)
    for x, r, dr, wv in zip(grads, res, dres, wires):
        w, rc = oracle.topk_compress(x, r, 0.01)
        assert wv.cpu().numpy()[:rc].tobytes() == w.tobytes()
        assert np.array_equal(bits(to_np(dr, F32)), bits(r))
    # buckets of one buffer, as many blocks as one launch may have (128 on 256 CUs), a short last bucket
    be, nb = 50_001, 32
    n = be * nb - 20_000
    g, r = student_t(rng, n), np.zeros(n, np.float32)
    dr = to_dev(r, F32)
    wire, stride = ops.topk_compress(to_dev(g, F32), dr, 0.01, bucket_elems=be)
    host = wire.cpu().numpy()
    for b in range(nb):
        s, e = b * be, min(n, (b + 1) * be)
        sub = r[s:e].copy()
        w, rc = oracle.topk_compress(g[s:e].copy(), sub, 0.01)
        r[s:e] = sub
        assert host[b * stride: b * stride + rc].tobytes() == w.tobytes(), b
    assert np.array_equal(bits(to_np(dr, F32)), bits(r))


def test_resident_list_longest_first(ops):
    """A list of every length class at once - one block, several with and without a sample, 128 -
    in an order that is not by length, up to the most buckets a call takes."""
    rng = np.random.default_rng(11)
    sizes = [5, 32_767, 600_001, 4097, 32_768, 16_385, 16_384, 700_003, 1, 65_537] + [1000 + 37 * i for i in range(54)]
    grads = [student_t(rng, n) for n in sizes]
    res = [(rng.standard_normal(n) * 1e-4).astype(np.float32) for n in sizes]
    dres = [to_dev(r, F32) for r in res]
    wires = ops.topk_compress_list([to_dev(x, F32) for x in grads], dres, 0.01)
    for x, r, dr, wv in zip(grads, res, dres, wires):
        w, rc = oracle.topk_compress(x, r, 0.01)
        assert wv.cpu().numpy()[:rc].tobytes() == w.tobytes(), x.size
        assert np.array_equal(bits(to_np(dr, F32)), bits(r)), x.size


def test_resident_list_in_several_launches(ops):
    """More waiting blocks than one launch may have: the longest bucket of all, whose 128 blocks fill
    a launch, others that share one, and the short ones that go with the first."""
    rng = np.random.default_rng(13)
    sizes = [700_003, 4096, 2_097_152, 16_385, 1_500_001, 3, 600_001, 1_048_577, 40_000]
    grads = [student_t(rng, n) for n in sizes]
    res = [(rng.standard_normal(n) * 1e-4).astype(np.float32) for n in sizes]
    dres = [to_dev(r, F32) for r in res]
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    for ratio in (0.01, 0.05):
        wires = ops.topk_compress_list([to_dev(x, F32) for x in grads], dres, ratio, status=status)
        for x, r, dr, wv in zip(grads, res, dres, wires):
            w, rc = oracle.topk_compress(x, r, ratio)
            assert wv.cpu().numpy()[:rc].tobytes() == w.tobytes(), (x.size, ratio)
            assert np.array_equal(bits(to_np(dr, F32)), bits(r)), (x.size, ratio)
    assert int(status) == 0
