"""hip_ops and the one-C-call functions beneath it: a call that has reached the library is raised
from its status and never made a second time, whatever the status says - folds and compress update
their operands in place."""
import pytest
import torch

from mccl_amd import _lib, hip_ops as ops

T = torch.zeros(8)
B = torch.zeros(64, dtype=torch.uint8)
CALLS = {
    "fold2": lambda: ops.fold2(T, T),
    "fold2_scale": lambda: ops.fold2_scale(T, T, 0.5),
    "fold2_batch": lambda: ops.fold2_batch([T], [T]),
    "ring_fold": lambda: ops.ring_fold(T, [T, T]),
    "topk_compress": lambda: ops.topk_compress(T, T, 0.5, bucket_elems=8, wire=B, workspace=B, wire_stride=36),
    "sparse_accumulate": lambda: ops.sparse_accumulate(T, [B], 36, bucket_elems=8, workspace=B),
}


class _Native:
    """Every fast function counts its call and returns one status."""

    def __init__(self, rc):
        self.rc, self.calls = rc, []

    def __getattr__(self, name):
        return lambda *args: (self.calls.append(name), self.rc)[1]


@pytest.mark.parametrize("rc", [-7, -6, -8])
@pytest.mark.parametrize("name", list(CALLS))
def test_an_error_is_raised_and_the_call_not_repeated(monkeypatch, name, rc):
    native = _Native(rc)
    monkeypatch.setattr(ops, "_native", native)
    monkeypatch.setattr(ops, "_stream", lambda: pytest.fail("called the library a second time"))
    monkeypatch.setattr(ops, "_dev", lambda *a, **k: None)
    with pytest.raises(_lib.MCCLHipError) as e:
        CALLS[name]()
    assert e.value.code == rc and name in str(e.value)
    assert native.calls == ["_fast_" + name]


@pytest.mark.parametrize("name", list(CALLS))
def test_none_goes_through_the_checks(monkeypatch, name):
    monkeypatch.setattr(ops, "_native", _Native(None))
    with pytest.raises(ValueError, match="must live on the GPU"):
        CALLS[name]()


def test_the_extension_leaves_what_is_not_well_formed():
    import torch.distributed  # noqa: F401
    from mccl_amd import _C
    assert _C._fast_fold2(T, T, 0) is None
    assert _C._fast_fold2_scale(T, T, 0.5) is None
    assert _C._fast_fold2_batch([T], [T], 0) is None
    assert _C._fast_ring_fold(T, [T], 0, 0, 8, None, 0) is None
    assert _C._fast_topk_compress(T, T, 0.5, 8, B, B, 36, None) is None
    assert _C._fast_sparse_accumulate(T, [B], 36, 8, None, None, B) is None


@pytest.mark.gpu
def test_in_place_calls_run_once_behind_an_error_left_by_another_call():
    dev = "cuda:0"
    lib = _lib.load()
    a, b = torch.full((1000,), 3.0, device=dev), torch.full((1000,), 2.0, device=dev)
    wire = torch.zeros(ops.topk_wire_stride(1000, 0.1), dtype=torch.uint8, device=dev)
    ws = ops.topk_workspace(1000, 1000, 0.1, dev)
    torch.cuda.synchronize()

    def behind_an_error(call):
        """call() on a thread whose last HIP error is set; what it does must happen once."""
        assert lib.hipSetDevice(100_000) != 0   # refused by the runtime: no such device
        try:
            call()
        except _lib.MCCLHipError as e:
            assert e.code == -7
        lib.hipGetLastError()
        torch.cuda.synchronize()

    d = a.clone()
    torch.cuda.synchronize()
    behind_an_error(lambda: ops.fold2(d, b))
    assert (d == 5.0).all()
    d = a.clone()
    behind_an_error(lambda: ops.fold2_scale(d, b, 0.5))
    assert (d == 2.5).all()
    d = a.clone()
    behind_an_error(lambda: ops.fold2_batch([d[:500], d[500:]], [b[:500], b[500:]]))
    assert (d == 5.0).all()
    r = a.clone()
    behind_an_error(lambda: ops.topk_compress(b, r, 0.1, bucket_elems=1000, wire=wire, workspace=ws, wire_stride=wire.numel()))
    assert (r[:100] == 0.0).all() and (r[100:] == 5.0).all()
    with pytest.raises(_lib.MCCLHipError) as e:
        ops.fold2(d, b, 5)   # no such op: refused by the library, nothing launched
    assert e.value.code == -1 and (d == 5.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [2 ** 62, 2 ** 62 + 4, 2 ** 63 - 4, 40])
def test_a_payload_buffer_shorter_than_its_rows_is_refused(stride):
    """Four rows of 2^62 bytes are 2^64, which 64 bits do not hold: nothing may be launched."""
    dev = "cuda:0"
    t, r = torch.ones(32, device=dev), torch.zeros(32, device=dev)
    wire = torch.zeros(4 * 36, dtype=torch.uint8, device=dev)
    ws = ops.topk_workspace(32, 8, 0.5, dev)
    with pytest.raises(ValueError, match="wire holds 144 elements"):
        ops.topk_compress(t, r, 0.5, bucket_elems=8, wire=wire, workspace=ws, wire_stride=stride)
    with pytest.raises(ValueError, match="holds 144 elements"):
        ops.sparse_accumulate(r, [wire], stride, bucket_elems=8, workspace=ws)
    torch.cuda.synchronize()
    assert (r == 0.0).all() and (wire == 0).all()
