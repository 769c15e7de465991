"""What the compressors allocate for payloads and results is seen by dispatch modes and profilers, and filled where new memory
is to be filled, as any tensor of torch's own."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tests._gpu_util import DEV

pytestmark = pytest.mark.gpu


class _Empties(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        if func is torch.ops.aten.empty.memory_format:
            self.seen.append((out.numel(), out.dtype))
        return out


@pytest.fixture()
def compressors():
    from mccl_amd import _C
    return _C.make_compressor(_C.CompressionMode.TOPK, 0.01), _C.make_compressor(_C.CompressionMode.FP16)


def test_a_dispatch_mode_sees_them(compressors):
    topk, half = compressors
    x = torch.randn(5000, device=DEV)
    topk.compress(x, stable_id=1)
    with _Empties() as mode:
        wire = topk.compress(x, stable_id=1)
        topk.decompress(wire, 5000)
        topk.compress_many([x, x[:1000]], [1, 2])
        half.decompress(half.compress(x), 5000)
    for want in [(404, torch.uint8), (5000, torch.float32), (84, torch.uint8), (half.max_compressed_size(20_000), torch.uint8)]:
        assert want in mode.seen, (want, mode.seen)


def test_a_profiler_sees_them(compressors):
    _, half = compressors
    x = torch.randn(5000, device=DEV)
    half.compress(x)
    with torch.autograd.profiler.profile() as prof:
        half.compress(x)
    assert any(e.name == "aten::empty" for e in prof.function_events)


def test_new_memory_is_filled_where_that_is_asked_for(compressors):
    _, half = compressors
    x = torch.randn(5000, device=DEV)
    fill = torch.utils.deterministic.fill_uninitialized_memory
    torch.use_deterministic_algorithms(True)
    torch.utils.deterministic.fill_uninitialized_memory = True
    try:
        wire = half.compress(x, capacity=20_000)
    finally:
        torch.use_deterministic_algorithms(False)
        torch.utils.deterministic.fill_uninitialized_memory = fill
    behind = torch.empty(0, dtype=torch.uint8, device=DEV).set_(wire.untyped_storage())[10_000:20_000]
    assert bool((behind == 255).all())
