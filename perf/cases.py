"""Workloads by which this package's speed is judged: what one rank of a data-parallel job does
to its gradient buckets, called through the public entry points, from the smallest bucket (a few
thousand elements, where launches and host time count) to a whole 96.5 M-element gradient held by
eight ranks.

A case is a dict of plain values.  ``listed()`` gives the fixed ones, ``draw(rng)`` one more out of
the same ranges, ``prepare`` what a program holds before the call (gradients, residuals, payloads,
workspaces), ``run`` one pass, ``work`` the bytes and operations the pass cannot do without and
``tolerance`` how far another correct implementation may be off.

kinds
  ring       hip_ops.ring_fold: the reduce half of a ring allreduce over `ws` rank buffers, AVG
             fused where asked for
  fold       hip_ops.fold2 / fold2_scale: one inbound chunk folded into the local one, in place
  foldlist   hip_ops.fold2_batch: the folds of one ring step over all buckets of a gradient
  topk       hip_ops.topk_compress: the top-k payloads of all buckets of a gradient in one call,
             error feedback in the caller's residual
  topklist   TopKCompressor.compress_many: a list of separate buckets of different lengths
  wire_topk  TopKCompressor.compress and .decompress: a bucket to its payload and back, as an
             exchange with a peer does
  wire_fp16  FP16Compressor.compress and .decompress: the half-precision transport, both ways
  sparse     hip_ops.sparse_accumulate: `ws` ranks' top-k payloads into one dense gradient
"""
import math

import torch
import torch.distributed  # noqa: F401  (registers the c10d types the extension builds on)

from mccl_amd import _C, hip_ops

GRADIENT = 96_510_024  # elements: the gradient of the benchmark's model
BUCKET = 6_553_600     # elements: 25 MiB of fp32, the default bucket of data-parallel training

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
           "i32": torch.int32, "i64": torch.int64}
_OPS = {"sum": hip_ops.SUM, "avg": hip_ops.AVG, "min": hip_ops.MIN, "max": hip_ops.MAX}


def listed():
    return [
        # the headline: eight ranks' fp32 gradients reduced in ring order, averaged
        {"name": "ring_f32_w8_gradient", "kind": "ring", "dtype": "f32", "ws": 8, "n": GRADIENT, "bucket": BUCKET,
         "op": "avg", "chunked": False, "stepwise": False},
        # mixed-precision training: four ranks' bf16 gradients, rounded after every step as on the wire
        {"name": "ring_bf16_w4_gradient", "kind": "ring", "dtype": "bf16", "ws": 4, "n": GRADIENT,
         "bucket": 2 * BUCKET, "op": "avg", "chunked": False, "stepwise": True},
        # a layer of odd length over three ranks, the largest magnitude wanted (gradient scaling)
        {"name": "ring_f16_w3_max_odd", "kind": "ring", "dtype": "f16", "ws": 3, "n": 1_000_003, "bucket": 1_000_003,
         "op": "max", "chunked": True, "stepwise": False},
        # one ring step of one bucket over eight ranks: one chunk folded
        {"name": "fold_f32_chunk", "kind": "fold", "dtype": "f32", "n": BUCKET // 8, "op": "sum"},
        # the smallest calls: a bias-sized bucket of odd length, averaged between two ranks
        {"name": "fold_bf16_tiny", "kind": "fold", "dtype": "bf16", "n": 4099, "op": "avg"},
        # the folds of one ring step over all fifteen buckets, eight chunks each, as one list
        {"name": "foldlist_f32_ring_step", "kind": "foldlist", "dtype": "f32", "n": GRADIENT, "bucket": BUCKET,
         "chunks": 8, "op": "sum"},
        # top-k 1 % with error feedback over the whole gradient, bucket by bucket in one call
        {"name": "topk_gradient", "kind": "topk", "n": GRADIENT, "bucket": BUCKET, "ratio": 0.01},
        # the tensor list of a coalesced allreduce: layers of very different, odd lengths
        {"name": "topklist_ragged", "kind": "topklist", "buckets": 24, "smallest": 1001, "largest": 1_500_001,
         "ratio": 0.01},
        # one default bucket to its payload and back
        {"name": "wire_topk_bucket", "kind": "wire_topk", "n": BUCKET, "ratio": 0.01},
        # a small bucket of odd length to its payload and back
        {"name": "wire_topk_small", "kind": "wire_topk", "n": 65_537, "ratio": 0.01},
        # one default bucket, a few elements short, as halves to the peer and back
        {"name": "wire_fp16_bucket", "kind": "wire_fp16", "n": BUCKET - 5},
        # eight ranks' payloads added up into the dense gradient, averaged
        {"name": "sparse_w8_gradient", "kind": "sparse", "ws": 8, "n": GRADIENT, "bucket": BUCKET, "ratio": 0.01},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm; odd in half of the draws."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v |= 1
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["ring", "ring", "fold", "fold", "foldlist", "topk", "topklist", "wire_topk", "wire_topk",
                       "wire_fp16", "sparse"])
    if kind == "ring":
        n = _log_int(rng, 1000, GRADIENT)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "bf16", "f16"]), "ws": rng.randint(2, 8), "n": n,
                "bucket": min(n, BUCKET), "op": rng.choice(["sum", "avg", "avg", "max", "min"]),
                "chunked": rng.random() < 0.5, "stepwise": rng.random() < 0.5}
    if kind == "fold":
        dtype = rng.choice(["f32", "f32", "bf16", "f16", "i64", "i32"])
        ops = ["sum", "max", "min"] if dtype[0] == "i" else ["sum", "sum", "avg", "max", "min"]
        return {"kind": kind, "dtype": dtype, "n": _log_int(rng, 64, BUCKET if dtype[0] == "i" else 4 * BUCKET),
                "op": rng.choice(ops)}
    if kind == "foldlist":
        n = _log_int(rng, BUCKET // 8, GRADIENT)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "bf16", "f16"]), "n": n, "bucket": min(n, BUCKET),
                "chunks": rng.randint(2, 16), "op": rng.choice(["sum", "sum", "max", "min"])}
    if kind == "topk":
        n = _log_int(rng, BUCKET, GRADIENT)
        return {"kind": kind, "n": n, "bucket": rng.choice([BUCKET, BUCKET, _log_int(rng, BUCKET // 4, 2 * BUCKET)]),
                "ratio": rng.choice([0.001, 0.01, 0.01, 0.01, 0.05])}
    if kind == "topklist":
        return {"kind": kind, "buckets": rng.randint(2, 30), "smallest": _log_int(rng, 200, 20_000),
                "largest": _log_int(rng, 100_000, BUCKET), "ratio": rng.choice([0.001, 0.01, 0.01, 0.05])}
    if kind == "wire_topk":
        return {"kind": kind, "n": _log_int(rng, 1000, 2 * BUCKET), "ratio": rng.choice([0.001, 0.01, 0.01, 0.05])}
    if kind == "wire_fp16":
        return {"kind": kind, "n": _log_int(rng, 1000, 4 * BUCKET)}
    return {"kind": kind, "ws": rng.randint(2, 12), "n": _log_int(rng, 200_000, GRADIENT), "bucket": BUCKET,
            "ratio": rng.choice([0.001, 0.01, 0.01, 0.02])}


def _buckets(n, bucket):
    return [(lo, min(n, lo + bucket)) for lo in range(0, n, bucket)]


def _lengths(case):
    """Lengths of a ragged bucket list: spread evenly over the logarithm, in no order of size."""
    count, a, b = case["buckets"], math.log(case["smallest"]), math.log(case["largest"])
    sizes = [int(round(math.exp(a + (b - a) * i / (count - 1)))) for i in range(count)]
    return sizes[::2] + sizes[1::2][::-1]


def _gen(dev, seed):
    return torch.Generator(device=dev).manual_seed(seed)


def _normal(n, gen, dev, scale):
    return torch.randn(n, generator=gen, device=dev).mul_(scale)


def _values(n, dtype, gen, dev):
    """Gradient values: N(0, 1e-3), in half formats with 0.1 % outliers a thousand times as large."""
    if dtype in (torch.int32, torch.int64):
        return torch.randint(-10 ** 6, 10 ** 6, (n,), generator=gen, device=dev, dtype=dtype)
    x = _normal(n, gen, dev, 1e-3)
    if dtype == torch.float32:
        return x
    m = torch.rand(n, generator=gen, device=dev) < 1e-3
    return torch.where(m, x * 1e3, x).to(dtype)


def _heavy_tailed(n, gen, dev):
    """Gradient values for the sparsifier: Student-t with three degrees of freedom, 1e-3 wide, 1 %
    of them exact duplicates (in magnitude) of others, so that ties occur."""
    x = torch.randn(n, generator=gen, device=dev)
    chi = torch.zeros(n, device=dev)
    for _ in range(3):
        chi += torch.randn(n, generator=gen, device=dev).square_()
    x.div_(chi.div_(3).sqrt_()).mul_(1e-3)
    m = n // 100
    if m:
        # every m-th element takes over the magnitude of the element drawn for it
        dst = torch.arange(m, device=dev) * (n // m)
        src = torch.randint(0, n, (m,), generator=gen, device=dev)
        x[dst] = x[src].neg()
    return x


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    gen = _gen(dev, seed)
    s = {"case": case}
    if kind == "ring":
        dtype, n, ws = _DTYPES[case["dtype"]], case["n"], case["ws"]
        s["ins"] = [_values(n, dtype, gen, dev) for _ in range(ws)]
        s["out"] = torch.empty(n, dtype=dtype, device=dev)
        s["scale"] = 1.0 / ws if case["op"] == "avg" else None
    elif kind == "fold":
        dtype = _DTYPES[case["dtype"]]
        s["dst"] = _values(case["n"], dtype, gen, dev)
        s["src"] = _values(case["n"], dtype, gen, dev)
    elif kind == "foldlist":
        dtype, n, c = _DTYPES[case["dtype"]], case["n"], case["chunks"]
        s["dst"] = _values(n, dtype, gen, dev)
        s["src"] = _values(n, dtype, gen, dev)
        s["dsts"], s["srcs"] = [], []
        for lo, hi in _buckets(n, case["bucket"]):
            ce = (hi - lo + c - 1) // c
            for a in range(lo, hi, ce):
                b = min(hi, a + ce)
                s["dsts"].append(s["dst"][a:b])
                s["srcs"].append(s["src"][a:b])
    elif kind == "topk":
        n, bucket, ratio = case["n"], min(case["bucket"], case["n"]), case["ratio"]
        s["grad"] = _heavy_tailed(n, gen, dev)
        s["residual"] = _normal(n, gen, dev, 1e-4)
        s["stride"] = hip_ops.topk_wire_stride(bucket, ratio)
        s["wire"] = torch.zeros(len(_buckets(n, bucket)) * s["stride"], dtype=torch.uint8, device=dev)
        s["workspace"] = hip_ops.topk_workspace(n, bucket, ratio, dev)
    elif kind == "topklist":
        s["grads"] = [_heavy_tailed(n, gen, dev) for n in _lengths(case)]
        s["ids"] = list(range(1, len(s["grads"]) + 1))
        s["compressor"] = _C.make_compressor(_C.CompressionMode.TOPK, case["ratio"])
    elif kind == "wire_topk":
        s["grad"] = _heavy_tailed(case["n"], gen, dev)
        s["compressor"] = _C.make_compressor(_C.CompressionMode.TOPK, case["ratio"])
    elif kind == "wire_fp16":
        s["grad"] = _normal(case["n"], gen, dev, 1e-3)
        s["compressor"] = _C.make_compressor(_C.CompressionMode.FP16)
    else:
        n, bucket, ratio, ws = case["n"], min(case["bucket"], case["n"]), case["ratio"], case["ws"]
        s["stride"] = hip_ops.topk_wire_stride(bucket, ratio)
        workspace = hip_ops.topk_workspace(n, bucket, ratio, dev)
        # large elements that the ranks share, so that about 30 % of their picks coincide
        shared = torch.rand(n, generator=gen, device=dev) < 0.4 * ratio
        s["wires"] = []
        for _ in range(ws):
            g = _normal(n, gen, dev, 1e-2)
            g = torch.where(shared, g * 50.0, g)
            wire = torch.zeros(len(_buckets(n, bucket)) * s["stride"], dtype=torch.uint8, device=dev)
            hip_ops.topk_compress(g, torch.zeros(n, device=dev), ratio, bucket_elems=bucket, wire=wire,
                                  workspace=workspace, wire_stride=s["stride"])
            s["wires"].append(wire)
        s["acc"] = torch.empty(n, device=dev)
        s["status"] = torch.zeros(1, dtype=torch.int32, device=dev)
        s["workspace"] = hip_ops.sparse_workspace(n, bucket, ws, dev)
    return s


def _residual(s, ident):
    """The compressor's error-feedback buffer, which it keeps in place from the first pass on."""
    kept = s.setdefault("residuals", {})
    if ident not in kept:
        kept[ident] = s["compressor"].error_feedback_buffer(ident)
    return kept[ident]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ring":
        return hip_ops.ring_fold(s["out"], s["ins"], _OPS[case["op"]],
                                 hip_ops.RING_CHUNKED if case["chunked"] else hip_ops.RING_BASIC,
                                 bucket_elems=case["bucket"], scale_by=s["scale"], stepwise=case["stepwise"])
    if kind == "fold":
        if case["op"] == "avg":
            return hip_ops.fold2_scale(s["dst"], s["src"], 0.5)
        return hip_ops.fold2(s["dst"], s["src"], _OPS[case["op"]])
    if kind == "foldlist":
        hip_ops.fold2_batch(s["dsts"], s["srcs"], _OPS[case["op"]])
        return s["dst"]
    if kind == "topk":
        hip_ops.topk_compress(s["grad"], s["residual"], case["ratio"], bucket_elems=case["bucket"], wire=s["wire"],
                              workspace=s["workspace"], wire_stride=s["stride"])
        return {"wire": s["wire"], "residual": s["residual"]}
    if kind == "topklist":
        wires = s["compressor"].compress_many(s["grads"], s["ids"])
        return {"wires": wires, "residuals": [_residual(s, i) for i in s["ids"]]}
    if kind == "wire_topk":
        wire = s["compressor"].compress(s["grad"], stable_id=1)
        dense = s["compressor"].decompress(wire, case["n"])
        return {"wire": wire, "dense": dense, "residual": _residual(s, 1)}
    if kind == "wire_fp16":
        wire = s["compressor"].compress(s["grad"])
        return {"wire": wire, "dense": s["compressor"].decompress(wire, case["n"])}
    hip_ops.sparse_accumulate(s["acc"], s["wires"], s["stride"], bucket_elems=case["bucket"],
                              scale_by=1.0 / case["ws"], status=s["status"], workspace=s["workspace"])
    return {"acc": s["acc"], "status": s["status"]}


def _k(count, ratio):
    return max(1, int(count * ratio))


def work(case):
    """Each input read once and each output written once; one operation per addition or comparison."""
    kind = case["kind"]
    if kind == "ring":
        es = _DTYPES[case["dtype"]].itemsize
        return {"bytes": (case["ws"] + 1) * es * case["n"], "flops": case["ws"] * case["n"]}
    if kind in ("fold", "foldlist"):
        return {"bytes": 3 * _DTYPES[case["dtype"]].itemsize * case["n"], "flops": case["n"]}
    if kind == "topk":
        ks = sum(_k(b - a, case["ratio"]) * 8 + 4 for a, b in _buckets(case["n"], case["bucket"]))
        return {"bytes": 12 * case["n"] + ks, "flops": case["n"]}
    if kind == "topklist":
        return {"bytes": sum(12 * n + 8 * _k(n, case["ratio"]) + 4 for n in _lengths(case)),
                "flops": sum(_lengths(case))}
    if kind == "wire_topk":
        pairs = 8 * _k(case["n"], case["ratio"]) + 4
        return {"bytes": 12 * case["n"] + pairs + 4 * case["n"] + pairs, "flops": case["n"]}
    if kind == "wire_fp16":
        return {"bytes": 12 * case["n"], "flops": 2 * case["n"]}
    pairs = sum(_k(b - a, case["ratio"]) * 8 + 4 for a, b in _buckets(case["n"], case["bucket"]))
    return {"bytes": 4 * case["n"] + case["ws"] * pairs, "flops": case["ws"] * pairs // 8}


def tolerance(case):
    """Every result is defined bit for bit: folds are single IEEE operations in ring order, picks
    are ordered by magnitude with ties to the lower index, casts round to nearest even."""
    return "exact"
