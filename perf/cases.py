"""What the framework's speed is measured on: the calls its users make, over the range of sizes they make them at.

A case is a dict of plain values. Its "kind" names the public entry point a pass goes through:

* ``kernel``: a single-table pooled lookup from the kernel factories (``ops.generate_embedding_spmdm*``), the form in
  which host code written against the core library calls it: synchronous, with the reference's ``bool``;
* ``module``: ``IntNBitTableBatchedEmbeddingBagsCodegen.forward``, what a serving process calls once per request
  batch: bounds check, pruned-row remap and the lookup over all tables;
* ``operator``: ``torch.ops.fbgemm.int_nbit_split_embedding_codegen_lookup_function``, what an exported or scripted
  model calls (with ``fast``, the Python operator with a plan in the tolerance-grade mode, which only it can select);
* ``quantize`` / ``dequantize``: float rows to the fused row formats and back, what a model publisher runs over whole
  tables, and what a consumer of the 8-bit rows runs.

Sizes are those of the five benchmark workloads (``fbgemm_amd/bench_configs.py``), of ``bench.py``'s side operators and
of the core library's microbenchmark shape, smaller where tables had to shrink so that several sets of inputs fit one
GPU. Tables, indices, lengths and per-sample weights are drawn on the GPU from the seed.
"""
import math

import numpy as np
import torch

from fbgemm_amd import module as tbe
from fbgemm_amd import ops
from fbgemm_amd.build import TORCH_OP_OUT

_TYPES = {"fp32": ops.FP32, "fp16": ops.FP16, "int8": ops.INT8, "int4": ops.INT4, "int2": ops.INT2, "fp8": ops.FP8, "bf16": ops.BF16}
_BITS = {"fp32": 32, "fp16": 16, "int8": 8, "int4": 4, "int2": 2, "fp8": 8}
_TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_OUT_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}

# the table sets of the table-batched cases: (row types, row widths), one of each drawn per table
_SETS = {
    "mixed": (("int4", "int4", "int8", "fp16"), (64, 128, 256)),              # config 3's mix
    "int4": (("int4",), (64,)),                                               # config 4's pruned tables
    "wide": (("int4",) * 12 + ("int2",), (256,)),                             # config 5: mostly int4 x 256, some int2 x 32
    "sequence": (("int4",), (128,)),
    "ragged": (("int2", "int4", "int8", "int8", "fp16", "fp32", "fp8"), (4, 12, 20, 36, 52, 100, 200, 300)),
}


def listed():
    return [
        # The core library's own microbenchmark shape: ten long bags of a 4-bit table. The smallest call a user makes;
        # launches and the chain of dependent loads inside a bag are all there is to it.
        {"name": "kernel_few_bags", "kind": "kernel", "type": "int4", "dim": 128, "rows": 4_000_000, "bags": 10, "length": 101,
         "spread": "uniform", "alpha": 0.0, "weighted": False, "mean": False, "output": "fp32", "lengths": False, "index": "int64"},
        # Config 1: one fused 8-bit table, an ordinary CPU-side batch.
        {"name": "kernel_8bit", "kind": "kernel", "type": "int8", "dim": 128, "rows": 100_000, "bags": 1024, "length": 20,
         "spread": "fixed", "alpha": 0.0, "weighted": False, "mean": False, "output": "fp32", "lengths": False, "index": "int64"},
        # Config 2: one 4-bit table of 4 M rows, skewed indices, ragged bags, fp16 output.
        {"name": "kernel_4bit", "kind": "kernel", "type": "int4", "dim": 128, "rows": 4_000_000, "bags": 4096, "length": 20,
         "spread": "uniform", "alpha": 1.05, "weighted": False, "mean": False, "output": "fp16", "lengths": False, "index": "int64"},
        # A width that fills no whole 16-byte chunks, Caffe2-style lengths, 32-bit indices, weighted mean.
        {"name": "kernel_odd", "kind": "kernel", "type": "int8", "dim": 100, "rows": 1_000_000, "bags": 10_000, "length": 25,
         "spread": "poisson", "alpha": 1.1, "weighted": True, "mean": True, "output": "fp32", "lengths": True, "index": "int32"},
        # One small request batch against 64 mixed tables through the module, bounds check on as by default.
        {"name": "module_request", "kind": "module", "set": "mixed", "tables": 64, "min_rows": 20_000, "max_rows": 1_000_000, "batch": 32,
         "length": 30, "spread": "poisson", "alpha": 1.1, "weighted": True, "pooling": "sum", "output": "fp16", "pruned": False,
         "check": True, "index": "int32"},
        # Config 4: half of the rows pruned through an index mapping, mean pooling, fp32 output, through the module.
        {"name": "module_pruned", "kind": "module", "set": "int4", "tables": 32, "min_rows": 1_000_000, "max_rows": 1_000_000, "batch": 4096,
         "length": 27, "spread": "uniform", "alpha": 1.05, "weighted": False, "pooling": "mean", "output": "fp32", "pruned": True,
         "check": True, "index": "int64"},
        # Tables of every row type at widths that are no power of two: the shapes the general kernel takes.
        {"name": "module_ragged", "kind": "module", "set": "ragged", "tables": 40, "min_rows": 10_000, "max_rows": 1_000_000, "batch": 1000,
         "length": 12, "spread": "poisson", "alpha": 1.1, "weighted": False, "pooling": "mean", "output": "fp32", "pruned": False,
         "check": True, "index": "int32"},
        # Config 3, the headline workload: 64 mixed tables, 2 048 bags each, weighted sum, fp16 output.
        {"name": "operator_mixed", "kind": "operator", "set": "mixed", "tables": 64, "min_rows": 100_000, "max_rows": 10_000_000,
         "batch": 2048, "length": 30, "spread": "poisson", "alpha": 1.1, "weighted": True, "pooling": "sum", "output": "fp16",
         "fast": False, "index": "int64"},
        # Config 5 at a quarter of its tables: int4 rows of 256 columns, 16 384 bags per table, bf16 output, tolerance grade.
        {"name": "operator_large", "kind": "operator", "set": "wide", "tables": 104, "min_rows": 3_000_000, "max_rows": 3_000_000,
         "batch": 16384, "length": 15, "spread": "poisson", "alpha": 1.2, "weighted": False, "pooling": "sum", "output": "bf16",
         "fast": True, "index": "int64"},
        # Sequence output: one row per index, as attention-style consumers of the embeddings take them.
        {"name": "operator_sequence", "kind": "operator", "set": "sequence", "tables": 32, "min_rows": 1_000_000, "max_rows": 1_000_000,
         "batch": 4096, "length": 27, "spread": "uniform", "alpha": 0.0, "weighted": False, "pooling": "none", "output": "fp16",
         "fast": False, "index": "int64"},
        # A trained fp32 table becomes 4-bit rows in the table-batched layout.
        {"name": "quantize_4bit", "kind": "quantize", "type": "int4", "rows": 1 << 20, "cols": 128, "input": "fp32", "front": True},
        # 8-bit rows with fp32 scale and bias become fp16 rows.
        {"name": "dequantize_8bit", "kind": "dequantize", "type": "int8", "rows": 1 << 20, "cols": 128, "output": "fp16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["kernel", "kernel", "kernel", "module", "module", "module", "operator", "operator", "quantize", "dequantize"])
    if kind == "kernel":
        ty = rng.choice(["int4", "int4", "int8", "int8", "int2", "fp16"])
        bags = _log(rng, 1, 16384)
        length = min(_log(rng, 2, 200), max(2, 1_000_000 // bags))
        return {"kind": kind, "type": ty, "dim": rng.choice([32, 64, 128, 256, 4 * rng.randint(1, 128)]), "rows": _log(rng, 10_000, 4_000_000),
                "bags": bags, "length": length, "spread": rng.choice(["fixed", "uniform", "poisson"]), "alpha": rng.choice([0.0, 1.05, 1.2]),
                "weighted": rng.random() < 0.4, "mean": rng.random() < 0.3, "output": rng.choice(["fp32", "fp16"]),
                "lengths": rng.random() < 0.3, "index": rng.choice(["int64", "int32"])}
    if kind in ("module", "operator"):
        tables = _log(rng, 1, 96)
        batch = _log(rng, 1, 8192)
        length = min(_log(rng, 2, 100), max(2, 5_000_000 // (tables * batch)))
        min_rows = _log(rng, 1000, 1_000_000)
        case = {"kind": kind, "set": rng.choice(["mixed", "mixed", "int4", "wide", "ragged"]), "tables": tables, "min_rows": min_rows,
                "max_rows": min(2_000_000, min_rows * rng.choice([1, 10])), "batch": batch, "length": length,
                "spread": rng.choice(["fixed", "uniform", "poisson"]), "alpha": rng.choice([0.0, 1.05, 1.1, 1.2]),
                "weighted": rng.random() < 0.4, "pooling": rng.choice(["sum", "sum", "mean"]), "output": rng.choice(["fp32", "fp16", "bf16"]),
                "index": rng.choice(["int64", "int32"])}
        if kind == "module":
            case["pruned"] = rng.random() < 0.4
            case["check"] = rng.random() < 0.7
        else:
            case["fast"] = rng.random() < 0.4
            if rng.random() < 0.3:
                case.update({"set": "sequence", "pooling": "none", "fast": False, "weighted": False,
                             "length": min(length, max(2, 2_000_000 // (tables * batch)))})
        return case
    cols = rng.choice([32, 64, 128, 256, 8 * rng.randint(1, 128)])
    rows = min(_log(rng, 100, 2_000_000), (1 << 27) // cols)
    if kind == "quantize":
        return {"kind": kind, "type": rng.choice(["int4", "int8", "int2"]), "rows": rows, "cols": cols, "input": rng.choice(["fp32", "fp16"]),
                "front": rng.random() < 0.5}
    return {"kind": kind, "type": rng.choice(["int4", "int8", "int2"]), "rows": rows, "cols": cols, "output": rng.choice(["fp32", "fp16"])}


# ---- inputs ------------------------------------------------------------------------------------------------------


def _tables(case):
    """(row type, width, rows) of every table of a table-batched case: a function of the case alone."""
    types, dims = _SETS[case["set"]]
    rng = np.random.default_rng(4321 + case["tables"])
    specs = []
    for t in range(case["tables"]):
        ty = types[t % len(types)]
        dim = 32 if case["set"] == "wide" and ty == "int2" else int(rng.choice(dims))
        u = rng.uniform()
        rows = int(round(math.exp(math.log(case["min_rows"]) * (1 - u) + math.log(case["max_rows"]) * u)))
        specs.append((ty, dim, rows))
    return specs


def _bag_lengths(case, n, gen):
    mean = case["length"]
    if case["spread"] == "fixed":
        return torch.full((n,), mean, dtype=torch.int64, device="cuda")
    if case["spread"] == "uniform":
        return torch.randint(1, 2 * mean, (n,), generator=gen, device="cuda")
    return torch.poisson(torch.full((n,), float(mean), device="cuda"), generator=gen).clamp_(max=200).long()


def _row_ids(rows, alpha, gen):
    """One row id for every entry of ``rows`` (the row count of the entry's table). alpha 0: uniform. Otherwise the rank
    is Zipf-like (P(rank >= k) = k^(1 - alpha)), ranks past the table spread evenly over it, and a multiplication by a
    prime scatters neighbouring ranks over the table."""
    n = rows.numel()
    even = (torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) * rows).long()
    if alpha == 0.0:
        return torch.minimum(even, rows - 1)
    u = 1.0 - torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    rank = u.pow_(-1.0 / (alpha - 1.0)).clamp_(max=1e15).long() - 1
    rank = torch.where(rank < rows, rank, even)
    return (rank * 2_654_435_761 + 40_503) % rows


def _scales(n, fp16, gen):
    pair = torch.empty(n, 2, device="cuda")
    pair[:, 0].uniform_(0.001, 0.05, generator=gen)
    pair[:, 1].uniform_(-1.0, 1.0, generator=gen)
    return pair.half() if fp16 else pair


def _prepare_kernel(case, gen):
    ty, dim, rows = case["type"], case["dim"], case["rows"]
    if ty == "fp16":
        table = torch.empty(rows, dim, dtype=torch.float16, device="cuda").normal_(generator=gen)
    else:
        data, pair = (dim * _BITS[ty] + 7) // 8, _scales(rows, ty != "int8", gen).view(torch.uint8)
        table = torch.randint(0, 256, (rows, data + pair.size(1)), dtype=torch.uint8, generator=gen, device="cuda")
        table[:, data:] = pair
    lens = _bag_lengths(case, case["bags"], gen)
    total = int(lens.sum())
    index = torch.int64 if case["index"] == "int64" else torch.int32
    indices = _row_ids(torch.full((total,), rows, device="cuda"), case["alpha"], gen).to(index)
    if case["lengths"]:
        where = lens.to(torch.int32)
    else:
        where = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)
    weights = torch.rand(total, generator=gen, device="cuda") if case["weighted"] else None
    args = (case["weighted"], case["mean"])
    if ty in ("int4", "int2"):
        kernel = ops.generate_embedding_spmdm_nbit(_BITS[ty], dim, *args, use_offsets=not case["lengths"], out_ty=_TYPES[case["output"]])
    else:
        kernel = ops.generate_embedding_spmdm(_TYPES[ty], dim, *args, use_offsets=not case["lengths"], out_ty=_TYPES[case["output"]])
    out = torch.empty(case["bags"], dim, dtype=_TORCH[case["output"]], device="cuda")
    return {"kind": "kernel", "kernel": kernel, "args": (case["bags"], total, rows, table, indices, where, weights, out)}


def _fill_tables(m, specs, gen):
    m.initialize_weights()
    m.weights_dev.view(torch.int32).random_(-(1 << 31), (1 << 31) - 1, generator=gen)
    for (ty, _, rows), (whole, _, _) in zip(specs, m.split_embedding_weights_with_scale_bias(0)):
        if ty in ("int8", "int4", "int2"):
            whole.view(torch.int32)[:, 0] = _scales(rows, True, gen).view(torch.int32).view(-1)
        elif ty in ("fp16", "fp32"):
            whole.view(_TORCH[ty]).normal_(generator=gen)


def _prepare_tables(case, gen):
    specs = _tables(case)
    pooling = {"sum": tbe.PoolingMode.SUM, "mean": tbe.PoolingMode.MEAN, "none": tbe.PoolingMode.NONE}[case["pooling"]]
    fp8 = {"fp8_exponent_bits": 4, "fp8_exponent_bias": 7} if any(ty == "fp8" for ty, _, _ in specs) else {}
    m = tbe.IntNBitTableBatchedEmbeddingBagsCodegen(
        [("", rows, dim, tbe.SparseType(ty), tbe.EmbeddingLocation.DEVICE) for ty, dim, rows in specs], pooling_mode=pooling,
        bounds_check_mode=tbe.BoundsCheckMode.WARNING if case.get("check", True) else tbe.BoundsCheckMode.NONE,
        output_dtype=tbe.SparseType(case["output"]), **fp8)
    _fill_tables(m, specs, gen)
    logical = torch.tensor([rows for _, _, rows in specs], device="cuda")
    if case.get("pruned"):
        # of every two neighbouring rows one, drawn at random, is kept: the mapping numbers the kept ones in order
        logical = logical * 2
        maps = []
        for _, _, rows in specs:
            pairs = torch.full((rows, 2), -1, dtype=torch.int32, device="cuda")
            keep = torch.randint(0, 2, (rows, 1), generator=gen, device="cuda")
            pairs.scatter_(1, keep, torch.arange(rows, dtype=torch.int32, device="cuda").view(-1, 1))
            maps.append(pairs.view(-1))
        m.set_index_remappings(maps)
    bags = case["tables"] * case["batch"]
    # without pooling the output has a row per index: the bag lengths then belong to the case, so that every seed's has one shape
    lens = _bag_lengths(case, bags, gen if case["pooling"] != "none" else torch.Generator(device="cuda").manual_seed(1))
    index = torch.int64 if case["index"] == "int64" else torch.int32
    offsets = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(index)
    indices = _row_ids(logical.repeat_interleave(lens.view(case["tables"], -1).sum(1)), case["alpha"], gen).to(index)
    weights = torch.rand(indices.numel(), generator=gen, device="cuda") if case["weighted"] else None
    if case["kind"] == "module":
        return {"kind": "module", "module": m, "args": (indices, offsets, weights)}
    args = (m.weights_dev, m.weights_uvm, m.weights_placements, m.weights_offsets, m.weights_tys, m.D_offsets, m.total_D,
            m.max_int2_D, m.max_int4_D, m.max_int8_D, m.max_float16_D, m.max_float32_D, indices, offsets, int(pooling), weights,
            m.output_dtype)
    fp8 = {"max_float8_D": m.max_float8_D, "fp8_exponent_bits": m.fp8_exponent_bits, "fp8_exponent_bias": m.fp8_exponent_bias}
    if case["fast"]:
        plan = ops.TbePlan(m.weights_offsets, m.weights_tys, m.D_offsets, m.weights_placements, m.weights_dev.numel(), 0, 16)
        return {"kind": "fast", "args": args, "more": dict(fp8, row_alignment=16, status=ops.Status(), plan=plan, accumulate=ops.ACC_FAST)}
    torch.ops.load_library(TORCH_OP_OUT)
    return {"kind": "operator", "args": args, "more": dict(fp8, row_alignment=16)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if case["kind"] == "kernel":
        return _prepare_kernel(case, gen)
    if case["kind"] in ("module", "operator"):
        return _prepare_tables(case, gen)
    bits, sb_float = _BITS[case["type"]], case["type"] == "int8" and not case.get("front", False)
    dtype = torch.float16 if case.get("input") == "fp16" else torch.float32
    rows = torch.empty(case["rows"], case["cols"], dtype=dtype, device="cuda").normal_(generator=gen)
    layout = ops.QLAYOUT_TBE if case.get("front") else ops.QLAYOUT_TRAILER
    if case["kind"] == "quantize":
        return {"kind": "quantize", "args": (rows, bits, sb_float, layout)}
    coded = ops.quantize_rowwise(rows, bits, sb_float, layout)
    return {"kind": "dequantize", "args": (coded, case["cols"], bits, sb_float, layout, _TORCH[case["output"]])}


def run(state):
    kind = state["kind"]
    if kind == "kernel":
        return state["kernel"](*state["args"]), state["args"][-1]
    if kind == "module":
        return state["module"](*state["args"])
    if kind == "operator":
        return torch.ops.fbgemm.int_nbit_split_embedding_codegen_lookup_function(*state["args"], **state["more"])
    if kind == "fast":
        return ops.int_nbit_split_embedding_codegen_lookup_function(*state["args"], **state["more"])
    if kind == "quantize":
        return ops.quantize_rowwise(*state["args"])
    return ops.dequantize_rowwise(*state["args"])


# ---- what a pass cannot do without ----------------------------------------------------------------------------------


def _distinct(rows, n, alpha):
    """Rows that ``n`` lookups are expected to touch (a row that is looked up twice has to be read once)."""
    if n <= 0:
        return 0.0
    if alpha == 0.0:
        return rows * -math.expm1(n * math.log1p(-1.0 / (rows + 1)))
    a = alpha - 1.0
    edges = np.unique(np.floor(np.geomspace(1, rows + 1, 4000)))
    count = np.diff(edges)
    p = (edges[:-1] ** -a - edges[1:] ** -a) / count + (rows + 1.0) ** -a / rows
    return float(np.sum(count * -np.expm1(n * np.log1p(-np.minimum(p, 1 - 1e-12)))))


def work(case):
    isz = 8 if case.get("index") == "int64" else 4
    if case["kind"] == "kernel":
        n = case["bags"] * case["length"]
        row = case["dim"] * _BITS[case["type"]] / 8 + {"int8": 8, "fp16": 0}.get(case["type"], 4)
        reads = _distinct(case["rows"], n, case["alpha"]) * row + n * (isz + 4 * case["weighted"]) + case["bags"] * 4
        return {"bytes": reads + case["bags"] * case["dim"] * _OUT_BYTES[case["output"]], "flops": 2 * n * case["dim"]}
    if case["kind"] in ("module", "operator"):
        per_table, specs = case["batch"] * case["length"], _tables(case)
        n, bags = per_table * len(specs), case["batch"] * len(specs)
        total, flops = n * (isz + 4 * case["weighted"]) + bags * isz, 0
        for ty, dim, rows in specs:
            row = dim * _BITS[ty] / 8 + (4 if ty in ("int8", "int4", "int2") else 0)
            if case.get("pruned"):
                touched = _distinct(2 * rows, per_table, case["alpha"])
                total += touched / 2 * row + touched * 4
            else:
                total += _distinct(rows, per_table, case["alpha"]) * row
            out_rows = per_table if case["pooling"] == "none" else case["batch"]
            total += out_rows * dim * _OUT_BYTES[case["output"]]
            flops += 2 * per_table * dim
        return {"bytes": total, "flops": flops}
    coded = case["cols"] * _BITS[case["type"]] / 8 + (8 if case["type"] == "int8" and not case.get("front") else 4)
    floats = case["cols"] * _OUT_BYTES[case.get("input") or case["output"]]
    return {"bytes": case["rows"] * (coded + floats), "flops": 4 * case["rows"] * case["cols"]}


def tolerance(case):
    """Quantized bytes are defined to the bit. A pooled sum of 20 .. 100 fp32 additions differs from the same sum in 64
    bits by rel 6e-8 .. 1.1e-7, max 5e-7; rounded to fp16 by rel 2.1e-4, max 4.9e-4 (half a unit in the last place); bf16
    is eight times coarser than fp16. About four times that."""
    if case["kind"] == "quantize":
        return "exact"
    return {"fp32": {"rel": 5e-7, "max": 2.5e-6}, "fp16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 6e-3, "max": 1.6e-2}}[case["output"]]
