"""The measured work of this library: what its users have it do, through the
public calls of ``ilgpu_amd.capi``.

Twelve listed cases cover the primitives (sort of keys, sort of pairs, scan,
reduce, histogram, unique) from latency-bound calls on a few thousand elements
over ordinary, ragged lengths to views of a gibibyte; ``draw`` spreads further
cases over the same ranges of length, element type, order, option and
distribution.

A sort and a Unique work in place.  The cases keep the column they start from
and produce the working copy with the library's own ``transform``, as a program
does that goes on using the unsorted column; a histogram adds to its bins, which
``initialize`` clears first.
"""
from __future__ import annotations

import numpy as np
import torch

from ilgpu_amd import capi, datagen

GIB = 1 << 30
DEVICE = "cuda:0"


def listed():
    return [
        # A whole column of 32-bit hashes or ids, the headline length.
        {"name": "sort_u32_2p28", "op": "sort", "type": "uint32", "n": 1 << 28,
         "values": "uniform", "descending": False, "total_order": False},
        # One million keys: the length at which a sort is called inside a loop.
        {"name": "sort_u32_2p20", "op": "sort", "type": "uint32", "n": 1 << 20,
         "values": "uniform", "descending": False, "total_order": False},
        # Ranking scores: floating-point keys, largest first, a ragged length.
        {"name": "sort_f32_descending_20m", "op": "sort", "type": "float32", "n": 20_000_003,
         "values": "normal", "descending": True, "total_order": False},
        # A short list of 64-bit time stamps or counters: latency only.
        {"name": "sort_i64_2000", "op": "sort", "type": "int64", "n": 2000,
         "values": "uniform", "descending": False, "total_order": False},
        # Argsort of a large 64-bit column: the index values are generated.
        {"name": "pairs_u64_index_2p27", "op": "pairs", "type": "uint64", "value_type": "uint32",
         "n": 1 << 27, "values": "uniform", "descending": False, "from_index": True},
        # A join's build side: 32-bit keys carrying 32-bit row numbers.
        {"name": "pairs_u32_u32_3m", "op": "pairs", "type": "uint32", "value_type": "uint32",
         "n": 3_000_017, "values": "uniform", "descending": False, "from_index": False},
        # Offsets from a column of counts, the largest view of one call.
        {"name": "scan_exclusive_i32_2p28", "op": "scan", "type": "int32", "n": 1 << 28,
         "functor": "add", "inclusive": False},
        # Running totals of a million 64-bit amounts.
        {"name": "scan_inclusive_i64_1m", "op": "scan", "type": "int64", "n": 1_000_003,
         "functor": "add", "inclusive": True},
        # Sum of a large column of floats.
        {"name": "reduce_add_f32_2p28", "op": "reduce", "type": "float32", "n": 1 << 28,
         "functor": "add"},
        # Byte histogram of a gibibyte (images, entropy).
        {"name": "histogram_u8_2p30", "op": "histogram", "type": "uint8", "n": 1 << 30,
         "bins": 256, "bin_type": "int32", "values": "uniform", "modulo": False},
        # Distribution of a measured quantity over a few thousand bins.
        {"name": "histogram_i32_4096_8m", "op": "histogram", "type": "int32", "n": 8_000_009,
         "bins": 4096, "bin_type": "int32", "values": "mixture", "modulo": False},
        # Distinct values of a sorted column with frequent and rare values.
        {"name": "unique_u32_zipf_2p26", "op": "unique", "type": "uint32", "n": 1 << 26,
         "values": "zipf"},
    ]


def _length(rng, smallest, largest):
    """Log-uniform over [smallest, largest]; exact powers of two now and then."""
    n = int(round(smallest * (largest / smallest) ** rng.random()))
    if rng.random() < 0.2:
        n = 1 << (n.bit_length() - 1)
    return max(smallest, min(largest, n))


def draw(rng):
    op = rng.choice(["sort", "sort", "sort", "pairs", "pairs", "scan", "scan", "reduce",
                     "histogram", "unique"])
    if op == "sort":
        kind = rng.choice(["uint32", "int32", "float32", "uint64", "int64", "float64", "uint16"])
        values = "normal" if kind.startswith("float") else rng.choice(
            ["uniform", "uniform", "narrow", "zipf"] if kind != "uint16" else ["uniform", "zipf"])
        size = np.dtype(kind).itemsize
        return {"op": op, "type": kind, "n": _length(rng, 1000, GIB // max(size, 4)),
                "values": values, "descending": rng.random() < 0.4,
                "total_order": kind.startswith("float") and rng.random() < 0.5}
    if op == "pairs":
        kind = rng.choice(["uint32", "int32", "float32", "uint64", "int64"])
        value = rng.choice(["uint32", "uint32", "uint64"])
        values = "normal" if kind.startswith("float") else rng.choice(["uniform", "uniform", "narrow", "zipf"])
        return {"op": op, "type": kind, "value_type": value,
                "n": _length(rng, 1000, 1 << (26 if value == "uint64" else 27)),
                "values": values, "descending": rng.random() < 0.4,
                "from_index": rng.random() < 0.5}
    if op in ("scan", "reduce"):
        kind = rng.choice(["int32", "uint32", "int64", "float32", "float64"])
        case = {"op": op, "type": kind, "n": _length(rng, 1000, GIB // np.dtype(kind).itemsize),
                "functor": rng.choice(["add", "add", "max", "min"])}
        if op == "scan":
            case["inclusive"] = rng.random() < 0.5
        return case
    if op == "histogram":
        kind, bins, values, modulo, largest = rng.choice([
            ("uint8", 256, "uniform", False, GIB),
            ("uint8", 256, "zipf", False, GIB),
            ("int32", 4096, "mixture", False, GIB // 4),
            ("int32", 1000, "uniform", True, GIB // 4),
            ("uint16", 65536, "uniform", False, 1 << 22),
        ])
        return {"op": op, "type": kind, "n": _length(rng, 1000, largest), "bins": bins,
                "bin_type": rng.choice(["int32", "int32", "int64", "float32"]),
                "values": values, "modulo": modulo}
    return {"op": "unique", "type": rng.choice(["uint32", "int32", "int64"]),
            "n": _length(rng, 1000, 1 << 27), "values": rng.choice(["zipf", "pairs", "distinct"])}


def _torch_type(name):
    """The torch type of the same width (torch has no arithmetic on wide unsigned ones)."""
    return {"uint8": torch.uint8, "uint16": torch.int16, "uint32": torch.int32,
            "uint64": torch.int64}.get(name) or getattr(torch, name)


def _values(case, seed):
    """The case's input column as a torch tensor on the GPU."""
    n, kind, values = case["n"], case["type"], case.get("values")
    to = _torch_type(kind)
    if case["op"] in ("scan", "reduce"):
        if not kind.startswith("float"):
            if case["functor"] == "add":  # counts
                return datagen.small_ints_i32_torch(n, seed).to(to)
            return datagen.splitmix64_torch(n, seed).to(to)
        if case["op"] == "scan" and case["functor"] == "add":  # weights
            return (datagen.small_ints_i32_torch(n, seed).to(to) + 1) / 16
        return datagen.normal_f32_torch(n, seed).to(to)
    if case["op"] == "unique":
        if values == "zipf":
            v = datagen.zipf_u32_torch(n, seed=seed)
        elif values == "pairs":  # every value about twice
            v = datagen.splitmix64_torch(n, seed).remainder(max(n // 2, 1)).to(torch.int32)
        else:
            return torch.arange(n, dtype=torch.int64, device=DEVICE).add_(seed & 0xFFFF).to(to)
        return torch.sort(v).values.to(to)
    if values == "normal":
        return datagen.normal_f32_torch(n, seed).to(to)
    if values == "zipf":
        distinct = 256 if kind == "uint8" else 1 << 15
        return datagen.zipf_u32_torch(n, distinct=distinct, seed=seed).to(to)
    if values == "mixture":
        return datagen.gaussian_mixture_i32_torch(n, seed=seed)
    if values == "narrow":  # ids of a table of a million rows
        return datagen.splitmix64_torch(n, seed).remainder(1_000_000).to(to)
    if kind == "uint8":
        return datagen.bytes_u8_torch(n, seed)
    return datagen.splitmix64_torch(n, seed).to(to)


def _device_array(tensor, name):
    """A DeviceArray that holds the tensor's elements."""
    out = capi.DeviceArray(tensor.numel(), name)
    out.bytes.copy_(tensor.contiguous().view(torch.uint8))
    return out


def _tensor(array):
    """The array's elements as a torch tensor on the same memory."""
    return array.bytes.view(_torch_type(str(array.dtype)))


_FUNCTORS = {"add": capi.OP_ADD, "max": capi.OP_MAX, "min": capi.OP_MIN}


def _input_seed(seed):
    """The generators' seed of one set of inputs."""
    return datagen.DEFAULT_SEED ^ (seed * 0x9E3779B97F4A7C15 & 0xFFFFFFFFFFFFFFFF)


def prepare(case, seed):
    n, kind, op = case["n"], case["type"], case["op"]
    state = {"case": case, "source": _device_array(_values(case, _input_seed(seed)), kind)}
    if op in ("sort", "pairs"):
        value_bytes = 0
        state["keys"] = capi.DeviceArray(n, kind)
        if op == "pairs":
            value_bytes = np.dtype(case["value_type"]).itemsize
            state["values"] = capi.DeviceArray(n, case["value_type"])
            if not case["from_index"]:
                rows = torch.arange(n, dtype=torch.int64, device=DEVICE).add_(seed & 0xFFFF)
                state["value_source"] = _device_array(rows.to(_torch_type(case["value_type"])),
                                                      case["value_type"])
        state["temp"] = capi.temp_buffer(capi.radix_sort_temp_bytes(n, kind, value_bytes))
    elif op == "scan":
        state["out"] = capi.DeviceArray(n, kind)
        state["temp"] = capi.temp_buffer(capi.scan_temp_bytes(n, kind))
    elif op == "reduce":
        state["out"] = capi.DeviceArray(1, kind)
        state["temp"] = capi.temp_buffer(capi.reduce_temp_bytes(n, kind))
    elif op == "histogram":
        state["bins"] = capi.DeviceArray(case["bins"], case["bin_type"])
        state["overflow"] = capi.DeviceArray.zeros(1, np.int32)
    elif op == "unique":
        state["data"] = capi.DeviceArray(n, kind)
        state["length"] = capi.DeviceArray.zeros(1, np.int64)
        state["temp"] = capi.temp_buffer(capi.unique_temp_bytes(n, kind))
    return state


def run(state):
    case = state["case"]
    op, source = case["op"], state["source"]
    if op == "sort":
        keys = state["keys"]
        capi.transform(source, keys)
        capi.radix_sort_keys(keys, state["temp"], descending=case["descending"],
                             float_total_order=case["total_order"])
        return _tensor(keys)
    if op == "pairs":
        keys, values = state["keys"], state["values"]
        capi.transform(source, keys)
        if not case["from_index"]:
            capi.transform(state["value_source"], values)
        capi.radix_sort_pairs(keys, values, state["temp"], descending=case["descending"],
                              values_from_index=case["from_index"])
        return {"keys": _tensor(keys), "values": _tensor(values)}
    if op == "scan":
        capi.scan(source, state["out"], state["temp"], op=_FUNCTORS[case["functor"]],
                  kind=capi.SCAN_INCLUSIVE if case["inclusive"] else capi.SCAN_EXCLUSIVE)
        return _tensor(state["out"])
    if op == "reduce":
        capi.reduce(source, state["out"], state["temp"], op=_FUNCTORS[case["functor"]])
        return _tensor(state["out"])
    if op == "histogram":
        capi.initialize(state["bins"], 0)
        capi.histogram(source, state["bins"], state["overflow"],
                       locator=capi.LOCATOR_MODULO if case["modulo"] else capi.LOCATOR_IDENTITY)
        return {"bins": _tensor(state["bins"]), "overflow": _tensor(state["overflow"])}
    capi.transform(source, state["data"])
    capi.unique(state["data"], state["length"], state["temp"])
    return {"data": _tensor(state["data"]), "length": _tensor(state["length"])}


def work(case):
    """Bytes: the column read once, the result written once.  Operations: one
    functor application per element where there is arithmetic."""
    n, size, op = case["n"], np.dtype(case["type"]).itemsize, case["op"]
    if op == "sort":
        return {"bytes": 2 * n * size, "flops": 0}
    if op == "pairs":
        value = np.dtype(case["value_type"]).itemsize
        return {"bytes": 2 * n * size + n * value * (1 if case["from_index"] else 2), "flops": 0}
    if op == "scan":
        return {"bytes": 2 * n * size, "flops": n}
    if op == "reduce":
        return {"bytes": (n + 1) * size, "flops": n}
    if op == "histogram":
        return {"bytes": n * size + case["bins"] * np.dtype(case["bin_type"]).itemsize, "flops": 0}
    return {"bytes": 2 * n * size, "flops": 0}


def tolerance(case):
    """Orders, counts and integer arithmetic have one right answer.  A float sum
    is accumulated in double precision and rounded once: at most 6e-8, half a
    unit in the last place.  A prefix sum is rounded at every level of its
    tree: against the float64 one it was 4.8e-7 at 2^28 floats and less below;
    sums of doubles were within 7e-16."""
    if case["op"] in ("scan", "reduce") and case["functor"] == "add":
        if case["type"] == "float32":
            return {"rel": 2.5e-7} if case["op"] == "reduce" else {"rel": 2e-6}
        if case["type"] == "float64":
            return {"rel": 5e-15}
    return "exact"


def exact(case, seed):
    """Sums in 64 bits by torch, where the result is rounded; orders, counts and
    extrema have no rounding to compare."""
    if case["op"] not in ("scan", "reduce") or case["functor"] != "add" \
            or not case["type"].startswith("float"):
        return None
    column = _values(case, _input_seed(seed)).to(torch.float64)
    if case["op"] == "reduce":
        return column.sum().reshape(1)
    total = torch.cumsum(column, 0)
    return total if case["inclusive"] else torch.cat([total.new_zeros(1), total[:-1]])
