"""Performance cases of the range-predicate engine.

Each case is one piece of work that a program gives the engine, through the entry points of
rtscan_amd, on tables whose columns have the distributions of the engine's workloads: column
0 uniform on [0, 2^32), column 1 normal (mean 2^31, sd 2^28), columns 2 and 3 Zipf (s = 1.1
and 1.5) over 2^20 keys.  Bitmaps, counts and indexes are whole numbers: two builds of the
engine give the same ones.

kind     what a pass is
scan     `queries` closed ranges over one column, one rts_scan_range call each (bitmap, and
         with `count` the number of rows)
ranges   `queries` closed ranges over one column in one rts_scan_ranges call
conj     `queries` conjunctions over `cols` columns, read directly
query    `queries` conjunctions over `cols` indexed columns, one rts_bindex_query call each
build    a BinDex over a column and the first query's answer from it
batch    `queries` queries of 1..cols columns over an indexed table in one launch of a batch
         plan; with `fresh` they are new to the plan (planned in the pass), else the plan
         already holds them and is launched again
encode   the value encoding of a column (rank form, or `dispersed`) and its map; with `sorted`
         the rank form's sorted places and codes too
"""
import ctypes
import math

import numpy as np
import torch

import rtscan_amd as R

ZIPF_KEYS = 1 << 20
SAMPLE = 1 << 16  # sorted sample of a column that the ranges are drawn from


def listed():
    return [
        # a small table in cache, queried one range at a time: latency and launches
        {"name": "scan_64_of_2p20", "kind": "scan", "rows": 1 << 20, "queries": 64, "count": True},
        # the plain scan of a large column, one range per launch, the engine's headline
        {"name": "scan_8_of_1e8", "kind": "scan", "rows": 100_000_000, "queries": 8, "count": False},
        # the small table's ranges (one dashboard refresh) in one call
        {"name": "ranges_64_of_2p20", "kind": "ranges", "rows": 1 << 20, "queries": 64, "count": True},
        # many ranges over one large column in one call
        {"name": "ranges_64_of_1e8", "kind": "ranges", "rows": 100_000_000, "queries": 64, "count": True},
        # ad-hoc filters over a large table that has no index
        {"name": "conj_4_of_1e8x4", "kind": "conj", "rows": 100_000_000, "cols": 4, "queries": 4},
        # an indexed large column, one range at a time
        {"name": "query_32_of_1e8", "kind": "query", "rows": 100_000_000, "cols": 1, "queries": 32, "bins": 128},
        # filters over an indexed table of ordinary size whose row count fits no tile
        {"name": "query_32_of_2e7x3", "kind": "query", "rows": 20_000_003, "cols": 3, "queries": 32, "bins": 256},
        # indexing a large new column
        {"name": "build_1e8", "kind": "build", "rows": 100_000_000, "column": 0, "bins": 128},
        # indexing a small skewed column
        {"name": "build_1e6_zipf", "kind": "build", "rows": 1_000_003, "column": 2, "bins": 256},
        # a standing set of queries over a large indexed table, evaluated again and again
        {"name": "batch_1024_of_1e8x4", "kind": "batch", "rows": 100_000_000, "cols": 4, "queries": 1024,
         "bins": 256, "fresh": False},
        # a serving loop's batch: queries that have just arrived, planned and evaluated
        {"name": "batch_64_of_2p26x2", "kind": "batch", "rows": 1 << 26, "cols": 2, "queries": 64, "bins": 128,
         "fresh": True},
        # re-encoding a skewed column so that its codes are spread evenly
        {"name": "encode_1e8_zipf", "kind": "encode", "rows": 100_000_000, "column": 2, "dispersed": False,
         "sorted": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["scan", "ranges", "conj", "query", "query", "build", "batch", "batch", "encode"])
    rows = _log_int(rng, 1 << 20, 100_000_000)
    if kind == "scan":
        return {"kind": kind, "rows": rows, "queries": _log_int(rng, 1, max(1, min(64, 800_000_000 // rows))),
                "count": rng.random() < 0.5}
    if kind == "ranges":
        return {"kind": kind, "rows": rows, "queries": _log_int(rng, 4, min(256, 6_400_000_000 // rows)),
                "count": rng.random() < 0.5}
    if kind == "conj":
        return {"kind": kind, "rows": rows, "cols": rng.randint(2, 4), "queries": rng.randint(1, 8)}
    if kind == "query":
        return {"kind": kind, "rows": rows, "cols": rng.randint(1, 4), "queries": rng.randint(8, 64),
                "bins": rng.choice([128, 256, 512])}
    if kind == "build":
        return {"kind": kind, "rows": rows, "column": rng.randint(0, 3), "bins": rng.choice([128, 256])}
    if kind == "batch":
        rows = _log_int(rng, 1 << 22, 100_000_000)
        return {"kind": kind, "rows": rows, "cols": rng.randint(2, 4), "queries": _log_int(rng, 16, 1024),
                "bins": rng.choice([128, 256]), "fresh": rng.random() < 0.5}
    form = rng.choice(["rank", "sorted", "dispersed"])
    return {"kind": kind, "rows": rows, "column": rng.randint(0, 3), "dispersed": form == "dispersed",
            "sorted": form == "sorted"}


class Buffer:
    """A torch tensor as the engine's device buffer (its entry points read .ptr)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


class DeviceView:
    """Device memory that an index owns, for torch.as_tensor; keeps the index alive."""

    def __init__(self, index, ptr, rows, words, stride_words):
        self.index = index
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (rows, words), "typestr": "<i4",
                                         "strides": (4 * stride_words, 4), "version": 3}


def _empty(*shape, dtype=torch.int32):
    return Buffer(torch.empty(shape, dtype=dtype, device="cuda"))


def _column(gen, rows, column):
    """uint32 values in an int32 tensor (the same 32 bits)."""
    if column == 0:
        return torch.randint(-(1 << 31), 1 << 31, (rows,), dtype=torch.int32, device="cuda", generator=gen)
    if column == 1:
        x = torch.randn(rows, dtype=torch.float64, device="cuda", generator=gen)
        return x.mul_(2.0 ** 28).add_(2.0 ** 31).clamp_(0, 2.0 ** 32 - 1).to(torch.int64).to(torch.int32)
    weight = torch.arange(1, ZIPF_KEYS + 1, dtype=torch.float64, device="cuda").pow_(-1.1 if column == 2 else -1.5)
    cdf = torch.cumsum(weight, 0)
    cdf /= cdf[-1].clone()
    key = torch.randint(-(1 << 31), 1 << 31, (ZIPF_KEYS,), dtype=torch.int32, device="cuda", generator=gen)
    u = torch.rand(rows, dtype=torch.float64, device="cuda", generator=gen)
    return key[torch.searchsorted(cdf, u).clamp_(max=ZIPF_KEYS - 1)]


def _sample(values):
    """Sorted sample of a column's values (int64 on the host)."""
    step = max(1, values.numel() // SAMPLE)
    s = values[::step][:SAMPLE].cpu().numpy().view(np.uint32).astype(np.int64)
    return np.sort(s)


def _range(rng, sample, selectivity):
    """A closed range that holds about `selectivity` of the column's rows."""
    m = len(sample)
    width = max(1, int(round(selectivity * (m - 1))))
    at = int(rng.integers(0, m - width)) if width < m else 0
    lo, hi = int(sample[at]), int(sample[min(m - 1, at + width)])
    return lo, max(lo, hi - (1 if hi > lo else 0))


def _table(seed, rows, columns):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cols = [Buffer(_column(gen, rows, c)) for c in columns]
    return cols, [_sample(c.tensor) for c in cols]


def _conjunctions(rng, case, samples):
    """Per query, (los, his) over all of the case's columns: selectivities 0.01, 0.1, 0.5 as
    analysts filter, any for a single column."""
    out = []
    for _ in range(case["queries"]):
        sels = [rng.choice([0.01, 0.1, 0.5]) if len(samples) > 1 else rng.random() for _ in samples]
        r = [_range(rng, s, sel) for s, sel in zip(samples, sels)]
        out.append(([a for a, _ in r], [b for _, b in r]))
    return out


def _mixed_queries(rng, case, samples):
    """Queries of 1..cols distinct columns, each range's selectivity log-uniform in
    [1e-5, 0.9]: (column, lo, hi) per column."""
    out = []
    for _ in range(case["queries"]):
        cols = rng.permutation(case["cols"])[: int(rng.integers(1, case["cols"] + 1))]
        out.append([(int(c),) + _range(rng, samples[c], math.exp(rng.uniform(math.log(1e-5), math.log(0.9))))
                    for c in cols])
    return out


def _words(rows):
    return (rows + 31) // 32


def _stride(rows):
    return (_words(rows) + 3) // 4 * 4


def prepare(case, seed):
    kind, rows = case["kind"], case["rows"]
    columns = [case["column"]] if "column" in case else list(range(case.get("cols", 1)))
    cols, samples = _table(seed, rows, columns)
    rng = np.random.default_rng(seed)
    s = {"case": case, "cols": cols}
    if kind == "encode":
        for name in ("codes", "values", "starts") + (("places", "sorted_codes") if case["sorted"] else ()):
            s[name] = _empty(rows)
            s[name].tensor.zero_()  # the map fills as many entries as there are distinct values
        torch.cuda.synchronize()
        return s
    if kind == "build":
        lo, hi = _range(rng, samples[0], 0.3)
        s.update(lo=[lo], hi=[hi], out=_empty(_words(rows)), count=_empty(1, dtype=torch.int64))
        torch.cuda.synchronize()
        return s
    q = case["queries"]
    if kind == "batch":
        s["queries"] = _mixed_queries(rng, case, samples)
    else:
        s["ranges"] = _conjunctions(rng, case, samples)
    s["out"] = _empty(q, _stride(rows)) if kind != "ranges" else _empty(q, _words(rows))
    s["out"].tensor.zero_()
    s["counts"] = _empty(q, dtype=torch.int64)
    s["counts"].tensor.zero_()
    if kind in ("scan", "conj", "query"):
        s["outs"] = [Buffer(s["out"].tensor[i]) for i in range(q)]
        s["each"] = [Buffer(s["counts"].tensor[i:i + 1]) for i in range(q)]
    if kind == "ranges":
        s["lo"] = np.array([r[0][0] for r in s["ranges"]], np.uint32)
        s["hi"] = np.array([r[1][0] for r in s["ranges"]], np.uint32)
    torch.cuda.synchronize()
    if kind in ("query", "batch"):
        s["indexes"] = [R.BinDexIndex(c, rows, bins=case["bins"]) for c in cols]
    if kind == "batch":
        s["plan"] = R.BatchPlan(cols, s["indexes"], rows, q)
        if not case["fresh"]:
            s["plan"].set_queries(s["queries"])
    return s


def run(s):
    case = s["case"]
    kind, rows = case["kind"], case["rows"]
    if kind == "scan":
        col, counted = s["cols"][0], case["count"]
        for i, (lo, hi) in enumerate(s["ranges"]):
            R.scan_range(col, rows, lo[0], hi[0], s["outs"][i], s["each"][i] if counted else None)
    elif kind == "ranges":
        R.scan_ranges(s["cols"][0], rows, s["lo"], s["hi"], s["out"], _words(rows),
                      s["counts"] if case["count"] else None)
    elif kind == "conj":
        for i, (lo, hi) in enumerate(s["ranges"]):
            R.conjunction_scan(s["cols"], lo, hi, rows, s["outs"][i], s["each"][i])
    elif kind == "query":
        for i, (lo, hi) in enumerate(s["ranges"]):
            R.bindex_query(s["indexes"], lo, hi, s["outs"][i], s["each"][i])
    elif kind == "batch":
        if case["fresh"]:
            s["plan"].set_queries(s["queries"])
        s["plan"].launch(s["out"], _stride(rows), s["counts"])
    elif kind == "encode":  # the C ABI call: the map stays on the device, as a C++ caller has it
        distinct = ctypes.c_int64()
        if case["dispersed"]:
            R.check(R.lib().rts_encode_column_dispersed(s["cols"][0].ptr, rows, 0, 0xFFFFFFFF, 1, s["codes"].ptr,
                                                        s["values"].ptr, s["starts"].ptr, ctypes.byref(distinct),
                                                        None), "rts_encode_column_dispersed")
        else:
            R.check(R.lib().rts_encode_column(s["cols"][0].ptr, rows, 0, 0xFFFFFFFF, s["codes"].ptr,
                                              s["places"].ptr if case["sorted"] else None,
                                              s["sorted_codes"].ptr if case["sorted"] else None,
                                              s["values"].ptr, s["starts"].ptr, ctypes.byref(distinct), None),
                    "rts_encode_column")
        out = {k: s[k].tensor for k in ("codes", "values", "starts", "places", "sorted_codes") if k in s}
        return dict(out, distinct=distinct.value)
    else:
        index = R.BinDexIndex(s["cols"][0], rows, bins=case["bins"])
        R.bindex_query([index], s["lo"], s["hi"], s["out"], s["count"])
        fv, block = index.s.filterVectorsInGPU, index.s.areasInGPU[0].contents.blocks[0].contents
        vectors = DeviceView(index, fv[0], len(fv), _words(rows), (fv[1] - fv[0]) // 4)
        values = DeviceView(index, _address(block.val), 1, rows, rows)
        places = DeviceView(index, _address(block.pos), 1, rows, rows)
        return {"starts": index.start_values().astype(np.int64), "counts": index.area_counts(),
                "vectors": torch.as_tensor(vectors, device="cuda"),
                "values": torch.as_tensor(values, device="cuda"),
                "places": torch.as_tensor(places, device="cuda"),
                "bitmap": s["out"].tensor, "count": s["count"].tensor}
    return s["out"].tensor, s["counts"].tensor


def _address(pointer):
    return ctypes.cast(pointer, ctypes.c_void_p).value


def work(case):
    kind, n = case["kind"], case["rows"]
    bitmap, column, q = 4 * _words(case["rows"]), 4 * case["rows"], case.get("queries", 1)
    if kind == "scan":
        return {"bytes": q * (column + bitmap), "flops": 0}
    if kind == "ranges":
        return {"bytes": column + q * bitmap, "flops": 0}
    if kind == "conj":
        return {"bytes": q * (case["cols"] * column + bitmap), "flops": 0}
    if kind == "query":  # per column two filter vectors and the rows of two bins (8 bytes each)
        return {"bytes": q * (case["cols"] * (2 * bitmap + 16 * n // case["bins"]) + bitmap), "flops": 0}
    if kind == "build":  # the column; sorted values and places, filter vectors, bins' rows
        return {"bytes": column + 8 * n + (case["bins"] - 1) * bitmap + 8 * n, "flops": 0}
    if kind == "batch":  # the table once and every bitmap
        return {"bytes": case["cols"] * column + q * bitmap, "flops": 0}
    distinct = min(n, ZIPF_KEYS) if case["column"] >= 2 else n
    return {"bytes": (4 if case["sorted"] else 2) * column + 8 * distinct, "flops": 0}


def _pack(mask):
    """Row i of a bool tensor to bit 31 - i % 32 of word i // 32 (int32 words)."""
    rows = mask.numel()
    padded = torch.zeros(_words(rows) * 32, dtype=torch.bool, device=mask.device)
    padded[:rows] = mask
    octets = padded.view(-1, 8).to(torch.uint8)
    octets = sum(octets[:, b] << (7 - b) for b in range(8)).view(-1, 4).to(torch.int64)
    word = (octets[:, 0] << 24) | (octets[:, 1] << 16) | (octets[:, 2] << 8) | octets[:, 3]
    return word.to(torch.int32)


def exact(case, seed):
    """The bitmaps and counts from comparisons of 64-bit values; none for the kinds whose
    outputs are more than bitmaps, and where it would take long."""
    kind, rows = case["kind"], case["rows"]
    if kind in ("build", "encode") or rows * case["queries"] * case.get("cols", 1) > 8_000_000_000:
        return None
    cols, samples = _table(seed, rows, list(range(case.get("cols", 1))))
    rng = np.random.default_rng(seed)
    if kind == "batch":
        queries = _mixed_queries(rng, case, samples)
    else:
        queries = [[(c, a, b) for c, (a, b) in enumerate(zip(lo, hi))]
                   for lo, hi in _conjunctions(rng, case, samples)]
    values = [c.tensor.to(torch.int64) & 0xFFFFFFFF for c in cols]
    width = _words(rows) if kind == "ranges" else _stride(rows)
    out = torch.zeros((len(queries), width), dtype=torch.int32, device="cuda")
    counts = torch.zeros(len(queries), dtype=torch.int64, device="cuda")
    for i, query in enumerate(queries):
        mask = None
        for c, lo, hi in query:
            m = (values[c] >= lo) & (values[c] <= hi)
            mask = m if mask is None else mask & m
        out[i, :_words(rows)] = _pack(mask)
        if case.get("count", True):
            counts[i] = mask.sum()
    return out, counts
