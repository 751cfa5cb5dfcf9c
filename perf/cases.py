"""The calls whose speed matters to a program that uses this library, and the
inputs they are measured on.

Every case goes through the package's public entry points on device-resident
columns, as a query engine that embeds the library calls them.  Columns come
from the library's own seeded generator and outputs are torch tensors that
the calls write into; torch has to be imported before the package, so that
both use one HIP runtime.

All outputs are bytes and whole numbers (compact rows, 133-byte SUM images,
counts, text), which are exact.
"""
import numpy as np
import torch

import ultraprecise_amd as U
from ultraprecise_amd import workloads as W

SWEEP = W.CONFIG2["expr"]
# moduli of the RSA workload: (digits of the column, modulus)
RSA = {17: "514679589732349351",
       71: "273420351015258185841522860354335753665897876941082396543621156533322691"}
Q1_GROUPS = 16
SERVE_SEED = W.CONFIG5["seed"]


def listed():
    return [
        # latency of a small ungrouped aggregation: one page of a table
        {"name": "sum-10k", "kind": "sum", "rows": 10_007, "stats": False},
        # the headline query at its full size, with load-time column statistics
        {"name": "q1-60m", "kind": "q1", "rows": 60_000_000, "stats": True},
        # the same query where nobody gathered statistics, at an odd row count
        {"name": "q1-nostats-8m", "kind": "q1", "rows": 8_000_003, "stats": False},
        # projection of an expression with a division: ordinary, high and
        # extreme precision of the precision sweep
        {"name": "calc-p38-10m", "kind": "calc", "P": 38, "S": 10, "rows": 10_000_000},
        {"name": "calc-p150-2m", "kind": "calc", "P": 150, "S": 50, "rows": 2_000_001},
        {"name": "calc-p300-1m", "kind": "calc", "P": 300, "S": 100, "rows": 1_000_000},
        # modular arithmetic: the RSA workload, 16-limb modulus
        {"name": "rsa-71-3m", "kind": "rsa", "P": 71, "N": RSA[71], "rows": 3_000_000},
        # SUM over the output of a sort by two low-cardinality keys: few
        # large segments, rows gathered through the sort's permutation
        {"name": "segsum-gather-20m", "kind": "segsum", "P": 15, "S": 2, "rows": 20_000_000, "segments": 6,
         "gather": True},
        # SUM per key over a column already in key order: many small segments
        {"name": "segsum-300k", "kind": "segsum", "P": 38, "S": 10, "rows": 12_000_001, "segments": 300_000,
         "gather": False},
        # bulk load of a price column from text, and its output as text
        {"name": "parse-10m", "kind": "parse", "P": 15, "S": 2, "rows": 10_000_000},
        {"name": "format-10m", "kind": "format", "P": 15, "S": 2, "rows": 10_000_000, "hex": False},
        # one batch of the serving stream: 32 distinct queries as they arrive
        {"name": "serve-32", "kind": "serve", "first": 0, "queries": 32, "rows": 10_000_000},
    ]


def _log(rng, lo, hi):
    """a whole number spread evenly over the logarithm of [lo, hi]"""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sum", "q1", "calc", "rsa", "segsum", "parse", "format", "serve"])
    if kind == "sum":
        return {"kind": kind, "rows": _log(rng, 1_000, 5_000_000), "stats": rng.random() < 0.5}
    if kind == "q1":
        return {"kind": kind, "rows": _log(rng, 100_000, 60_000_000), "stats": rng.random() < 0.5}
    if kind == "calc":
        P = rng.randint(12, 300)
        return {"kind": kind, "P": P, "S": rng.randint(P // 6, P // 3),
                "rows": _log(rng, 10_000, int(10e6 * min(1.0, (38 / P) ** 1.2)))}
    if kind == "rsa":
        P = _log(rng, 10, 140)
        return {"kind": kind, "P": P, "N": str(rng.randrange(10 ** P, 10 ** (P + 1))),
                "rows": _log(rng, 10_000, int(10e6 * min(1.0, 20 / P)))}
    if kind == "segsum":
        rows = _log(rng, 50_000, 20_000_000)
        P = _log(rng, 9, 76)
        return {"kind": kind, "P": P, "S": rng.randint(0, P // 2), "rows": rows,
                "segments": _log(rng, 1, max(2, rows // 20)), "gather": rng.random() < 0.5}
    if kind in ("parse", "format"):
        P = _log(rng, 9, 76)
        c = {"kind": kind, "P": P, "S": rng.randint(0, P // 2), "rows": _log(rng, 10_000, int(10e6 * min(1.0, 15 / P)))}
        if kind == "format":
            c["hex"] = rng.random() < 0.4
        return c
    return {"kind": "serve", "first": rng.randrange(0, 9_900), "queries": _log(rng, 1, 16), "rows": 1_000_000}


# ---------------------------------------------------------------- inputs


class Out:
    """A torch tensor where the library takes a device buffer."""

    def __init__(self, nbytes):
        self.tensor = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
        self.ptr = self.tensor.data_ptr()
        self.nbytes = nbytes


class In(Out):
    def __init__(self, tensor):
        self.tensor = tensor.contiguous()
        self.ptr = self.tensor.data_ptr()
        self.nbytes = self.tensor.numel() * self.tensor.element_size()


def _digits(seed, cid, P, rows, neg=500):
    return U.gen_compact_device(U.gen_desc(U.GEN_DIGITS, P, seed, cid, digits=P, neg_permille=neg), rows)


def _named(spec, dev, rows, stats):
    """column descriptions, with the load-time statistic where it is kept"""
    return [(c[0], c[1], c[2], U.column_maxbits(d, c[1], rows)) if stats else (c[0], c[1], c[2])
            for c, d in zip(spec, dev)]


def _serve_queries(case):
    config = dict(W.CONFIG5, rows=(1e3, float(case["rows"])))
    return [W.random_query(SERVE_SEED, case["first"] + i, config=config) for i in range(case["queries"])]


def prepare(case, seed):
    U.init(0)
    kind = case["kind"]
    s = {"kind": kind, "rows": case.get("rows")}
    rows = case.get("rows")
    if kind == "sum":
        spec = W.CONFIG1["cols"]
        s["cols"] = [_column(seed, i, c, rows) for i, c in enumerate(spec)]
        s["agg"] = U.Agg(W.CONFIG1["exprs"], _named(spec, s["cols"], rows, case["stats"]))
        s["images"], s["counts"] = Out(2 * U.IMAGE_BYTES), Out(8)
    elif kind == "q1":
        C = W.CONFIG3
        s["cols"] = [_column(seed, i, c, rows) for i, c in enumerate(C["cols"])]
        s["f1"] = U.gen_byte_device(seed, W.COL_FLAG1, C["flag1"], rows)
        s["f2"] = U.gen_byte_device(seed, W.COL_FLAG2, C["flag2"], rows)
        s["ship"] = U.gen_int32_device(seed, W.COL_SHIP, C["ship"][0], C["ship"][1], rows)
        s["agg"] = U.Agg(C["exprs"], _named(C["cols"], s["cols"], rows, case["stats"]), filter=C["filter"], nkeys=2,
                         avg=(0, 1, 4))
        s["images"], s["counts"] = Out(Q1_GROUPS * 8 * U.IMAGE_BYTES), Out(Q1_GROUPS * 8)
    elif kind == "calc":
        P, S = case["P"], case["S"]
        s["cols"] = [_digits(seed, i, P, rows) for i in range(4)]
        s["expr"] = U.Expr(SWEEP, [(n, P, S) for n in "abcd"])
        s["out"] = Out(rows * s["expr"].out_bytes)
    elif kind == "rsa":
        P, N = case["P"], case["N"]
        s["cols"] = [_digits(seed, 0, P, rows, neg=0)]
        s["expr"] = U.Expr(f"col1 * col1 % {N} * col1 % {N}", [("col1", P, 0)])
        s["out"] = Out(rows * s["expr"].out_bytes)
    elif kind == "segsum":
        P, n = case["P"], case["segments"]
        s.update(P=P, S=case["S"], segments=n, col=_digits(seed, 0, P, rows), out=Out(n * U.IMAGE_BYTES))
        g = torch.Generator(device="cuda").manual_seed(seed)
        # the key of every row; a stable sort by key gives the order and the starts
        key = torch.randint(0, n, (rows,), generator=g, device="cuda", dtype=torch.int32)
        skey, order = torch.sort(key, stable=True)
        s["assoc"] = In(order.to(torch.int32)) if case["gather"] else None
        s["groups"] = In(torch.searchsorted(skey, torch.arange(n, device="cuda", dtype=torch.int32), out_int32=True))
    elif kind == "parse":
        P, S = case["P"], case["S"]
        slots = _slots(case, seed, False)
        text = slots != 0
        offs = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
        torch.cumsum(text.sum(1), 0, out=offs[1:])
        s.update(P=P, S=S, chars=In(slots[text]), offs=In(offs), out=Out(rows * U.compact_bytes(P)))
    elif kind == "format":
        P, S = case["P"], case["S"]
        form = U.FORMAT_HEX if case["hex"] else U.FORMAT_TEXT
        stride = U.format_stride(P, S, form)
        s.update(P=P, S=S, form=form, stride=stride, col=_values(case, seed), out=Out(rows * stride))
    else:
        qs = _serve_queries(case)
        s["queries"] = [(U.VmProgram(q["text"], q["cols"]), q["rows"],
                         [_digits(seed, 16 * i + k, q["P"], q["rows"]) for k in range(len(q["cols"]))])
                        for i, q in enumerate(qs)]
        s["batch"] = U.Batch(max_queries=64)
        s["images"], s["counts"] = Out(len(qs) * U.IMAGE_BYTES), Out(len(qs) * 8)
    return s


def _column(seed, i, spec, rows):
    return U.gen_compact_device(W.gen_desc(U, seed, i, spec), rows)


def _values(case, seed):
    """the price column at DECIMAL(15,2), else values of every digit count
    the precision allows, down to a few digits"""
    P, rows = case["P"], case["rows"]
    if P == 15:
        return _column(seed, 1, W.CONFIG3["cols"][1], rows)
    return U.gen_compact_device(U.gen_desc(U.GEN_DIGITS, P, seed, 1, digits=max(1, P - seed % 3), neg_permille=300), rows)


def _slots(case, seed, hexa):
    """the column's text, one NUL-padded slot a row"""
    form = U.FORMAT_HEX if hexa else U.FORMAT_TEXT
    stride = U.format_stride(case["P"], case["S"], form)
    out = Out(case["rows"] * stride)
    col = _values(case, seed)
    U.format_compact(col, case["rows"], case["P"], case["S"], form, out, stride)
    torch.cuda.synchronize()
    return out.tensor.view(case["rows"], stride)


# ---------------------------------------------------------------- one pass


def run(s):
    kind = s["kind"]
    if kind == "sum":
        s["agg"].run(s["cols"], s["rows"], s["images"], s["counts"], max_groups=1)
        return {"images": s["images"].tensor, "counts": s["counts"].tensor}
    if kind == "q1":
        n, keys = s["agg"].run(s["cols"], s["rows"], s["images"], s["counts"], filter_col=s["ship"], key0=s["f1"],
                               key1=s["f2"], max_groups=Q1_GROUPS)
        return {"images": s["images"].tensor, "counts": s["counts"].tensor, "groups": n,
                "keys": np.array(keys, dtype=np.int64)}
    if kind in ("calc", "rsa"):
        s["expr"].calc(s["cols"], s["rows"], s["out"])
        return s["out"].tensor
    if kind == "segsum":
        U.segsum_compact(s["col"], s["P"], s["S"], s["rows"], s["assoc"], s["groups"], s["segments"], s["out"])
        return s["out"].tensor
    if kind == "parse":
        U.parse_compact(s["chars"], s["offs"], s["rows"], s["P"], s["S"], s["out"])
        return s["out"].tensor
    if kind == "format":
        U.format_compact(s["col"], s["rows"], s["P"], s["S"], s["form"], s["out"], s["stride"])
        return s["out"].tensor
    b = s["batch"]
    for i, (prog, rows, cols) in enumerate(s["queries"]):
        b.add(prog, cols, rows, s["images"], s["counts"], image_offset=U.IMAGE_BYTES * i, count_offset=8 * i)
    b.launch(graph=True)
    return {"images": s["images"].tensor, "counts": s["counts"].tensor}


def exact(case, seed):
    """No floating-point output: bytes and counts are equal or wrong."""
    return None


# ---------------------------------------------------------------- work


def _limbs(digits):
    return max(1, -(-int(digits * 3.3219281) // 32))


def work(case):
    """Bytes: every input read and every output written once.  Operations:
    two for each 32-bit limb product of schoolbook multiplication and
    division on the values' own widths."""
    kind = case["kind"]
    rows = case.get("rows", 0)
    if kind == "sum":
        return {"bytes": rows * 21 + 2 * U.IMAGE_BYTES + 8, "flops": rows * 4}
    if kind == "q1":
        return {"bytes": rows * 34 + 6 * 8 * U.IMAGE_BYTES + 6 * 8, "flops": rows * 6}
    if kind == "calc":
        P, S = case["P"], case["S"]
        w, out = _limbs(P), U.Expr(SWEEP, [(n, P, S) for n in "abcd"]).out_bytes
        # (a+b)*c, the quotient's S + 5 digits by the divisor, and its alignment
        return {"bytes": rows * (4 * U.compact_bytes(P) + out),
                "flops": 2 * rows * (w * w + _limbs(S + 5) * w + _limbs(S + 5) * _limbs(S))}
    if kind == "rsa":
        P, N = case["P"], case["N"]
        w, out = _limbs(P), U.Expr(f"col1 * col1 % {N} * col1 % {N}", [("col1", P, 0)]).out_bytes
        return {"bytes": rows * (U.compact_bytes(P) + out), "flops": 2 * rows * 4 * w * w}
    if kind == "segsum":
        n = case["segments"]
        return {"bytes": rows * (U.compact_bytes(case["P"]) + (4 if case["gather"] else 0)) + n * (4 + U.IMAGE_BYTES),
                "flops": 0}
    if kind in ("parse", "format"):
        P, S = case["P"], case["S"]
        if kind == "parse":
            # mean text length: the digits, the point, a sign on some rows
            return {"bytes": rows * (U.compact_bytes(P) + 8 + (8 if P == 15 else P + 1)), "flops": 0}
        stride = U.format_stride(P, S, U.FORMAT_HEX if case["hex"] else U.FORMAT_TEXT)
        return {"bytes": rows * (U.compact_bytes(P) + stride), "flops": 0}
    total = 0
    for q in _serve_queries(case):
        total += q["rows"] * len(q["cols"]) * U.compact_bytes(q["P"]) + U.IMAGE_BYTES + 8
    return {"bytes": total, "flops": 0}
