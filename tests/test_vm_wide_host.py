"""CPU: the interpreter's wide evaluation (vm_wide.h) built for the host and
checked row by row against exact integer arithmetic over the plan -- the
seeded serving queries that need more than 32 limbs, and expressions that
reach each of its loops (casts up and down, truncation, constants, zero
divisors and vanishing differences, divisors of every register size and
past them)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from ultraprecise_amd import workloads as W

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ultraprecise_amd", "csrc")


@pytest.fixture(scope="session")
def vmw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("vmw") / "libvm_wide_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                           os.path.join(HERE, "vm_host", "vm_wide_host.cpp"), os.path.join(CSRC, "planner.cpp"),
                           "-o", out])
    lib = ctypes.CDLL(out)

    def run(text, cols, data, rows, mode=2):
        n = len(cols)
        names = (ctypes.c_char_p * n)(*[c[0].encode() for c in cols])
        P = (ctypes.c_int * n)(*[c[1] for c in cols])
        S = (ctypes.c_int * n)(*[c[2] for c in cols])
        ptrs = (ctypes.c_void_p * n)(*[d.ctypes.data for d in data])
        acc = np.zeros(1024, dtype=np.uint32)
        width = ctypes.c_int()
        err = ctypes.create_string_buffer(400)
        rc = lib.vmw_sum(text.encode(), names, P, S, n, ptrs, ctypes.c_int64(rows), acc.ctypes.data_as(ctypes.c_void_p),
                         ctypes.byref(width), err, 400, mode)
        if rc == 3:
            return None   # the register kernels' form only
        assert rc == 0, err.value
        v = int.from_bytes(acc.tobytes(), "little")
        return v - (1 << 32768 if v >> 32767 else 0), width.value

    return run


def stored_sum(U, O, text, cols, data, rows):
    """the low 32 limbs of the exact sum, as the oracle's wide sum has it"""
    e = U.Expr(text, cols, mode=U.MODE_EXTENDED)
    img, n = O.plan_sum_wide(e.plan, data, [c[1] for c in cols], [c[2] for c in cols], rows, mode=O.EXTENDED, threads=8)
    return img


def check(U, O, vmw, text, cols, data, rows):
    got, width = vmw(text, cols, data, rows)
    img = stored_sum(U, O, text, cols, data, rows)
    mag = int.from_bytes(img[5:133], "little")
    assert (1 if got < 0 else 0, abs(got) & ((1 << 1024) - 1)) == (img[1], mag), text
    return width


def columns(U, cols, rows, seed, digits=None):
    return [U.gen_compact_host(U.gen_desc(U.GEN_DIGITS, P, seed, 40 + i, digits=(digits or [P] * len(cols))[i],
                                          neg_permille=500), rows) for i, (_, P, S) in enumerate(cols)]


C300 = [(n, 300, 100) for n in "abcd"]
C150 = [(n, 150, 50) for n in "abcd"]
EXPRS = [
    ("(a+b)*c - a/d", C300), ("a*b*c*d", C300), ("a*b*c/d", C300), ("(a*b)/(c*d)", C300),
    ("(a-a)/b + (c-c)*d - b", C300), ("a/(b-b) + c*d", C300), ("(a-a)/(b-b) - c*d*a", C300),
    ("(a*b*c)/(b*c*d)", C300), ("(a/b)/(c/d) * a * b", C300), ("a*b*(c-d)/(a*d - b*c)", C150),
    ("cast(a*b*c, 400, 20) + truncate(a*b, 10) - truncate(c*d, -30)", C300),
    ("cast(a, 500, 300)*b*1.5 - 12345678901234567890.123456789 / c * a * b", C300),
]


@pytest.mark.parametrize("k", range(len(EXPRS)))
def test_expressions(U, O, vmw, k):
    text, cols = EXPRS[k]
    rows = 60
    for seed, digits in ((1, None), (2, [300, 40, 9, 130][:len(cols)] if cols is C300 else [150, 20, 3, 60])):
        data = columns(U, cols, rows, seed + 10 * k, digits)
        assert check(U, O, vmw, text, cols, data, rows) >= 64


@pytest.mark.parametrize("digits", [1, 9, 10, 19, 20, 38, 39, 77, 78, 150, 154, 155, 299, 300])
def test_divisor_lengths(U, O, vmw, digits):
    rows = 50
    data = columns(U, C300, rows, digits, [300, digits, 300, max(1, digits // 2)])
    check(U, O, vmw, "a*c/b + a/d*c", C300, data, rows)
    check(U, O, vmw, "a/(b*d) + a*c*c", C300, data, rows)


def test_serving_queries(U, O, vmw):
    widths, n = {}, 0
    cfg = dict(W.CONFIG5, rows=(1e1, 6e1))
    for i in range(4000):
        q = W.random_query(23, i, config=cfg)
        if q["P"] < 76:
            continue
        try:
            w = U.VmProgram(q["text"], q["cols"], mode=U.MODE_EXTENDED).width
        except U.UpdecError:
            continue
        if w < 64 or widths.get(w, 0) >= 12:
            continue
        rows = q["rows"]
        data = columns(U, q["cols"], rows, 100 + i)
        assert check(U, O, vmw, q["text"], q["cols"], data, rows) == w
        widths[w] = widths.get(w, 0) + 1
        n += 1
    assert set(widths) == {64, 128, 256, 512} and n >= 40, widths
