"""CPU: faithful divisions by one-word divisors (dec_device.h, built for the
host) against the reference's rules in Python integers, and the generated code
of such divisions, which needs one reciprocal."""
import ctypes
import os
import random
import re
import subprocess

import numpy as np
import pytest

from test_divmod_host import CSRC, HERE, _value, _words
from test_shift_code import assembly


@pytest.fixture(scope="session")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("ddiv") / "libddiv_word_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                           os.path.join(HERE, "quad_host", "ddiv_word_host.cpp"), "-o", out])
    return ctypes.CDLL(out)


def quotient(a, b, S):
    """|a| 10^S / |b| as DivOrMod rounds it (decimal.cu:2201-2333)"""
    if a == 0 or b == 0:
        return a
    est = S // 3 * 10 + (0, 4, 7)[S % 3]
    x = a * 10 ** S
    if a.bit_length() + est - 1 <= 64:     # uint64 throughout
        x &= (1 << 64) - 1
        return x // b + (2 * (x % b) % (1 << 64) >= b)
    return x // b + (2 * (x % b) % (1 << 32) >= b)


@pytest.mark.parametrize("wa", [1, 2])
@pytest.mark.parametrize("S", range(4, 11))
def test_rules(lib, wa, S):
    rng = random.Random(10 * S + wa)
    n = 8000
    a = [_value(rng, wa) if i % 3 else rng.getrandbits(rng.randint(0, 32 * wa)) for i in range(n)]
    b = [_value(rng, 1) if i % 2 else rng.getrandbits(rng.randint(0, 32)) for i in range(n)]
    A = np.array([_words(x, 2) for x in a], dtype=np.uint32)
    B = np.array(b, dtype=np.uint32)
    neg = np.array([[rng.randint(0, 1), rng.randint(0, 1)] for _ in range(n)], dtype=np.uint32)
    out = np.zeros((n, 4), dtype=np.uint32)
    p = [x.ctypes.data_as(ctypes.c_void_p) for x in (A, B, neg, out)]
    assert lib.ddiv_word_run(wa, S, p[0], p[1], p[2], n, p[3]) == 0
    for i in range(n):
        got = sum(int(w) << (32 * k) for k, w in enumerate(out[i, :3]))
        sign = int(neg[i, 0] ^ neg[i, 1]) if a[i] else 0
        assert (got, int(out[i, 3])) == (quotient(a[i], b[i], S) & ((1 << 96) - 1), sign), (a[i], b[i])


@pytest.mark.parametrize("P,text", [(5, "a/b"), (9, "a/b"), (15, "a/7"), (28, "a/7")])
def test_one_reciprocal(U, tmp_path, P, text):
    src = str(tmp_path / "k.hip")
    with open(src, "w") as f:
        f.write("#include <hip/hip_runtime.h>\n" + U.Expr(text, [(n, P, P // 3) for n in "ab"]).source)
    assert len(re.findall("v_rcp_f64", assembly(src, src + ".s"))) == 1
