"""CPU: the long division of dec_device.h (divmod) built for the host and
checked against Python integers, on operands whose limbs sit at the edges
of a word, so that saturated digits, add-backs and zero low words occur."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ultraprecise_amd", "csrc")
EDGES = [0, 1, 2, 0x7fffffff, 0x80000000, 0x80000001, 0xfffffffe, 0xffffffff]


@pytest.fixture(scope="session")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("divmod") / "libdivmod_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                           os.path.join(HERE, "quad_host", "divmod_host.cpp"), "-o", out])
    return ctypes.CDLL(out)


def _word(rng):
    return rng.choice(EDGES) if rng.random() < 0.7 else rng.getrandbits(32)


def _value(rng, n):
    return sum(_word(rng) << (32 * i) for i in range(rng.randint(1, n)))


def _words(v, n):
    return [(v >> (32 * i)) & 0xffffffff for i in range(n)]


def _number(w):
    return sum(int(x) << (32 * i) for i, x in enumerate(w))


@pytest.mark.parametrize("nx,nb", [(1, 1), (3, 1), (2, 2), (5, 2), (4, 3), (2, 3), (9, 5), (12, 8), (20, 17)])
def test_divmod_exact(lib, nx, nb):
    rng = random.Random(100 * nx + nb)
    pairs = []
    for _ in range(20_000):
        b = _value(rng, nb) or 1
        x = _value(rng, nx)
        if rng.random() < 0.4:  # next to a multiple of the divisor: top words equal, add-back
            x = min(max(0, b * _value(rng, nx) + rng.choice([-1, 0, 1])), (1 << (32 * nx)) - 1)
        pairs.append((x, b))
    n = len(pairs)
    X = np.array([_words(x, nx) for x, _ in pairs], dtype=np.uint32)
    B = np.array([_words(b, nb) for _, b in pairs], dtype=np.uint32)
    q = np.zeros((n, nx + 1), dtype=np.uint32)
    r = np.zeros((n, nb), dtype=np.uint32)
    ptr = ctypes.c_void_p
    assert lib.divmod_run(nx, nb, X.ctypes.data_as(ptr), B.ctypes.data_as(ptr), n, q.ctypes.data_as(ptr),
                          r.ctypes.data_as(ptr)) == 0
    for i, (x, b) in enumerate(pairs):
        assert (_number(q[i]), _number(r[i])) == divmod(x, b), (hex(x), hex(b))


def test_two_word_reciprocal(lib):
    lib.recip2_run.restype = ctypes.c_uint32
    rng = random.Random(5)
    tops = [0x80000000, 0x80000001, 0xfffffffe, 0xffffffff]
    for i in range(50_000):
        d1 = tops[i % 8] if i % 8 < 4 else rng.getrandbits(31) | 0x80000000
        d0 = _word(rng)
        assert lib.recip2_run(ctypes.c_uint32(d1), ctypes.c_uint32(d0)) == ((1 << 96) - 1) // (d1 << 32 | d0) - (1 << 32)


@pytest.mark.parametrize("bits", [1, 31, 32, 33, 63, 64, 65, 96])
@pytest.mark.parametrize("signs", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_zero_dividend_is_plus_zero(lib, bits, signs):
    """also where the reference's bisection would return 1: a divisor of up
    to 64 bits against a dividend of none"""
    b = np.array(_words((1 << bits) - 1, 3), dtype=np.uint32)
    out = np.zeros(5, dtype=np.uint32)
    lib.ddiv_run(ctypes.c_uint32(0), ctypes.c_uint32(signs[0]), b.ctypes.data_as(ctypes.c_void_p),
                 ctypes.c_uint32(signs[1]), out.ctypes.data_as(ctypes.c_void_p))
    assert not out.any()
