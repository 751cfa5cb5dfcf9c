"""GPU: text ingest of rows that end before their bytes do -- fixed-width slots
padded with NULs, whatever stands behind the NUL, rows that end in a '.' -- and
of long rows that are not numbers, whose characters add up to values of either
sign: against the oracle, at scales above, at and below the row's fraction."""
import random

import numpy as np
import pytest

from test_gpu_codec import text_column

pytestmark = pytest.mark.gpu

DIGITS = b"7081926354" * 8


def _check(U, O, rows, P, S):
    B = U.compact_bytes(P)
    dch, doff = text_column(U, rows)
    out = U.DeviceBuffer(len(rows) * B + 8).zero()
    U.parse_compact(dch, doff, len(rows), P, S, out)
    got = out.numpy(count=len(rows) * B + 8)
    bad = np.nonzero((got[:len(rows) * B] != O.parse_compact(rows, P, S)).reshape(-1, B).any(axis=1))[0]
    assert bad.size == 0, [rows[i] for i in bad[:5]]
    assert not got[len(rows) * B:].any()


@pytest.mark.parametrize("P,S", [(9, 0), (15, 2), (38, 10), (76, 40), (300, 3)])
def test_padded_slots(U, O, gpu, P, S):
    rows = []
    for width in (1, 4, 15, 16, 17, 20, 31, 32, 33, 48, 64):
        for n in sorted({0, 1, 2, 14, 15, 16, 17, 18, 30, 31, 32, 33, width - 1, width}):
            if not 0 <= n <= width:
                continue
            for sign in (b"", b"-"):
                for point in (None, 0, 1, n - 1, n):
                    body = sign + (DIGITS[:n] if point is None else DIGITS[:max(point, 0)] + b"." + DIGITS[max(point, 0):n])
                    for pad in (b"\0", b"\0.", b"\0x7"):
                        rows.append((body + pad * width)[:max(width, len(body))])
    _check(U, O, rows, P, S)


@pytest.mark.parametrize("P,S", [(9, 0), (15, 2), (38, 10), (76, 40), (300, 100)])
def test_odd_rows(U, O, gpu, P, S):
    rng = random.Random(P)
    rows = []
    for n in list(range(1, 40)) + [63, 64, 65, 100, 310, 400]:
        d = (DIGITS * 6)[:n]
        for c in (b" ", b"+", b"e", b"\xff", b"\x80", b"/", b"."):
            for at in {0, n // 2, n - 1, n}:
                rows.append(d[:at] + c + d[at:])
                rows.append(b"-" + d[:at] + c + b"." + d[at:])
        rows.append(bytes(rng.choice(b" +-./\x80\xff\x01") for _ in range(n)))
        rows.append(b"\x80" * n)
        rows.append(b" " * n + d)
    _check(U, O, rows, P, S)
