"""GPU: text ingest of plain rows (sixteen characters at a time) and of the
rows next to them that are not plain: every length around the pieces, the
point and the sign at every place, and a foreign byte at every place --
against the oracle, at scales above, at and below the row's fraction."""
import numpy as np
import pytest

from test_gpu_codec import text_column

pytestmark = pytest.mark.gpu

DIGITS = b"9081726354" * 5


def _rows():
    out = []
    for n in list(range(0, 20)) + [31, 32, 33, 34, 47, 48, 49]:
        d = DIGITS[:n]
        for sign in (b"", b"-"):
            out.append(sign + d)
            out.extend(sign + d[:k] + b"." + d[k:] for k in range(n + 1))
            out.append(sign + b"0" * n)
            out.append(sign + b"9" * n)
    for n in (3, 15, 16, 17, 33):
        for k in range(n):
            for c in (b"\0", b"-", b".", b"/", b":", b" ", b"\xff", b"0"):
                out.append(DIGITS[:k] + c + DIGITS[k + 1:n])
                out.append(b"-" + DIGITS[:k] + c + b".5" + DIGITS[k + 1:n])
    return out


@pytest.mark.parametrize("P,S", [(15, 2), (9, 0), (18, 18), (30, 7), (76, 40), (300, 0)])
def test_plain_and_near_plain_rows(U, O, gpu, P, S):
    rows = _rows()
    B = U.compact_bytes(P)
    dch, doff = text_column(U, rows)
    out = U.DeviceBuffer(len(rows) * B + 8).zero()
    U.parse_compact(dch, doff, len(rows), P, S, out)
    got = out.numpy(count=len(rows) * B + 8)
    want = O.parse_compact(rows, P, S)
    bad = np.nonzero((got[:len(rows) * B] != want).reshape(-1, B).any(axis=1))[0]
    assert bad.size == 0, [rows[i] for i in bad[:5]]
    assert not got[len(rows) * B:].any()


def test_rows_that_end_the_buffer(U, O, gpu):
    """the last row's characters end the allocation, at every alignment"""
    for n in range(1, 24):
        rows = [DIGITS[:n % 5 + 1], DIGITS[:n]]
        chars = np.frombuffer(b"".join(rows), dtype=np.uint8)
        offs = np.array([0, len(rows[0]), len(chars)], dtype=np.int64)
        dch, doff = U.DeviceBuffer.from_numpy(chars), U.DeviceBuffer.from_numpy(offs)
        out = U.DeviceBuffer(2 * 16)
        U.parse_compact(dch, doff, 2, 38, 3, out)
        assert np.array_equal(out.numpy(count=32), O.parse_compact(rows, 38, 3))
