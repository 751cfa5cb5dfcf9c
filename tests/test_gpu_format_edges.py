"""GPU: output formatting where the digits meet the point and the top: every
digit count and scale around the groups of four, both signs, and strides on
both sides of the copy's division rule -- against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _column(U, P):
    B = U.compact_bytes(P)
    vals = [0]
    for d in range(1, P + 1):
        vals += [10 ** (d - 1), 10 ** d - 1, int("1234567890" * 31) % 10 ** d]
    vals.append((1 << (8 * B - 1)) - 1)
    rows = []
    for v in vals:
        for neg in (0, 1):
            rows.append((v | (neg << (8 * B - 1))).to_bytes(B, "little"))
    return np.frombuffer(b"".join(rows), dtype=np.uint8), len(rows), B


@pytest.mark.parametrize("P", [1, 4, 9, 15, 18, 19, 38, 70, 150, 300])
@pytest.mark.parametrize("form", ["hex", "text"])
def test_every_length(U, O, gpu, P, form):
    col, n, B = _column(U, P)
    f = U.FORMAT_HEX if form == "hex" else U.FORMAT_TEXT
    dcol = U.DeviceBuffer.from_numpy(col)
    for S in sorted({s for s in (0, 1, 2, 3, 4, 5, 7, 8, 9, P // 2, P - 1, P) if 0 <= s <= P}):
        stride = U.format_stride(P, S, f) + (4 if S % 2 else 0)
        out = U.DeviceBuffer(n * stride + 16).zero()
        U.format_compact(dcol, n, P, S, f, out, stride)
        got = out.numpy()
        want = O.format_compact(col, n, P, S, form == "hex", stride)
        assert np.array_equal(got[:n * stride], want), (S, np.argmax(got[:n * stride] != want) // stride)
        assert not got[n * stride:].any()


@pytest.mark.parametrize("stride", [32764, 32768, 65540])
def test_wide_slots(U, O, gpu, stride):
    col, n, B = _column(U, 30)
    n = 70
    assert n * B <= col.size
    dcol = U.DeviceBuffer.from_numpy(col)
    out = U.DeviceBuffer(n * stride)
    U.format_compact(dcol, n, 30, 3, U.FORMAT_TEXT, out, stride)
    assert np.array_equal(out.numpy(), O.format_compact(col[:n * B], n, 30, 3, False, stride))
