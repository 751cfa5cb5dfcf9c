"""GPU: output of wide columns whose values have few digits -- all rows of a
wave short, one long among them, zeros -- at scales before and behind the last
digit, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [39, 77, 154, 300])
@pytest.mark.parametrize("S", [0, 1, 7, 8, 9, 26, 39])
@pytest.mark.parametrize("form", ["hex", "text"])
def test_short_values(U, O, gpu, P, S, form):
    B = U.compact_bytes(P)
    waves = []
    for digits in (0, 1, 3, 8, 9, 16, 17, 38):
        m = 10 ** digits - 1
        waves.append([max(m - i, 0) for i in range(64)])
        waves.append([min(i, m) for i in range(64)])
    waves.append([0] * 63 + [10 ** (P - 1)])
    waves.append([2 ** (32 * k) - (k & 1) for k in range(8 * B // 32)][:64] + [5])
    vals = [(v, (i & 1)) for i, v in enumerate(x for w in waves for x in w)]
    raw = b"".join(((v & ((1 << (8 * B - 1)) - 1)) | (s << (8 * B - 1))).to_bytes(B, "little") for v, s in vals)
    col = np.frombuffer(raw, dtype=np.uint8)
    f = U.FORMAT_HEX if form == "hex" else U.FORMAT_TEXT
    stride = U.format_stride(P, S, f) + 4
    out = U.DeviceBuffer(len(vals) * stride)
    U.format_compact(U.DeviceBuffer.from_numpy(col), len(vals), P, S, f, out, stride)
    got = out.numpy(count=len(vals) * stride)
    want = O.format_compact(col, len(vals), P, S, form == "hex", stride)
    bad = np.nonzero((got != want).reshape(-1, stride).any(axis=1))[0]
    assert bad.size == 0, (bad[:5], [vals[i] for i in bad[:5]])
