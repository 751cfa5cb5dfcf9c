"""GPU: text ingest with offsets that go down: a row whose end is not past its
start is empty, every other one is its own characters, wherever the last
offset lies -- against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TEXT = b"-81723.4650912837465.5501928374650192837465.0192837465"


@pytest.mark.parametrize("P,S", [(15, 2), (38, 10), (300, 100)])
@pytest.mark.parametrize("ends", [[9, 3], [9, 0], [6, 2, 20, 2, 36, 1], [54, 53, 54, 7, 23, 7, 0], [0, 0, 12, 12, 5]])
def test_offsets_that_go_down(U, O, gpu, P, S, ends):
    offs = np.array([0] + ends, dtype=np.int64)
    rows = [TEXT[a:b] if b > a else b"" for a, b in zip(offs[:-1], offs[1:])]
    B = U.compact_bytes(P)
    dch, doff = U.DeviceBuffer.from_numpy(np.frombuffer(TEXT, dtype=np.uint8)), U.DeviceBuffer.from_numpy(offs)
    out = U.DeviceBuffer(len(rows) * B + 8).zero()
    U.parse_compact(dch, doff, len(rows), P, S, out)
    got = out.numpy(count=len(rows) * B + 8)
    assert got[:len(rows) * B].tobytes() == O.parse_compact(rows, P, S).tobytes(), rows
    assert not got[len(rows) * B:].any()
