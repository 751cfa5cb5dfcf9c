"""GPU: shifts by amounts that lie in a wave's last register.  Kernels whose
registers end an allocation block with a 64-bit shift's amount in the last of
them gave wrong rows from the second wave of a SIMD on, so the rows here are
enough for several waves, against exact integers."""
import pytest

pytestmark = pytest.mark.gpu


def _values(raw, B, n):
    top = 8 * B - 1
    v = [int.from_bytes(raw[i * B:(i + 1) * B].tobytes(), "little") for i in range(n)]
    return [(x & ((1 << top) - 1), x >> top) for x in v]


@pytest.mark.parametrize("P", [70, 110, 120, 122, 130, 160])
def test_mod_of_columns(U, gpu, P):
    rows = 200_003
    B = U.compact_bytes(P)
    dev = [U.gen_compact_device(U.gen_desc(U.GEN_DIGITS, P, 11, k, digits=P, neg_permille=500), rows) for k in range(2)]
    a, b = (_values(d.numpy(count=rows * B), B, rows) for d in dev)
    e = U.Expr("a%b", [(n, P, P // 3) for n in "ab"], mode=U.MODE_EXTENDED)
    out = U.DeviceBuffer(rows * e.out_bytes)
    e.calc(dev, rows, out)
    got = _values(out.numpy(), e.out_bytes, rows)
    bad = [i for i in range(rows) if got[i] != (a[i][0] % b[i][0], a[i][1] ^ b[i][1])]
    assert not bad, (len(bad), bad[:3])
