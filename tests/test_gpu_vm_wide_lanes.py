"""GPU: the interpreter's workspace kernel where the lanes of a wave disagree --
zero divisors beside the faithful rules' edges, quotients and divisors of every
length in one wave -- where its settings are other than the default, and where a
query's partials are summed by several blocks; against the oracle."""
import numpy as np
import pytest

from test_vm_wide_narrow import EXPRS
from ultraprecise_amd import workloads as W

pytestmark = pytest.mark.gpu


def _column(U, P, rows, seed):
    """values of 1 to P digits, exact zeros, and the numbers next to 2^31, 2^32,
    2^63 and 2^64, each of them in every wave of 64 rows"""
    rng = np.random.default_rng(seed)
    B = U.compact_bytes(P)
    edges = [0, 1] + [2 ** k + d for k in (31, 32, 63, 64) for d in (-1, 0, 1)]
    out = bytearray()
    for i in range(rows):
        kind = (i * 37 + seed) % 64
        if kind < len(edges):
            v = edges[kind]
        else:
            d = 1 + (kind * 7 + seed) % P
            v = int("".join(rng.choice(list("0123456789"), d)))
        v %= 10 ** P
        neg = int(rng.integers(0, 2)) if v else 0
        out += (v | neg << (8 * B - 1)).to_bytes(B, "little")
    return np.frombuffer(bytes(out), dtype=np.uint8)


def _want(O, U, text, cols, host, rows, mode):
    e = U.Expr(text, cols, mode=mode)
    P, S = [c[1] for c in cols], [c[2] for c in cols]
    if e.faithful:
        return O.plan_sum(O.Plan(e.plan), host, P, S, rows, mode=O.FAITHFUL, threads=16)[0]
    return O.plan_sum_wide(e.plan, host, P, S, rows, mode=O.EXTENDED, threads=16)[0]


def _run(U, batch, items):
    images, counts = U.DeviceBuffer(133 * len(items)).zero(), U.DeviceBuffer(8 * len(items)).zero()
    for k, (prog, dev, rows) in enumerate(items):
        assert batch.add(prog, dev, rows, images, counts, image_offset=133 * k, count_offset=8 * k) == k
    batch.launch(graph=False)
    U.device_sync()
    assert counts.numpy("int64").tolist() == [rows for _, _, rows in items]
    return [bytes(x) for x in images.numpy().reshape(-1, 133)]


@pytest.mark.parametrize("P,S", [(9, 2), (15, 2), (19, 0), (20, 3), (38, 12), (76, 25)])
def test_lanes_that_disagree(U, O, gpu, P, S):
    rows = 64 + 37
    cols = [(n, P, S) for n in "abcd"]
    wide = "*".join("abcd"[i % 4] for i in range(300 * 3 // (10 * P) + 1))   # some 300 bits, so 16 limbs
    host = [_column(U, P, rows, 11 * P + i) for i in range(4)]
    dev = [U.DeviceBuffer.from_numpy(h) for h in host]
    items, want = [], []
    for text in EXPRS:
        for mode in (U.MODE_AUTO, U.MODE_EXTENDED):
            for t in (text + " + " + wide, text + " - (d/c)/(b/a)"):
                try:
                    prog = U.VmProgram(t, cols, mode=mode)
                except U.UpdecError:
                    continue
                if prog.workspace:
                    # one wave, two, and one row
                    for n in (rows, 64, 1):
                        items.append((prog, dev, n))
                        want.append((t, mode, n, _want(O, U, t, cols, host, n, mode)))
    assert items
    for k in range(0, len(items), 16):
        got = _run(U, U.Batch(max_queries=16, max_items=1 << 10), items[k:k + 16])
        for g, w in zip(got, want[k:k + 16]):
            assert g == w[3], w[:3]


@pytest.mark.parametrize("rows_per_item,blocks", [(64, 1), (192, 4), (4096, 12), (64, 64)])
def test_settings(U, O, gpu, rows_per_item, blocks):
    rows = 2500
    batch = U.Batch(max_queries=8, max_items=1 << 10)
    for c in range(U.VM_FIRST_MULTI_LANE, len(U.VM_CLASS_WIDTHS)):
        batch.tune(c, rows_per_item, blocks)
    items, want = [], []
    for k, text in enumerate(("(a+b)*c - a/d", "a*b*c*d/a", "((a-a)/b + c)*d*a*b")):
        cols = [(n, 300, 100) for n in "abcd"]
        host = [_column(U, 300, rows, 7 * k + i) for i in range(4)]
        items.append((U.VmProgram(text, cols), [U.DeviceBuffer.from_numpy(h) for h in host], rows))
        assert items[-1][0].width >= 64
        want.append(_want(O, U, text, cols, host, rows, U.MODE_AUTO))
    assert _run(U, batch, items) == want


@pytest.mark.parametrize("P,text,width", [(5, "a+b", 2), (15, "a*b", 4), (38, "a*b+c", 8), (76, "a*b*c", 32),
                                          (300, "a+b-c*a", 64), (300, "a*b*c*d", 128)])
def test_partials_summed_by_several_blocks(U, O, gpu, P, text, width):
    """1,024 items and more of one query (several blocks add them) against the
    oracle, and beside a small query"""
    rows = 64 * 1100 + 3 if width < 64 else 64 * 1030 + 3
    cols = [(n, P, P // 3) for n in "abcd"]
    host = [U.gen_compact_host(W.digits_desc(U, 3, i, P), rows) for i in range(4)]
    dev = [U.DeviceBuffer.from_numpy(h) for h in host]
    prog = U.VmProgram(text, cols)
    assert prog.width == width
    batch = U.Batch(max_queries=8, max_items=1 << 14)
    for c in range(len(U.VM_CLASS_WIDTHS)):
        batch.tune(c, 64, 4)
    want = [_want(O, U, text, cols, host, n, U.MODE_AUTO) for n in (rows, 100)]
    assert _run(U, batch, [(prog, dev, rows), (prog, dev, 100)]) == want
    # and as few items as one block adds
    few = U.Batch(max_queries=8, max_items=512)
    assert _run(U, few, [(prog, dev, rows)]) == want[:1]


def test_multi_lane_calc_at_512_limbs(U, O, gpu):
    """the generated kernel whose values take a whole wave, eight limbs a lane"""
    for i in (1297, 3425):
        q = W.random_query(91, i)
        e = U.Expr(q["text"], q["cols"])
        assert e.multi_lane_width == 512
        rows = 131
        n = len(q["cols"])
        host = [U.gen_compact_host(U.gen_desc(U.GEN_DIGITS, q["P"], 6, 40 + k, digits=q["P"], neg_permille=500), rows)
                for k in range(n)]
        want = O.plan_eval_wide(e.plan, host, [c[1] for c in q["cols"]], [c[2] for c in q["cols"]], rows, e.out_bytes,
                                mode=O.EXTENDED, threads=16)
        e.set_lanes(64)
        out = U.DeviceBuffer(rows * e.out_bytes + 4).zero()
        e.calc([U.DeviceBuffer.from_numpy(h) for h in host], rows, out)
        full = out.numpy()
        assert not full[rows * e.out_bytes:].any()
        bad = np.nonzero((full[:rows * e.out_bytes] != want).reshape(rows, -1).any(axis=1))[0]
        assert bad.size == 0, (q["text"], bad[:5])
