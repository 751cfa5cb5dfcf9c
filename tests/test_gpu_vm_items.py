"""GPU: how a batch cuts its queries into items and stages its tables, against
the oracle: batches with no item to spare, some, and many; one kernel's
queries alone and all kernels' together on the same batch object."""
import pytest

from ultraprecise_amd import workloads as W

pytestmark = pytest.mark.gpu
ROWS = [0, 1, 255, 257, 1_500, 4_097]


def _queries(U, widths, seed):
    seen, out = {}, []
    for i in range(400):
        q = W.random_query(seed, i)
        try:
            prog = U.VmProgram(q["text"], q["cols"])
        except U.UpdecError:
            continue
        if prog.width in widths and seen.get(prog.width, 0) < 2:
            seen[prog.width] = seen.get(prog.width, 0) + 1
            rows = ROWS[len(out) % len(ROWS)]
            host = [U.gen_compact_host(U.gen_desc(U.GEN_DIGITS, P, seed, 16 * i + k, digits=P, neg_permille=500),
                                       max(rows, 1)) for k, (_, P, S) in enumerate(q["cols"])]
            out.append((q, prog, rows, host, [U.DeviceBuffer.from_numpy(h) for h in host]))
    assert set(seen) == set(widths)
    return out


def _want(O, U, q, prog, rows, host):
    e = U.Expr(q["text"], q["cols"])
    P, S = [c[1] for c in q["cols"]], [c[2] for c in q["cols"]]
    if prog.faithful:
        return O.plan_sum(O.Plan(e.plan), host, P, S, rows, mode=O.FAITHFUL)[0]
    return O.plan_sum_wide(e.plan, host, P, S, rows, mode=O.EXTENDED)[0]


def _run(U, batch, queries, graph):
    images = U.DeviceBuffer(len(queries) * U.IMAGE_BYTES).zero()
    counts = U.DeviceBuffer(len(queries) * 8).zero()
    for k, (q, prog, rows, host, dev) in enumerate(queries):
        assert batch.add(prog, dev, rows, images, counts, image_offset=U.IMAGE_BYTES * k, count_offset=8 * k) is not None
    batch.launch(graph=graph)
    U.device_sync()
    assert [int(c) for c in counts.numpy("int64")] == [rows for _, _, rows, _, _ in queries]
    return [bytes(x) for x in images.numpy().reshape(-1, U.IMAGE_BYTES)]


@pytest.mark.parametrize("max_items", [64, 120, 1 << 16])
def test_items_and_kernels(U, O, gpu, max_items):
    every = _queries(U, (2, 4, 8, 16, 32, 64, 128), 37)
    want = [_want(O, U, q, prog, rows, host) for q, prog, rows, host, _ in every]
    batch = U.Batch(max_queries=16, max_items=max_items)
    for k in range(7):
        assert _run(U, batch, every[k:k + 1], True) == want[k:k + 1]
        assert _run(U, batch, every, k != 3) == want
