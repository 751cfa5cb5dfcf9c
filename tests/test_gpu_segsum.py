"""GPU: the segmented SUM at the places where its tiling can go wrong --
starts on tile and chunk boundaries, more starts in a tile than the block
sums at once, runs of empty segments, positions in no segment, one segment
over many chunks, and every row width class, in row order and gathered --
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(U, O, P, rows, groups, assoc=None, seed=1):
    S = P // 3
    host = U.gen_compact_host(U.gen_desc(U.GEN_DIGITS, P, seed, 3, digits=P, neg_permille=500), rows)
    groups = np.asarray(groups, dtype=np.int32)
    col, dg = U.DeviceBuffer.from_numpy(host), U.DeviceBuffer.from_numpy(groups)
    da = None if assoc is None else U.DeviceBuffer.from_numpy(assoc)
    out = U.DeviceBuffer(len(groups) * 133 + 8)
    out.zero()
    U.segsum_compact(col, P, S, rows, da, dg, len(groups), out)
    got = out.numpy()
    want = O.segsum_compact(host, P, S, rows, assoc, groups)
    assert np.array_equal(got[:len(groups) * 133].reshape(-1, 133), want)
    assert not got[len(groups) * 133:].any()


GROUPS = {
    "one": lambda n: [0],
    "late": lambda n: [n // 3],
    "last": lambda n: [0, n - 1],
    "tiles": lambda n: sorted({k for t in range(0, n, 1024) for k in (t, t + 1, t + 1023) if k < n}),
    "each": lambda n: list(range(n)),
    "dense": lambda n: [k for k in range(0, n, 3) for _ in range(1 + k % 4)],
    "empty": lambda n: sorted([0] * 70 + [min(5, n)] * 130 + [n // 2] * 64 + [n - 1] * 3 + [n] * 100),
}


@pytest.mark.parametrize("name", list(GROUPS))
@pytest.mark.parametrize("rows", [1, 3, 255, 1024, 1025, 5003])
@pytest.mark.parametrize("P", [2, 9, 15, 19, 38])
def test_starts(U, O, gpu, P, rows, name):
    _check(U, O, P, rows, GROUPS[name](rows), seed=rows)


@pytest.mark.parametrize("P", [4, 7, 12, 17, 21, 24, 26, 29, 31, 33, 36, 40, 76, 150, 300])
@pytest.mark.parametrize("gather", [False, True])
def test_widths(U, O, gpu, P, gather):
    rng = np.random.default_rng(P)
    rows = 20_011
    groups = np.sort(rng.integers(0, rows, size=700))
    groups[0] = 17
    _check(U, O, P, rows, np.sort(groups), rng.permutation(rows).astype(np.int32) if gather else None, seed=P)


@pytest.mark.parametrize("gather", [False, True])
def test_segments_over_many_chunks(U, O, gpu, gather):
    """rows enough for several tiles a block: segments that span chunks,
    begin and end inside one, and end exactly on a chunk's end"""
    rng = np.random.default_rng(9)
    rows = 5_000_003
    assoc = rng.permutation(rows).astype(np.int32) if gather else None
    cuts = np.sort(rng.integers(1, rows, size=300))
    groups = np.unique(np.concatenate([[0, 3072, 6144, 1_000_000, 1_000_001, 4_000_000], cuts])).astype(np.int32)
    _check(U, O, 15, rows, groups, assoc, seed=4)
    _check(U, O, 15, rows, groups[groups >= 1_000_000][:2], assoc, seed=5)
