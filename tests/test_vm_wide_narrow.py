"""The interpreter's workspace evaluation (vm_wide.h) on
programs of few limbs, faithful and extended, on the CPU against the oracle:
its divisions at the lines between the faithful rules."""
import pytest

from test_vm_wide_host import check, columns, vmw  # noqa: F401
from ultraprecise_amd import workloads as W

CLASSES = (16, 32)
EXPRS = ["a*b/c - d/a + c/b", "(a+b)*c/d - a/d - b/c", "a/(b-b) + c/d - d/b", "(a-a)/b + c/d - b/(a-a)",
         "(a/b)*(c/d) + a/(c-d)", "a/(b*c*d) - d/b + a/(c*d)", "cast(a/b, 40, 3) + truncate(c/d, 2) - 7.25*d/b",
         "(a*b)/(c*d) + (a/c)/(b/d)"]


def same(U, O, vmw, text, cols, data, rows):  # noqa: F811
    """the workspace form's sum of a program as compiled is the oracle's;
    returns the width (None: the program has no such form)"""
    e = U.Expr(text, cols)
    if not e.faithful:
        return check(U, O, vmw, text, cols, data, rows) if vmw(text, cols, data, rows) else None
    r = vmw(text, cols, data, rows, 1)
    if r is None:
        return None
    img = O.plan_sum(O.Plan(e.plan), data, [c[1] for c in cols], [c[2] for c in cols], rows, mode=O.FAITHFUL)[0]
    assert (1 if r[0] < 0 else 0, abs(r[0]) & ((1 << 1024) - 1)) == (img[1], int.from_bytes(img[5:133], "little")), text
    return r[1]


@pytest.mark.parametrize("P,S", [(4, 1), (7, 0), (9, 2), (10, 0), (15, 2), (18, 6), (19, 0), (20, 3), (38, 12), (76, 25)])
def test_expressions(U, O, vmw, P, S):  # noqa: F811
    """digits of one, two and three words, so that divisors and dividends meet
    the faithful rules' lines at 32 and 64 bits; one row each, so that no sum
    hides a row"""
    cols = [(n, P, S) for n in "abcd"]
    wide = "*".join("abcd"[i % 4] for i in range(300 * 3 // (10 * P) + 1))   # some 300 bits, so 16 limbs
    done = 0
    for k, text in enumerate(EXPRS):
        text += " + " + wide
        for digits in (None, [P, 1, P // 2, P], [1, P, P, P], [P, min(P, 10), min(P, 10), min(P, 19)],
                       [min(P, 7), min(P, 20), min(P, 19), 1]):
            data = columns(U, cols, 60, 7 * k + P, digits)
            if same(U, O, vmw, text, cols, data, 60) is None:
                break
            B = U.compact_bytes(P)
            for r in range(60):
                same(U, O, vmw, text, cols, [d[r * B:(r + 1) * B].copy() for d in data], 1)
            done += 1
    assert done


def test_serving_queries(U, O, vmw):  # noqa: F811
    widths = {}
    for i in range(600):
        q = W.random_query(29, i, config=dict(W.CONFIG5, rows=(1e1, 4e1)))
        try:
            w = U.VmProgram(q["text"], q["cols"]).width
        except U.UpdecError:
            continue
        if w not in CLASSES or widths.get(w, 0) >= 15:
            continue
        if same(U, O, vmw, q["text"], q["cols"], columns(U, q["cols"], q["rows"], 300 + i), q["rows"]) == w:
            widths[w] = widths.get(w, 0) + 1
    assert set(widths) == set(CLASSES), widths
