"""CPU: generated calc kernels read their columns before they compute, where the
columns are narrow enough to wait in registers, and as the plan needs them where
they are wide."""
import re

import pytest


@pytest.mark.parametrize("P,first", [(5, True), (38, True), (50, False), (300, False)])
def test_loads_first(U, P, first):
    src = U.Expr("(a+b)*c - a/d", [(n, P, P // 3) for n in "abcd"]).source
    body = src[src.index("// plan"):]
    loads = [m.start() for m in re.finditer(r"col_load<", body)]
    assert len(loads) == 4
    assert (loads[-1] < body.index("dadd<")) == first
