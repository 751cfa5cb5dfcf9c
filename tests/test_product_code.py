"""CPU: generated products of wide operands hold one row of limb products at a
time: no scratch memory, and registers for the operands, the result and a row,
not for every limb product."""
import concurrent.futures
import re

from test_shift_code import assembly


def test_wide_products_in_registers(U, tmp_path):
    cases = [("a*b", P, m) for P in (76, 110, 130, 200) for m in (U.MODE_AUTO, U.MODE_EXTENDED)]
    cases += [("a*b", 300, U.MODE_AUTO), ("a*b*c", 95, U.MODE_AUTO), ("a*b*c", 130, U.MODE_AUTO)]

    def build(k):
        text, P, mode = cases[k]
        src = str(tmp_path / f"{k}.hip")
        e = U.Expr(text, [(n, P, P // 3) for n in "abc"], mode=mode)
        with open(src, "w") as f:
            f.write("#include <hip/hip_runtime.h>\n" + e.source)
        s = assembly(src, src + ".s")
        return [int(re.search(rf"\.amdhsa_{what} (\d+)", s).group(1))
                for what in ("private_segment_fixed_size", "next_free_vgpr")], e.out_bytes

    with concurrent.futures.ThreadPoolExecutor(8) as ex:
        for (text, P, mode), ((scratch, regs), out) in zip(cases, ex.map(build, range(len(cases)))):
            # the operands and the result, and as much again for the row
            limbs = (out + 3) // 4 + text.count("*") * ((out + 3) // 4)
            assert scratch == 0 and regs <= 64 + 2 * limbs, (text, P, mode, scratch, regs)
