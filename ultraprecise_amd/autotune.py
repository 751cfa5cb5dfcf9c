"""Autotuner for the interpreter's persistent kernels.

Per register-width class (W = 2 .. 32 limbs in registers, W = 64 .. 512 limbs
in a workspace) it times representative queries of that width -- seeded
serving queries whose programs land in the class and run on its kernel -- over
every candidate (rows per work item, resident blocks per compute unit) and
keeps the fastest.  The classes from 64 limbs on share one kernel, whose blocks
are single waves: each of them is timed with that kernel's blocks set for all,
and the blocks that are best over all of them are kept, each class with its
own best rows for those.  Results are cached per device name in a JSON file so
a process pays the search once.
"""
import json
import os

DEFAULT_CANDIDATES = ((1024, 4), (2048, 4), (4096, 2), (4096, 4), (8192, 4), (8192, 8), (16384, 4), (32768, 4))
WIDE_BLOCKS = (8, 10, 12)
WIDE_ROWS = (64, 128, 256, 512, 1024)
# of what the file holds and the kernels it was measured on: another number,
# another file
CACHE_VERSION = 2


def class_rows(width, rows):
    """rows timed per query of a class: fewer for the costly wide classes"""
    return rows if width <= 32 else max(100_000, rows * 32 // (width * 2))


def candidates_for(U, cls, candidates):
    return list(candidates) if cls < U.VM_FIRST_MULTI_LANE else [(r, b) for b in WIDE_BLOCKS for r in WIDE_ROWS]


def cache_path(device_name):
    base = os.environ.get("UPDEC_TUNE_DIR", os.path.join(os.path.expanduser("~"), ".cache", "ultraprecise_amd"))
    safe = "".join(ch if ch.isalnum() else "_" for ch in device_name)
    return os.path.join(base, f"vm_tuning_v{CACHE_VERSION}_{safe}.json")


def representative_queries(U, W, per_class=2, seed=77, max_draws=12000):
    """seeded serving queries, `per_class` of each width class (as drawn) that
    run on that class's kernel"""
    found = {c: [] for c in range(len(U.VM_CLASS_WIDTHS))}
    for i in range(max_draws):
        q = W.random_query(seed, i)
        try:
            prog = U.VmProgram(q["text"], q["cols"])
        except U.UpdecError:
            continue
        cls = prog.width_class
        if bool(prog.workspace) != (cls >= U.VM_FIRST_MULTI_LANE):
            continue
        if len(found[cls]) < per_class:
            found[cls].append(q)
        if all(len(v) >= per_class for v in found.values()):
            break
    return found


def apply(U, batch, cls, cand):
    """one class's candidate, with the blocks of the kernel that runs it"""
    batch.tune(cls, cand[0], cand[1])
    if cls >= U.VM_FIRST_MULTI_LANE:
        for c in range(U.VM_FIRST_MULTI_LANE, len(U.VM_CLASS_WIDTHS)):
            if c != cls:
                batch.tune(c, cand[0], cand[1])


def choose(U, times):
    """{class: {(rows, blocks): ms}} -> {class: (rows, blocks)}: the fastest of
    each register class; of the classes that share the wide kernel, the blocks
    with the least total of each class's time against its own best"""
    result = {c: min(t, key=t.get) for c, t in times.items() if c < U.VM_FIRST_MULTI_LANE}
    wide = {c: t for c, t in times.items() if c >= U.VM_FIRST_MULTI_LANE}
    if wide:
        def best(t, blocks):
            return min((ms, cand) for cand, ms in t.items() if cand[1] == blocks)
        every = sorted({b for t in wide.values() for _, b in t})
        blocks = min(every, key=lambda b: sum(best(t, b)[0] / min(t.values()) for t in wide.values()))
        result.update({c: best(t, blocks)[1] for c, t in wide.items()})
    return result


def load(path, classes):
    """a cached result, or None where there is none of this form"""
    try:
        with open(path) as f:
            data = {int(k): tuple(int(x) for x in v) for k, v in json.load(f).items()}
    except (OSError, ValueError, AttributeError, TypeError):
        return None
    ok = all(0 <= c < classes and len(v) == 2 and v[0] >= 64 and 1 <= v[1] <= 64 for c, v in data.items())
    return data if data and ok else None


def tune(U, rows=2_000_000, candidates=DEFAULT_CANDIDATES, reps=3, use_cache=True):
    """returns {class: (rows_per_item, blocks_per_cu)}"""
    from . import workloads as W
    name = U.device_info()["name"]
    path = cache_path(name)
    if use_cache:
        known = load(path, len(U.VM_CLASS_WIDTHS))
        if known:
            return known
    reps = max(1, reps)
    times = {}
    for cls, qs in representative_queries(U, W).items():
        if not qs:
            continue
        progs, cols = [], []
        crows = class_rows(U.VM_CLASS_WIDTHS[cls], rows)
        for q in qs:
            progs.append(U.VmProgram(q["text"], q["cols"]))
            cols.append([U.gen_compact_device(U.gen_desc(U.GEN_DIGITS, q["P"], 77, 900 + k, digits=q["P"],
                                                         neg_permille=500), crows) for k in range(len(q["cols"]))])
        img = U.DeviceBuffer(133 * len(qs))
        cnt = U.DeviceBuffer(8 * len(qs))
        times[cls] = {}
        for cand in candidates_for(U, cls, candidates):
            b = U.Batch(max_queries=len(qs), max_items=1 << 16)
            apply(U, b, cls, cand)

            def launch():
                for k, (p, c) in enumerate(zip(progs, cols)):
                    if b.add(p, c, crows, img, cnt, image_offset=133 * k, count_offset=8 * k) is None:
                        raise RuntimeError("tuning batch overflow")
                b.launch(graph=False)

            launch()
            U.device_sync()
            e0, e1 = U.Event(), U.Event()
            e0.record()
            for _ in range(reps):
                launch()
            e1.record()
            times[cls][tuple(cand)] = e0.elapsed_ms(e1) / reps
        del cols
    result = choose(U, times)
    if use_cache:
        os.makedirs(os.path.dirname(path), exist_ok=True)
        with open(path, "w") as f:
            json.dump({str(k): list(v) for k, v in result.items()}, f)
    return result


def tune_expr_lanes(U, expr, columns, rows, out, reps=3, sample_rows=1_000_000):
    """Lanes per row of a JIT calc expression with a multi-lane form: times
    calc over the first `sample_rows` rows at one row per lane and at W/4
    and W/8 lanes per row (at most 64), keeps the fastest on `expr` and
    returns {lanes: ms}.  An expression without the form keeps one row per
    lane."""
    w = expr.multi_lane_width
    if not w:
        return {1: None}
    n = min(rows, sample_rows)
    times = {}
    for lanes in sorted({1, w // 4, w // 8}):
        if lanes > 64:
            continue
        expr.set_lanes(lanes)
        expr.calc(columns, n, out)      # compile and warm up
        U.device_sync()
        ev0, ev1 = U.Event(), U.Event()
        ev0.record()
        for _ in range(reps):
            expr.calc(columns, n, out)
        ev1.record()
        ev1.sync()
        times[lanes] = ev0.elapsed_ms(ev1) / reps
    best = min(times, key=times.get)
    expr.set_lanes(best)
    return times
