"""CPU: the interpreter's tuner -- what a candidate sets, which queries stand for
a class, how the result is chosen, and which cached files are taken."""
import json

from test_batch_host import fake  # noqa: F401
from ultraprecise_amd import autotune
from ultraprecise_amd import workloads as W


def test_candidate_sets_the_blocks_of_the_shared_kernel(fake):  # noqa: F811
    fake("""
for cls in range(U.VM_FIRST_MULTI_LANE, len(U.VM_CLASS_WIDTHS)):
    for blocks in autotune.WIDE_BLOCKS:
        b = U.Batch(max_queries=8, max_items=1 << 16)
        autotune.apply(U, b, cls, (64, blocks))
        assert add(b, WIDE, 10_000_000) is not None
        fake.fake_clear()
        b.launch(graph=False)
        grid = [int(l.split()[-1]) for l in log("k_vm_sum_wide")]
        assert grid == [256 * blocks], (cls, blocks, grid)
""")


def test_representatives_run_on_their_class_kernel(U):
    found = autotune.representative_queries(U, W, per_class=2, max_draws=3000)
    for cls, qs in found.items():
        assert qs or U.VM_CLASS_WIDTHS[cls] == 512, cls
        for q in qs:
            p = U.VmProgram(q["text"], q["cols"])
            assert p.width_class == cls and bool(p.workspace) == (cls >= U.VM_FIRST_MULTI_LANE)


def test_choice(U):
    times = {0: {(1024, 4): 2.0, (2048, 4): 1.0},
             5: {(64, 8): 1.0, (128, 8): 0.9, (64, 12): 1.2, (128, 12): 1.0},
             6: {(64, 8): 5.0, (128, 8): 6.0, (64, 12): 2.0, (128, 12): 3.0}}
    assert autotune.choose(U, times) == {0: (2048, 4), 5: (128, 12), 6: (64, 12)}
    assert autotune.choose(U, {4: {(64, 4): 1.0}}) == {4: (64, 4)}


def test_cached_files(U, tmp_path, monkeypatch):
    monkeypatch.setenv("UPDEC_TUNE_DIR", str(tmp_path))
    path = autotune.cache_path("AMD Instinct MI355X")
    # the name that files of the multi-lane kernels had
    assert not path.endswith("vm_tuning_AMD_Instinct_MI355X.json")
    n = len(U.VM_CLASS_WIDTHS)
    assert autotune.load(path, n) is None
    for data in ({"5": [512, 4, 16]}, {"0": [8192, 4], "5": [512, 4, 16]}, {"9": [64, 4]}, {"0": [1, 4]}, {}, []):
        with open(path, "w") as f:
            json.dump(data, f)
        assert autotune.load(path, n) is None, data
    with open(path, "w") as f:
        f.write('{"0": [8192')
    assert autotune.load(path, n) is None
    with open(path, "w") as f:
        json.dump({"0": [8192, 4], "5": [512, 12]}, f)
    assert autotune.load(path, n) == {0: (8192, 4), 5: (512, 12)}
