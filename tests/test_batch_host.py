"""CPU: what an interpreter batch asks of the HIP runtime, seen through a
runtime without a device (hip_stub/fake_hip.cpp): on which device it
allocates, what it frees and when, and what it does with little memory."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_room.argtypes = [ctypes.c_size_t]
fake.fake_pinned.restype = ctypes.c_void_p
sys.path.insert(0, sys.argv[2])
import ultraprecise_amd as U
from ultraprecise_amd import autotune

class Buf:
    def __init__(self, ptr=4096): self.ptr = ptr

def log(word=""):
    return [l for l in fake.fake_log().decode().splitlines() if word in l]

def device(d=None):
    v = ctypes.c_int()
    if d is not None: fake.hipSetDevice(d)
    fake.hipGetDevice(ctypes.byref(v))
    return v.value

COLS = [(n, 38, 12) for n in "abcd"]
C300 = [(n, 300, 100) for n in "abcd"]
NARROW = U.VmProgram("a+b", COLS)
# 16 limbs with three divisions: the wide kernel, or registers
MIDDLE = U.VmProgram("a/b + c/d + b/a + " + "*".join("abc"), COLS)
WIDE = U.VmProgram("(a+b)*c - a/d", C300)                       # 64 limbs
WIDER = U.VmProgram("a*b*c*d*a*b*c/d", C300)
assert (MIDDLE.width, WIDE.width) == (16, 64) and WIDER.width > 128, (MIDDLE.width, WIDE.width, WIDER.width)

def add(b, prog, rows=1000):
    return b.add(prog, [Buf() for _ in prog.cols], rows, Buf(), Buf())
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "hip_stub", "fake_hip.cpp"),
                           "-o", out])

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE + code, out, ROOT], capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stdout + p.stderr
        return p.stdout

    return run


def test_workspace_lies_on_the_batch_device(fake):
    """queries staged by a thread whose current device is another one"""
    fake("""
b = U.Batch(max_queries=8, max_items=64)
device(3)
fake.fake_clear()
assert add(b, WIDE) == 0 and add(b, WIDER) == 1
assert log("hipMalloc") and all(" dev0 " in l for l in log("hipMalloc")), log()
assert device() == 3
""")


def test_a_larger_workspace_frees_nothing(fake):
    """hipFree waits for every stream of the device, and a captured launch may
    still be replayed on the old workspace"""
    fake("""
b = U.Batch(max_queries=8, max_items=64)
fake.fake_clear()
for prog in (MIDDLE, WIDE, WIDER):
    assert add(b, prog) is not None
    b.launch(graph=False)
got = [int(l.split()[2]) for l in log("hipMalloc")]
assert len(got) >= 2 and all(y >= 2 * x or y == 1 << 30 for x, y in zip(got, got[1:])), log()
assert not log("hipFree"), log()
del b
assert len(log("hipFree")) >= len(got)
""")


def test_queries_are_staged_while_a_stream_is_captured(fake):
    """by this thread or another: the allocation is in relaxed mode, and the
    thread's own mode is back afterwards"""
    fake("""
b = U.Batch(max_queries=8, max_items=64)
fake.fake_capturing(1)
for mode in (0, 1, 2):
    m = ctypes.c_int(mode)
    fake.hipThreadExchangeStreamCaptureMode(ctypes.byref(m))
    assert add(b, (MIDDLE, WIDE, WIDER)[mode]) is not None
    m = ctypes.c_int(0)
    fake.hipThreadExchangeStreamCaptureMode(ctypes.byref(m))
    assert m.value == mode
assert len(log("hipMalloc")) >= 2
""")


def test_little_memory_is_asked_for_once(fake):
    """a workspace smaller than wanted serves the queries of one batch; the
    next batch asks again"""
    fake("""
b = U.Batch(max_queries=64, max_items=1 << 12)
fake.fake_room(100 << 20)
for prog in (WIDE, WIDE, WIDER, WIDE):
    assert add(b, prog) is not None
asked = len(log("hipMalloc"))
first = [l for l in log("hipMalloc") if l.endswith("-> 0")][-1]
assert int(first.split()[2]) <= 100 << 20
for prog in (WIDE, WIDER, MIDDLE) * 5:
    assert add(b, prog) is not None
assert len(log("hipMalloc")) == asked and not log("hipFree"), log()
b.launch(graph=False)
assert [l for l in log("launch") if "k_vm_sum_wide" in l]
fake.fake_room(4 << 30)
assert add(b, WIDER) is not None
assert int(log("hipMalloc")[-1].split()[2]) > 500 << 20, log()
""")


def test_memory_for_one_block(fake):
    """programs that have no register class run on one block; the others take
    registers"""
    fake("""
b = U.Batch(max_queries=64, max_items=1 << 12)
fake.fake_room(1 << 20)
assert add(b, WIDE) is not None and add(b, MIDDLE) is not None
b.launch(graph=False)
names = " ".join(log("launch"))
assert "k_vm_sum_wide" in names and "k_vm_sumILi16" in names, names
assert [l for l in log("hipMalloc") if l.endswith("-> 0") and int(l.split()[2]) <= 1 << 20]
""")


def test_no_memory_at_all(fake):
    fake("""
b = U.Batch(max_queries=64, max_items=1 << 12)
fake.fake_room(0)
assert add(b, MIDDLE) is not None
try:
    add(b, WIDE)
    raise SystemExit("accepted without a workspace")
except U.UpdecError as e:
    assert "workspace" in str(e)
assert b.pending == 1 and add(b, NARROW) is not None
b.launch(graph=False)
names = " ".join(log("launch"))
assert "k_vm_sum_wide" not in names and "k_vm_sumILi16" in names, names
""")


def test_kernel_time_is_read_on_the_run_device(fake):
    """the aggregation's clock, asked for by a thread whose current device is
    another one (the fake's kernels write no reading)"""
    fake("""
a = U.Agg(["a+b"], COLS)
a.run([Buf() for _ in COLS], 1000, Buf(), Buf(), max_groups=1)
device(2)
fake.fake_clear()
try:
    a.last_kernel_ms()
except U.UpdecError:
    pass
assert log() and all(" dev0" in l for l in log()), log()
assert log("hipDeviceSynchronize") and device() == 2
# a captured run has no time
fake.fake_capturing(1)
a.run([Buf() for _ in COLS], 1000, Buf(), Buf(), max_groups=1)
fake.fake_clear()
try:
    a.last_kernel_ms()
    raise SystemExit("a captured run was timed")
except U.UpdecError as e:
    assert "no timed run" in str(e) and not log(), log()
""")


def test_items_of_wide_programs_whatever_the_register_class_is_tuned_to(fake):
    """a 16-limb program that runs on the wide kernel takes items for its
    waves, and as many as the batch has to spare"""
    fake("""
b = U.Batch(max_queries=8, max_items=1 << 16)

def items(tuned, max_items_left=None):
    if tuned: b.tune(3, tuned, 4)
    for k in range(5):
        assert add(b, MIDDLE, 10_000_000) is not None
    b.launch(graph=False)
    raw = ctypes.string_at(fake.fake_pinned(2), 24 * 65536)
    rows = []
    for i in range(65536):
        r0, r1 = (int.from_bytes(raw[24 * i + o:24 * i + o + 8], "little") for o in (8, 16))
        rows.append(r1 - r0)
        if sum(rows) == 50_000_000: return rows
    raise SystemExit("items do not cover the rows")

assert max(items(None)) <= 2048
assert max(items(16384)) <= 2048 and max(items(32768)) <= 2048
assert max(items(512)) <= 1024
""")
