"""GPU: a query that needs a larger workspace is staged while a stream is being
captured: the capture stays whole and the batch gives what it gives otherwise."""
import ctypes

import pytest

from ultraprecise_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_add_during_a_capture(U, gpu):
    hip = ctypes.CDLL("libamdhip64.so.7")
    rows = 3000
    cols = [(n, 300, 100) for n in "abcd"]
    progs = [U.VmProgram("(a+b)*c - a/d", cols), U.VmProgram("a*b*c*d*a*b*c/d", cols)]
    assert progs[0].width < progs[1].width
    dev = [U.gen_compact_device(W.digits_desc(U, 1, i, 300), rows) for i in range(4)]

    def results(capture):
        b = U.Batch(max_queries=8, max_items=1 << 10)
        img, cnt = U.DeviceBuffer(2 * U.IMAGE_BYTES).zero(), U.DeviceBuffer(16).zero()
        st, src, dst = U.Stream(), U.DeviceBuffer(4096), U.DeviceBuffer(4096)
        U.copy_kernel(dst, src, 4096, stream=st)
        U.device_sync()
        graph = ctypes.c_void_p()
        if capture:
            assert hip.hipStreamBeginCapture(ctypes.c_void_p(st.handle), 0) == 0
            U.copy_kernel(dst, src, 4096, stream=st)
        for k, p in enumerate(progs):
            assert b.add(p, dev, rows, img, cnt, image_offset=U.IMAGE_BYTES * k, count_offset=8 * k) == k
        if capture:
            assert hip.hipStreamEndCapture(ctypes.c_void_p(st.handle), ctypes.byref(graph)) == 0 and graph.value
            assert hip.hipGraphDestroy(graph) == 0
        b.launch(graph=True)
        U.device_sync()
        assert cnt.numpy("int64").tolist() == [rows, rows]
        return img.numpy().tobytes()

    assert results(True) == results(False)
