"""GPU: the aggregation's kernel time is there when its run is: work on other
streams is not waited for, nor is a stream that has been destroyed."""
import pytest

from ultraprecise_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1000, 2_000_000])
def test_other_streams_are_not_waited_for(U, gpu, rows):
    dev = U.gen_compact_device(W.digits_desc(U, 5, 0, 18), rows)
    agg = U.Agg(["a+a"], [("a", 18, 2)])
    images, counts = U.DeviceBuffer(133), U.DeviceBuffer(8)
    agg.run([dev], rows, images, counts, max_groups=1)
    assert agg.last_kernel_ms() > 0
    big = 2 << 30
    src, dst = U.DeviceBuffer(big), U.DeviceBuffer(big)
    mine, other = U.Stream(), U.Stream()
    U.device_sync()
    done = U.Event()
    for _ in range(400):     # some 0.4 s of copies
        U.copy_kernel(dst, src, big, stream=other)
    done.record(other)
    agg.run([dev], rows, images, counts, max_groups=1, stream=mine)
    assert 0.0 < agg.last_kernel_ms() < 100.0
    assert not done.done()
    done.sync()


def test_stream_destroyed_after_the_run(U, gpu):
    rows = 500_000
    dev = U.gen_compact_device(W.digits_desc(U, 5, 0, 18), rows)
    agg = U.Agg(["a*a"], [("a", 18, 2)])
    images, counts = U.DeviceBuffer(133), U.DeviceBuffer(8)
    for _ in range(5):
        st = U.Stream()
        agg.run([dev], rows, images, counts, max_groups=1, stream=st)
        del st
        assert 0.0 < agg.last_kernel_ms() < 100.0
