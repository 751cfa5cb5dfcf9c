"""The aggregation's own kernel time, read from the device's clock: positive,
never more than the wall time of the run it belongs to, and refused while
there is none."""
import time

import numpy as np
import pytest

from ultraprecise_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 1025, 3_000_000])
@pytest.mark.parametrize("nkeys", [0, 1])  # the two-pass form's clock and the one-pass form's
def test_kernel_time_lies_within_the_run(U, gpu, rows, nkeys):
    dev = U.gen_compact_device(W.digits_desc(U, 5, 0, 18), rows)
    key = U.DeviceBuffer.from_numpy((np.arange(rows) % 3).astype(np.uint8))
    agg = U.Agg(["a+a"], [("a", 18, 2)], nkeys=nkeys)
    with pytest.raises(U.UpdecError):
        agg.last_kernel_ms()
    images, counts = U.DeviceBuffer(4 * 133), U.DeviceBuffer(4 * 8)
    args = dict(key0=key, max_groups=4) if nkeys else dict(max_groups=1)
    agg.run([dev], rows, images, counts, **args)
    U.device_sync()
    for _ in range(3):
        t0 = time.perf_counter()
        agg.run([dev], rows, images, counts, **args)
        U.device_sync()
        wall = 1000.0 * (time.perf_counter() - t0)
        assert 0.0 < agg.last_kernel_ms() <= wall
