"""Reading back behind ticks that are still running: the threads that copy do not spend
the wait in loops."""
import time

import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def test_frame_behind_a_long_step(gpu):
    from fallingsand3d_amd import render as R
    dims = (1024, 1024, 512)
    announce(f"frame of {dims} behind 0.3 s of ticks")
    with gpu.World(dims, flags=gpu.DENSE) as w:
        w.fuse = False
        w.fill_rain(3, gpu.threshold(3, 10))
        cam = R.orbit_camera(dims, 0.4, 1.6, 0.4, 16 / 9)
        R.render(w, cam, 640, 360)
        w.step(100)
        w.sync()
        shares = []
        for _ in range(3):
            w.step(1500)
            t0, c0 = time.perf_counter(), time.process_time()
            R.render(w, cam, 640, 360)
            wall, cpu = time.perf_counter() - t0, time.process_time() - c0
            print(f"wall {wall * 1e3:.0f} ms, processor {cpu * 1e3:.0f} ms")
            assert wall > 0.05
            shares.append(cpu / wall)
        # one thread that waits in the runtime, whose way of waiting is its own
        assert min(shares) < 1.3
