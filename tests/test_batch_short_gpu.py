"""Batch runs of one and two ticks, which take the wide kernel from 2^17 cells on, between
longer ones: hashes and grids against the oracle, and no slower than that kernel."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

FEW = [(20, 9, 11), (64, 30, 30), (7, 40, 33)]
MORE = FEW + [(70, 41, 39), (130, 17, 20)]  # over 2^17 cells


@pytest.mark.parametrize("dims", [FEW, MORE], ids=["few", "more"])
def test_short_and_long_runs(gpu, O, dims):
    rng = np.random.default_rng(len(dims))
    announce(f"batch of {len(dims)} worlds, short and long runs")
    cur = [rng.choice(np.array([0, 0, 1, 2, 3, 90], np.uint8), size=d[::-1]) for d in dims]
    with gpu.Batch(dims) as b:
        for i, g in enumerate(cur):
            b.upload(i, g)
        t = 0
        for n in (1, 2, 5, 1, 1, 2, 3, 0, 2, 7):
            got = b.run(n)
            for i, g in enumerate(cur):
                cur[i], _ = O.run(g, t, n, use_lut=True)
                assert int(got[i]) == O.state_hash(cur[i]), (n, t, i)
                assert (b.download(i) == cur[i]).all()
            t += n
            assert b.tick_count == t


def test_one_tick_is_as_fast_as_the_wide_kernel(gpu):
    dims = [(8, 128, 128)] * 300
    announce("one tick of 300 worlds of 8 x 128 x 128")
    with gpu.Batch(dims) as b:
        b.fill_rain(np.arange(300, dtype=np.uint64), np.full(300, gpu.threshold(3, 10), np.uint64))
        times = {}
        for mode in (gpu.batch.PERSISTENT, gpu.batch.WIDE) * 8:
            b.run(1, mode=mode)
            times.setdefault(mode, []).append(b.last_run_ms())
        short, wide = (min(times[m]) for m in (gpu.batch.PERSISTENT, gpu.batch.WIDE))
        print(f"{short:.3f} ms, wide {wide:.3f} ms")
        assert short < 1.5 * wide
