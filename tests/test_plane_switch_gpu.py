"""Changes between ticks of the active items and ticks of everything on one large world,
against the byte kernels: an odd and an even number of dense passes in between, and
runs that begin at either parity."""
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPE = (1024, 1031, 517)
NEAR = (704, 640, 600)  # the fewest voxels, 2^28, whose items are listed


def same(a, b, what):
    assert a.tick_count == b.tick_count
    assert a.hash() == b.hash(), what


@pytest.mark.parametrize("shape", [SHAPE, NEAR], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("t0", [0, 1])
def test_runs_between_changes_of_schedule(gpu, shape, t0):
    announce(f"changes of schedule between runs of {shape}, from tick {t0}")
    with gpu.World(shape) as a, gpu.World(shape, flags=gpu.DENSE) as b:
        b.fuse = False  # single byte ticks of every row quad
        for w in (a, b):
            w.fill_boxes(7, side_min=5, side_max=60)
            w.tick_count = t0
        for dense in (3, 4, 5):
            for items in (3, 4):
                for skip, n in ((gpu.SKIP_AUTO, 4), (gpu.SKIP_OFF, dense), (gpu.SKIP_AUTO, items)):
                    a.skip = skip
                    a.run(n, 0)
                    b.run(n, 0)
                    same(a, b, (dense, items, skip, a.tick_count))


@pytest.mark.parametrize("t0", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3])
def test_short_runs_after_a_change_of_schedule(gpu, n, t0):
    announce(f"runs of {n} after a change of schedule, from tick {t0}")
    with gpu.World(SHAPE, flags=gpu.DENSE) as a, gpu.World(SHAPE, flags=gpu.DENSE) as b:
        b.fuse = False
        for w in (a, b):
            w.fill_boxes(8, side_min=5, side_max=60)
            w.tick_count = t0
            w.run(10, 0)
        for skip, first in ((gpu.SKIP_AUTO, n), (gpu.SKIP_OFF, n), (gpu.SKIP_AUTO, n), (gpu.SKIP_OFF, 4), (gpu.SKIP_AUTO, n)):
            a.skip = skip
            for k in (first, n, 1, 1, n):
                a.step(k)
                b.step(k)
            same(a, b, (skip, a.tick_count))
