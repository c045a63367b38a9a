"""Grids of so many thin layers that a launch with a workgroup for every two of them
would have 2^32 threads or more."""
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dense", [False, True], ids=["default", "dense"])
def test_runs_of_very_many_layers(gpu, dense):
    shape = (24, 1, 45_000_000)
    announce(f"runs of {shape} dense={dense}")
    with gpu.World(shape, flags=gpu.DENSE if dense else 0) as a, gpu.World(shape, flags=gpu.DENSE) as b:
        b.fuse = False  # byte ticks
        for w in (a, b):
            w.fill_rain(3, gpu.threshold(3, 10))
        assert list(a.run(4, 2)) == list(b.run(4, 2))
        a.step(3)
        b.step(3)
        assert a.hash() == b.hash()
