"""Hashes inside runs of plane ticks against the oracle: after every tick, after
every second or third one, on either side of the sizes up to which a word takes
sixteen lanes and the sum one slot, with reserved bytes."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [1, 2, 3])
@pytest.mark.parametrize("shape", [(16, 1, 1), (64, 64, 64), (65, 7, 70), (200, 30, 41), (100, 60, 64), (100, 62, 64),
                                   (1000, 30, 62), (1000, 31, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_hashes_match_oracle(gpu, O, shape, every):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + every)
    g = rng.choice(np.array([0, 0, 0, 1, 2, 3, 3, 250], np.uint8), size=(nz, ny, nx))
    announce(f"hashed plane runs {shape} every {every}")
    with gpu.World(shape) as w:
        w.upload(g)
        t = 0
        for n in (9, 4):
            g, want = O.run(g, t, n, every, use_lut=True)
            assert [int(h) for h in w.run(n, every)] == [int(h) for h in want]
            t += n
        assert (w.download() == g).all()
