"""An editor's calls, one cell or one hash at a time, against the oracle: sizes around
the largest that is hashed by one launch, cells at every edge, reserved bytes, and
worlds whose state is bytes or planes."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

# 2^18 cells are hashed by one launch
SHAPES = [(1, 1, 1), (5, 3, 2), (48, 37, 29), (64, 64, 64), (257, 255, 4), (64, 65, 64)]


@pytest.mark.parametrize("planes", [False, True], ids=["bytes", "planes"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_pokes_and_single_ticks(gpu, O, shape, planes):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + planes)
    cur, t = rng.choice(np.array([0, 0, 1, 2, 3], np.uint8), size=(nz, ny, nx)), 0
    announce(f"edits and single ticks {shape} planes={planes}")
    with gpu.World(shape) as w:
        w.upload(cur)
        if planes:
            w.run(4, 0)
            cur, _ = O.run(cur, t, 4, use_lut=True)
            t += 4
        for k in range(9):
            for _ in range(4):
                x, y, z = (int(rng.choice([0, n - 1, int(rng.integers(0, n))])) for n in shape)
                v = int(rng.choice([0, 1, 2, 3, 200]))
                w.set_voxel(x, y, z, v)
                cur[z, y, x] = v
                assert w.get_voxel(x, y, z) == v
            assert w.hash() == O.state_hash(cur)
            if k % 2:
                w.step(1)
                cur, _ = O.run(cur, t, 1, use_lut=True)
                t += 1
                assert w.get_voxel(nx - 1, ny - 1, nz - 1) == cur[-1, -1, -1]
            cur, want = O.run(cur, t, 1, 1, use_lut=True)
            t += 1
            assert w.tick() == int(want[0])
        assert (w.download() == cur).all()
