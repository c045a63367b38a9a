"""Runs of ticks through the bit planes against the oracle, bit for bit: word and
row edges, odd sizes, both start parities, reserved bytes, hashes inside a run,
host edits between runs and switches to and from the byte kernels."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPES = [(16, 1, 1), (16, 5, 9), (17, 9, 11), (31, 2, 2), (63, 6, 7), (64, 1, 5), (64, 8, 8), (65, 7, 6), (100, 33, 37),
          (127, 4, 19), (128, 17, 5), (129, 5, 40), (320, 21, 13), (512, 9, 10), (1000, 6, 20), (1024, 5, 6),
          (2048, 7, 35), (2100, 3, 9), (4033, 3, 4), (4096, 5, 4)]


def scene(rng, shape, reserved=0.02):
    nx, ny, nz = shape
    g = rng.choice(np.array([0, 0, 0, 1, 2, 2, 3, 3], np.uint8), size=(nz, ny, nx))
    g[rng.random(g.shape) < reserved] = 201
    return g


@pytest.mark.parametrize("dense", [False, True], ids=["default", "dense"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_runs_match_oracle(gpu, O, shape, dense):
    rng = np.random.default_rng(sum(shape) * 3 + dense)
    for t0, reserved in ((6, 0.02), (11, 0.0)):
        announce(f"plane runs {shape} t0={t0} dense={dense}")
        g = scene(rng, shape, reserved)
        with gpu.World(shape, flags=gpu.DENSE if dense else 0) as w:
            w.upload(g)
            w.tick_count = t0
            cur, want = O.run(g, t0, 23, 4, use_lut=True)
            assert [int(h) for h in w.run(23, 4)] == [int(h) for h in want]
            assert (w.download() == cur).all()
            w.step(5)
            cur, _ = O.run(cur, t0 + 23, 5, use_lut=True)
            assert (w.download() == cur).all()
            cur, want = O.run(cur, t0 + 28, 1, 1, use_lut=True)
            assert w.tick() == int(want[0]) == w.hash()
            assert w.tick_count == t0 + 29


def test_edits_and_path_switches(gpu, O):
    shape = (200, 30, 41)
    rng = np.random.default_rng(5)
    cur, t = scene(rng, shape), 0
    announce("plane runs with host edits, single byte ticks and schedule switches between them")
    with gpu.World(shape) as w:
        w.upload(cur)
        for k in range(10):
            n = int(rng.integers(1, 9))
            if k % 2:
                w.run(n, 0)
            else:
                w.step(n)
            cur, _ = O.run(cur, t, n, use_lut=True)
            t += n
            assert (w.download() == cur).all(), k
            for _ in range(12):
                x, y, z = int(rng.integers(0, 200)), int(rng.integers(0, 30)), int(rng.integers(0, 41))
                x = int(rng.choice([0, 63, 64, 127, 128, 199, x]))
                v = int(rng.choice([0, 1, 2, 3, 90]))
                w.set_voxel(x, y, z, v)
                cur[z, y, x] = v
            if k == 3:
                w.skip = gpu.SKIP_WAVES  # byte kernels
            if k == 5:
                w.skip = gpu.SKIP_AUTO
            if k == 6:
                t += 3
                w.tick_count = t
            if k == 7:
                cur[8:12, :, 20:90] = 3
                w.upload(cur)
            if k == 8:
                w.step(1)
                cur, _ = O.run(cur, t, 1, use_lut=True)
                t += 1
        assert (w.download() == cur).all()
        assert w.hash() == O.state_hash(cur)


def test_plane_graph_replays(gpu, O):
    dims = (192, 100, 90)
    announce("plane graphs replayed from both parities and buffers")
    with gpu.World(dims) as w:
        w.fill_boxes(5, side_min=6, side_max=40)
        cur, t = w.download(), 0
        for n, every in ((20, 5), (21, 7), (20, 5), (20, 5), (21, 7), (21, 7), (20, 5), (7, 0), (20, 5)):
            got = [int(h) for h in w.run(n, every)]
            cur, want = O.run(cur, t, n, every, use_lut=True)
            t += n
            assert got == [int(h) for h in want], (n, t)
        assert (w.download() == cur).all()
