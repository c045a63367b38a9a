"""Planes take no memory of their own where the byte buffer that is not current holds
them, and that buffer's use by ticks on bytes, loads and saves in between goes on."""
import ctypes

import numpy as np
import pytest

from conftest import announce
from fallingsand3d_amd._lib import lib

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0  # (of the runtime it is linked with)
    return free.value


def test_runs_take_no_more_memory(gpu):
    dims = (1024, 1024, 600)
    announce(f"memory of a run of {dims}")
    for dense in (False, True):
        with gpu.World(dims, flags=gpu.DENSE if dense else 0) as w:
            w.fill_rain(1, gpu.threshold(3, 10))
            w.step(2)
            w.sync()
            before = free_bytes()
            w.run(10, 5)
            assert before - free_bytes() < w.size // 16  # (lists of what moves, graphs)


# rows whose planes fit the other byte buffer, and rows whose planes do not
@pytest.mark.parametrize("shape", [(130, 40, 33), (33, 60, 41), (65, 30, 30), (1100, 9, 40)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dense", [False, True], ids=["default", "dense"])
def test_bytes_and_planes_in_turn(gpu, O, tmp_path, shape, dense):
    rng = np.random.default_rng(shape[0])
    nx, ny, nz = shape
    announce(f"ticks on bytes, planes, loads and edits in turn {shape} dense={dense}")
    cur = rng.choice(np.array([0, 0, 0, 1, 2, 2, 3, 222], np.uint8), size=(nz, ny, nx))
    path = tmp_path / "w.fs3d"
    with gpu.World(shape, flags=gpu.DENSE if dense else 0) as w:
        w.upload(cur)
        t, saved = 0, None
        for k in range(60):
            op = int(rng.integers(0, 9))
            if op == 0:
                w.save(path)
                saved = (cur, t)
            elif op == 1 and saved:
                w.load(path)
                cur, t = saved
            elif op == 2:
                w.prepare_run(int(rng.integers(3, 6)), 0)
            elif op == 3:
                x, y, z, v = int(rng.integers(0, nx)), int(rng.integers(0, ny)), int(rng.integers(0, nz)), int(rng.integers(0, 5))
                w.set_voxel(x, y, z, v)
                cur = cur.copy()
                cur[z, y, x] = v
            elif op == 4 and not dense:
                w.skip = [gpu.SKIP_AUTO, gpu.SKIP_SEGS, gpu.SKIP_WAVES, gpu.SKIP_LISTED][int(rng.integers(0, 4))]
            else:
                n = int(rng.choice([1, 1, 2, 3, 4, 7]))
                if op % 2:
                    w.run(n, 0)
                else:
                    w.step(n)
                cur, _ = O.run(cur, t, n, use_lut=True)
                t += n
            assert w.tick_count == t and w.hash() == O.state_hash(cur), (k, op)
        assert (w.download() == cur).all()
