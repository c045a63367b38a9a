"""Copies to host memory through the staging slots: around the sizes at which the
slots, the pieces and the helper threads begin and end, odd sizes, pinned
destinations, several threads at once, and images of the sphere tracer cut into
pieces anywhere."""
import ctypes
import threading

import numpy as np
import pytest

from conftest import announce
from fallingsand3d_amd._lib import check, lib

pytestmark = pytest.mark.gpu

# 64 KiB, 512 KiB (the calling thread alone), 1 MiB a slot, 12 slots in use
SIZES = [1, 65535, 65536, 65537, 524287, 524288, 524301, (1 << 20) + 16383, 12 << 20, (12 << 20) + 1, 33 * (1 << 20) + 5]


@pytest.mark.parametrize("n", SIZES)
def test_download_sizes(gpu, n):
    rng = np.random.default_rng(n)
    dims = {1: (1, 1, 1)}.get(n) or next((d, n // d, 1) for d in range(min(4096, n), 0, -1) if n % d == 0)
    g = rng.integers(0, 4, n, dtype=np.uint8).reshape(dims[::-1])
    announce(f"download of {dims}")
    with gpu.World(dims) as w:
        w.upload(g)
        assert (w.download() == g).all()
        hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so.7")
        pinned = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(n), 0) == 0
        check(lib().fs3d_world_download(w.handle, pinned, n))
        assert ctypes.string_at(pinned, n) == g.tobytes()
        assert hip.hipHostFree(pinned) == 0


def test_downloads_from_threads(gpu):
    announce("four threads downloading and rendering at once")
    from fallingsand3d_amd import render as R
    want = R.render_sdf(W=700, H=500)
    bad = []

    def one(seed):
        rng = np.random.default_rng(seed)
        g = rng.integers(0, 4, (37, 300, 301), dtype=np.uint8)
        with gpu.World((301, 300, 37)) as w:
            w.upload(g)
            for _ in range(6):
                if not (w.download() == g).all() or not np.array_equal(R.render_sdf(W=700, H=500), want):
                    bad.append(seed)

    ts = [threading.Thread(target=one, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_sdf_pieces(gpu, O):
    from fallingsand3d_amd import render as R
    announce("sphere tracer images cut into pieces")
    for W, H in ((1, 1), (3, 700), (701, 3), (257, 255), (1023, 311)):
        img = R.render_sdf((0.1, 0.2, -1.5), aspect=1.25, W=W, H=H)
        assert img.tobytes() == O.raymarch_sdf(np.array((0.1, 0.2, -1.5), np.float32), 1.25, W, H).tobytes()
