"""Device memory of a trainer per key of its budget (opts.entriesCap): the
sort's key and id buffers, and nothing beside them. The raster's record of
taken keys lies in those once they are free."""
import ctypes as C

import numpy as np
import pytest

import gsabi

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _setup(keys, W=160, H=96, n=500, trainer=None, **kw):
    rng = np.random.default_rng(1)
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / 100.0 * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / 100.0 * z
    p[:, 2] = z
    p[:, 3:6] = -2.0
    p[:, 6] = 1.0
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 100.0, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": rng.random((W * H, 3)).astype(np.float32)}]
    t = trainer or gsabi.GSTrainer(shDeg=0, maxSplats=n, entriesCap=keys, **kw)
    t.setup({"data": p, "n": n}, cams, images, W, H, 2.0)
    return t


@pytest.mark.parametrize("name,bytes_per_key,kw", [
    # keys and scratch of 8 bytes, ids and scratch of 4
    ("segments", 24, {}),
    ("segments_32", 24, {"tile": 32}),
    ("global64", 24, {"sortMode": gsabi.GS_SORT_GLOBAL64}),
    ("radix", 16, {"sortMode": gsabi.GS_SORT_DEPTH_THEN_TILE}),
    # three views more with ids, keys and scratch of their own
    ("views", 24 + 3 * 20, {"viewsPerStep": 4}),
    ("views_32", 24 + 3 * 20, {"viewsPerStep": 4, "tile": 32}),
    # the overlapped launches record the first view's taken keys apart: 2 bytes at 16 pixels, 8 at 32
    ("overlap", 24 + 3 * 20 + 2, {"viewsPerStep": 4, "viewsLaunch": gsabi.GS_VIEWS_OVERLAP}),
    ("overlap_32", 24 + 3 * 20 + 8, {"viewsPerStep": 4, "viewsLaunch": gsabi.GS_VIEWS_OVERLAP, "tile": 32}),
], ids=lambda v: v if isinstance(v, str) else "")
def test_memory_per_budgeted_key(name, bytes_per_key, kw):
    """Free memory with two budgets 64M keys apart; allocations come in pages
    of 2 MB, 30 at most here: 1 byte per key of margin."""
    left = []
    for keys in (16 << 20, 80 << 20):
        t = _setup(keys, **kw)
        t.stepOnce(0)
        t.readLoss()
        left.append(_free_bytes())
        t.destroy()
    per_key = (left[0] - left[1]) / (64 << 20)
    print(name, per_key, flush=True)
    assert abs(per_key - bytes_per_key) <= 1.0


@pytest.mark.parametrize("launch", [gsabi.GS_VIEWS_PERSISTENT, gsabi.GS_VIEWS_OVERLAP])
def test_raster_shapes_changed_between_batched_steps(launch):
    """Batched steps, graph replays among them, as the tiles go from 16 pixels
    to 32, 8 and back: the record of taken keys grows with the tile, and the
    sums stay those of a trainer that runs the views in one launch without a
    graph. Single steps run in between on the same buffers."""
    kw = dict(viewsPerStep=3, seed=5)
    a, b = _setup(1 << 20, viewsLaunch=launch, graph=1, **kw), _setup(1 << 20, graph=0, **kw)
    for tile in (16, 32, 8, 16):
        for t in (a, b):
            t.setRasterShape(tile, 128)
            for _ in range(3):
                t.stepViews([0, 0, 0])
            t.stepOnce(0)
            t.stepViews([0, 0])
        x, y = a.readGaussians()["data"], b.readGaussians()["data"]
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32), err_msg=f"tile {tile}")
    a.destroy()
    b.destroy()


def test_second_setup_past_the_batched_binning_limit():
    """15 further slots of 107.3M keys take 25.76 GB of binning buffers, just
    under the 24 GiB that batched binning may have; with 100k Gaussians the
    same trainer's second setup passes that, and its views bin one after
    another. Its steps are those of a trainer that was set up once."""
    kw = dict(viewsPerStep=16, seed=5)
    keys = 107_300_000
    a = _setup(keys, n=500, **kw)
    a.stepViews([0, 0])
    _setup(keys, n=100000, trainer=a)
    b = _setup(1 << 22, n=100000, **kw)
    for t in (a, b):
        for _ in range(3):
            t.stepViews([0, 0, 0])
    x, y = a.readGaussians()["data"], b.readGaussians()["data"]
    a.destroy()
    b.destroy()
    np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))
