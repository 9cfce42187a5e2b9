"""States to the device and back: what comes back is what went up, at sizes
below one thread's share, of one slab, of many slabs on many threads, and with
rows wider than a slab (FP32 storage rounds)."""
import numpy as np
import pytest

import hydro_amd

pytestmark = pytest.mark.gpu

# (600000 doubles a row are wider than a staging buffer, 1100000 floats too)
SIZES = [(1, 1), (61, 7), (250, 125), (1021, 767), (2999, 1501), (600000, 3), (1100000, 2)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("form", [hydro_amd.FP64, hydro_amd.MIXED])
def test_round_trip(nx, ny, form):
    p = hydro_amd.Params(nx=nx, ny=ny, dx=0.1, tend=1e30, precision=form)
    u = np.random.default_rng(nx + ny).uniform(-3.0, 3.0, p.shape())
    want = u if form == hydro_amd.FP64 else u.astype(np.float32).astype(np.float64)
    with hydro_amd.Grid(p) as g:
        g.upload(u)
        assert np.array_equal(g.download(), want)
        g.upload(-u)  # (staging buffers are reused)
        assert np.array_equal(g.download(), -want)
    with hydro_amd.Batch(form) as b:
        ids = [b.add(p), b.add(p)]
        b.upload(ids[0], u)
        b.upload(ids[1], -u)
        assert np.array_equal(b.download(ids[0]), want)
        assert np.array_equal(b.download(ids[1]), -want)
