"""The march kernel on states far from smooth ones (near-vacuum and huge cells,
signed zeros, infinities and NaN) against the two sweep kernels, bit for bit (a
NaN matching a NaN), on grids large enough to take it.  The steps have a given
dt: the maximum behind a computed one depends on the order of its cells where
some are NaN."""
import numpy as np
import pytest

import hydro_amd
from tests.helpers import bits_differ
from tests.test_gpu_whole_step import params, smooth

pytestmark = pytest.mark.gpu

SHAPES = [(hydro_amd.FP64_FAST, 1021, 1100), (hydro_amd.MIXED, 2101, 4200)]


def blocks(rng, p, n, side=40):
    for _ in range(n):
        j, i = rng.integers(0, p.ny + 4), rng.integers(0, p.nx + 4)
        yield (slice(None), slice(j, j + rng.integers(1, side)), slice(i, i + rng.integers(1, side)))


def state(kind, p):
    u, rng = smooth(p), np.random.default_rng(5)
    big = 1e30 if p.precision == hydro_amd.MIXED else 1e200
    for b in blocks(rng, p, 60):
        v = u[b]
        if kind == "vacuum":
            v[0], v[3] = 10.0 ** rng.uniform(-30, -8), 10.0 ** rng.uniform(-40, -10)
            v[1:3] *= v[0]
        elif kind == "huge":
            v[3] = rng.choice([1e12, big, -big])
            v[1] *= rng.choice([1e6, -1e10])
        elif kind == "zeros":
            for k in (1, 2, 3):
                v[k] = rng.choice([0.0, -0.0], size=v[k].shape)
        else:
            v[rng.integers(0, 4)] = rng.choice([np.nan, np.inf, -np.inf])
    return u


@pytest.mark.parametrize("form,nx,ny", SHAPES)
@pytest.mark.parametrize("kind", ["vacuum", "huge", "zeros", "nonfinite"])
def test_same_bits_as_two_sweeps(form, nx, ny, kind):
    p = params(nx, ny, form)
    u0, out = state(kind, p), []
    for two in (False, True):
        with hydro_amd.Grid(p) as g:
            if two:
                g.set_tune(2, 1, 1, 1)
            g.upload(u0)
            for n in range(4):
                g.godunov(1 + n % 2, 1e-5)
            out.append(g.download())
    assert bits_differ(*out) == 0, (p, kind)
