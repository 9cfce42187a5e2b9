"""The whole-step kernel (small grids) against the two sweep kernels, bit for
bit in every form, at sizes around its tiles (60 columns, 4 or 12 rows); and
the calls that have to know which buffer the state is in after odd numbers of
its steps, against the oracle."""
import numpy as np
import pytest

import hydro_amd
import oracle
from tests.helpers import bits_differ, to_oracle

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3), (4, 4), (59, 5), (60, 12), (61, 13), (120, 24), (121, 25), (180, 96), (300, 211),
          (500, 500), (517, 8), (9, 700)]


def params(nx, ny, form, **kw):
    return hydro_amd.Params(nx=nx, ny=ny, dx=1.0 / max(nx, ny), courant_factor=0.7, tend=1e30,
                            precision=form, **kw)


def smooth(p, seed=3):
    rng = np.random.default_rng(seed)
    x, y = np.arange(p.nx + 4) / p.nx, np.arange(p.ny + 4) / p.ny

    def w(a):
        return a * np.outer(np.cos(12.0 * y + rng.uniform(0, 6)), np.cos(9.0 * x + rng.uniform(0, 6)))
    r, u, v, pr = np.exp(w(0.4)), w(0.8), w(0.8), np.exp(w(0.4))
    return np.ascontiguousarray(
        np.stack([r, r * u, r * v, pr / (p.gamma - 1) + 0.5 * r * (u * u + v * v)]))


@pytest.mark.parametrize("form", [hydro_amd.FP64, hydro_amd.FP64_FAST, hydro_amd.MIXED])
@pytest.mark.parametrize("bounds,slope,iorder,scheme", [
    ((1, 1, 1, 1), 1.0, 2, 1), ((3, 3, 3, 3), 2.0, 2, 1), ((2, 2, 2, 2), 1.0, 2, 2),
    ((0, 1, 2, 0), 1.5, 1, 3)])
def test_same_bits_as_two_sweeps(form, bounds, slope, iorder, scheme):
    for nx, ny in SHAPES:
        p = params(nx, ny, form, slope_type=slope, iorder=iorder, scheme=scheme,
                   boundary_left=bounds[0], boundary_right=bounds[1], boundary_down=bounds[2],
                   boundary_up=bounds[3])
        u0 = smooth(p)
        out = []
        for two in (False, True):
            with hydro_amd.Grid(p) as g:
                if two:
                    g.set_tune(2, 1, 1, 1)
                g.upload(u0)
                dts = np.concatenate([g.run(3), g.run(1), g.run(4)])
                out.append((dts, g.download(), g.image(100)))
        assert bits_differ(out[0][0], out[1][0]) == 0, (nx, ny)
        assert bits_differ(out[0][1], out[1][1]) == 0, (nx, ny)
        assert np.array_equal(out[0][2], out[1][2]), (nx, ny)


def test_calls_between_odd_numbers_of_steps():
    p = params(130, 70, hydro_amd.FP64)
    port, po = oracle.Port(), to_oracle(p)
    u0 = smooth(p)
    u = u0.copy()
    dts, (t, n, dt) = port.run(po, u, 3)

    def more(steps):
        nonlocal t, n, dt
        d, (t, n, dt) = port.run(po, u, steps, (t, n, dt))
        return d

    with hydro_amd.Grid(p) as g:
        g.upload(u0)
        assert np.array_equal(g.run(3), dts)
        assert bits_differ(g.download(), u) == 0
        assert np.array_equal(g.run(2), more(2))          # odd step first
        g.make_boundary(1)
        port.make_boundary(1, po, u)
        assert bits_differ(g.download(), u) == 0
        g.set_tune(4, 1, 4, 2)                            # the sweeps from here ...
        assert np.array_equal(g.run(3), more(3))
        assert g.compute_deltat() == port.compute_deltat(po, u)
        g.autotune(1)                                     # ... or either
        assert np.array_equal(g.run(1), more(1))
        g.run_async(1)
        g.run_async(2)
        more(3)
        assert bits_differ(g.download(), u) == 0          # (without a sync)
        assert g.state()[:2] == (t, n)
        d = g.compute_deltat()
        g.godunov(1, d)
        g.godunov(2, d)
        g.godunov(2, d)
        for k in (1, 2, 2):
            port.godunov(k, d, po, u)
        assert bits_differ(g.download(), u) == 0
        assert g.compute_deltat() == port.compute_deltat(po, u)
        g.upload(u0)
        assert bits_differ(g.download(), u0) == 0
