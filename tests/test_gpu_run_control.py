"""The device time loop on a grid that was used before: the CFL maxima of an
earlier state must not reach a later one's dt, whatever calls lie between."""
import numpy as np
import pytest

import hydro_amd
import oracle
from tests.helpers import bits_differ, to_oracle

pytestmark = pytest.mark.gpu

# tiles, two sweeps (FP64)
SIZES = [(96, 70), (900, 801)]


def params(nx, ny):
    return hydro_amd.Params(nx=nx, ny=ny, dx=1.0 / nx, courant_factor=0.7, tend=1e30)


def quiet(p):
    """A state with wave speeds far below a blast's."""
    i, j = np.meshgrid(np.arange(p.nx + 4), np.arange(p.ny + 4))
    rho = 1.0 + ((3 * i + j) % 17) / 40.0
    u, v = ((i + 2 * j) % 13) / 130.0, ((5 * i + j) % 11) / 120.0
    pr = 0.01 + ((i + j) % 7) / 1000.0
    e = pr / (p.gamma - 1.0) + 0.5 * rho * (u * u + v * v)
    return np.ascontiguousarray(np.stack([rho, rho * u, rho * v, e]))


def check(g, p, u, state, steps):
    """Runs g on, and the oracle from the same state, dt sequence and state compared."""
    dts = g.run(steps)
    ref, _ = oracle.Port().run(to_oracle(p), u, steps, state)
    assert bits_differ(dts, ref) == 0, (dts, ref)
    assert bits_differ(g.download(), u) == 0


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("before", ["run", "godunov"])
def test_odd_step_after_another_run(nx, ny, before):
    p = params(nx, ny)
    with hydro_amd.Grid(p) as g:
        g.init_blast(nx // 2, ny // 2, 1.0 / p.dx / p.dx)
        if before == "run":
            g.run(2)
        else:
            g.godunov(2, g.compute_deltat())
        u = quiet(p)
        g.upload(u)
        g.set_state(0.25, 3, 1e-4)
        check(g, p, u, (0.25, 3, 1e-4), 6)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_new_state_over_queued_steps(nx, ny):
    p = params(nx, ny)
    weak = (nx // 3, ny // 3, 1e-3 / p.dx / p.dx)
    with hydro_amd.Grid(p) as g:
        g.init_blast(nx // 2, ny // 2, 1.0 / p.dx / p.dx)
        g.run(1)
        g.run_async(1)  # the odd step, whose maxima are in the slots when it is done
        g.init_blast(*weak)
        check(g, p, oracle.Port().init_blast(to_oracle(p), *weak), None, 5)
