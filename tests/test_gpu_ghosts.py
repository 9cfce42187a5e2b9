"""Ghost cells formed inside the sweeps: every pair of boundary types in each
direction, at the widths where a row piece or a segment ends on them, bit for
bit against the oracle, ghost cells of the whole array included (uploaded
ghosts hold values of their own, which types 0 and 2 keep or read)."""
import numpy as np
import pytest

import hydro_amd
import oracle
from tests.helpers import bits_differ, to_oracle

pytestmark = pytest.mark.gpu

TYPES = [(lo, hi) for lo in (0, 1, 2, 3) for hi in (0, 1, 2, 3)]
SHAPES = [(1, 1), (2, 3), (3, 2), (3, 3), (4, 5), (60, 3), (61, 17), (62, 16), (120, 9), (122, 33),
          (250, 6), (252, 4), (254, 7), (505, 3)]


def state(p, seed):
    rng = np.random.default_rng(seed)
    r = rng.uniform(0.5, 2.0, p.shape()[1:])
    u, v = rng.uniform(-0.5, 0.5, (2,) + r.shape)
    e = rng.uniform(0.5, 2.0, r.shape) / (p.gamma - 1) + 0.5 * r * (u * u + v * v)
    return np.ascontiguousarray(np.stack([r, r * u, r * v, e]))


def cases():
    for k, (nx, ny) in enumerate(SHAPES):
        for m, x in enumerate(TYPES):
            y = TYPES[(5 * m + k) % 16]
            yield hydro_amd.Params(nx=nx, ny=ny, dx=0.02, courant_factor=0.5, tend=1e30,
                                   boundary_left=x[0], boundary_right=x[1],
                                   boundary_down=y[0], boundary_up=y[1]), 16 * k + m


@pytest.mark.parametrize("steps", [1, 3, 4])
def test_ghosts_grid_and_batch(steps):
    port = oracle.Port()
    batch = hydro_amd.Batch()
    want = {}
    for p, seed in cases():
        u0 = state(p, seed)
        u = u0.copy()
        dts, _ = port.run(to_oracle(p), u, steps)
        with hydro_amd.Grid(p) as g:
            g.upload(u0)
            got = g.run(steps)
            assert np.array_equal(got, dts), (p, got, dts)
            assert bits_differ(g.download(), u) == 0, p
        i = batch.add(p)
        batch.upload(i, u0)
        want[i] = (p, u)
    batch.run(steps)
    for i, (p, u) in want.items():
        assert bits_differ(batch.download(i), u) == 0, p
    batch.close()
