"""A batch advances its instances in two groups on streams of their own, small
loads in one: loads of one, two and many instances, even and lopsided, with instances that come and
go at either step parity and runs queued behind one another, each state bit for
bit that of the same run on a grid of its own."""
import numpy as np
import pytest

import hydro_amd
from tests.helpers import bits_differ

pytestmark = pytest.mark.gpu

LOADS = [[(70, 50)], [(64, 60), (61, 65)], [(700, 500), (2, 3)], [(600, 380), (598, 381)],
         [(300, 200), (8, 8), (122, 64), (1, 40), (65, 129), (250, 6), (33, 33)]]
FORMS = [hydro_amd.FP64, hydro_amd.FP64_FAST, hydro_amd.MIXED]


def params(nx, ny, k, form):
    return hydro_amd.Params(nx=nx, ny=ny, dx=1.0 / max(nx, ny), courant_factor=0.8, tend=1e30,
                            boundary_left=1 + k % 3, boundary_right=1 + k % 3,
                            boundary_down=1 + k // 3 % 3, boundary_up=1 + k // 3 % 3,
                            slope_type=1.0 + k % 2, precision=form)


def alone(p, k, steps):
    with hydro_amd.Grid(p) as g:
        g.init_blast(p.nx // 2, p.ny // 3, 1.0 + k)
        g.run(steps)
        return g.download()


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("load", LOADS, ids=lambda x: "%dx%d" % x[0])
def test_groups(load, form):
    with hydro_amd.Batch(form) as b, hydro_amd.Batch(form) as other:
        for x in (b, other):
            x.ids = []
            for k, (nx, ny) in enumerate(load):
                p = params(nx, ny, k, form)
                i = x.add(p)
                x.init_blast(i, nx // 2, ny // 3, 1.0 + k)
                x.ids.append((i, p, k))
        for n in (3, 4):  # queued behind one another, beside the other batch
            b.run_async(n)
            other.run_async(n)
        late = params(96, 40, 7, form)  # joins at the other parity
        i = b.add(late)
        b.init_blast(i, 48, 13, 8.0)
        b.run(5)
        for j, p, k in b.ids:
            assert bits_differ(b.download(j), alone(p, k, 12)) == 0, (p, "12 steps")
        gone = b.ids.pop(0)  # the largest of most loads leaves
        b.remove(gone[0])
        b.run(2)
        for j, p, k in b.ids:
            assert bits_differ(b.download(j), alone(p, k, 14)) == 0, (p, "14 steps")
        assert bits_differ(b.download(i), alone(late, 7, 7)) == 0
        for j, p, k in other.ids:
            assert bits_differ(other.download(j), alone(p, k, 7)) == 0, (p, "7 steps")


@pytest.mark.parametrize("form", [hydro_amd.FP64_FAST, hydro_amd.MIXED])
def test_whole_steps(form):
    """Loads large enough for whole steps, whose states change buffers with each
    step: odd and even counts, runs that end on their own at either parity, a
    load that falls below the line and one whose narrow grid rules them out."""
    big = [(1900, 2300), (700, 3001), (61, 5000), (500, 7)]
    big += [(2001, 1200)] if form == hydro_amd.MIXED else []
    with hydro_amd.Batch(form) as b:
        ids = []
        for k, (nx, ny) in enumerate(big):
            p = params(nx, ny, k, form)
            p.nstepmax = (2**31 - 1, 2**31 - 1, 5, 6)[k % 4]
            i = b.add(p)
            b.init_blast(i, nx // 2, ny // 3, 1.0 + k)
            ids.append((i, p, k))

        def check(steps):
            for i, p, k in ids:
                want = alone(p, k, min(steps, p.nstepmax))
                assert bits_differ(b.download(i), want) == 0, (p, steps)
        b.run(3)
        check(3)
        b.autotune(1)
        b.run_async(1)
        check(4)  # (without a sync)
        b.run_async(3)
        u = b.download(ids[2][0])
        b.sync()
        assert np.array_equal(u, b.download(ids[2][0]))
        check(7)
        thin = params(2, 90, 5, form)  # rules whole steps out
        t = b.add(thin)
        b.init_blast(t, 1, 30, 6.0)
        b.run(2)
        check(9)
        b.remove(t)
        b.run(1)
        check(10)
        b.remove(ids.pop(0)[0])  # (fast: below the line from here)
        b.run(3)
        check(13)
        b.set_tune(2, 4, 8)
        b.run(1)
        check(14)
        i, p, k = ids[0]
        b.init_blast(i, p.nx // 2, p.ny // 3, 1.0 + k)
        b.run(1)
        assert bits_differ(b.download(i), alone(p, k, 1)) == 0
