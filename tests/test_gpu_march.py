"""The march kernel (both sweeps of a large grid's step in one launch, fast and
mixed forms) against the two sweep kernels, bit for bit: widths around its 60
columns, segments of a few rows and of many, grids of one column block and of
one segment, every boundary type."""
import numpy as np
import pytest

import hydro_amd
from tests.helpers import bits_differ
from tests.test_gpu_whole_step import params, smooth

pytestmark = pytest.mark.gpu

# (bounds left, right, down, up), slope_type, iorder, scheme
SETUPS = [((1, 1, 1, 1), 1.0, 2, 1), ((3, 3, 3, 3), 2.0, 2, 1), ((2, 2, 2, 2), 1.0, 2, 2),
          ((0, 1, 2, 0), 1.5, 1, 3)]
FAST, MIXED = hydro_amd.FP64_FAST, hydro_amd.MIXED
SHAPES = [(FAST, s) for s in [(3, 16001), (59, 16003), (61, 8003), (120, 8001), (121, 5400),
                              (2047, 470), (16300, 61), (30001, 33), (245820, 5)]]
SHAPES += [(MIXED, s) for s in [(60, 150001), (2101, 4200), (8188, 1101), (126000, 73)]]


@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_same_bits_as_two_sweeps(k):
    form, (nx, ny) = SHAPES[k]
    for m in (k % 4, (k + 1 + k // 4) % 4):
        b, slope, iorder, scheme = SETUPS[m]
        p = params(nx, ny, form, slope_type=slope, iorder=iorder, scheme=scheme,
                   boundary_left=b[0], boundary_right=b[1], boundary_down=b[2], boundary_up=b[3])
        u0 = smooth(p)
        out = []
        for two in (False, True):
            with hydro_amd.Grid(p) as g:
                if two:
                    g.set_tune(2, 1, 1, 1)
                g.upload(u0)
                dts = np.concatenate([g.run(3), g.run(2)])
                out.append((dts, g.download()))
        assert bits_differ(out[0][0], out[1][0]) == 0, (p, m)
        assert bits_differ(out[0][1], out[1][1]) == 0, (p, m)
