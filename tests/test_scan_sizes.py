"""Grids on both sides of the sizes where the cell scans change their form (one workgroup up to
6,144 cells, tiles of 8,192 in it and of 2,048 behind it): the same cells, ghosts and forces as the
oracle's."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64
from tests.helpers import RCUT, SKIN, assert_same_layout, make_pair_domain

pytestmark = pytest.mark.gpu

CELL = RCUT + SKIN


# inner cells per side; with the ghost layers 3^3, 2,040, 2,048, 2,052, 6,120, 6,144, 6,160, 8,192 and 8,208 cells
@pytest.mark.parametrize("dims", [(1, 1, 1), (10, 15, 8), (6, 14, 14), (10, 17, 7), (15, 16, 18), (14, 14, 22), (12, 18, 20), (14, 14, 30),
                                  (16, 17, 22)])
def test_cells_ghosts_and_forces(dims):
    rng = np.random.default_rng(sum(dims))
    sites = np.stack(np.meshgrid(*[np.arange(2 * k) for k in dims], indexing="ij"), -1).reshape(-1, 3)
    sites = sites[rng.random(len(sites)) < 0.4] if len(sites) > 8 else sites
    r = (sites + 0.5 + rng.uniform(-0.15, 0.15, sites.shape)) * (0.5 * CELL)
    ids = rng.permutation(len(r)).astype(np.uint64)
    size = tuple(CELL * k for k in dims)
    dom = dict(bounds_min=(0.0,) * 3, bounds_max=size, grid_dims=dims, cell_size=CELL, periodic=(1, 1, 1))
    o, b = make_pair_domain(r, 0.3 * rng.standard_normal(r.shape), ids, dom)
    o.init(1.0, 1.0, RCUT, SKIN)
    b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
    for _ in range(2):
        oe, ge = o.export(ghosts=True), b.export(ghosts=True)
        assert_same_layout(oe, ge)
        for k in ("f", "ep"):
            np.testing.assert_array_equal(o.export()[k].view(np.uint64), b.export()[k].view(np.uint64), err_msg=k)
        assert len(ge["id"]) > len(r)
        for x in (o, b):
            x.run(5, 0.004, 1.0, 1.0, RCUT, SKIN, rebuild_every=5)
