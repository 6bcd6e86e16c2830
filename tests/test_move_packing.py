"""Re-binning against the oracle's order bit for bit: cells below, at and past the packing's 64
and 128 particles, few to nearly all of them leaving, and grids at the edge of the one-workgroup
scan."""
import numpy as np
import pytest

from exanbody_amd import Box
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

EDGE = 3.0


def pair_of(dims, n, seed):
    rng = np.random.default_rng(seed)
    hi = np.array(dims, float) * EDGE
    r = rng.uniform(0.0, 1.0, (n, 3)) * hi
    v = rng.standard_normal((n, 3))
    ids = np.arange(n, dtype=np.uint64)
    o = Oracle((0, 0, 0), tuple(hi), dims, EDGE, ghost_dist=2.8)
    o.set_particles(r, v, ids)
    b = Box((0, 0, 0), tuple(hi), dims, EDGE)
    b.nbh_dist(2.5, 0.3)
    b.set_particles(r, v, ids)
    return o, b


def same(o, b):
    eo, eb = o.export(), b.export()
    for k in ("cell", "id", "r", "v"):
        np.testing.assert_array_equal(np.ascontiguousarray(eo[k]).view(np.uint8), np.ascontiguousarray(eb[k]).view(np.uint8), err_msg=k)


# particles a cell: 1, 20, 64 around the one-word edge, 128 around the two-word edge, 200
@pytest.mark.parametrize("per_cell", [1, 20, 63, 66, 127, 130, 200])
@pytest.mark.parametrize("dt", [0.02, 0.3, 1.5])
def test_cells(per_cell, dt):
    o, b = pair_of((4, 3, 5), 60 * per_cell, per_cell)
    for _ in range(3):
        o.push_f_v_r(dt)
        b.push_f_v_r(dt)
        o.move_particles()
        b.move_particles()
        same(o, b)
        o.rebuild_amr()
        b.rebuild_amr()
        same(o, b)


# with the ghost layer: 32,768 cells, and the next cubic grid; and one of several scan tiles
@pytest.mark.parametrize("dims", [(30, 30, 30), (31, 31, 31), (19, 20, 21), (1, 1, 1)])
def test_grids(dims):
    o, b = pair_of(dims, 3000, 7)
    o.push_f_v_r(0.7)
    b.push_f_v_r(0.7)
    o.move_particles()
    b.move_particles()
    same(o, b)
    o.ghost_update_all()
    b.ghost_update_all()
    assert o.num_ghost_particles() == b.num_particles()[1]
    eo, eb = o.export(ghosts=True), b.export(ghosts=True)
    np.testing.assert_array_equal(eo["id"], eb["id"])
    np.testing.assert_array_equal(eo["r"].view(np.uint64), eb["r"].view(np.uint64))
