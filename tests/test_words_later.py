"""chunk_neighbors of a large box leaves the staging words to the first force: the forces, runs and
lists that follow are those of lists built with them."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Box, cubic_domain
from tests.helpers import RCUT, SKIN, fcc_inputs

pytestmark = pytest.mark.gpu


def _boxes(precision):
    r, v, ids, L = fcc_inputs(73, temperature=1.0, seed=9)  # 1,556,068 atoms
    assert len(r) >= 1_500_000
    d = cubic_domain(L, RCUT + SKIN)
    out = []
    for _ in range(2):
        b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
        b.nbh_dist(RCUT, SKIN)
        b.set_particles(r, v, ids)
        b.init(1.0, 1.0, RCUT, SKIN, precision)
        out.append(b)
    return out


def _same(a, c):
    ea, ec = a.export(ghosts=True), c.export(ghosts=True)
    for k in ("cell", "id", "r", "v", "f", "ep"):
        assert np.array_equal(ea[k].view(np.uint8), ec[k].view(np.uint8)), k


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
def test_forces_and_runs_after_lists(precision):
    a, c = _boxes(precision)
    a.chunk_neighbors(RCUT + SKIN)
    for b in (a, c):
        b.zero_particle_force()
        b.lennard_jones_force(1.0, 1.0, RCUT, precision=precision)
    _same(a, c)
    a.chunk_neighbors(RCUT + SKIN)
    for b in (a, c):
        b.run(3, 0.004, 1.0, 1.0, RCUT, SKIN, precision=precision, rebuild_every=2)
    _same(a, c)
    # lists with a filter in between, twice without a force
    a.chunk_neighbors(RCUT + SKIN, half_symmetric=1)
    a.chunk_neighbors(RCUT + SKIN)
    a.chunk_neighbors(RCUT + SKIN)
    for b in (a, c):
        b.zero_particle_force()
        b.gravitational_force(0.5, [1.0], RCUT)
    _same(a, c)


def test_half_lists():
    """The force over half lists: the words are written for them as well."""
    a, c = _boxes(PRECISION_FP64)
    a.chunk_neighbors(RCUT + SKIN, half_symmetric=1)
    a.zero_particle_force()
    a.lennard_jones_force(1.0, 1.0, RCUT)
    c.zero_particle_force()
    c.lennard_jones_force(1.0, 1.0, RCUT)
    # every inner pair once: the energies (each pair counted by one of its atoms) are near half
    ea, ec = a.export()["ep"].sum(), c.export()["ep"].sum()
    assert 0.45 < ea / ec < 0.55
