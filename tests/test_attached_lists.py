"""A box whose lists outgrow their capacity when it is attached to a batch (the batch builds them
again and does not wait): whoever uses the lists next, the batch's first step, an operator on the
box, or the box alone after the batch is gone, finds them complete."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Batch, Box, cubic_domain

pytestmark = pytest.mark.gpu

RCUT, SKIN = 2.5, 0.3
KEYS = ("cell", "id", "r", "v", "f", "ep")


def _fallen_in(precision):
    """2,744 atoms at density 0.6 (lists of about 55, capacity 96) that fell freely towards the
    middle of the box by a factor of 0.62, without a rebuild: lists of the present positions are
    longer than the capacity."""
    rng = np.random.default_rng(8)
    m, a = 14, 0.6 ** (-1.0 / 3.0)
    q = np.arange(m ** 3)
    r = (np.stack([q % m, q // m % m, q // (m * m)], 1) + 0.5 + rng.uniform(-0.05, 0.05, (m ** 3, 3))) * a
    v = (0.5 * m * a - r) * 0.38
    d = cubic_domain(m * a, RCUT + SKIN)
    b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
    b.nbh_dist(RCUT, SKIN)
    b.set_particles(r, v)
    b.init(0.0, 1.0, RCUT, SKIN, precision)
    _, first = b.streams()
    assert first < 96
    b.run(4, 0.25, 0.0, 1.0, RCUT, SKIN, precision=precision, rebuild_every=1000)
    return b


def _attach(batch, b, precision):
    return batch.attach(b, 7, 1e-3, 1e-4, 1.0, RCUT, SKIN, precision=precision, rebuild_every=5)


def _same(a, c):
    ea, ec = a.export(ghosts=True), c.export(ghosts=True)
    for k in KEYS:
        np.testing.assert_array_equal(ea[k].view(np.uint8), ec[k].view(np.uint8), err_msg=k)


def _same_streams(a, c):
    (sa, ma), (sc, mc) = a.streams(), c.streams()
    assert ma == mc > 96
    np.testing.assert_array_equal(np.concatenate(sa), np.concatenate(sc))


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("use", ["step", "streams", "batch gone"])
def test_lists_outgrown_at_attach(use, lanes, precision, monkeypatch):
    monkeypatch.setenv("XNB_BRICKS", f"0,0,0,{lanes}")
    a, c = _fallen_in(precision), _fallen_in(precision)
    c.chunk_neighbors(RCUT + SKIN)  # the present positions, like the attach's build
    batch = Batch()
    slot = _attach(batch, a, precision)
    if use == "batch gone":
        batch.close()
        _same_streams(a, c)
        for b in (a, c):
            b.zero_particle_force()
            b.lennard_jones_force(1e-4, 1.0, RCUT, precision=precision)
        _same(a, c)
        for b in (a, c):
            b.run(7, 1e-3, 1e-4, 1.0, RCUT, SKIN, precision=precision, rebuild_every=5)
        _same(a, c)
        return
    if use == "streams":
        _same_streams(a, c)
    while batch.step(3):
        pass
    batch.detach(slot)
    batch.close()
    c.run(7, 1e-3, 1e-4, 1.0, RCUT, SKIN, precision=precision, rebuild_every=5)
    _same(a, c)
