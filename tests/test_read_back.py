"""Read-back of particles and neighbour streams: whole chunks, remainders, several threads."""
import threading

import numpy as np
import pytest

from exanbody_amd import Box, cubic_domain

pytestmark = pytest.mark.gpu

RHO = 0.8


def make(n, seed):
    rng = np.random.default_rng(seed)
    length = max((n / RHO) ** (1.0 / 3.0), 6.0)
    r, v = rng.uniform(0.0, length, (n, 3)), rng.standard_normal((n, 3))
    types = rng.integers(0, 256, n).astype(np.uint8)
    ids = rng.permutation(n).astype(np.uint64)
    d = cubic_domain(length, 2.8)
    b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
    b.nbh_dist(2.5, 0.3)
    b.set_particles(r, v, ids, types, extra=[v[:, 0] * 3.0])
    return b, r, v, ids, types, d


def check(b, r, v, ids, types, e):
    at = np.argsort(ids)[e["id"].astype(np.int64)]  # input index of every exported particle
    np.testing.assert_array_equal(np.sort(e["id"]), np.arange(len(ids), dtype=np.uint64))
    np.testing.assert_array_equal(e["r"], r[at])
    np.testing.assert_array_equal(e["v"], v[at])
    np.testing.assert_array_equal(e["type"], types[at])
    np.testing.assert_array_equal(e["extra"][0], v[at, 0] * 3.0)
    assert not e["f"].any() and not e["ep"].any()


# a workgroup packs 256 particles, half a pinned block holds 11,264 on the way out, 16,384 on the way in; from 64 MiB on several threads
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 11263, 11264, 11265, 16384, 16385, 33793, 800001])
def test_export(n):
    b, r, v, ids, types, d = make(n, n)
    e = b.export()
    check(b, r, v, ids, types, e)
    counts = b.cell_counts()
    np.testing.assert_array_equal(e["cell"], np.repeat(np.arange(len(counts), dtype=np.uint32), counts))
    b.move_particles()
    b.rebuild_amr()
    b.ghost_update_all()
    counts = b.cell_counts()
    inner, g = b.export(), b.export(ghosts=True)
    assert g["r"].shape[0] == sum(b.num_particles())
    np.testing.assert_array_equal(g["cell"], np.repeat(np.arange(len(counts), dtype=np.uint32), counts))
    dims, gl, _ = b.grid_info()
    i, j, k = g["cell"] % dims[0], g["cell"] // dims[0] % dims[1], g["cell"] // (dims[0] * dims[1])
    own = np.all([(x >= gl) & (x < m - gl) for x, m in ((i, dims[0]), (j, dims[1]), (k, dims[2]))], axis=0)
    for q in ("cell", "r", "v", "f", "ep", "id", "type"):
        np.testing.assert_array_equal(g[q][own], inner[q])
    # an image is its source shifted by whole box edges, one rounding away
    src = np.empty(n, np.int64)
    src[inner["id"].astype(np.int64)] = np.arange(n)
    s = src[g["id"].astype(np.int64)]
    shift = (g["r"] - inner["r"][s]) / (d["grid_dims"][0] * d["cell_size"])
    assert np.abs(shift - np.round(shift)).max() < 1e-14
    np.testing.assert_array_equal(g["v"], inner["v"][s])
    np.testing.assert_array_equal(g["type"], inner["type"][s])


def test_boxes_read_back_from_several_threads():
    boxes = [make(30000 + 710000 * (q % 2) + 1111 * q, q) for q in range(4)]
    got = [None] * 4

    def read(q):
        got[q] = [boxes[q][0].export() for _ in range(3)]

    th = [threading.Thread(target=read, args=(q,)) for q in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for q in range(4):
        for e in got[q]:
            check(*boxes[q][:5], e)
