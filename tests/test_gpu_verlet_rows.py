"""Verlet rows as the device stores them, against brute force: row lengths on
both sides of each register sort (64, 128 and 256 entries) and beyond it, boxes
of five cells and more per direction, open and mixed directions, a skewed box,
atoms a little outside their periodic box, rows ordered by global ids that
fit 32 bits, that do not, and that repeat, and the cell grids of each way the
cells are made."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import errors, gpu_compute, to_dev
from oracle import OracleNEP, neighbor_rows

pytestmark = pytest.mark.gpu

REACH = 5.2  # radial cutoff 4.2 and skin 1 of the model


def _atoms(h, density, seed, spill):
    """A jittered grid of the density in the box, its atoms moved by up to spill outside it."""
    rng = np.random.default_rng(seed)
    thick = np.array([abs(np.linalg.det(h)) / np.linalg.norm(np.cross(h[:, (d + 1) % 3], h[:, (d + 2) % 3]))
                      for d in range(3)])
    m = np.maximum(1, np.round(thick * density ** (1 / 3)).astype(int))
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, 3)
    u = (g + 0.5 + rng.uniform(-0.3, 0.3, g.shape)) / m
    x = u[rng.permutation(len(u))] @ h.T
    return np.ascontiguousarray((x + rng.uniform(-spill, spill, x.shape) * (spill > 0)).T)


BOXES = {
    "five_cells": (np.diag([13.1, 13.4, 15.5]), (1, 1, 1), 0.0),
    "six_cells": (np.diag([15.6, 16.0, 18.3]), (1, 1, 1), 1.5),
    "mixed": (np.diag([21.0, 14.0, 17.0]), (1, 0, 1), 0.0),
    "open": (np.diag([14.0, 19.0, 12.0]), (0, 0, 0), 0.0),
    "skewed": (np.array([[17.0, 3.0, -2.0], [0.0, 16.0, 2.5], [0.0, 0.0, 15.0]]), (1, 1, 1), 0.0),
}


@pytest.mark.parametrize("ids", [None, "small", "large", "repeated"])
@pytest.mark.parametrize("density", [0.02, 0.105, 0.16, 0.22, 0.42, 0.6])
@pytest.mark.parametrize("name", sorted(BOXES))
def test_rows_match_brute_force(dmgx, name, density, ids):
    h, pbc, spill = BOXES[name]
    pos = _atoms(h, density, 11, spill)
    n = pos.shape[1]
    rng = np.random.default_rng(4)
    gid = {None: None, "small": rng.permutation(n) * 5 + 1, "large": rng.permutation(n) * (1 << 33) + 2,
           "repeated": rng.integers(0, max(1, n // 3), n)}[ids]
    nep = dmgx.NEP(os.path.join(POTENTIALS, "nep_carbon.txt"))
    assert nep.info.rc_radial_max + 1.0 == pytest.approx(REACH)
    kw = {} if gid is None else {"global_id": to_dev(gid.astype(np.int64), __import__("torch").int64),
                                 "sort_by_gid": True}
    gpu_compute(dmgx, nep, dmgx.Box(h, pbc), np.zeros(n, np.int32), pos, **kw)
    rows = nep.verlet_rows(0, n)
    ref = neighbor_rows(h, pbc, pos, nep.info.rc_radial_max + 1.0, max_nb=1024)
    for i in range(n):
        want = np.sort(np.asarray(ref[i]))
        if gid is not None:
            want = want[np.lexsort((want, gid[want]))]
        assert np.array_equal(rows[i], want), (i, len(rows[i]), len(want))


def _elongated(n, edges, seed):
    rng = np.random.default_rng(seed)
    return np.ascontiguousarray(rng.uniform(0.02, 0.98, (n, 3)).T * np.asarray(edges)[:, None])


# (atoms, box, directions): either side of the size up to which one workgroup
# makes the cells, more cells than its LDS holds, several tiles of the scan
# with a rest, rows of cells longer than a tile, and rows of a single cell
CELLS = [(1, (40.0, 40.0, 40.0), (0, 0, 0)), (6144, (38.0, 38.0, 38.0), (1, 1, 1)),
         (6145, (38.0, 38.0, 38.0), (1, 1, 1)), (3000, (80.0, 90.0, 70.0), (1, 0, 1)),
         (4000, (110.0, 30.0, 141.0), (0, 1, 0)), (7000, (61.0, 59.0, 83.0), (1, 1, 1)),
         (6500, (23000.0, 14.0, 14.0), (0, 0, 0)), (6500, (5.0, 60.0, 61.0), (0, 1, 1))]


@pytest.mark.parametrize("n,edges,pbc", CELLS)
def test_rows_over_cell_grids(dmgx, n, edges, pbc):
    nep = dmgx.NEP(os.path.join(POTENTIALS, "nep_carbon.txt"))
    h, pos = np.diag(edges), _elongated(n, edges, n)
    for _ in range(2):  # the second rebuild starts from the counts the first one left
        gpu_compute(dmgx, nep, dmgx.Box(h, pbc), np.zeros(n, np.int32), pos, force_rebuild=True)
        rows = nep.verlet_rows(0, n)
    ref = neighbor_rows(h, pbc, pos, nep.info.rc_radial_max + 1.0, max_nb=1024)
    for i in range(n):
        assert np.array_equal(rows[i], np.sort(np.asarray(ref[i]))), i


@pytest.mark.parametrize("n", [8192, 8193])
def test_reverse_entries_around_the_wide_search(dmgx, n):
    """Forces (which read every edge's reverse entry) against the oracle on both sides of the size up to which a
    wavefront searches a centre's reverse entries, at the parity tests' bars."""
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(m ** 3)[:n]]
    pos = np.ascontiguousarray((5.0 + 2.3 * g + rng.uniform(-0.15, 0.15, (n, 3))).T)
    edge = 10.0 + 2.3 * m
    path = os.path.join(POTENTIALS, "nep_carbon.txt")
    h, pbc, types = np.diag([edge] * 3), (0, 0, 0), np.zeros(n, np.int32)
    ref = OracleNEP(path, round_params_to_float=True).compute(h, pbc, types, pos)
    e = errors(gpu_compute(dmgx, dmgx.NEP(path), dmgx.Box(h, pbc), types, pos), ref)
    assert e["force"] <= 1e-4 and e["energy_atom_max"] <= 2e-5 and e["virial"] <= 2e-4, e
