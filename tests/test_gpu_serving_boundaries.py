"""The periodic images that a served request brings along: every mix of periodic and open directions, straight and
sheared boxes, thin ones with several images a side, atoms exactly on a face, wrapped in from outside, and beyond the
box in an open direction.  Single points against the FP64 oracle, which takes any positions."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import errors
from oracle import OracleNEP

pytestmark = pytest.mark.gpu

CARBON = os.path.join(POTENTIALS, "nep_carbon.txt")
TOL_F, TOL_EA, TOL_V = 1e-4, 2e-5, 2e-4


def _frac(cells, seed):
    """Jittered cubic sites in fractions of a box of `cells`, some exactly on its faces."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(c) for c in cells], indexing="ij"), -1).reshape(-1, 3).astype(float)
    s = (g + 0.5 + rng.uniform(-0.06, 0.06, g.shape)) / np.array(cells)
    for d in range(3):
        k = np.flatnonzero(g[:, d] == 0)[:: 3]
        s[k, d] = 0.0
    return s


@pytest.mark.parametrize("shear", [False, True], ids=["straight", "sheared"])
@pytest.mark.parametrize("pbc", [(1, 1, 1), (1, 1, 0), (0, 1, 0), (1, 0, 1), (0, 0, 0)])
@pytest.mark.parametrize("cells", [(1, 2, 5), (3, 4, 4), (1, 1, 1)])
def test_images_of_a_request(dmgx, shear, pbc, cells):
    a = 2.2
    h = np.diag(a * np.array(cells, float))
    if shear:
        h = h @ np.array([[1, 0.3, -0.2], [0, 1, 0.15], [0.1, 0, 1]])
    s = _frac(cells, sum(cells))
    n = len(s)
    rng = np.random.default_rng(3)
    shifts = np.zeros((n, 3))
    for d in range(3):
        if pbc[d]:  # face atoms at either end, and atoms a box or two away
            on_face = np.flatnonzero(s[:, d] == 0.0)
            shifts[on_face[::2], d] = 1.0
            shifts[rng.integers(0, n, max(n // 8, 1)), d] = rng.integers(-2, 3)
    pos = np.ascontiguousarray(h @ (s + shifts).T)
    srv = dmgx.Server(dmgx.NEP(CARBON), max_atoms=200_000)
    types = np.zeros(n, np.int32)
    out = srv.poll(srv.submit(dmgx.Box(h, pbc), types, np.full(n, 12.0), pos), wait=True)
    ref = OracleNEP(CARBON, round_params_to_float=True).compute(h, pbc, types, np.ascontiguousarray(h @ s.T))
    e = errors((out["potential"], out["force"], out["virial"]), ref)
    assert e["force"] <= max(TOL_F, 2e-6 * np.abs(ref["force"]).max()), e
    assert e["energy_atom_max"] <= TOL_EA and e["virial"] <= max(TOL_V, 2e-6 * np.abs(ref["virial"]).max()), e


@pytest.mark.parametrize("steps", [0, 1])
def test_atoms_beyond_an_open_face(dmgx, steps):
    """A slab periodic in x and y whose atoms lie 9 to 16 A outside the box in the open direction."""
    h = np.diag([6.6, 8.8, 4.0])
    s = _frac((3, 4, 3), 8)
    pos = np.ascontiguousarray((np.diag([6.6, 8.8, 6.6]) @ s.T) - np.array([[0.0], [0.0], [16.0]]))
    n = len(s)
    types = np.zeros(n, np.int32)
    srv = dmgx.Server(dmgx.NEP(CARBON), max_atoms=200_000)
    box = dmgx.Box(h, (1, 1, 0))
    v = np.zeros((3, n)) if steps else None
    out = srv.poll(srv.submit(box, types, np.full(n, 12.0), pos, v, steps=steps, dt_fs=1e-9), wait=True)
    ref = OracleNEP(CARBON, round_params_to_float=True).compute(h, (1, 1, 0), types, pos)
    e = errors((out["potential"], out["force"], out["virial"]), ref)
    assert e["force"] <= TOL_F and e["energy_atom_max"] <= TOL_EA and e["virial"] <= TOL_V, e
