"""Periodic boxes whose thickness divides 2.5 (rc + skin), the thickness that their supercell has to exceed: whichever
way their computed thickness is rounded, they are evaluated, as the FP64 oracle does."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import errors, gpu_compute
from oracle import OracleNEP

pytestmark = pytest.mark.gpu

CARBON = os.path.join(POTENTIALS, "nep_carbon.txt")
NEED = 2.5 * (4.2 + 1.0)


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("a,c", [(10.93, 6.1), (6.55, 9.74), (6.49, 8.33), (6.06, 7.91), (10.88, 5.36)])
def test_boxes_that_divide_the_supercell(dmgx, a, c, parts):
    rng = np.random.default_rng(parts)
    edges = np.array([a, NEED / parts, c])
    m = np.maximum(1, (edges / 2.4).astype(int))
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, 3)
    pos = np.ascontiguousarray(((g + 0.5 + rng.uniform(-0.05, 0.05, g.shape)) / m * edges).T)
    types = np.zeros(len(g), np.int32)
    box = dmgx.Box.orthogonal(*edges)
    ref = OracleNEP(CARBON, round_params_to_float=True).compute(box.h, box.pbc, types, pos)
    e = errors(gpu_compute(dmgx, dmgx.NEP(CARBON), box, types, pos), ref)
    assert e["force"] <= 1e-4 and e["energy_atom_max"] <= 2e-5 and e["virial"] <= 2e-4, e
