"""The descriptor with sixteen lanes per atom, which the smallest systems take unless lanes were set: every kind of
instance against the FP64 oracle and against one lane per atom (the same products, another FP32 summation order)."""
import os

import numpy as np
import pytest

from conftest import BASELINE, POTENTIALS
from gpu_helpers import errors, gpu_compute
from oracle import OracleNEP

pytestmark = pytest.mark.gpu

INPUTS = os.path.join(BASELINE, "inputs", "potentials")
MODELS = [os.path.join(POTENTIALS, f) for f in (
    "nep_carbon.txt", "nep_cu.txt", "nep_carbon_zbl.txt", "nep_water.txt", "nep5_ch.txt", "nep4_typecut_ch.txt",
    "nep5_zbl_typewise_ch.txt", "nep4_zbl_flexible_ch.txt", "nep4_lmax2_ch.txt", "nep4_lmax3_ch.txt", "nep4_big_ch.txt",
    "nep4_lmax6_ch.txt")] + [os.path.join(INPUTS, f) for f in ("nep_C.txt", "nep_water.txt", "nep_BaTiO3_zbl.txt")]


def _system(n, seed=17, spacing=2.4):
    """n atoms on jittered sites in the middle of an open box, from atoms with many neighbours to a lone one."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil((n - 1) ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n - 1].astype(float)
    pos = np.concatenate([8.0 + g * spacing + rng.uniform(-0.2, 0.2, (n - 1, 3)), [[1.0, 1.0, 1.0]]])
    return np.ascontiguousarray(pos.T), 16.0 + m * spacing


@pytest.mark.parametrize("n", [17, 600])
@pytest.mark.parametrize("path", MODELS, ids=lambda p: os.path.relpath(p, os.path.dirname(POTENTIALS)).replace("/", "_"))
def test_sixteen_lanes_against_oracle_and_one(dmgx, path, n):
    pos, edge = _system(n)
    by_size, one = dmgx.NEP(path), dmgx.NEP(path)
    one.set_desc_lanes(1)
    types = (np.arange(n) % by_size.num_types).astype(np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    ref = OracleNEP(path, round_params_to_float=True).compute(box.h, box.pbc, types, pos)
    a, b = (gpu_compute(dmgx, h, box, types, pos) for h in (by_size, one))
    fmax, emax, vmax = (np.abs(ref[k]).max() for k in ("force", "pe", "virial"))
    e = errors(a, ref)
    # the bars of the parity tests: absolute, or the FP32 floor of large values (1e-5 of a site energy, as the
    # reference's manifest has it)
    assert e["force"] <= max(1e-4, 2e-6 * fmax), (e, fmax)
    assert e["energy_atom_max"] <= max(2e-5, 1e-5 * emax), (e, emax)
    assert e["virial"] <= max(2e-4, 2e-6 * vmax), (e, vmax)
    # between the two orders twice as much at most
    for x, y, tol in zip(a, b, (max(4e-5, 2e-5 * emax), max(2e-4, 4e-6 * fmax), max(4e-4, 4e-6 * vmax))):
        assert np.abs(x - y).max() <= tol
    if n == 600:
        assert not np.array_equal(a[0], b[0])  # sixteen lanes ran, not one
