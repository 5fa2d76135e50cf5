"""Two atoms at the same place (a duplicate at both faces of a box, say) have no direction between them: their site
energies, and the forces and virials of every atom that sees them, are not numbers, and the others' are.  Against the
FP64 oracle's pattern on every form of the network: matrix cores with the operands in registers and through LDS,
bfloat16 operands, the vector ALUs, groups of lanes, and the candidate rows."""
import os

import numpy as np
import pytest

from conftest import BASELINE, POTENTIALS
from gpu_helpers import gpu_compute
from oracle import OracleNEP

pytestmark = pytest.mark.gpu

INPUTS = os.path.join(BASELINE, "inputs", "potentials")


@pytest.mark.parametrize("path", [os.path.join(POTENTIALS, f) for f in (
    "nep_carbon.txt", "nep_cu.txt", "nep_carbon_zbl.txt", "nep_water.txt", "nep4_typecut_ch.txt", "nep4_big_ch.txt",
    "nep4_lmax6_ch.txt")] + [os.path.join(INPUTS, "nep_C.txt"), os.path.join(INPUTS, "nep_BaTiO3_zbl.txt")],
    ids=os.path.basename)
def test_energies_are_not_numbers(dmgx, path):
    rng = np.random.default_rng(5)
    n = 125
    g = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(float)
    pos = 5.0 + g * 2.9 + rng.uniform(-0.15, 0.15, (n, 3))
    pos[70] = pos[3]
    pos = np.ascontiguousarray(pos.T)
    nep = dmgx.NEP(path)
    types = (np.arange(n) % nep.num_types).astype(np.int32)
    box = dmgx.Box.orthogonal(40.0, 40.0, 40.0, pbc=(0, 0, 0))
    ref = OracleNEP(path, round_params_to_float=True).compute(box.h, box.pbc, types, pos)
    assert list(np.flatnonzero(~np.isfinite(ref["pe"]))) == [3, 70]
    assert 2 < (~np.isfinite(ref["force"])).any(0).sum() < n  # neighbours see them, others do not
    for split in (False, True):
        nep.set_split(split)
        for lanes in (0, 1, 4):  # 0: sixteen lanes per atom at this size
            nep.set_desc_lanes(lanes)
            for mode in ({}, {"ann_valu": True}, {"ann_bf16": True}, {"ann_bf16_split": True}):
                out = gpu_compute(dmgx, nep, box, types, pos, **mode)
                for a, b in zip(out, (ref["pe"], ref["force"], ref["virial"])):
                    assert np.array_equal(np.isfinite(a), np.isfinite(b)), (split, lanes, mode)
