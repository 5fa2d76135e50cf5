"""Edge rows interleaved by tiles of 64 centres, and the descriptor's lane
groups that read them: centre ranges that start and end inside a tile, systems
of a tile's size and one atom to either side, and the sizes where the lanes per
atom change, against the FP64 oracle (the bars of the parity tests)."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import errors, gpu_compute
from oracle import OracleNEP

pytestmark = pytest.mark.gpu

TOL_F, TOL_EA, TOL_V = 1e-4, 2e-5, 2e-4


def _cluster(n, seed, spacing=2.3, side=60.0):
    """n carbon atoms on a jittered grid in the middle of an open box."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n].astype(float)
    return 5.0 + g * spacing + rng.uniform(-0.15, 0.15, (n, 3)), max(side, 10.0 + m * spacing)


def _check(out, ref, n=None):
    e = errors(out, ref, n)
    assert e["force"] <= TOL_F and e["energy_atom_max"] <= TOL_EA and e["virial"] <= TOL_V, e


@pytest.mark.parametrize("model", ["nep_carbon.txt", "nep_carbon_zbl.txt", "nep4_typecut_ch.txt"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 193])
def test_systems_around_a_tile(dmgx, model, n):
    path = os.path.join(POTENTIALS, model)
    nep = dmgx.NEP(path)
    pos, edge = _cluster(n, n)
    types = (np.arange(n) % nep.num_types).astype(np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    ref = OracleNEP(path, round_params_to_float=True).compute(box.h, box.pbc, types, np.ascontiguousarray(pos.T))
    for lanes in (0, 1, 4):
        nep.set_desc_lanes(lanes)
        _check(gpu_compute(dmgx, nep, box, types, pos.T), ref)


@pytest.mark.parametrize("nd1,n1,n2,nd2", [(0, 0, 300, 300), (1, 5, 250, 299), (63, 64, 128, 300), (65, 70, 71, 200),
                                           (37, 37, 101, 164)])
def test_centre_ranges_inside_tiles(dmgx, nd1, n1, n2, nd2):
    """Ranges [nd1, nd2) and [n1, n2) against the oracle's ranges, and slots outside [n1, n2) left as they were."""
    path = os.path.join(POTENTIALS, "nep_carbon.txt")
    n = 300
    pos, edge = _cluster(n, 7)
    types = np.zeros(n, np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    nep = dmgx.NEP(path)
    orc = OracleNEP(path, round_params_to_float=True)
    ref = orc.compute(box.h, box.pbc, types, np.ascontiguousarray(pos.T), n1=n1, n2=n2, nd1=nd1, nd2=nd2)
    for lanes in (0, 1, 4):
        nep.set_desc_lanes(lanes)
        pe, f, v = gpu_compute(dmgx, nep, box, types, pos.T, n1=n1, n2=n2, nd1=nd1, nd2=nd2)
        assert np.abs(f[:, n1:n2] - ref["force"][:, n1:n2]).max() <= TOL_F
        assert np.abs(v[:, n1:n2] - ref["virial"][:, n1:n2]).max() <= TOL_V
        assert np.abs(pe[nd1:nd2] - ref["pe"][nd1:nd2]).max() <= TOL_EA
        out = np.ones(n, bool)
        out[n1:n2] = False
        assert not f[:, out].any() and not v[:, out].any()


@pytest.mark.parametrize("material,cells", [("carbon", 10), ("carbon", 11), ("cu", 12), ("cu", 13)])
def test_lane_rule_sizes(dmgx, workloads, material, cells):
    """Systems to either side of the sizes where the untuned lanes per atom change (8,000 and 10,648 carbon
    atoms, 6,912 and 8,788 Cu atoms): FP32 rounding apart, the result of one lane per atom."""
    s = workloads.vacancy_lattice(material, cells, np.random.default_rng(3), vacancies=False)
    path = os.path.join(POTENTIALS, f"nep_{material}.txt")
    nep = dmgx.NEP(path)
    auto = gpu_compute(dmgx, nep, s["box"], s["types"], s["pos"])
    nep.set_desc_lanes(1)
    one = gpu_compute(dmgx, nep, s["box"], s["types"], s["pos"])
    for a, b, tol in zip(auto, one, (TOL_EA, TOL_F, TOL_V)):
        assert np.abs(a - b).max() <= tol


@pytest.mark.parametrize("n", [6144, 6145, 12288, 12289, 36864, 36865])
def test_untuned_lanes_give_the_set_lanes_results(dmgx, n):
    """The filter's and gather's lanes by size, on both sides of each limit: the edges of the rows exactly those of
    16 and 8 lanes, and the forces to the rounding of their FP64 sums (1e-12 of the largest term of about 10)."""
    pos, edge = _cluster(n, n)
    types = np.zeros(n, np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    path = os.path.join(POTENTIALS, "nep_carbon.txt")
    by_size, as_set = dmgx.NEP(path), dmgx.NEP(path)
    as_set.set_tiles(16, 8)
    a = gpu_compute(dmgx, by_size, box, types, pos.T)
    b = gpu_compute(dmgx, as_set, box, types, pos.T)
    assert np.array_equal(a[0], b[0])
    assert np.abs(a[1] - b[1]).max() <= 1e-11 and np.abs(a[2] - b[2]).max() <= 1e-11
