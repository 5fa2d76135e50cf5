"""What the autotuner and the lane setters leave in a handle, seen through results: the FP32 sums of the descriptor
and the FP64 sums of the gather differ in their last bits with the lanes that form them."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import gpu_compute, to_dev

pytestmark = pytest.mark.gpu

CARBON = os.path.join(POTENTIALS, "nep_carbon.txt")


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def _autotune(nep, s, types, **kw):
    import torch
    n = len(types)
    t, x = to_dev(types, torch.int32), to_dev(s["pos"], torch.float64)
    out = [torch.zeros(k * n, dtype=torch.float64, device="cuda") for k in (1, 3, 9)]
    return nep.autotune(s["box"], t, x, *out, **kw)


def test_refused_autotune_leaves_the_lanes_by_size(dmgx, workloads):
    s = workloads.carbon_diamond_4096(seed=4)
    nep = dmgx.NEP(CARBON)
    with pytest.raises(dmgx.DmgxError):
        _autotune(nep, s, np.full(len(s["types"]), nep.num_types, np.int32))
    fresh, by_hand = dmgx.NEP(CARBON), dmgx.NEP(CARBON)
    by_hand.set_tiles(16, 8)
    a, b, c = (gpu_compute(dmgx, h, s["box"], s["types"], s["pos"]) for h in (nep, fresh, by_hand))
    assert not _same(b, c)
    assert _same(a, b)


def test_bfloat16_autotune_keeps_the_descriptor_lanes_set(dmgx, workloads):
    """Autotuning BF16 requests does not time the descriptor's lanes, so exactly four stay exactly four."""
    s = workloads.carbon_diamond_4096(seed=4)
    nep, four, by_size = dmgx.NEP(CARBON), dmgx.NEP(CARBON), dmgx.NEP(CARBON)
    nep.set_desc_lanes(4)
    tune = _autotune(nep, s, s["types"], ann_bf16=True)
    assert tune["desc_lanes"] == 4
    four.set_desc_lanes(4)
    if tune["split"]:
        pytest.skip("candidate rows keep one lane per atom")
    a, b, c = (gpu_compute(dmgx, h, s["box"], s["types"], s["pos"])[0] for h in (nep, four, by_size))
    assert not np.array_equal(b, c)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("cells,lanes", [(4, (32, 16)), (10, (16, 16)), (12, (16, 8)), (17, (16, 4))])
def test_reported_lanes_are_those_launched(dmgx, workloads, cells, lanes):
    """An untuned handle reports the lanes that its last evaluation launched, so that pinning what it reports changes
    nothing."""
    s = workloads.vacancy_lattice("carbon", cells, np.random.default_rng(3), vacancies=False)
    nep, pinned = dmgx.NEP(CARBON), dmgx.NEP(CARBON)
    t = nep.tuning()
    assert (t["filter_lanes"], t["gather_lanes"]) == (16, 8)
    a = gpu_compute(dmgx, nep, s["box"], s["types"], s["pos"])
    t = nep.tuning()
    assert (t["filter_lanes"], t["gather_lanes"], t["tuned"]) == (*lanes, False)
    pinned.set_tiles(t["filter_lanes"], t["gather_lanes"])
    assert _same(a, gpu_compute(dmgx, pinned, s["box"], s["types"], s["pos"]))
    nep.set_tiles(8, 4)
    gpu_compute(dmgx, nep, s["box"], s["types"], s["pos"])
    t = nep.tuning()
    assert (t["filter_lanes"], t["gather_lanes"]) == (8, 4)


def test_tuned_descriptor_group_is_not_taken_for_larger_systems(dmgx, workloads):
    """Four lanes per atom tuned on 39,304 atoms stay for them; 110,592 atoms take one lane, as the rule by size has
    it."""
    small, large = (workloads.vacancy_lattice("carbon", c, np.random.default_rng(3), vacancies=False) for c in (17, 24))
    nep = dmgx.NEP(CARBON)
    tune = _autotune(nep, small, small["types"])
    if tune["desc_lanes"] != 4 or tune["split"]:
        pytest.skip("the autotuner chose no group here")
    pinned = dmgx.NEP(CARBON)
    for s, lanes in ((small, 4), (large, 1)):
        pinned.set_desc_lanes(lanes)
        a, b = (gpu_compute(dmgx, h, s["box"], s["types"], s["pos"])[0] for h in (nep, pinned))
        assert np.array_equal(a, b), lanes
