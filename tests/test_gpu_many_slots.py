"""More than 2^27 slots: an edge record's word has no room for the neighbour's type above such a slot, so its readers
look the type up.  300 centres with neighbours on both sides of slot 2^27, and the slots between far away, give bit for
bit what the same atoms give in a few slots."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS
from gpu_helpers import gpu_compute

pytestmark = pytest.mark.gpu

MODEL = os.path.join(POTENTIALS, "nep4_typecut_ch.txt")


def test_untyped_edge_words(dmgx):
    import torch
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 64 GiB of free device memory")
    n, ghosts = 300, 200
    N = (1 << 27) + ghosts // 2
    edge = 420.0
    rng = np.random.default_rng(9)
    g = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n + ghosts].astype(float)
    g = rng.permutation(g)
    pos = np.ascontiguousarray((5.0 + 2.0 * g + rng.uniform(-0.2, 0.2, g.shape)).T)
    types = rng.integers(0, 2, n + ghosts).astype(np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    slots = np.concatenate([np.arange(n), np.arange(N - ghosts, N)])  # of the same atoms among the N
    assert (slots[n:] < 1 << 27).any() and (slots >= 1 << 27).any()
    few, many = dmgx.NEP(MODEL), dmgx.NEP(MODEL)
    x = torch.empty(3 * N, dtype=torch.float64, device="cuda")
    x[:N].uniform_(60.0, edge - 5.0)
    x[N:].uniform_(5.0, edge - 5.0)
    t = torch.ones(N, dtype=torch.int32, device="cuda")
    at = torch.tensor(slots, device="cuda")
    for d in range(3):
        x[d * N + at] = torch.tensor(pos[d], device="cuda")
    t[at] = torch.tensor(types, device="cuda")
    pe, f, v = (torch.zeros(k * N, dtype=torch.float64, device="cuda") for k in (1, 3, 9))
    for split in (False, True):
        few.set_split(split)
        many.set_split(split)
        ref = gpu_compute(dmgx, few, box, types, pos, n1=0, n2=n, nd1=0, nd2=n)
        many.compute_domain(box, N, t, x, pe, f, v, n1=0, n2=n, nd1=0, nd2=n)
        torch.cuda.synchronize()
        for got, want, k in zip((pe, f, v), ref, (1, 3, 9)):
            assert np.array_equal(got.view(k, N)[:, :n].cpu().numpy(), want.reshape(k, -1)[:, :n]), split
        for rows in ("radial_rows", "angular_rows"):
            a, b = getattr(few, rows)(0, n), getattr(many, rows)(0, n)
            assert all(np.array_equal(slots[p], q) for p, q in zip(a, b)), (split, rows)
    del x, t, pe, f, v, many
    torch.cuda.empty_cache()
