"""Models beyond the padded descriptor sizes (more radial functions, wider bases or higher 3-body orders): the generic
descriptor instances on every number of lanes per atom and on the candidate rows, against the FP64 oracle at the bars
of the parity tests; and the lanes that untuned handles of each kind of instance take."""
import numpy as np
import pytest

from gpu_helpers import errors, gpu_compute
from oracle import OracleNEP

pytestmark = pytest.mark.gpu


def write_model(path, symbols, n_max, basis, l_max, sample, cutoff=(4.2, 3.7), neurons=30, seed=7):
    """A random NEP4 model with the descriptor scaler of `sample` (box, types, pos)."""
    rng = np.random.default_rng(seed)
    T, (L, q222, q1111) = len(symbols), l_max
    dim = n_max[0] + 1 + (n_max[1] + 1) * (L + bool(q222) + bool(q1111))
    weights = rng.normal(0.0, 0.1, (dim + 2) * neurons * T + 1)
    coeffs = rng.normal(0.0, 0.1, T * T * ((n_max[0] + 1) * (basis[0] + 1) + (n_max[1] + 1) * (basis[1] + 1)))
    head = [f"nep4 {T} {' '.join(symbols)}", f"cutoff {cutoff[0]} {cutoff[1]} 128 96", f"n_max {n_max[0]} {n_max[1]}",
            f"basis_size {basis[0]} {basis[1]}", "l_max " + " ".join(map(str, l_max)), f"ANN {neurons} 0"]

    def save(scaler):
        values = np.concatenate([weights, coeffs, scaler])
        path.write_text("\n".join(head + [f"{np.float32(v):.9e}" for v in values]) + "\n")

    save(np.ones(dim))
    box, types, pos = sample
    q = OracleNEP(str(path)).compute(box.h, box.pbc, types, pos, want_descriptor=True)["q"]
    span = q.max(0) - q.min(0)
    save(np.where(span > 0, 1.0 / np.where(span > 0, span, 1.0), 1.0))
    return str(path)


def lattice(dmgx, workloads, cells, num_types, seed=5):
    s = workloads.vacancy_lattice("carbon", cells, np.random.default_rng(seed), vacancies=False)
    n = len(s["types"])
    return s["box"], (np.arange(n) % num_types).astype(np.int32), np.ascontiguousarray(s["pos"])


@pytest.mark.parametrize("num_types", [1, 2])
@pytest.mark.parametrize("n_max,basis,l_max", [((4, 4), (16, 12), (4, 2, 1)), ((15, 9), (8, 16), (4, 0, 0)),
                                               ((4, 3), (6, 6), (5, 2, 0)), ((2, 1), (3, 2), (8, 0, 1))])
def test_generic_instances_against_oracle(dmgx, workloads, tmp_path, num_types, n_max, basis, l_max):
    box, types, pos = lattice(dmgx, workloads, 4, num_types)
    path = write_model(tmp_path / "nep.txt", ["C", "H"][:num_types], n_max, basis, l_max, (box, types, pos))
    ref = OracleNEP(path, round_params_to_float=True).compute(box.h, box.pbc, types, pos)
    nep = dmgx.NEP(path)
    for split in (False, True):
        nep.set_split(split)
        for lanes in (0, 1, 4):
            nep.set_desc_lanes(lanes)
            e = errors(gpu_compute(dmgx, nep, box, types, pos), ref)
            assert e["force"] <= max(1e-4, 2e-6 * np.abs(ref["force"]).max()), (split, lanes, e)
            assert e["energy_atom_max"] <= max(2e-5, 2e-7 * np.abs(ref["pe"]).max()), (split, lanes, e)
            assert e["virial"] <= max(2e-4, 2e-6 * np.abs(ref["virial"]).max()), (split, lanes, e)


def _cluster(n, seed=11, spacing=2.3):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n].astype(float)
    return np.ascontiguousarray((5.0 + g * spacing + rng.uniform(-0.15, 0.15, (n, 3))).T), 10.0 + m * spacing


@pytest.mark.parametrize("n_max,basis,l_max,n,desc,gather", [
    ((4, 4), (16, 12), (4, 2, 1), 8192, None, 16),  # None: sixteen lanes, which cannot be set
    ((4, 4), (16, 12), (4, 2, 1), 8193, 4, 16), ((4, 4), (16, 12), (4, 2, 1), 36865, 4, 8),
    ((4, 4), (16, 12), (4, 2, 1), 49151, 4, 8), ((4, 4), (16, 12), (4, 2, 1), 49152, 1, 8),
    ((4, 4), (8, 8), (6, 2, 1), 5121, 4, 16), ((4, 4), (8, 8), (6, 2, 1), 36863, 4, 8),
    ((4, 4), (8, 8), (6, 2, 1), 36865, 1, 4),
    ((4, 4), (11, 8), (4, 2, 1), 36865, 4, 4), ((4, 4), (12, 8), (4, 2, 1), 36865, 4, 8),
    ((4, 4), (12, 8), (4, 2, 1), 6144, None, 16), ((4, 4), (12, 8), (4, 2, 1), 6145, 4, 16),
    ((4, 4), (12, 8), (4, 2, 1), 57343, 4, 8), ((4, 4), (12, 8), (4, 2, 1), 57344, 1, 8),
    ((4, 4), (8, 8), (4, 2, 1), 8192, None, 16), ((4, 4), (8, 8), (4, 2, 1), 8193, 4, 16),
    ((4, 4), (8, 8), (4, 2, 1), 36863, 4, 8), ((4, 4), (8, 8), (4, 2, 1), 36865, 1, 4)])
def test_untuned_lanes_by_the_instance(dmgx, workloads, tmp_path, n_max, basis, l_max, n, desc, gather):
    """The lanes of an untuned handle follow the kind of descriptor instance and the width of the gather's adjoint rows:
    bit for bit the results of the lanes set by hand."""
    path = write_model(tmp_path / "nep.txt", ["C"], n_max, basis, l_max, lattice(dmgx, workloads, 4, 1))
    pos, edge = _cluster(n)
    types = np.zeros(n, np.int32)
    box = dmgx.Box.orthogonal(edge, edge, edge, pbc=(0, 0, 0))
    untuned, by_hand = dmgx.NEP(path), dmgx.NEP(path)
    a = gpu_compute(dmgx, untuned, box, types, pos)
    by_hand.set_tiles(16, gather)
    if desc:
        by_hand.set_desc_lanes(desc)
    b = gpu_compute(dmgx, by_hand, box, types, pos)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    if desc is None:  # neither of the others
        for lanes in (1, 4):
            by_hand.set_desc_lanes(lanes)
            assert not np.array_equal(a[0], gpu_compute(dmgx, by_hand, box, types, pos)[0])
