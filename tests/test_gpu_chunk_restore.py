"""A chunk of MD steps that outgrows its Verlet rows goes back to its checkpoint and runs again with longer rows: the
state afterwards is, bit for bit, that of a handle whose rows were long enough from the start."""
import os

import numpy as np
import pytest

from conftest import POTENTIALS

pytestmark = pytest.mark.gpu

CARBON = os.path.join(POTENTIALS, "nep_carbon.txt")
FS = 10.18051  # femtoseconds in the engine's time unit


def _model(tmp_path, rows):
    lines = open(CARBON).read().splitlines()
    i = next(k for k, l in enumerate(lines) if l.startswith("cutoff"))
    lines[i] = " ".join(lines[i].split()[:3] + [str(rows), str(rows)])
    path = tmp_path / f"nep_{rows}.txt"
    path.write_text("\n".join(lines) + "\n")
    return str(path)


def _cloud(n, seed=6, spacing=4.0, side=120.0):
    """Sparse atoms that fall towards the middle of the box (velocities per fs): 6 neighbours become about 30 after
    20 fs."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n].astype(float)
    pos = (g - (m - 1) / 2) * spacing + rng.uniform(-0.1, 0.1, (n, 3))
    vel = -0.02 * pos
    return np.ascontiguousarray((pos + side / 2).T), np.ascontiguousarray(vel.T), side


@pytest.mark.parametrize("ensemble", ["nve", "nvt_ber", "nvt_bdp", "npt_ber", "npt_scr"])
@pytest.mark.parametrize("n", [124, 125, 343])
def test_restored_chunk_equals_long_rows(dmgx, tmp_path, ensemble, n):
    pos, vel, side = _cloud(n)
    types, mass = np.zeros(n, np.int32), np.full(n, 12.011)
    kw = {} if ensemble == "nve" else dict(t_init=300.0, t_coupling=50.0)
    if ensemble.startswith("npt"):
        kw.update(p_target_gpa=0.0, bulk_modulus_gpa=100.0, p_coupling=500.0)
    out, rows = {}, {}
    for cap in (4, 100):
        nep = dmgx.NEP(_model(tmp_path, cap))
        md = dmgx.MD(nep, dmgx.Box.orthogonal(side, side, side), types, mass, pos, vel * FS)
        md.run(0, 0.5, "nve")
        rows[cap] = nep.tuning()["row_capacity"]
        th = md.run(40, 0.5, ensemble, **kw)
        out[cap] = (md.arrays(), th, md.box().h, nep.neighbor_stats()["max_verlet"], nep.tuning()["row_capacity"])
    assert out[4][3] > rows[4] and out[4][4] > rows[4]  # the short rows overflowed inside the run
    assert rows[100] == out[100][4]
    for k in out[4][0]:
        assert np.array_equal(out[4][0][k], out[100][0][k]), k
    assert np.array_equal(out[4][1], out[100][1]) and np.array_equal(out[4][2], out[100][2])


def test_restored_chunk_keeps_unwrapped_positions(dmgx, tmp_path):
    """The same through a run directory that writes unwrapped positions, with an odd number of atoms."""
    import importlib
    from xyz_io import read_xyz
    cli = importlib.import_module("dmg-md_amd.cli")
    n = 125
    pos, vel, side = _cloud(n)
    frames = {}
    for cap in (4, 100):
        d = tmp_path / str(cap)
        d.mkdir()
        lines = [f"C {p[0]:.17g} {p[1]:.17g} {p[2]:.17g} {v[0]:.17g} {v[1]:.17g} {v[2]:.17g}" for p, v in zip(pos.T, vel.T)]
        (d / "model.xyz").write_text(f'{n}\nLattice="{side} 0 0 0 {side} 0 0 0 {side}" '
                                     "Properties=species:S:1:pos:R:3:vel:R:3\n" + "\n".join(lines) + "\n")
        (d / "nep.txt").write_text(open(_model(tmp_path, cap)).read())
        (d / "run.in").write_text("potential nep.txt\ntime_step 0.5\nensemble nve\n"
                                  "dump_xyz 20 g.xyz precision double unwrapped_position velocity\nrun 40\n")
        cli.run_directory(str(d), "run.in", "model.xyz")
        frames[cap] = [read_xyz(str(d / "g.xyz"), frame=k) for k in range(2)]
    for a, b in zip(frames[4], frames[100]):
        for k in ("pos", "vel", "unwrapped_position"):
            assert np.array_equal(a[k], b[k]), k
