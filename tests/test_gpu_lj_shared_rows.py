"""lj1g and lj terms of the same rows in one pass: species and orders in which
an lj1g finds no lj list of its rows, one, or two, against the oracle (FP64
forces and energies within 1e-10), with the shared launches and with separate
ones, at every lane count of the shared launches.  (The mixed path's shared
launches are held to the separate ones in test_gpu_fusion.py.)"""
import numpy as np
import pytest

from pfmds_amd import configs
from pfmds_amd.system import Interaction
from tests.harness import gpu_ctx, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu

R = (6.5, 7.5)
ROW = lambda a, b: (a, b, 160, 8.5, 20)  # noqa: E731


def lj1g(g, eps=0.0104, sig=3.4):
    return Interaction("lj1g", [eps, sig, *R], [ROW(g, g)])


def lj(a, b, eps=0.012, sig=3.5):
    return Interaction("lj", [eps, sig, *R], [ROW(a, b), ROW(b, a)])


# groups: 1 A, 2 B, 3 C, 4 all, 5 A+B, 6 empty
CASES = {
    "gas": [lj1g(1), lj1g(2), lj(1, 2)],
    "lj first": [lj(1, 2), lj1g(2, 0.014, 3.65), lj1g(1)],
    "one side": [lj1g(1), lj(1, 2), lj(2, 3)],
    "two of one row group": [lj1g(1), lj(1, 2), lj(1, 3, 0.009, 3.3), lj1g(3)],
    "no partner": [lj1g(5), lj(3, 5, 0.01, 3.45)],
    "alone": [lj1g(5), lj1g(3, 0.02, 3.2)],
}


def gas(name, n=700):
    s = configs.lj_gas_lattice(n, 0.02, 17, 120.0)
    rng = np.random.default_rng(4)
    s.species = [("A", "B", "C")[k] for k in rng.integers(0, 3, n)]
    s.groups = [["A"], ["B"], ["C"], ["A", "B", "C"], ["A", "B"], ["#"]]
    s.all_moving = s.xyz_moving = s.all_atoms = s.traj = 4
    s.z_moving = 6
    s.interactions = CASES[name]
    return s


@pytest.mark.parametrize("name", list(CASES))
def test_shared_rows(name):
    s = gas(name)
    o = oracle_ctx(s)
    o.run("nve", 0.5, 0, 0, True)
    o.run("nve", 0.5, 1, 15, True)
    po, _, fo = o.state()
    eo = o.energies()["e_inter"]
    for lanes in (4, 8, 16):
        for fuse in (True, False):
            c = gpu_ctx(s)
            c.set_tuning(lanes, 256)
            c.set_fusion(fuse)
            c.run("nve", 0.5, 0, 0, True)
            c.run("nve", 0.5, 1, 15, True)
            p, _, f = c.state()
            assert rel_inf(f, fo) < 1e-10, (name, lanes, fuse)
            assert rel_inf(p, po) < 1e-10
            np.testing.assert_allclose(c.energies()["e_inter"], eo, rtol=1e-10)
            c.close()
