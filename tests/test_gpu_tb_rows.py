"""Tersoff-Brenner rows of more than one chunk of four bonds, and of one to
four: carbon clusters with up to nine neighbours inside the cutoff, in the
switching zone too, against the oracle (forces within 1e-11 of the largest in
FP64, 1e-4 eV/A RMS in the mixed path at these strained geometries' scale).
"""
import numpy as np
import pytest

from pfmds_amd import capi, configs
from pfmds_amd.system import Integrator, Interaction, System
from tests.harness import gpu_ctx, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu


def clusters(a, jitter, m, seed=3):
    """Blocks of m^3 carbon atoms on a cubic lattice of spacing a, 8 A apart."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * a
    o = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3) * (8.0 + a * m)
    pos = (o[:, None, :] + g[None]).reshape(-1, 3) + 2.0 + jitter * (2 * rng.random((len(o) * len(g), 3)) - 1)
    n = len(pos)
    box = np.full(3, 3 * (8.0 + a * m))
    return System(box=box, pos=np.mod(pos, box), vel=np.zeros((n, 3)), mass=np.full(n, 12.011), species=["C"] * n,
                  groups=[["C"], ["#"]],
                  interactions=[Interaction("tb", list(configs.TB_BRENNER_I), [(1, 1, 16, 2.3, 10)])],
                  integrators=[Integrator("nve", 0.5, 10, 10**9, 10**9)], z_moving=2)


@pytest.mark.parametrize("a,m", [(1.75, 2), (1.8, 1), (1.6, 2), (1.35, 2), (1.7, 3)])
def test_rows_against_oracle(a, m):
    s = clusters(a, 0.06, m)
    g, o, x = gpu_ctx(s), oracle_ctx(s), gpu_ctx(s, capi.MIXED)
    for c in (g, o, x):
        c.run("nve", 0.5, 0, 0, True)
    nnum = g.get_list(1, 1, stride=16)[0]
    print(f"[tb rows] a={a} m={m} neighbours {nnum.min()}..{nnum.max()}", flush=True)
    fo = o.state()[2]
    if m == 1:
        assert not g.state()[2].any()
        return
    assert rel_inf(g.state()[2], fo) < 1e-11
    np.testing.assert_allclose(g.energies()["e_inter"], o.energies()["e_inter"], rtol=1e-11)
    assert rel_inf(x.state()[2], fo) < 1e-4


@pytest.mark.parametrize("r1,r2", [(2.0, 2.0), (1.7, 1.7), (2.1, 2.0)])
def test_cutoff_without_a_switching_zone(r1, r2):
    """R1 = R2 (and R1 beyond R2, which the reference's branches also take):
    the cutoff is 1 with derivative 0 below R1, against the oracle within the
    same 1e-11."""
    s = clusters(1.45, 0.06, 2)
    s.interactions[0].params[8:10] = [r1, r2]
    g, o = gpu_ctx(s), oracle_ctx(s)
    for c in (g, o):
        c.run("nve", 0.5, 0, 0, True)
    assert np.abs(o.state()[2]).max() > 1.0
    assert rel_inf(g.state()[2], o.state()[2]) < 1e-11
    np.testing.assert_allclose(g.energies()["e_inter"], o.energies()["e_inter"], rtol=1e-11)


def test_coincident_carbons_stop_the_run():
    """Two atoms on one point with no other neighbour: as in the oracle the
    forces are not numbers, the energy is one, and the next step's position
    check stops the run."""
    s = clusters(1.8, 0.0, 1)
    s.pos[1] = s.pos[0]
    g, o = gpu_ctx(s), oracle_ctx(s)
    for c in (g, o):
        c.run("nve", 0.5, 0, 0, True)
    np.testing.assert_array_equal(np.isnan(g.state()[2]), np.isnan(o.state()[2]))
    assert np.isnan(g.state()[2][:2]).any()
    np.testing.assert_allclose(g.energies()["e_inter"], o.energies()["e_inter"], rtol=1e-11)
    with pytest.raises(capi.PfmError) as e:
        g.run("nve", 0.5, 1, 2, False)
    assert e.value.code == capi.E_OUT_OF_CELL
