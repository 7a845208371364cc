"""Nose-Hoover chains of every length class (1, 2, 3 and the longest, 16), one
and two of them, one of length 1 with an infinite mass (a thermostat that does not
move), on sizes about one workgroup: positions, velocities, chain states and
chain energies against the oracle in FP64, after steps with nothing to report
(chains advanced by the next step's first half) and one that reports.

Bound: 1e-10 of the largest value, as in the other FP64 comparisons with the
oracle over some tens of steps."""
import numpy as np
import pytest

from pfmds_amd import configs
from pfmds_amd.system import NHC, KB
from tests.harness import gpu_ctx, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,chains", [(255, [1]), (256, [2]), (257, [3, 1]), (513, [16, 2]), (300, [16]), (300, [0])])
def test_chains(n, chains):
    s = configs.lj_gas_lattice(n, 0.02, 71, 150.0)
    s.nhcs = []
    for k, M in enumerate(chains):
        g = 3 if len(chains) == 1 else k + 1
        m = n if g == 3 else n // 2
        q = 3 * m * KB * 100.0 * 20.0 ** 2
        s.nhcs.append(NHC(g, 100.0, M or 1, q if M else float("inf")))
    res = []
    for make in (oracle_ctx, gpu_ctx):
        c = make(s)
        c.run("nvt", 0.5, 0, 0, True)
        c.run("nvt", 0.5, 1, 40, False)
        c.run("nvt", 0.5, 41, 55, True)
        res.append((c.state(), c.energies(), [c.get_chain(k + 1, h.M) for k, h in enumerate(s.nhcs)]))
        c.close()
    (so, eo, co), (sg, eg, cg) = res
    for x, y in zip(sg, so):
        assert rel_inf(x, y) < 1e-10
    if chains != [0]:
        np.testing.assert_allclose(eg["e_nhc"], eo["e_nhc"], rtol=1e-10)
    for (xg, vg), (xo, vo) in zip(cg, co):
        assert rel_inf(xg, xo) < 1e-10 and rel_inf(vg, vo) < 1e-10


@pytest.mark.parametrize("n", [300, 8193, 32752, 32784])
@pytest.mark.parametrize("groups", [(3,), (1, 2)])
def test_energies_in_the_force_launch(n, groups):
    """The force launch of a gas forms the kinetic energies up to 1,024 blocks
    (32,768 atoms of 8 lanes); with separate launches (pfm_set_fusion(h, 0))
    k_kick2_ke forms them: the same run within 1e-10."""
    s = configs.lj_gas_lattice(n, 0.02, 72, 150.0)
    s.nhcs = [NHC(g, 100.0, 3, 3 * n * KB * 100.0 * 20.0 ** 2) for g in groups]
    res = []
    for fuse in (True, False):
        c = gpu_ctx(s)
        c.set_fusion(fuse)
        c.run("nvt", 0.5, 0, 0, True)
        c.run("nvt", 0.5, 1, 30, False)
        c.run("nvt", 0.5, 31, 40, True)
        res.append((c.state(), c.energies(), [c.get_chain(k + 1, 3) for k in range(len(groups))]))
        c.close()
    (sa, ea, ca), (sb, eb, cb) = res
    for x, y in zip(sa, sb):
        assert rel_inf(x, y) < 1e-10
    np.testing.assert_allclose(ea["e_nhc"], eb["e_nhc"], rtol=1e-10)
    for (xa, va), (xb, vb) in zip(ca, cb):
        assert rel_inf(xa, xb) < 1e-10 and rel_inf(va, vb) < 1e-10


def test_forces_carried_over_outside_all_atoms():
    """Atoms outside all_atoms keep their forces between steps (zero_forces
    clears that group only): the kinetic energies then come from the whole
    force, as in the oracle."""
    s = configs.lj_gas_lattice(300, 0.02, 73, 150.0)
    s.all_atoms = 1
    s.nhcs = [NHC(3, 100.0, 3, 3 * 300 * KB * 100.0 * 20.0 ** 2)]
    res = []
    for make in (oracle_ctx, gpu_ctx):
        c = make(s)
        c.run("nvt", 0.2, 0, 0, True)
        c.run("nvt", 0.2, 1, 8, False)
        c.run("nvt", 0.2, 9, 10, True)
        res.append((c.state(), c.get_chain(1, 3)))
        c.close()
    (so, co), (sg, cg) = res
    for x, y in zip(sg, so):
        assert rel_inf(x, y) < 1e-10
    for x, y in zip(cg, co):
        assert rel_inf(x, y) < 1e-10


@pytest.mark.parametrize("q,M", [(1e-3, 1), (1e-12, 3), (1e-30, 1), (1e-30, 3), (1e-300, 1)])
def test_small_masses_at_zero_temperature(q, M):
    """A light thermostat at T = 0: its velocity takes the scale's exponent far
    past the exponential's range, where the scale is 0 as in the oracle."""
    s = configs.lj_gas_lattice(300, 0.02, 73, 150.0)
    s.nhcs = [NHC(3, 0.0, M, q)]
    res = []
    for make in (oracle_ctx, gpu_ctx):
        c = make(s)
        c.run("nvt", 0.5, 0, 0, True)
        c.run("nvt", 0.5, 1, 2, True)
        c.run("nvt", 0.5, 3, 8, False)
        res.append((c.state(), c.get_chain(1, M)))
        c.close()
    (so, co), (sg, cg) = res
    for x, y in zip(sg, so):
        np.testing.assert_allclose(x, y, rtol=0, atol=1e-10 * max(np.abs(y).max(), 1.0))
    for x, y in zip(cg, co):
        np.testing.assert_allclose(x, y, rtol=1e-9)
