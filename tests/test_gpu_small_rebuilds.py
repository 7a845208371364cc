"""Rebuilds of few atoms (binning in one workgroup, group rows in one launch)
about their limits: lists, velocities after the zero-momentum step and a run
over three rebuilds against the oracle (FP64: velocities 1e-12 after the one
subtraction, positions, forces and energies 1e-10 as elsewhere), for 1 to 8,193 atoms
about the steps of 256, 1,024 and 8,192, and for replicas."""
import numpy as np
import pytest

from pfmds_amd import capi, configs, system
from tests.harness import gpu_ctx, list_sets, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [165, 255, 257, 1024, 1025, 8191, 8192, 8193])
def test_small_rebuild(n):
    s = configs.lj_gas_lattice(n, 0.02, 13, 100.0, period=4)
    o, c = oracle_ctx(s), gpu_ctx(s)
    for x in (o, c):
        x.run("nve", 0.5, 0, 0, True)
    assert rel_inf(c.state()[1], o.state()[1]) < 1e-12
    for x in (o, c):
        x.run("nve", 0.5, 1, 9, True)
    for ii, it in enumerate(s.interactions):
        for k in range(len(it.lists)):
            assert list_sets(c, ii + 1, k + 1)[0] == list_sets(o, ii + 1, k + 1)[0], (ii, k)
    po, _, fo = o.state()
    p, _, f = c.state()
    assert rel_inf(p, po) < 1e-10 and rel_inf(f, fo) < 1e-10
    o.close()
    c.close()


@pytest.mark.parametrize("sizes", [(170, 855), (4096, 4096), (4096, 4097), (2047, 2049, 257)])
def test_small_rebuild_of_replicas(sizes):
    reps = [configs.lj_gas_lattice(n, 0.02, 20 + k, 100.0, period=4) for k, n in enumerate(sizes)]
    b = system.build_batch_context(system.merge_replicas(reps), capi.FP64)
    b.run("nve", 0.5, 0, 9, True)
    p, v, f = b.state()
    e = b.replica_energies()
    at = 0
    for r, s in enumerate(reps):
        c = gpu_ctx(s)
        c.run("nve", 0.5, 0, 9, True)
        q, w, g = c.state()
        for x, y in ((p, q), (v, w), (f, g)):
            assert rel_inf(x[at:at + s.n], y) < 1e-10
        one = c.energies()
        for name in ("pe", "ke", "temp"):
            np.testing.assert_allclose(e[name][r], one[name], rtol=1e-10)
        at += s.n
        c.close()
    b.close()
