"""The row lanes a handle starts with: 16 for few atoms, 8 for more, at the
sizes where that changes: the same bits as with the lanes set, and the other
count within the rounding of the sums (1e-12 of the largest force in FP64, and
2e-5 in the mixed path, a few float roundings of the largest pair term)."""
import numpy as np
import pytest

from pfmds_amd import capi, configs, system
from tests.harness import gpu_ctx, rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n,lanes", [(capi.FP64, 15000, 16), (capi.FP64, 15001, 8), (capi.MIXED, 8192, 16),
                                          (capi.MIXED, 8193, 8)])
def test_row_lanes(prec, n, lanes):
    s = configs.lj_gas_lattice(n, 0.02, 41, 100.0)
    f = {}
    for L in (0, 8, 16):
        c = gpu_ctx(s, prec)
        if L:
            c.set_tuning(L, 256)
        c.run("nve", 0.5, 0, 3, True)
        f[L] = c.state()[2]
        c.close()
    np.testing.assert_array_equal(f[0], f[lanes])
    assert rel_inf(f[8], f[16]) < (1e-12 if prec == capi.FP64 else 2e-5)


@pytest.mark.parametrize("prec", [capi.FP64, capi.MIXED])
def test_replica_bits_follow_the_lanes(prec):
    """A batch starts with the lanes of its whole size, a replica of it alone
    with those of its own: with the same lanes set on both, the forces of the
    first step have the same bits, without within the rounding above."""
    reps = [configs.fcc_cu_rgl(nx=k, ny=10, nz=k + 2, seed=90 + k, dt=0.5) for k in (9, 11, 12)]
    b = system.merge_replicas(reps)
    assert b.system.n > 8192 and max(s.n for s in reps) < 8192
    f = {}
    for lanes in (0, 8, 16):
        c = system.build_batch_context(b, prec)
        if lanes:
            c.set_tuning(lanes, 256)
        c.run("nve", 0.5, 0, 0, True)
        f[lanes] = c.state()[2]
        for r, s in enumerate(reps):
            o = gpu_ctx(s, prec)
            if lanes:
                o.set_tuning(lanes, 256)
            o.run("nve", 0.5, 0, 0, True)
            got, want = f[lanes][b.replica_slice(r)], o.state()[2]
            if lanes:
                np.testing.assert_array_equal(got, want)
            assert rel_inf(got, want) < (1e-12 if prec == capi.FP64 else 2e-5)
