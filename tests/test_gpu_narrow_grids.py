"""List search of boxes under three cells wide in some direction (their cells
take every pair's nearest image), and the pair and quad passes of the
workgroup-per-cell kernel: every list of a binary gas equal to the oracle's as
sets, single systems of each grid shape and a batch that mixes them.
"""
import numpy as np
import pytest

from pfmds_amd import capi, configs, system
from tests.harness import gpu_ctx, list_sets, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu


def gas(sides, seed, spacing=3.6, jitter=0.25):
    """Binary gas (lj1g A, lj1g B, lj A-B; list cutoff 8.5 A) on a jittered
    lattice filling a box of the given sides, atoms up to its faces."""
    s = configs.lj_gas_lattice(64, 0.02, seed, 100.0)
    rng = np.random.default_rng(seed)
    L = np.asarray(sides, float)
    m = np.maximum(1, np.floor(L / spacing).astype(int))
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, 3)
    pos = g * (L / m) + jitter * (2 * rng.random((len(g), 3)) - 1)
    pos = np.mod(pos, L)
    n = len(pos)
    s.box, s.pos, s.vel = L, pos, np.zeros((n, 3))
    s.species = ["A" if x else "B" for x in rng.random(n) < 0.5]
    s.mass = np.where(np.array(s.species) == "A", 39.95, 83.80)
    return s


SHAPES = [(9.0, 9.0, 9.0), (18.0, 18.0, 18.0), (9.0, 18.0, 35.0), (18.0, 26.0, 43.0), (26.0, 26.0, 26.0),
          (40.0, 17.2, 26.0), (60.0, 60.0, 10.0)]


@pytest.mark.parametrize("sides", SHAPES)
def test_lists_equal_oracle(sides):
    s = gas(sides, 5)
    g, o = gpu_ctx(s), oracle_ctx(s)
    for c in (g, o):
        c.run("nve", 0.5, 0, 0, True)
    for k, it in enumerate(s.interactions, start=1):
        for li in range(1, len(it.lists) + 1):
            assert list_sets(g, k, li)[0] == list_sets(o, k, li)[0], f"{sides}: list {k}.{li}"
    assert rel_inf(g.state()[2], o.state()[2]) < 1e-10


def test_batch_of_shapes():
    """Narrow and wide grids in one handle, each replica against the oracle."""
    reps = [gas(x, 11 + k) for k, x in enumerate(SHAPES)]
    reps += [configs.fcc_cu_rgl(nx=c, ny=4, nz=c, seed=40 + c, dt=0.5, nmax=128) for c in (4, 5, 7)]
    b = system.merge_replicas(reps)
    g = system.build_batch_context(b, capi.FP64)
    g.run("nve", 0.5, 0, 0, True)
    g.run("nve", 0.5, 1, 20, True)
    pos, _, frc = g.state()
    for r, s in enumerate(reps):
        o = oracle_ctx(s)
        o.run("nve", 0.5, 0, 0, True)
        o.run("nve", 0.5, 1, 20, True)
        po, _, fo = o.state()
        sl = b.replica_slice(r)
        assert rel_inf(pos[sl], po) < 1e-10, r
        assert rel_inf(frc[sl], fo) < 1e-8, r
