"""List search one wave per cell: a dilute binary gas (2,197 cells of 2.7
atoms), its four lists in one pass, two of them in one pass and one by one,
alone, beside a larger Cu crystal (the candidates under half of the atoms:
compacted staging) and beside a box under three cells wide, whose cells go to
the workgroup-per-cell kernel in a launch of their own.  Every list equal to
the oracle's as sets.
"""
import functools

import numpy as np
import pytest

from pfmds_amd import capi, configs, system
from pfmds_amd.system import Interaction
from tests.harness import gpu_ctx, list_sets, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu


def gas(n, density, seed, variant):
    s = configs.lj_gas_lattice(n, density, seed, 100.0, dt=1.0, period=10)
    a = np.random.default_rng(seed).random(n) < 0.3
    s.species = ["A" if x else "B" for x in a]
    s.mass = np.where(a, 39.95, 83.80)
    lj1g_a, lj1g_b, lj = s.interactions
    s.interactions = {"quad": [lj1g_a, lj1g_b, lj], "pair": [lj1g_a, lj], "single": [lj]}[variant]
    return s


@functools.lru_cache(maxsize=None)
def oracle_lists(n, density, seed, variant):
    s = gas(n, density, seed, variant)
    o = oracle_ctx(s)
    o.run("nve", 1.0, 0, 0, True)
    out = {}
    for k, it in enumerate(s.interactions, start=1):
        for li in range(1, len(it.lists) + 1):
            out[k, li] = list_sets(o, k, li)[0]
    return out, o.state()[2]


@pytest.mark.parametrize("beside", ["", "cu", "narrow", "cu narrow"])
@pytest.mark.parametrize("variant", ["quad", "pair", "single"])
def test_lists_equal_oracle(variant, beside):
    gases = [(6000, 0.0036, 81, variant)] + [(170, 0.03, 82, variant)] * ("narrow" in beside)
    reps = [gas(*g) for g in gases]
    if "cu" in beside:
        reps.append(configs.fcc_cu_rgl(nx=13, ny=12, nz=13, seed=83, dt=1.0))
    wide = np.floor(reps[0].box / 8.5).astype(int)
    assert wide.prod() >= 2048 and reps[0].n < 10 * wide.prod()
    if "narrow" in beside:
        assert (reps[1].box / 8.5 < 3).all()
    b = system.merge_replicas(reps) if len(reps) > 1 else None
    g = system.build_batch_context(b, capi.FP64) if b else gpu_ctx(reps[0])
    g.run("nve", 1.0, 0, 0, True)
    frc = g.state()[2]
    for k, it in enumerate(reps[0].interactions, start=1):
        for li in range(1, len(it.lists) + 1):
            got = list_sets(g, k, li)[0]
            want, first, sp = [], 0, "AB"[it.lists[li - 1][1] - 1]  # entries count their group's atoms
            for r, q in enumerate(gases):
                want += [tuple(x + first for x in row) for row in oracle_lists(*q)[0][k, li]]
                first += reps[r].species.count(sp)
            assert got == want, f"list {k}.{li}"
    for r, q in enumerate(gases):
        f = frc[b.replica_slice(r)] if b else frc
        assert rel_inf(f, oracle_lists(*q)[1]) < 1e-10
