"""The FP64 pair terms over their whole distance range: isolated dimers from
short separations to past the list's cutoff, with both edges of the switching
zone to one part in 1e12, against the pair formulas in long double.

Tolerance, set before the first run: u = 2^-53; the distance, the cutoff and
the products round a few times each (32 u of every bracket, with the cutoff
at 1 because its half-angle form rounds in absolute terms), and an
exponential of argument a adds 4 u |a|.  The ljc / morsec exponents that are
not whole numbers go through the same power function: against the oracle
within 1e-12 of the largest force.
"""
import numpy as np
import pytest

from pfmds_amd import capi, configs
from pfmds_amd.system import Integrator, Interaction, System
from tests.harness import gpu_ctx, oracle_ctx, rel_inf

pytestmark = pytest.mark.gpu
LD = np.longdouble
PI = LD(3.14159265358979)
U = 2.0 ** -53


def dimers(name, params, lo, hi, rc, nmax=4):
    """Isolated dimers along x, 25 A apart on a grid, of 60 separations."""
    R1, R2 = params[-2], params[-1]
    d = np.concatenate([np.linspace(lo, hi, 54), [R1 * (1 - 1e-12), R1, R1 * (1 + 1e-12), 0.5 * (R1 + R2),
                                                  R2 * (1 - 1e-12), R2 * (1 + 1e-9)]])
    g = np.stack(np.meshgrid(np.arange(4), np.arange(4), np.arange(4), indexing="ij"), -1).reshape(-1, 3)[:len(d)]
    a = g * 25.0 + 3.1
    b = a.copy()
    b[:, 0] += d
    pos = np.stack([a, b], 1).reshape(-1, 3)
    n = len(pos)
    sp = ["A", "B"] * len(d) if name == "lj" else ["A"] * n
    lists = [(1, 2, nmax, rc, 10), (2, 1, nmax, rc, 10)] if name == "lj" else [(1, 1, nmax, rc, 10)]
    groups = [["A"], ["B"], ["A", "B"], ["#"]]
    s = System(box=np.full(3, 100.0), pos=pos, vel=np.zeros((n, 3)), mass=np.full(n, 40.0), species=sp,
               groups=groups, interactions=[Interaction(name, params, lists)],
               integrators=[Integrator("nve", 1.0, 10, 10**9, 10**9)], all_moving=3, xyz_moving=3, z_moving=4,
               all_atoms=3)
    return s, (b[:, 0].astype(LD) - a[:, 0].astype(LD))


def switch(r, R1, R2):
    x = np.clip((r - R1) / (R2 - R1), LD(0), LD(1))
    return (1 + np.cos(PI * x)) / 2, -PI * np.sin(PI * x) / (2 * (R2 - R1)), x


@pytest.mark.parametrize("name", ["lj", "lj1g", "rjl"])
def test_dimer_scan(name):
    if name == "rjl":
        params, lo, hi, rc = list(configs.RJL_CU), 1.9, 5.99, 6.5
    else:
        params, lo, hi, rc = [0.0104, 3.4, 6.5, 7.5], 2.6, 7.9, 8.5
    s, r = dimers(name, params, lo, hi, rc)
    c = gpu_ctx(s)
    c.run("nve", 1.0, 0, 0, True)
    f = c.state()[2].reshape(-1, 2, 3)
    p = [LD(x) for x in params]
    R1, R2 = p[-2], p[-1]
    if name == "rjl":
        A0, xi, pp, q, r0 = p[:5]
        fc, df, _ = switch(r, R1, R2)
        ep, eq = np.exp(-pp * (r / r0 - 1)), np.exp(-2 * q * (r / r0 - 1))
        with np.errstate(all="ignore"):
            att = xi * eq / np.sqrt(eq * fc)
            want = -2 * A0 * (pp / r0 * fc - df) * ep + 2 * (q / r0 * fc - df / 2) * att
        # each bracket's rounding, the cutoff's in absolute terms
        wb = np.abs(PI / (R2 - R1))
        arg = 32 + 4 * np.abs(pp * (r / r0 - 1))
        scale = arg * (2 * A0 * (pp / r0 + wb) * ep + 2 * (q / r0 + wb) * att)
        want, scale = -want, scale
    else:
        eps, sig = p[:2]
        V = (sig / r) ** 6
        if name == "lj":
            fc, df, _ = switch(r, R1, R2)
        else:
            x = np.clip((r - R1) / (R2 - R1), LD(0), LD(1))
            fc = 1 - 10 * x ** 3 + 15 * x ** 4 - 6 * x ** 5
            df = r * 0 + (-30 * x ** 2 + 60 * x ** 3 - 30 * x ** 4) / 1
        want = 4 * eps * (V * (12 * V - 6) * fc / r - V * (V - 1) * df)
        scale = 64 * 4 * eps * V * ((12 * V + 6) / r + (V + 1) * 30 / (R2 - R1))
    inside = r < R2
    got = -f[:, 0, 0]  # repulsion pushes the first atom towards -x
    ok = inside & np.isfinite(want.astype(float))
    assert ok.sum() >= 50
    err = np.abs(got[ok] - want[ok]) / (U * scale[ok])
    assert float(err.max()) < 1.0, float(err.max())
    assert not f[~inside].any()
    np.testing.assert_array_equal(f[:, 0], -f[:, 1])


@pytest.mark.parametrize("kind,delt", [("morsec", 0.5), ("morsec", 1.0), ("morsec", 2.0), ("morsec", 3.3), ("ljc", 2.7), ("ljc", 3.0),
                                       ("ljc", 4.0), ("ljc", 5.0)])
def test_cosine_exponents(kind, delt):
    s = configs.graphene_on_cu(cx=14, cy=8, gx=14, gy=8, layers=4, seed=31, jitter=0.1)
    lists = s.interactions[2].lists
    params = [0.025, 3.05, 1.30, delt, 6.0, 7.0, 0.0] if kind == "morsec" else [0.005, 3.2, delt, 6.0, 7.0, 0.0]
    s.interactions[2] = Interaction(kind, params, lists)
    g, o = gpu_ctx(s), oracle_ctx(s)
    for c in (g, o):
        c.run("nve", 0.5, 0, 0, True)
    assert rel_inf(g.state()[2], o.state()[2]) < 1e-12
    np.testing.assert_allclose(g.energies()["e_inter"], o.energies()["e_inter"], rtol=1e-12)


@pytest.mark.parametrize("name", ["lj", "lj1g", "rjl"])
def test_coincident_atoms_stop_the_run(name):
    """Two atoms on one point: the forces are not numbers and the next step's
    position check stops the run."""
    params = list(configs.RJL_CU) if name == "rjl" else [0.0104, 3.4, 6.5, 7.5]
    s, _ = dimers(name, params, 2.6, 5.9, 6.5 if name == "rjl" else 8.5)
    s.pos[1] = s.pos[0]
    c = gpu_ctx(s)
    c.run("nve", 1.0, 0, 0, False)
    assert np.isnan(c.state()[2][:2]).any()
    with pytest.raises(capi.PfmError) as e:
        c.run("nve", 1.0, 1, 2, False)
    assert e.value.code == capi.E_OUT_OF_CELL


@pytest.mark.parametrize("name", ["lj", "lj1g", "rjl"])
def test_coincident_atoms_energy(name):
    """Two atoms on one point: their rows' energies are those of the formulas,
    infinite for the powers of 1/r (and the interaction's sum then is no
    number, as its compensated sum cannot be) and finite for the exponentials
    (the sum is the oracle's)."""
    params = list(configs.RJL_CU) if name == "rjl" else [0.0104, 3.4, 6.5, 7.5]
    s, _ = dimers(name, params, 2.6, 5.9, 6.5 if name == "rjl" else 8.5)
    s.pos[1] = s.pos[0]
    g, o = gpu_ctx(s), oracle_ctx(s)
    for c in (g, o):
        c.run("nve", 1.0, 0, 0, True)
    np.testing.assert_array_equal(np.isnan(g.state()[2][:2]), np.isnan(o.state()[2][:2]))
    if name == "rjl":
        np.testing.assert_allclose(g.energies()["e_inter"], o.energies()["e_inter"], rtol=1e-12)
    else:
        e = g.row_energies(1)
        assert not np.isnan(e).any() and np.isposinf(e).sum() == 1 and o.energies()["e_inter"][0] == np.inf


def rjl_row_energies(r, p, r0, R1, R2):
    """Energies of isolated rjl dimers along x with A0 = 1 and xi = 0, so that
    each of a dimer's two rows holds exp(-(r - r0) p/r0) f(r), in ascending
    order; separations r are multiples of 2^-40."""
    m = int(np.ceil(len(r) ** (1 / 3)))
    step = float(2 ** np.ceil(np.log2(2.2 * R2 + 4.0)))
    g = np.stack(np.meshgrid(np.arange(m), np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 3)[:len(r)]
    a = g * step + 1.0
    b = a.copy()
    b[:, 0] += r
    assert (b[:, 0] - a[:, 0] == r).all()
    pos = np.stack([a, b], 1).reshape(-1, 3)
    n = len(pos)
    s = System(box=np.full(3, m * step), pos=pos, vel=np.zeros((n, 3)), mass=np.full(n, 63.546), species=["Cu"] * n,
               groups=[["Cu"], ["#"]],
               interactions=[Interaction("rjl", [1.0, 0.0, p, 0.0, r0, R1, R2], [(1, 1, 4, R2 + 0.25, 10)])],
               integrators=[Integrator("nve", 1.0, 10, 10**9, 10**9)], z_moving=2)
    c = gpu_ctx(s)
    c.run("nve", 1.0, 0, 0, True)
    e = np.sort(c.row_energies(1)).reshape(-1, 2)
    np.testing.assert_array_equal(e[:, 0], e[:, 1])
    return e[:, 0]


def separations(lo, hi, k, seed):
    return np.round(np.random.default_rng(seed).uniform(lo, hi, k) * 2.0 ** 40) / 2.0 ** 40


def test_exponential_is_no_less_accurate_than_the_library():
    """The argument r0 - r is exact for p = r0 = 1, so the rows hold the
    exponential alone: within the 0.87 ulp that the library's has over
    [-25, 12] (4 million arguments)."""
    r = separations(0.1, 20.0, 8000, 1)
    e = rjl_row_energies(r, 1.0, 1.0, 20.5, 21.0)
    want = np.sort(np.exp(1 - r.astype(LD)))
    err = np.abs(e - want) / np.spacing(want.astype(float))
    print(f"[exp] max {float(err.max()):.3f} ulp", flush=True)
    assert float(err.max()) < 0.87


@pytest.mark.parametrize("R1,R2", [(1.7, 2.0), (5.5, 6.0), (6.1, 7.3), (6.5, 7.5)])
def test_cutoff_is_no_less_accurate_than_the_library(R1, R2):
    """p = 0 leaves the cutoff alone: its RMS error over the switching zone
    within 0.51 u, that of (1 + cos(pi x))/2 with the library's cosine over
    random zones."""
    r = separations(R1, R2, 8000, 2)
    r = r[(r > R1) & (r < R2)]
    e = rjl_row_energies(r, 0.0, 1.0, R1, R2)
    want = np.sort(switch(r.astype(LD), LD(R1), LD(R2))[0])
    err = ((e - want) / U).astype(float)
    print(f"[cutoff] max {np.abs(err).max():.3f} u, rms {np.sqrt((err ** 2).mean()):.3f} u", flush=True)
    assert np.sqrt((err ** 2).mean()) < 0.51
