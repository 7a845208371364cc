"""pfm_set_state / pfm_get_state through their pinned chunks: what goes in
comes back bit for bit in original order, for sizes below, at and past the
chunks' edges (512 KiB: 21,845 atoms of one array), with absent arrays, before
the first sort and after one, repeatedly and from a second thread.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from pfmds_amd import capi, configs
from tests.harness import gpu_ctx

pytestmark = pytest.mark.gpu
D = C.POINTER(C.c_double)


def bare(n):
    rng = np.random.default_rng(n)
    return capi.Context.gpu(np.full(3, 50.0), rng.random((n, 3)) * 50, rng.random((n, 3)), np.full(n, 2.0)), rng


@pytest.mark.parametrize("n", [1, 255, 7281, 7282, 21845, 21846, 200001])
def test_round_trip_and_absent_arrays(n):
    c, rng = bare(n)
    p, v = rng.random((n, 3)) * 50, rng.random((n, 3))
    c.set_state(p, v)
    for _ in range(2):
        gp, gv, gf = c.state()
        np.testing.assert_array_equal(gp, p)
        np.testing.assert_array_equal(gv, v)
        assert not gf.any()
    # one array at a time: the other keeps its values
    v2 = rng.random((n, 3))
    assert c.lib.pfm_set_state(c.h, None, v2.ctypes.data_as(D)) == capi.OK
    out = np.full((n, 3), -1.0)
    assert c.lib.pfm_get_state(c.h, None, out.ctypes.data_as(D), None) == capi.OK
    np.testing.assert_array_equal(out, v2)
    p2 = rng.random((n, 3)) * 50
    assert c.lib.pfm_set_state(c.h, p2.ctypes.data_as(D), None) == capi.OK
    gp, gv, _ = c.state()
    np.testing.assert_array_equal(gp, p2)
    np.testing.assert_array_equal(gv, v2)
    assert c.lib.pfm_get_state(c.h, None, None, None) == capi.OK


def test_after_sorts_and_from_a_thread():
    """Reading the state leaves the run as it is; a read from another thread
    gives the same arrays."""
    s = configs.fcc_cu_rgl(nx=9, ny=8, nz=7, seed=3)
    a, b = gpu_ctx(s), gpu_ctx(s)
    for c in (a, b):
        c.run("nve", 1.0, 0, 0, True)
    got = []
    for k in range(4):
        for c in (a, b):
            c.run("nve", 1.0, 1 + 15 * k, 15 * (k + 1), False)
        t = threading.Thread(target=lambda: got.append(a.state()))
        t.start()
        t.join()
    for x, y in zip(got[-1], b.state()):
        np.testing.assert_array_equal(x, y)
    # the same state set back re-sorts and gives the same forces to rounding
    p, v, f = b.state()
    b.set_state(p, v)
    b.run("nve", 1.0, 0, 0, False)
    assert np.abs(b.state()[2] - f).max() < 1e-12 * np.abs(f).max()


def test_copy_state_around_nvms_blocks():
    """The staging of pfm_copy_state outlives the first nvms block of its
    handle (whose ring once released it)."""
    s = configs.fcc_cu_rgl(nx=6, seed=9, temperature=80.0)
    a, b = gpu_ctx(s), gpu_ctx(s)
    a.run("nve", 1.0, 0, 5, False)
    b.run("nve", 1.0, 0, 0, False)
    for _ in range(2):
        b.copy_state_from(a)
        p, v, _ = a.state()
        q, w, _ = b.state()
        np.testing.assert_array_equal(p, q)
        np.testing.assert_array_equal(v, w)
        b.run("nvms", 1.0, 0, 25, True, 1e-30)


@pytest.mark.parametrize("n", [64, 5000])
def test_state_arrays_own_their_memory(n):
    """A program that keeps the positions of many frames holds no more than
    those: the three arrays share no block."""
    s = configs.lj_gas_lattice(n, 0.02, 7, 100.0)
    c = gpu_ctx(s)
    a, b = c.state(), c.state()
    for x in (*a, *b):
        assert x.flags.owndata and x.base is None and x.shape == (n, 3) and x.flags.c_contiguous
    for i, x in enumerate((*a, *b)):
        assert not any(np.shares_memory(x, y) for y in (*a, *b)[i + 1:])
