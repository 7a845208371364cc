"""The end of an nvms step inside a block, one kernel (k_spec_step), against
the separate kernels of the step-by-step path, bit for bit: sizes about one
workgroup and beyond the largest grid (1,024 workgroups of 256), 3, 4 and 5
interactions (their sums and the kinetic energy go four to an exchange), xyz-
and z-moving atoms, both precisions."""
import numpy as np
import pytest

from pfmds_amd import capi, configs
from pfmds_amd.system import Interaction
from tests.harness import gpu_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ni,steps", [(255, 3, 60), (256, 4, 60), (257, 5, 60), (262145, 3, 9)])
@pytest.mark.parametrize("prec", [capi.FP64, capi.MIXED])
def test_spec_step(n, ni, steps, prec):
    s = configs.lj_gas_lattice(n, 0.02, 31, 60.0)
    s.xyz_moving, s.z_moving = 1, 2
    a, b = (s.interactions[k].lists[0] for k in (0, 1))
    s.interactions = s.interactions + [Interaction("lj1g", [0.001, 3.2, 6.5, 7.5], [r]) for r in (a, b)][:ni - 3]
    res = []
    for spec in (False, True):
        c = gpu_ctx(s, prec)
        c.set_speculation(spec)
        last = c.run("nvms", 0.5, 0, steps // 3, True, 1e-30)
        last = c.run("nvms", 0.5, steps // 3 + 1, steps, True, 1e-30)
        res.append((last, c.state(), c.energies()))
        c.close()
    (la, sa, ea), (lb, sb, eb) = res
    assert la == lb
    for x, y in zip(sa, sb):
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(ea["e_inter"], eb["e_inter"])
    for k in ("pe", "ke", "temp"):
        assert ea[k] == eb[k], k
