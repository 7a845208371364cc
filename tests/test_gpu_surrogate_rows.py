"""The surrogate's row passes where the rows are split (sur_split): few rows
(32 lanes each), more than a round of those (8 lanes each) and more than a full
round of workgroups (8 lanes, the rest 32), against the float64 textbook sums
over neighbours found by a k-d tree: descriptors, forces and, at the middle
size, the loss gradient (whose tangent pass takes the same split), with the
bounds of test_gpu_surrogate.py; and the fused pass against the separate
kernels bit for bit."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import tests.sur_ref as S
from pfmds_amd import capi, configs
from tests.test_gpu_surrogate import RC, emulate, forces_from_gG, groups, sur_ctx, theta_for

pytestmark = pytest.mark.gpu


def tree_pairs(s, g1, g2):
    """sur_ref.pairs by a k-d tree."""
    tree = cKDTree(np.mod(s.pos[g2], s.box), boxsize=s.box)
    near = tree.query_ball_point(np.mod(s.pos[g1], s.box), RC)
    ri = np.repeat(np.arange(len(g1)), [len(x) for x in near])
    ia, ja = g1[ri], g2[np.concatenate([np.asarray(x, dtype=int) for x in near])]
    d = s.pos[ja] - s.pos[ia]
    shift = np.round(d / s.box)
    d -= s.box * shift
    ok = ((d * d).sum(-1) < RC * RC) & (ia != ja)
    return ri[ok], ia[ok], ja[ok], shift[ok]


# rows: 4 gx gy; 256 CUs: 6,144 rows in a round of the wide ones, 24,576 in a full one
@pytest.mark.parametrize("cells", [(3, 2), (13, 11), (52, 30), (104, 60)])
def test_row_split(cells):
    import torch
    gx, gy = cells
    cx, cy = max(10, int(round(gx * 100 / 104))), max(6, int(round(gy * 58 / 60)))
    gx, gy = (10, 6) if gx < 10 else (gx, gy)
    s = configs.graphene_on_cu(cx=cx, cy=cy, gx=gx, gy=gy, layers=2, frozen=1, seed=59, jitter=0.1)
    g1, g2 = groups(s)
    P = tree_pairs(s, g1, g2)
    G = S.descriptors(torch.tensor(s.pos), s.box, g1, g2, RC, P, brute=False).numpy()
    theta = theta_for(G, seed=4)
    for precision in (capi.MIXED, capi.FP64):
        ctx, _ = sur_ctx(s, theta, precision)
        Gg = ctx.sur_descriptors(1, len(g1))
        assert (np.abs(Gg - G) / np.maximum(np.abs(G).max(0), 1e-12)).max() < 1e-4
        f = ctx.state()[2]
        Ei, gG = emulate(Gg, theta)
        f_emu = forces_from_gG(s, P, gG)
        assert np.sqrt(np.mean((f - f_emu) ** 2)) < 1e-3 * np.sqrt(np.mean(f_emu ** 2))
        ctx.set_fusion(False)
        ctx.run("nve", 0.5, 0, 0, True)
        np.testing.assert_array_equal(ctx.state()[2], f)
        if len(g1) == 6240 and precision == capi.MIXED:
            f_ref = np.random.default_rng(6).normal(size=s.pos.shape) * 0.5
            e_ref = float(S.unpack(theta)["b3"]) * len(g1) + 3.0
            loss, grad = ctx.sur_loss_grad(1, f_ref, e_ref, 0.7, 1.3)
            lref, gref = S.loss_and_grad(s.pos, s.box, g1, g2, RC, S.round_weights(theta), f_ref, e_ref, 0.7, 1.3, P)
            np.testing.assert_allclose(loss, lref, rtol=3e-2)
            assert np.linalg.norm(grad - gref) < 3e-2 * np.linalg.norm(gref)
        ctx.close()
