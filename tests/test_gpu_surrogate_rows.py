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


def with_loners(s, k):
    """The system and k carbon atoms without neighbours, 7.5 A apart in the empty
    part of its tall box, 30 A from the rest: they add rows and nothing else."""
    nx, ny = (np.floor(s.box[:2] / 7.5)).astype(int)
    z0 = s.pos[:, 2].max() + 30.0
    i = np.arange(k)
    p = np.stack([(i % nx) * 7.5, (i // nx % ny) * 7.5, z0 + (i // (nx * ny)) * 7.5], 1) + 1.0
    assert k == 0 or p[:, 2].max() < s.box[2] - 30.0
    s.pos = np.concatenate([s.pos, p])
    s.vel = np.concatenate([s.vel, np.zeros((k, 3))])
    s.mass = np.concatenate([s.mass, np.full(k, 12.011)])
    s.species = list(s.species) + ["C"] * k
    return s


@pytest.mark.parametrize("precision", [capi.MIXED, capi.FP64])
def test_lanes_give_the_same_bits(precision):
    """The rows of one system among few rows (32 lanes each), among more than a
    round of those (8 lanes) and among a full round of workgroups with a rest
    (8 lanes, and 32 for the rest): descriptors are equal bit for bit, forces
    within 1e-12 of the largest (an atom's own share is an FP64 sum over its
    row's lanes), the fused pass and the separate kernels bit for bit, and the
    force loss's gradient within 1e-5 (its sums over the rows are split anew; a
    descriptor or tangent off in its last bit moves a BF16 input and the
    gradient by several times that)."""
    rng = np.random.default_rng(61)
    res, theta, n0, rows0 = [], None, None, None
    for total in (0, 7000, 24576 + 500):
        s = configs.graphene_on_cu(cx=12, cy=11, gx=13, gy=11, layers=2, frozen=1, seed=60, jitter=0.1, lz=9000.0)
        if n0 is None:
            n0, rows0 = s.n, len(groups(s)[0])
            f_ref = 0.5 * rng.normal(size=(n0, 3))
        s = with_loners(s, max(0, total - rows0))
        g1, g2 = groups(s)
        if theta is None:
            P = tree_pairs(s, g1, g2)
            import torch
            theta = theta_for(S.descriptors(torch.tensor(s.pos), s.box, g1, g2, RC, P, brute=False).numpy(), seed=4)
        ctx, _ = sur_ctx(s, theta, precision)
        G = ctx.sur_descriptors(1, len(g1))
        f = ctx.state()[2]
        assert not f[n0:].any()
        target = np.concatenate([f_ref, f[n0:]])
        _, grad = ctx.sur_loss_grad(1, target, 0.0, 0.0, 1.3 * len(g2) / n0)
        ctx.set_fusion(False)
        ctx.run("nve", 0.5, 0, 0, True)
        res.append((G[:rows0], f[:n0], ctx.state()[2][:n0], grad[:-1]))
        ctx.close()
    for a, b, c, grad in res[1:]:
        np.testing.assert_array_equal(a, res[0][0])
        np.testing.assert_array_equal(b, c)
        assert np.abs(b - res[0][1]).max() < 1e-12 * np.abs(b).max()
        d = float(np.linalg.norm(grad - res[0][3]) / np.linalg.norm(res[0][3]))
        print(f"[sur lanes] gradient {d:.2e}", flush=True)
        assert d < 1e-5
