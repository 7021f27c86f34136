"""Forests in mixed precision on target tiles.  The translations are FP64 and
carry no cell radius, so no pair is left to the per-target kernel for its
cells' radii: none at all where the systems' groups are concatenated (plans
prepared on the host, plans built on the device, whose groups hold no pairs,
and both together), and only those off the first system's lattice, as in FP64,
where the upload groups a forest whose levels do not share a radius.  A system's potentials and accelerations are then those it has alone: the same
FP32 partial sums in P2P, the same FP64 translations summed in another order
(1e-12, the request loop's bound).  Systems of other sizes, one without any
M2L pair."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [4, 10])
@pytest.mark.parametrize("how", ["device", "prepared", "both", "plain"])
def test_forest_groups_every_pair(how, P):
    import exafmm_amd as F
    systems = [F.make_bodies(n, d, 7 + n) for n, d in ((9000, "cube1"), (30, "cube1"), (12001, "plummer1"), (4000, "sphere"))]
    with F.FMM(P=P, precision=F.FMM_MIXED) as f:
        plans, alone = [], []
        for i, (x, q) in enumerate(systems):
            x *= 1.0 + 0.37 * i
            p = F.Plan(x, lists_on=f if how == "device" or (how == "both" and i % 2 == 0) else None)
            if how != "plain":
                p.prepare(P, F.FMM_MIXED)
            f.set_bodies_plan(p, q)
            assert f.stats()["m2l_ungrouped"] == 0
            f.evaluate()
            plans.append(p)
            alone.append(f.targets())
        forest, q = F.Plan.merge(plans), np.concatenate([q for _, q in systems])
        with F.FMM(P=P) as g:
            g.set_bodies_plan(forest, q)
            off = g.stats()["m2l_ungrouped"]
        assert how == "plain" or off == 0
        f.set_bodies_plan(forest, q)
        st = f.stats()
        assert st["m2l_path"] == F.M2L_TILES and st["m2l_ungrouped"] == off
        f.evaluate()
        t, at = f.targets(), 0
        for a in alone:
            b = t[at:at + len(a)]
            at += len(a)
            assert np.linalg.norm(b[:, 0] - a[:, 0]) <= 1e-12 * np.linalg.norm(a[:, 0])
            assert np.linalg.norm(b[:, 1:] - a[:, 1:]) <= 1e-12 * np.linalg.norm(a[:, 1:])
