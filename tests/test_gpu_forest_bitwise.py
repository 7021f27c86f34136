"""A system sums the same way alone and in a forest.  P2M and P2P deal a leaf to
more lanes in systems of few leaves, by the system's own count: with the M2L per
target (fixed order, no atomic additions) and orders above 12 (one form of M2M
and L2L) the targets are the same bits, whatever the forest holds.  Forests with
more leaves than the lines (8192 and 12000) of systems below them, and with a
system above them; leaves of 16 bodies and more and smaller ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,sizes,ncrit", [(13, (9000, 5001, 8999), 3), (14, (40000, 3000, 40), 3),
                                           (13, (60000, 100, 50001, 55000), 28)])
def test_same_bits_alone_and_in_a_forest(P, sizes, ncrit):
    import exafmm_amd as F
    systems = [F.make_bodies(n, "cube1", 11 + i) for i, n in enumerate(sizes)]
    plans = [F.Plan(x, ncrit=ncrit) for x, _ in systems]
    leaves = [p.stats()["nleaf"] for p in plans]
    assert sum(leaves) > 12000
    alone = []
    with F.FMM(P=P, ncrit=ncrit, m2l_mode=F.M2L_TARGET) as f:
        for p, (_, q) in zip(plans, systems):
            f.set_bodies_plan(p, q)
            f.evaluate()
            alone.append(f.targets())
        f.set_bodies_plan(F.Plan.merge(plans), np.concatenate([q for _, q in systems]))
        f.evaluate()
        t = f.targets()
    at = 0
    for a, k in zip(alone, leaves):
        assert np.array_equal(t[at:at + len(a)], a), k
        at += len(a)
