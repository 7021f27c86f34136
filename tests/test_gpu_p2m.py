"""P2M of leaves of every size (empty groups of lanes, one body, more than a
wavefront's) at the orders' edges (odd orders: a middle column of its own) and
on both sides of the rule that deals a leaf's bodies to lanes (8192 leaves),
against multipoles in extended precision: FP64 recurrences of at most P steps
and sums of at most ncrit bodies, 1e-13 per degree of the leaf multipoles."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [2, 3, 4, 7, 8, 11, 12, 13, 20])
@pytest.mark.parametrize("n,ncrit", [(1, 64), (70, 64), (300, 3), (2000, 100)])
def test_leaf_multipoles(P, n, ncrit):
    import exafmm_amd as F
    x, q = F.make_bodies(n, "plummer1", P)
    many = F.Plan(F.make_bodies(60000, "cube1", 3)[0], ncrit=4)
    assert many.stats()["nleaf"] > 8192
    plan = F.Plan(x, ncrit=ncrit)
    t = plan.tree()
    leaf = np.flatnonzero(t["nchild"] == 0)
    ref = np.zeros((len(leaf), P * (P + 1) // 2), np.clongdouble)
    LD = np.longdouble
    for i, c in enumerate(leaf):
        b = slice(t["ibody"][c], t["ibody"][c] + t["nbody"][c])
        dx, dy, dz = (x[t["perm"][b]].astype(LD) - t["X"][c].astype(LD)).T
        w = q[t["perm"][b]].astype(LD)
        r2 = dx * dx + dy * dy + dz * dz
        rmm = np.ones(len(w), np.clongdouble)
        for m in range(P):
            if m > 0:
                rmm = rmm * (dx + 1j * dy) * (-LD(1) / (2 * m))
            r0, r1 = np.zeros(len(w), np.clongdouble), rmm
            for k in range(m, P):
                if k > m:
                    r0, r1 = r1, (r1 * (2 * k - 1) * dz - r0 * r2) / LD(k * k - m * m)
                s = np.sqrt(LD(math.factorial(k - m)) * LD(math.factorial(k + m)))
                ref[i, k * (k + 1) // 2 + m] = (w * np.conj(r1)).sum() * s
    with F.FMM(P=P) as f:
        for p, c in ((plan, q), (F.Plan.merge([plan, many]), np.concatenate([q, np.ones(60000)]))):
            f.set_bodies_plan(p, c)
            f.upward()
            M = f.expansions()[0][: len(t["R"])][leaf]
            for k in range(P):
                u = slice(k * (k + 1) // 2, (k + 1) * (k + 2) // 2)
                assert np.linalg.norm(M[:, u] - ref[:, u]) <= 1e-13 * np.linalg.norm(ref[:, u]), k
