"""The target-tile M2L (rotate, shift, rotate back) at the sizes where its
layout changes: every order it takes (P = 2..12: one to three tiles of four
degrees, with and without a shared last row), tiles stored whole and split
over work items, reflections (the lattice holds offsets along every axis) and
periodic images.
Against the per-target kernel, which evaluates each pair's harmonics directly,
on the same multipoles: both are FP64 sums of the same terms, a few hundred
per coefficient with condition numbers below 1e2, so they agree to 1e-12."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _F():
    import exafmm_amd
    return exafmm_amd


def _locals(F, x, q, mode, **kw):
    with F.FMM(m2l_mode=mode, nspawn=1000, **kw) as f:
        f.set_bodies(x, q)
        f.upward()
        f.m2l()
        f.synchronize()
        return f.expansions()[1], f.stats()


def _check(F, x, q, **kw):
    t, st = _locals(F, x, q, F.M2L_TILES, **kw)
    r, _ = _locals(F, x, q, F.M2L_TARGET, **kw)
    assert st["m2l_path"] == F.M2L_TILES and st["m2l_pairs"] > 0 and st["m2l_ungrouped"] == 0
    assert np.all(np.isfinite(t.view(np.float64)))
    # per degree: the coefficients of different degrees differ by many orders
    P = kw["P"]
    for n in range(P):
        u = slice(n * (n + 1) // 2, (n + 1) * (n + 2) // 2)
        assert np.linalg.norm(t[:, u] - r[:, u]) <= 1e-12 * np.linalg.norm(r[:, u]), n


@pytest.mark.parametrize("P", range(2, 13))
@pytest.mark.parametrize("dist,n,ncrit", [("cube1", 200, 8), ("plummer1", 3001, 16)])
def test_every_order_matches_per_target(P, dist, n, ncrit):
    F = _F()
    x, q = F.make_bodies(n, dist, P)
    _check(F, x, q, P=P, theta=0.5, ncrit=ncrit)


@pytest.mark.parametrize("P", [5, 8, 9, 10, 12])
def test_periodic_images_match_per_target(P):
    F = _F()
    rng = np.random.default_rng(P)
    x = rng.random((1500, 3)) - 0.5
    q = rng.random(1500) - 0.5
    _check(F, x, q, P=P, theta=0.4, ncrit=32, images=1, cycle=1.0)


def test_device_plan_of_another_order():
    """a device-built plan holds the tiles of its context's order; a context
    of another order builds its own"""
    F = _F()
    x, q = F.make_bodies(5000, "cube1", 1)
    with F.FMM(P=10) as a, F.FMM(P=8) as b:
        plan = F.Plan(x, lists_on=a)
        b.set_bodies_plan(plan, q)
        b.evaluate()
        t = b.targets()
        plan.prepare(P=8)
        b.set_bodies_plan(plan, q)
        b.evaluate()
        t2 = b.targets()
        b.set_bodies(x, q)
        b.evaluate()
        r = b.targets()
    for v in (t, t2):
        assert np.all(np.linalg.norm(v - r, axis=0) <= 1e-12 * np.linalg.norm(r, axis=0))


def _multipoles(x, q, t, P):
    """every cell's multipole from its bodies (extended precision)"""
    LD, CL = np.longdouble, np.clongdouble
    M = np.zeros((len(t["R"]), P * (P + 1) // 2), CL)
    xs, qs = x[t["perm"]].astype(LD), q[t["perm"]].astype(LD)
    for c, (b, n) in enumerate(zip(t["ibody"], t["nbody"])):
        dx, dy, dz = (xs[b:b + n] - t["X"][c].astype(LD)).T
        r2 = dx * dx + dy * dy + dz * dz
        rmm = np.ones(n, CL)
        for m in range(P):
            if m > 0:
                rmm = rmm * (dx + 1j * dy) * (-LD(1) / (2 * m))
            r0, r1 = np.zeros(n, CL), rmm
            for k in range(m, P):
                if k > m:
                    r0, r1 = r1, (r1 * (2 * k - 1) * dz - r0 * r2) / LD(k * k - m * m)
                s = np.sqrt(LD(math.factorial(k - m)) * LD(math.factorial(k + m)))
                M[c, k * (k + 1) // 2 + m] = (qs[b:b + n] * np.conj(r1)).sum() * s
    return M


@pytest.mark.parametrize("P", range(2, 13))
@pytest.mark.parametrize("n,ncrit", [(90, 8), (2999, 16)])
def test_m2m_l2l_every_order(P, n, ncrit):
    """M2M and L2L by rotation: multipoles of every cell against its bodies'
    (a cell's own P2M; the scalar M2M kernel itself is 1.1e-12 from them at
    P = 12), local expansions against the scalar L2L, which the same tree given
    by the caller takes with one radius a part in 1e12 off.  FP64 sums chained
    over at most 6 levels: 1e-12 per degree."""
    F = _F()
    x, q = F.make_bodies(n, "plummer1", P)
    out = []
    with F.FMM(P=P, theta=0.5, ncrit=ncrit, m2l_mode=F.M2L_TARGET) as f:
        f.set_bodies(x, q)
        t = f.tree()
        for scale in (1.0, 1.0 + 1e-12):
            R = t["R"].copy()
            R[-1] *= scale
            f.set_tree(x[t["perm"]], q[t["perm"]], {**t, "R": R})
            f.upward()
            f.m2l()
            f.downward()
            f.synchronize()
            out.append((f.expansions(), f.lists()))
    assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))
    M = _multipoles(x, q, t, P)
    for a, b in ((out[0][0][0], M), (out[0][0][1], out[1][0][1])):
        for k in range(P):
            u = slice(k * (k + 1) // 2, (k + 1) * (k + 2) // 2)
            assert np.linalg.norm(a[:, u] - b[:, u]) <= 1e-12 * np.linalg.norm(b[:, u]), k


@pytest.mark.parametrize("cycle", [1.0, (1.0, 1.5, 2.0)])
def test_periodic_groups_on_the_device(cycle):
    """the offset classes of periodic lists, built on the device: every image,
    a rectangular cycle, the far images' operator added at images = 2"""
    F = _F()
    rng = np.random.default_rng(5)
    c = np.broadcast_to(np.asarray(cycle), (3,))
    x = (rng.random((2003, 3)) - 0.5) * c
    q = rng.random(2003) - 0.5
    q -= q.mean()
    _check(F, x, q, P=7, theta=0.5, ncrit=20, images=1, cycle=cycle)
    _check(F, x, q, P=10, theta=0.4, ncrit=50, images=2, cycle=cycle)


@pytest.mark.parametrize("n,theta,ncrit", [(24, 0.5, 1), (500, 0.5, 8), (20000, 0.3, 64)])
def test_group_numbering(n, theta, ncrit):
    """Groups and classes numbered on the device, from a few to thousands of
    distinct offsets over a table of 2^20 slots: as many as the host finds."""
    F = _F()
    x, q = F.make_bodies(n, "plummer1", n)
    _check(F, x, q, P=4, theta=theta, ncrit=ncrit)
    st = {}
    for mode in (F.M2L_TILES, F.M2L_GROUPED):
        with F.FMM(P=4, theta=theta, ncrit=ncrit, m2l_mode=mode) as f:
            f.set_bodies(x, q)
            st[mode] = f.stats()["m2l_groups"]
    assert st[F.M2L_TILES] == st[F.M2L_GROUPED] > 1
