"""The lists of fmm_set_bodies walked on the device (trees of many cells): the
same pairs, in the same order, as the host's recursive walk of the same tree
(which an adopted tree takes).  Single and double splits, the order of a split
of up to 8 x 8 children, sorted and uneven trees, and the 27 periodic images;
all whole numbers, so they are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(F, dist, n):
    if dist != "line":
        return F.make_bodies(n, dist, 5)
    rng = np.random.default_rng(n)  # cells with few children, deep
    x = rng.random((n, 3)) * [1.0, 1e-3, 1e-3]
    x[: n // 2, 0] = x[: n // 2, 0] ** 4
    return x, rng.random(n) - 0.5


@pytest.mark.parametrize("dist,n,theta,ncrit,nspawn,images", [
    ("cube1", 20000, 0.4, 8, 5000, 0),
    ("cube1", 9000, 0.6, 1, 1, 0),
    ("plummer1", 30000, 0.35, 16, 1000000, 0),
    ("plummer1", 30011, 0.5, 7, 64, 0),
    ("line", 20000, 0.4, 4, 1000, 0),
    ("cube1", 9001, 0.4, 4, 5000, 1),
    ("plummer1", 12000, 0.5, 6, 100, 2),
])
def test_lists_in_the_host_order(dist, n, theta, ncrit, nspawn, images):
    import exafmm_amd as F
    x, q = _bodies(F, dist, n)
    kw = dict(P=4, theta=theta, ncrit=ncrit, nspawn=nspawn)
    if images:
        kw.update(images=images, cycle=float(2 * abs(x).max()))
    with F.FMM(**kw) as f, F.FMM(**kw) as h:
        f.set_bodies(x, q)
        t = f.tree()
        h.set_tree(x[t["perm"]], q[t["perm"]], t)
        assert f.stats()["ncell"] >= 600
        for k in ("m2l_pairs", "p2p_pairs", "p2p_body_pairs"):
            assert f.stats()[k] == h.stats()[k] > 0, k
        for a, b in zip(f.lists(), h.lists()):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("dist,n,ncrit,images", [("cube1", 50000, 64, 0), ("plummer1", 50021, 10, 0),
                                                 ("line", 60000, 32, 0), ("plummer1", 50000, 64, 1)])
def test_tree_of_many_bodies(dist, n, ncrit, images):
    """From 50000 bodies the tree of fmm_set_bodies is built on the device too:
    the host's cells, numbers and body order, and its lists."""
    import exafmm_amd as F
    x, q = _bodies(F, dist, n)
    x[7] = x[5]
    kw = dict(images=images, cycle=float(2 * abs(x).max())) if images else {}
    h = F.Plan(x, ncrit=ncrit, theta=0.5)
    with F.FMM(P=4, theta=0.5, ncrit=ncrit, **kw) as f:
        f.set_bodies(x, q)
        a, b = f.tree(), h.tree()
        for k in ("perm", "iparent", "ichild", "nchild", "ibody", "nbody", "X", "R"):
            assert np.array_equal(a[k], b[k]), k
        if not images:
            for u, v in zip(f.lists(), h.lists()):
                assert np.array_equal(u, v)
