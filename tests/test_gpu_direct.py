"""The direct sum at the edges of its blocks (64 targets) and source runs (a
multiple of 256 bodies, split when few targets leave the GPU idle), against an
extended-precision sum.  FP64 sums of n terms in runs of at most a few
thousand: within 1e-13 of the sum of the terms' magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nt", [(1, 1), (3, 200), (255, 63), (257, 65), (4096, 64), (70001, 1), (20000, 129)])
def test_direct_blocks_and_runs(n, nt):
    import exafmm_amd as F
    rng = np.random.default_rng(n)
    x, q = rng.random((n, 3)), rng.random(n) - 0.5
    xt = np.concatenate([x[:nt], rng.random((max(0, nt - n), 3)) + 0.25])  # sources themselves first
    with F.FMM(P=4) as f:
        f.set_bodies(x, q)
        got = f.direct(xt)
        again = f.direct(xt[: (nt + 1) // 2])
    X, Q = x.astype(np.longdouble), q.astype(np.longdouble)
    for i in range(nt):
        d = xt[i].astype(np.longdouble) - X
        r2 = (d * d).sum(1)
        k = r2 > 0
        w = Q[k] / np.sqrt(r2[k])
        g = -d[k] * (w / r2[k])[:, None]
        assert abs(got[i, 0] - w.sum()) <= 1e-13 * max(abs(w).sum(), 1e-300)
        assert np.all(abs(got[i, 1:] - g.sum(0)) <= 1e-13 * np.maximum(abs(g).sum(0), 1e-300))
    assert np.allclose(again, got[: (nt + 1) // 2], rtol=1e-11, atol=1e-11)
