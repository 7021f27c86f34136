"""P2P with one and with four wavefronts a leaf (by the number of leaves): a
system alone (few leaves) and in a forest of more than 12000 leaves, at leaf
sizes on both sides of the kernel's bounds (16 bodies: targets per lane; 256:
more than one pass over the targets; lists of less and more than a window of
64 entries and a chunk of 256 bodies).  The same sums in another order: FP64
rounding, 1e-13 (the FP32 partial sums of the mixed kernel are the same)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ncrit", [(1, 8), (40, 64), (700, 8), (3001, 24), (6000, 400)])
@pytest.mark.parametrize("prec", [0, 1])
def test_wavefronts_per_leaf(n, ncrit, prec):
    import exafmm_amd as F
    x, q = F.make_bodies(n, "plummer1", n)
    fx, fq = F.make_bodies(80000, "cube1", 3)
    filler = F.Plan(fx, ncrit=4)
    assert filler.stats()["nleaf"] > 12000
    plan = F.Plan(x, ncrit=ncrit)
    with F.FMM(P=4, precision=prec) as f:
        out = []
        for p, c in ((plan, q), (F.Plan.merge([plan, filler]), np.concatenate([q, fq]))):
            f.set_bodies_plan(p, c)
            f.p2p()
            out.append(f.targets()[:n])
    assert np.any(out[0]) or n == 1
    assert np.all(np.linalg.norm(out[0] - out[1], axis=0) <= 1e-13 * np.linalg.norm(out[0], axis=0))
