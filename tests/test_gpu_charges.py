"""fmm_set_charges on both sides of the size where the host stops putting the
charges into tree order: the solve that follows is that of a context given the
bodies with those charges (1e-13: the order of atomic additions), called again
and again without a wait between the calls, and replayed from a captured graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 1000, 32767, 32768, 32769, 70001])
def test_new_charges(n):
    import exafmm_amd as F
    x, q = F.make_bodies(n, "plummer1", 5)
    rng = np.random.default_rng(n)
    qs = [rng.standard_normal(n) for _ in range(3)]
    with F.FMM(P=5) as f, F.FMM(P=5) as g:
        f.set_bodies(x, q)
        for graph in (False, True):
            f.evaluate(graph=graph)
            for c in qs:
                f.set_charges(np.zeros(n))
                f.set_charges(c)
                f.evaluate(graph=graph)
                g.set_bodies(x, c)
                g.evaluate()
                a, b = f.targets(), g.targets()
                assert np.linalg.norm(a[:, 0] - b[:, 0]) <= 1e-13 * np.linalg.norm(b[:, 0])
                assert np.linalg.norm(a[:, 1:] - b[:, 1:]) <= 1e-13 * np.linalg.norm(b[:, 1:])
