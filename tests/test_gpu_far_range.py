"""Far images at the smallest theta they take: supercells of 2 x 17 + 1 boxes a
side (35^6 offsets, which an int still counts).  One charge's potential is the
sum of 1 / |w| over its images: 26 near ones and those of the cube |w| <= 17 x
35 + 17 = 612 without |w| <= 17, which the integral of 1 / r over the cubes
gives to 1e-5 (8 x 1.19003868 a^2 for a cube of half side a; the midpoint rule
of a harmonic function errs at the inner faces only, 2e-6 there).  Below that
theta bodies are refused, whatever the size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

X, Q = np.zeros((1, 3)), np.ones(1)


def test_largest_range():
    import exafmm_amd as F
    with F.FMM(P=2, theta=0.0296, images=2, cycle=1.0) as f:
        f.set_bodies(X, Q)
        f.evaluate()
        pot = f.targets()[0, 0]
    near = 6 + 12 / np.sqrt(2) + 8 / np.sqrt(3)
    assert abs(pot - near - 8 * 1.19003868 * (612.5 ** 2 - 17.5 ** 2)) < 1e-5 * pot


# 2 prange + 1 = 37 (its sixth power wraps an int to a negative number), 53 and 63 (to positive ones)
@pytest.mark.parametrize("theta", [0.0294, 0.02, 0.0165, 1e-4, 1e-12])
def test_smaller_theta_is_refused(theta):
    import exafmm_amd as F
    xs, qs = F.make_bodies(300, "cube1", 1)
    with F.FMM(P=4, theta=theta, images=2, cycle=8.0) as f, F.FMM(P=4, theta=theta, images=1, cycle=8.0) as g:
        for x, q in ((X, Q), (xs, qs)):
            with pytest.raises(F.FMMError, match="theta"):
                f.set_bodies(x, q)
            with pytest.raises(F.FMMError, match="theta"):
                f.md_evaluate(x, q)
        f.set_bodies(np.zeros((0, 3)), np.zeros(0))  # no images to sum
        g.set_bodies(X, Q)  # nor with the 27 near ones alone
        g.evaluate()
        assert np.isfinite(g.targets()).all()
