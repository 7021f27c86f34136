"""The Ewald sum at the sizes where its kernels change: one body, the edges of a
wavefront and of the tiles of 1024 sources, cutoffs that list none, some and
all of the sources, a box of three lengths, bodies outside the box, coincident
bodies.  Against the same sums in numpy, wave vectors and the C library's erfc.
A term carries a few roundings (its phase up to |k.x| < 40 of them, 1e-14 of
the term), so every result lies within 1e-13 of the sum of its terms'
magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(x, q, ksize, alpha, sigma, cutoff, L):
    from scipy.special import erfc
    x = np.where(x < -L / 2, x + L, x)
    x = np.where(x > L / 2, x - L, x)
    d = x[:, None] - x[None]
    d = np.where(d < -L / 2, d + L, d)
    d = np.where(d > L / 2, d - L, d)
    r2 = (d * d).sum(2)
    r2 = np.where((r2 > 0) & (r2 < cutoff * cutoff), r2, np.inf)
    s = np.sqrt(r2) * alpha
    pt = q * erfc(s) / s * alpha
    w = q * (2 / np.sqrt(np.pi) * np.exp(-s * s) / s ** 2 + erfc(s) / s ** 3) * alpha ** 3
    self_ = 2 / np.sqrt(np.pi) * q * alpha
    out = np.column_stack([pt.sum(1) - self_, -(np.where(np.isinf(r2)[..., None], 0, d) * w[..., None]).sum(1)])
    mag = np.column_stack([abs(pt).sum(1) + abs(self_),
                           (np.where(np.isinf(r2)[..., None], 0, abs(d)) * abs(w)[..., None]).sum(1)])
    r = range(-ksize, ksize + 1)
    kv = np.array([(a, b, c) for a in range(ksize + 1) for b in r for c in r
                   if 0 < a * a + b * b + c * c <= ksize * ksize and (a > 0 or b > 0 or (b == 0 and c > 0))], float)
    for k in kv * (2 * np.pi / L):
        k2 = k @ k
        f = 2 / sigma / np.prod(L) * np.exp(-k2 / (4 * alpha * alpha)) / k2
        e = np.exp(1j * (x @ k))
        S = (q * e).sum() * f
        z = e.conj() * S
        out[:, 0] += z.real
        out[:, 1:] += z.imag[:, None] * k
        m = abs(q).sum() * f
        mag[:, 0] += m
        mag[:, 1:] += m * abs(k)
    return out, mag


@pytest.mark.parametrize("n", [1, 3, 63, 65, 1023, 1025, 2050])
@pytest.mark.parametrize("cut", [1e-3, 0.2, 0.5, 0.9])
def test_ewald_against_numpy(n, cut):
    import exafmm_amd as F
    rng = np.random.default_rng(n)
    L = np.array([3.0, 4.0, 5.0]) if cut == 0.2 else np.array([3.0, 3.0, 3.0])
    x = (rng.random((n, 3)) * 1.2 - 0.6) * L
    q = rng.random(n) - 0.5
    if n > 3:
        x[n // 2] = x[1]
    args = (5, 1.3, 0.25 / np.pi, cut * L.min())
    with F.FMM(P=4, images=1, cycle=tuple(L)) as f:
        p, g = f.ewald(x, q, *args)
    ref, mag = _reference(x, q, *args, L)
    assert np.all(abs(np.column_stack([p, g]) - ref) <= 1e-13 * mag)
