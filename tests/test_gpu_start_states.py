"""GPU: the start states of the adjoint's segments, through the m = 0 spectra of
single polar rings against extended precision.

Near a pole the recurrence amplifies a step's rounding by min(l, 1 / theta).  Its
result and its product are rounded once per step, together 0.8 2^-53 (rms), so L
steps leave at most about 2^-53 sqrt(L) min(L, 1 / theta).  A drift of x^2 = cos^2
theta in the states, rounding by rounding the same, grows with l instead:
sqrt(L) / 3.5 times that bound at l = L.
"""
import numpy as np
import pytest

import cosmopp_amd as cm

pytestmark = pytest.mark.gpu


def legendre_m0(x, L):
    """lambda_l0(x), l = 0 .. L, in extended precision."""
    x = np.longdouble(x)
    p = [np.longdouble(1), x]
    for l in range(2, L + 1):
        p.append(((2 * l - 1) * x * p[-1] - (l - 1) * p[-2]) / l)
    l = np.arange(L + 1, dtype=np.longdouble)
    return np.array(p) * np.sqrt((2 * l + 1) / (4 * np.longdouble(np.pi)))


@pytest.mark.parametrize("nside,lmax", [(256, 700), (512, 1000)])
def test_polar_rings(nside, lmax):
    print("case start states", nside, lmax, flush=True)
    mp = cm.Map(nside, lmax)
    npix = 12 * nside * nside
    rng = np.random.default_rng(nside)
    l = np.arange(lmax + 1)
    ratio = []
    for i in range(2, 34):  # ring i: 4 i pixels from 2 i (i - 1)
        v = np.zeros(npix)
        ring = slice(2 * i * (i - 1), 2 * i * (i + 1))
        v[ring] = 1.0 + rng.random(4 * i)
        got = mp.map2alm_quadrature(v)[l * l]
        x = 1.0 - i * i / (3.0 * nside * nside)
        want = legendre_m0(x, lmax) * v[ring].astype(np.longdouble).sum() * (4 * np.longdouble(np.pi) / npix)
        err = np.linalg.norm((got - want).astype(float)) / np.linalg.norm(want.astype(float))
        ratio.append(err / (2.0**-53 * np.sqrt(lmax) * min(lmax, 1.0 / np.arccos(x))))
    rms = float(np.sqrt(np.mean(np.square(ratio))))
    print("rms error over its bound %.2f, largest %.2f" % (rms, max(ratio)), flush=True)
    assert rms < 1.0
    mp.close()
