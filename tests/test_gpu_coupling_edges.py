"""GPU: the coupling matrix at the edges of its blocks (4 distances l1 - l2, 256
degrees, 16 steps) against the oracle, and which entries a non-finite W_l3
reaches (those of its own triangles).

Tolerance 1e-12 for the whole matrix as for the other sizes; the sums have
positive terms only, each within a few roundings, so single entries keep it too.
"""
import numpy as np
import pytest

import cosmopp_amd as cm
import oracle

pytestmark = pytest.mark.gpu


def w3j2_table(L):
    """oracle.w3j2_table in extended precision (its differences of log-gammas of
    size 5e3 keep 1e-12 only): h(a) h(b) h(c) / ((2g+1) h(g)), h(n) = (2n)!/(4^n n!^2)."""
    n = np.arange(1, 2 * L + 2, dtype=np.longdouble)
    h = np.concatenate([[np.longdouble(1)], np.cumprod((2 * n - 1) / (2 * n))])
    out = np.zeros((L + 1,) * 3)
    l2, l3 = np.meshgrid(np.arange(L + 1), np.arange(L + 1), indexing="ij")
    for l1 in range(L + 1):
        ok = ((l1 + l2 + l3) % 2 == 0) & (l3 >= abs(l1 - l2)) & (l3 <= l1 + l2)
        g = (l1 + l2[ok] + l3[ok]) // 2
        out[l1][ok] = h[g - l1] * h[g - l2[ok]] * h[g - l3[ok]] / ((2 * g + 1) * h[g])
    return out


@pytest.mark.parametrize("lmax", [0, 1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 33, 255, 256, 257, 300])
def test_coupling_block_edges(lmax):
    print("case coupling edges", lmax, flush=True)
    rng = np.random.default_rng(lmax)
    w = np.abs(rng.standard_normal(lmax + 1)) / (1.0 + np.arange(lmax + 1)) ** 2
    got, want = cm.coupling_matrix(w, lmax), oracle.coupling(w, lmax, table=w3j2_table(lmax))
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=0)


@pytest.mark.parametrize("lmax,l3", [(40, 0), (40, 7), (300, 290)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_coupling_non_finite(lmax, l3, bad):
    print("case coupling non-finite", lmax, l3, bad, flush=True)
    w = 1.0 / (1.0 + np.arange(lmax + 1))
    clean = cm.coupling_matrix(w, lmax)
    w[l3] = bad
    got = cm.coupling_matrix(w, lmax)
    l = np.arange(lmax + 1)
    l1, l2 = l[:, None], l[None, :]
    hit = (abs(l1 - l2) <= l3) & (l3 <= l1 + l2) & ((l1 + l2 + l3) % 2 == 0)
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit], clean[~hit])
