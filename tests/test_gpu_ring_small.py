"""GPU: the ring stage of small maps (all transforms at most 1024 points) in its
four modes against the oracle: power-of-two rings from 4 samples, Bluestein
lengths 32 to 1024 (even and odd powers of two), rings shorter and longer than
the workgroup, aliased bins.

Tolerance 1e-10, the framework's bar; a transform's rounding is of the order of
1e-16 log2 of its length.
"""
import numpy as np
import pytest

import cosmopp_amd as cm
import oracle
from cases import Case
from test_gpu_gibbs import problem, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside", [1, 2, 4, 8, 16, 32, 64, 128])
@pytest.mark.parametrize("ratio", [1, 3, 4])
def test_ring_modes(nside, ratio):
    lmax = max(2, ratio * nside)
    print("case ring small", nside, lmax, flush=True)
    c = Case(nside, lmax, 5400.0 / lmax / 60.0, 20.0, 20.0, seed=nside + lmax)
    mp = c.make_map()
    assert rel(mp.forward(c.x), oracle.synthesis(nside, lmax, c.x, c.beam)) < 1e-10
    f, g = mp.value_and_grad(c.x)
    fo, go = oracle.neg2lnL(nside, lmax, c.x, c.beam, c.cl, c.d, c.w)
    assert abs(f - fo) < 1e-10 * abs(fo)
    assert rel(g, go) < 1e-10
    assert rel(mp.map2alm_quadrature(c.d), oracle.quadrature(nside, lmax, c.d)) < 1e-10
    mp.close()
    rng, cl, beam, mask, sigma = problem(nside, lmax, nside + lmax)
    gb = cm.Gibbs(nside, lmax, cl, beam, mask, sigma)
    x = rng.standard_normal((lmax + 1) ** 2)
    assert rel(gb.multiply_by_matrix(x), oracle.gibbs_apply(nside, lmax, x, cl, beam, mask, sigma)) < 1e-10
    gb.close()
