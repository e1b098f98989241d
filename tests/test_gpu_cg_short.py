"""GPU: the Gibbs solve at the sizes where its vector work changes form: one
element to one wave, one block's 256, 1024, the last size that one workgroup
holds (4096 = 64^2) and the first that it does not.

Both solves stop at |r| <= 1e-9 |b|; tolerances as for the other solves.
"""
import numpy as np
import pytest

import cosmopp_amd as cm
import oracle
from test_gpu_gibbs import problem, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside,lmax", [(2, 2), (4, 7), (8, 15), (16, 31), (16, 32), (32, 63), (32, 64)])
def test_gibbs_solve_sizes(nside, lmax):
    print("case gibbs sizes", nside, lmax, flush=True)
    rng, cl, beam, mask, sigma = problem(nside, lmax, 3 * nside + lmax)
    npix = 12 * nside * nside
    g = cm.Gibbs(nside, lmax, cl, beam, mask, sigma)
    b = g.rhs(rng.standard_normal(npix) * 30.0, rng.standard_normal(npix), rng.standard_normal(npix))
    prec = 1e-9 * np.linalg.norm(b)
    x, it = g.solve(b, precision=prec)
    xo, ito = oracle.cg_solve(lambda v: oracle.gibbs_apply(nside, lmax, v, cl, beam, mask, sigma),
                              lambda v: oracle.gibbs_precondition(lmax, v, cl, beam, mask, sigma), b, precision=prec)
    assert abs(it - ito) <= 2
    assert rel(x, xo) < 1e-8
    # a second solve on the same context gives the same iterates
    x2, it2 = g.solve(b, precision=prec)
    assert it2 == it and np.array_equal(x, x2)
    g.close()
