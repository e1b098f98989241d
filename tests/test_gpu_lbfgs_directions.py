"""GPU: every direction of the device L-BFGS against the two-loop recursion of
the run's own iterates on the host, from sizes of one wave's work to many blocks.

Three minimisations on one context, so that the ten history slots come round at
every position.  Tolerance 1e-8: both sides form at most 20 products of n <= 2e5
terms, each to n eps = 4e-11 of the sum of its terms' magnitudes; a pair that is
lost or held twice changes a direction by far more than 1e-3.  The values fall
(sufficient decrease), and a run without a callback, whose history updates share
the directions' launches, gives the same bits.
"""
import numpy as np
import pytest

import cosmopp_amd as cm
from cases import Case

pytestmark = pytest.mark.gpu

M = 10


def download(ptr, n):
    out = np.empty(n)
    assert cm.lib().cmbl_copy_to_host(out.ctypes.data, ptr, n * 8) == 0
    return out


def recursion(g, S, Y):
    """Two-loop recursion, newest pair first."""
    if not S:
        return g.copy()
    q, alpha = g.copy(), []
    for s, y in zip(S, Y):
        alpha.append(s @ q / (s @ y))
        q -= alpha[-1] * y
    z = (S[0] @ Y[0]) / (Y[0] @ Y[0]) * q
    for s, y, a in zip(S[::-1], Y[::-1], alpha[::-1]):
        z += (a - y @ z / (s @ y)) * s
    return z


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("nside,lmax", [(2, 7), (64, 55), (128, 256), (512, 432)])
def test_directions(nside, lmax, graphs):
    import torch

    print("case lbfgs directions", nside, lmax, graphs, flush=True)
    c = Case(nside, lmax, 5400.0 / lmax / 60.0, 20.0, 20.0, seed=nside + lmax)
    mp = c.make_map()
    n = c.x.size
    x0 = torch.from_numpy(c.x).to("cuda:0")
    res = torch.empty_like(x0)
    lb = cm.LBFGS(mp, x0.data_ptr(), m=M, graphs=graphs)
    ends = []
    for run in range(3):
        seen = []

        def step(i, f, gn, x, g, z):
            seen.append((f, download(x, n), download(g, n), download(z, n) if i else None))

        lb.set_starting(x0.data_ptr())
        f, its, _ = lb.minimize(res.data_ptr(), epsilon=1e-30, gnorm_tol=1e-30, max_iter=12, callback=step)
        assert len(seen) == its + 1 >= 13
        S, Y = [], []
        for (f0, xa, ga, _), (f1, xb, gb, z) in zip(seen, seen[1:]):
            assert f1 < f0
            want = recursion(ga, S, Y)
            assert np.linalg.norm(z - want) <= 1e-8 * np.linalg.norm(want)
            S, Y = [xb - xa] + S[:M - 1], [gb - ga] + Y[:M - 1]
        ends.append((f, res.cpu().numpy()))
        lb.set_starting(x0.data_ptr())
        f, _, _ = lb.minimize(res.data_ptr(), epsilon=1e-30, gnorm_tol=1e-30, max_iter=12)
        ends.append((f, res.cpu().numpy()))
    for f, x in ends[1:]:
        assert f == ends[0][0] and np.array_equal(x, ends[0][1])
    lb.close()
    mp.close()


@pytest.mark.parametrize("side", [False, True])
def test_set_starting_waits_for_the_callers_stream(side):
    """A point still being written on the caller's stream: the value at the start
    is that of the finished point."""
    import torch

    print("case lbfgs set_starting in flight", side, flush=True)
    c = Case(16, 32, 5400.0 / 32 / 60.0, 20.0, 20.0, seed=5)
    mp = c.make_map()
    want, _ = mp.value_and_grad(c.x)
    x1 = torch.from_numpy(c.x).to("cuda:0")
    x0 = torch.zeros_like(x1)
    lb = cm.LBFGS(mp, x0.data_ptr(), m=M)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.current_stream()):
        torch.cuda._sleep(20_000_000)  # about 10 ms
        x0.copy_(x1)
        lb.set_starting(x0.data_ptr())
    assert lb.state()["f"] == want
    lb.close()
    mp.close()
