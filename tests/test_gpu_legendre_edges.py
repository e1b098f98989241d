"""GPU: the Legendre stages at the edges of their blocks (synthesis: 16 l-steps
from an item's first l; adjoint: rows of eight, 64-pair groups joining at their
own rows, segments; matrix-core tiles of 32) against the oracle.

Tolerance 1e-10, the framework's bar: both sides run about lmax rounded steps
per l in FP64, 1e-16 each, over at most 400 of them."""
import numpy as np
import pytest

import cosmopp_amd as cm
import oracle
from cases import Case

pytestmark = pytest.mark.gpu


def make_map(c, k_synth, k_adj):
    mp = cm.Map(c.nside, c.lmax, tuning=(k_synth, k_adj, 4096))
    mp.set_beam(c.beam)
    mp.set_cl(c.cl)
    mp.set_data(c.d, c.w)
    return mp


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(b), 1e-300)


# lmax about multiples of 8, 16 and 32, and 4 nside; one 64-pair block and less,
# several blocks, a partial last block of K = 8
@pytest.mark.parametrize("nside,lmax", [(1, 2), (1, 4), (2, 7), (4, 8), (8, 15), (8, 31), (16, 16), (16, 17),
                                        (32, 128), (64, 33), (128, 145), (128, 400), (256, 130)])
@pytest.mark.parametrize("k_synth,k_adj", [(1, 1), (2, 8), (4, 2), (8, 4)])
def test_block_edges(nside, lmax, k_synth, k_adj):
    print("case edges", nside, lmax, k_synth, k_adj, flush=True)
    c = Case(nside, lmax, 5400.0 / lmax / 60.0, 20.0, 20.0, seed=nside + lmax)
    mp = make_map(c, k_synth, k_adj)
    f, g = mp.value_and_grad(c.x)
    fo, go = oracle.neg2lnL(c.nside, c.lmax, c.x, c.beam, c.cl, c.d, c.w)
    assert abs(f - fo) < 1e-10 * abs(fo)
    assert rel(g, go) < 1e-10
    mp.close()


# a pair; a pair and a single map; a partial group; a full group with a pair; two
# full groups with a single map
@pytest.mark.parametrize("nmaps", [2, 3, 6, 10, 17])
@pytest.mark.parametrize("nside,lmax,k_synth", [(8, 31, 1), (64, 65, 2), (128, 145, 1)])
def test_batch_groups(nmaps, nside, lmax, k_synth):
    import torch

    print("case groups", nmaps, nside, lmax, k_synth, flush=True)
    cases = [Case(nside, lmax, 5400.0 / lmax / 60.0, 10.0 + i, 12.0, seed=31 * i + nmaps) for i in range(nmaps)]
    maps = [make_map(c, k_synth, 1) for c in cases]
    dev = torch.device("cuda:0")
    xs = [torch.from_numpy(c.x).to(dev) for c in cases]
    gs = [torch.empty_like(x) for x in xs]
    f = torch.empty(nmaps, dtype=torch.float64, device=dev)
    b = cm.Batch(maps)
    b.value_and_grad_device([x.data_ptr() for x in xs], f.data_ptr(), [g.data_ptr() for g in gs],
                            torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for i, c in enumerate(cases):
        fo, go = oracle.neg2lnL(c.nside, c.lmax, c.x, c.beam, c.cl, c.d, c.w)
        assert abs(f[i].item() - fo) < 1e-10 * abs(fo)
        assert rel(gs[i].cpu().numpy(), go) < 1e-10
    b.close()
    for mp in maps:
        mp.close()


# the spin-2 synthesis at the same edges, each tuning's item split into blocks
@pytest.mark.parametrize("nside,lmax,k_synth", [(1, 2, 1), (2, 8, 2), (16, 17, 1), (64, 33, 4), (128, 144, 8)])
def test_pol_edges(nside, lmax, k_synth):
    print("case pol edges", nside, lmax, k_synth, flush=True)
    rng = np.random.default_rng(nside + lmax)
    t, e, b = (rng.standard_normal((lmax + 1) ** 2) for _ in range(3))
    mp = cm.Map(nside, lmax, tuning=(k_synth, 1, 4096))
    for got, want in zip(mp.alm2map_pol(t, e, b), oracle.alm2map_pol(nside, lmax, t, e, b)):
        assert rel(got, want) < 1e-10
    mp.close()


# the rest of a batch beside a full matrix-core group: one map up to nside 128 and
# three at nside 256 form a group of their own, fewer and larger maps do not
@pytest.mark.parametrize("nside,lmax,nmaps", [(64, 65, 9), (128, 100, 11), (256, 130, 10), (256, 130, 11), (512, 60, 13),
                                              (512, 60, 14)])
def test_batch_rest_beside_a_group(nside, lmax, nmaps):
    import torch

    print("case rest", nside, lmax, nmaps, flush=True)
    cases = [Case(nside, lmax, 5400.0 / lmax / 60.0, 10.0 + i, 12.0, seed=17 * i + nmaps) for i in range(nmaps)]
    maps = [make_map(c, 1, 1) for c in cases]
    xs = [torch.from_numpy(c.x).to("cuda:0") for c in cases]
    gs = [torch.empty_like(x) for x in xs]
    f = torch.empty(nmaps, dtype=torch.float64, device="cuda:0")
    b = cm.Batch(maps)
    b.value_and_grad_device([x.data_ptr() for x in xs], f.data_ptr(), [g.data_ptr() for g in gs],
                            torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for i in (0, 7, 8, nmaps - 1):
        c = cases[i]
        fo, go = oracle.neg2lnL(c.nside, c.lmax, c.x, c.beam, c.cl, c.d, c.w)
        assert abs(f[i].item() - fo) < 1e-10 * abs(fo)
        assert rel(gs[i].cpu().numpy(), go) < 1e-10
    b.close()
    for mp in maps:
        mp.close()


# batches whose maps share no geometry, on both sides of the lines between 2, 4 and 8
# ring pairs per lane, against the maps one by one
@pytest.mark.parametrize("sizes", [[(64, 130), (128, 133), (256, 300)], [(64, 130), (512, 520), (8, 20)],
                                   [(256, 140), (128, 60)], [(512, 900)], [(32, 64), (512, 1500), (512, 1400)]])
def test_batch_ring_pairs_per_lane(sizes):
    import torch

    print("case ring pairs", sizes, flush=True)
    cases = [Case(n, l, 5400.0 / l / 60.0, 10.0 + n, 12.0, seed=n + l) for n, l in sizes]
    maps = [make_map(c, 1, 1) for c in cases]
    xs = [torch.from_numpy(c.x).to("cuda:0") for c in cases]
    gs = [torch.empty_like(x) for x in xs]
    f = torch.empty(len(maps), dtype=torch.float64, device="cuda:0")
    b = cm.Batch(maps)
    b.value_and_grad_device([x.data_ptr() for x in xs], f.data_ptr(), [g.data_ptr() for g in gs],
                            torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for i, (c, mp) in enumerate(zip(cases, maps)):
        fo, go = mp.value_and_grad(c.x)
        assert abs(f[i].item() - fo) < 1e-10 * abs(fo)
        assert rel(gs[i].cpu().numpy(), go) < 1e-10
    b.close()
    for mp in maps:
        mp.close()
