"""The backward at every kind of step count: fewer steps than a group of 8, whole
groups, a partial group, both register capacities (64 and 104 steps) up to the
step cap, with full LDS bins, the LDS cell cache (2D [48, 48]) and rows beyond
the recovery bound; the image and chain backwards, which keep other bins, at step
counts of the trail body; and adaptive substeps, whose step counts other than 50
take the segmented body; against the oracle at the tolerances of the other
backward tests."""
import numpy as np
import pytest
import torch

from cpab.pytorch._native import native
from oracle import oracle as orc

from helpers import (assert_adjoint_close, assert_grad_close, cpab_for, meshgrid, seeded_theta,
                     uniform_points)
from test_gpu_kernels import _As_gpu, _backward_case, _dev, _image_order

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nstep", [1, 5, 7, 8, 9, 16, 63, 64, 65, 96, 97, 100])
@pytest.mark.parametrize("tess", [[7], [4, 3], [3, 4, 2]])
def test_backward_step_counts(cuda, tess, nstep):
    _check(tess, nstep, 1500, 0.5, cuda)


@pytest.mark.parametrize("tess,nstep,n,scale", [([48, 48], 50, 9000, 0.5), ([48, 48], 66, 3000, 0.5),
                                                ([10, 10, 10], 70, 3000, 0.5), ([20, 20], 20, 3000, 6.0),
                                                ([50], 13, 3000, 10.0), ([4, 4, 4], 90, 2000, 6.0),
                                                # bins of doubles without the reverse table, float bins
                                                ([22, 22], 50, 9000, 0.5), ([32, 32], 50, 9000, 0.5),
                                                ([32, 32], 30, 3000, 0.5), ([7, 7, 7], 50, 3000, 0.5)])
def test_backward_step_counts_cache_and_strong(cuda, tess, nstep, n, scale):
    _check(tess, nstep, n, scale, cuda)


@pytest.mark.parametrize("tess,nstep,n,scale", [([30, 30], 1, 3000, 0.5), ([30, 30], 4, 20000, 0.5),
                                                ([30, 30], 5, 20000, 0.5), ([41, 41], 8, 3000, 0.5),
                                                ([41, 41], 9, 3000, 0.5), ([36, 36], 3, 3000, 6.0),
                                                ([20, 20], 3, 3000, 0.5), ([20, 20], 8, 16384, 0.5),
                                                ([20, 20], 8, 16385, 0.5), ([19, 19], 1, 3000, 0.5),
                                                ([18, 18], 1, 3000, 0.5), ([48, 48], 5, 3000, 6.0)])
def test_backward_few_steps_large_table(cuda, tess, nstep, n, scale):
    # the segmented body without adaptive substeps, and both sides of its line
    _check(tess, nstep, n, scale, cuda)


def test_backward_rounding_many_tables(cuda):
    # one row over as many workgroups as there are compute units, each with a table of
    # its own: their sum takes one rounding, not one for each table
    _check_rounding([50], 1, 1, 60000, cuda)


@pytest.mark.parametrize("nstep", [1, 5, 8])
@pytest.mark.parametrize("tess", [[50], [16, 16], [48, 48], [5, 5, 5]])
def test_backward_rounding(cuda, tess, nstep):
    # the reverse sweep's positions are the replay's own
    _check_rounding(tess, nstep, 4, 10000, cuda)


def _check_rounding(tess, nstep, n_theta, n, cuda):
    # The oracle replays the same float positions and adds in double.  What is left is
    # the roundings of the adjoint, one for each step, and those of a workgroup's table,
    # of the tables' sum and of the moments formed from it.  Each is at most 2^-24 of its
    # value, 2^-24 / sqrt(3) in the mean of squares, and over this many points they are
    # independent of each other.
    T = cpab_for(tess)
    theta = seeded_theta(T, n_theta, 0.5, 5)
    pts = uniform_points(len(tess), n, 6)
    g = np.ones((n_theta, len(tess), n), np.float32)
    As, mom, _ = _backward_case(T, theta, pts, g, cuda, nstep=nstep)
    ref, _ = orc.backward(pts, As, g, tess, nstep)
    err = np.linalg.norm(mom - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert (err <= np.sqrt((nstep + 3) / 3.0) * 2.0 ** -24).all(), err * 2.0 ** 24


@pytest.mark.parametrize("nstep", [5, 20, 37, 70])
@pytest.mark.parametrize("tess", [[50], [6, 5], [20, 20], [48, 48], [3, 3, 3], [10, 10, 10]])
def test_adaptive_step_counts(cuda, tess, nstep):
    # the segmented body: full bins with and without the affine table in LDS, the
    # cell cache
    _check(tess, nstep, 3000, 0.5, cuda, adaptive=1)


@pytest.mark.parametrize("nstep", [5, 20, 70])
@pytest.mark.parametrize("tess,ins,outs,C,adaptive,scale", [
    ([10], (50,), (1500,), 2, 0, 0.5), ([6, 5], (40, 48), (36, 48), 1, 0, 0.5),
    ([6, 5], (37, 23), (29, 31), 3, 0, 0.5), ([6, 5], (40, 48), (36, 48), 1, 1, 0.5),
    ([36, 36], (20, 30), (64, 80), 1, 0, 0.5),      # no room for the reverse table; few steps
    ([48, 48], (20, 30), (64, 80), 2, 0, 0.5),      # the cell cache
    ([3, 3, 3], (10, 12, 9), (11, 9, 13), 2, 0, 0.5), ([10, 10, 10], (10, 12, 9), (16, 8, 32), 1, 0, 0.5),
    ([6, 5], (40, 48), (36, 48), 2, 0, 8.0), ([3, 3, 3], (10, 12, 9), (6, 8, 32), 1, 0, 8.0)])
def test_image_step_counts(cuda, tess, ins, outs, C, adaptive, scale, nstep):
    # the fused transform_data backward against the resampling backward at the
    # oracle's final points and the points' backward from there
    T = cpab_for(tess)
    p, nd, B = T.params, len(tess), 2
    theta = seeded_theta(T, B, scale, 710)
    rng = np.random.default_rng(711)
    data = rng.random((B, C, *ins)).astype(np.float32)
    gout = rng.standard_normal((B, C, *outs)).astype(np.float32)
    grid = T.uniform_meshgrid(list(outs)).cpu().numpy()
    As = _As_gpu(T, theta, cuda)
    Tr = torch.empty_like(As)
    native().expm(nd, As, 1.0 / nstep, Tr)
    A, nP = As.cpu().numpy(), int(np.prod(outs))
    fin = torch.empty((B, nd, nP), device=cuda)
    seed = torch.empty((B, nd, nP), device=cuda) if C == 1 else None
    native().transform_data_forward(nd, _dev(data, cuda), T._uniform_axes(list(outs)), list(outs),
                                    nstep, p.nc, adaptive, Tr, As, torch.empty((B, C, *outs), device=cuda),
                                    fin, seed_grad=seed)
    if nd == 1:
        xT = orc.forward_closed_1d(grid, A, p.nc)
    else:
        xT = orc.forward_trels(grid, Tr.cpu().numpy(), A, p.nc, nstep, adaptive=bool(adaptive))
    np.testing.assert_array_equal(fin.cpu().numpy(), _image_order(xT, outs))
    mom = torch.full((B, p.nC, nd * (nd + 1)), float("nan"), device=cuda)
    ws = torch.empty(native().transform_data_backward_workspace_size(nd, B, list(outs), p.nC),
                     dtype=torch.uint8, device=cuda)
    native().transform_data_backward(nd, _dev(data, cuda), T._uniform_axes(list(outs)), list(outs),
                                     nstep, p.nc, adaptive, fin, As, _dev(gout, cuda), mom, None, ws,
                                     seed_grad=seed)
    rg, _ = orc.interp_backward(nd, data, xT, outs, gout)
    ref_m, _ = orc.backward(grid, A, rg, p.nc, nstep, adaptive=bool(adaptive))
    assert_grad_close(mom.cpu().numpy(), ref_m, rtol=2e-5)


@pytest.mark.parametrize("nstep", [5, 20, 70])
@pytest.mark.parametrize("tess,K,adaptive,scale", [([50], 4, 0, 0.3), ([16, 16], 3, 0, 0.3),
                                                   ([16, 16], 3, 1, 0.3), ([48, 48], 3, 0, 0.3),
                                                   ([4, 4, 4], 4, 0, 0.3), ([10, 10, 10], 3, 0, 0.3),
                                                   ([16, 16], 3, 0, 8.0)])
def test_chain_step_counts(cuda, tess, K, adaptive, scale, nstep):
    # every stage's sums and the adjoint handed from stage to stage
    T = cpab_for(tess)
    p, nd, nb = T.params, len(tess), 2
    theta = (np.random.default_rng(720).standard_normal((K * nb, p.d)) * scale).astype(np.float32)
    pts = uniform_points(1, 3000, 721) if nd == 1 else meshgrid([40, 33] if nd == 2 else [17, 13, 11])
    nP = pts.shape[-1]
    As = _As_gpu(T, theta, cuda)
    Tr = torch.empty_like(As)
    native().expm(nd, As, 1.0 / nstep, Tr)
    out, gp = (torch.empty((nb, nd, nP), device=cuda) for _ in range(2))
    sp = torch.empty((K - 1, nb, nd, nP), device=cuda)
    native().chain_forward(nd, _dev(pts, cuda), False, nb, K, nP, nstep, p.nc, adaptive, Tr, As, out, sp)
    g = np.random.default_rng(722).standard_normal((nb, nd, nP)).astype(np.float32)
    mom = torch.full((K * nb, p.nC, nd * (nd + 1)), float("nan"), device=cuda)
    ws = torch.empty(native().chain_backward_workspace_size(nd, nP, nb, K, p.nC), dtype=torch.uint8,
                     device=cuda)
    native().chain_backward(nd, _dev(pts, cuda), False, nb, K, nP, nstep, p.nc, adaptive, sp, As,
                            _dev(g, cuda), mom, gp, ws)
    A = As.cpu().numpy().reshape(K, nb, p.nC, nd, nd + 1)
    M = mom.cpu().numpy().reshape(K, nb, p.nC, -1)
    xs, lam = [pts] + [sp[s].cpu().numpy() for s in range(K - 1)], g
    for s in reversed(range(K)):
        ref_m, lam = orc.backward(xs[s], A[s], lam, p.nc, nstep, adaptive=bool(adaptive))
        assert_grad_close(M[s], ref_m, rtol=2e-5)
    # lambda is rounded once for each of the K T steps in either form of the sweep:
    # beside assert_adjoint_close's relative part, K T 2^-24 of the largest adjoint
    # (its own 1e-6 is 17 steps' worth; K T = 280 needs 1.1e-5)
    assert_grad_close(gp.cpu().numpy(), lam, rtol=1e-5, atol_frac=max(1e-6, K * nstep * 2.0 ** -24))


def _check(tess, nstep, n, scale, cuda, adaptive=0):
    T = cpab_for(tess)
    theta = seeded_theta(T, 2, scale, 700 + nstep)
    pts = uniform_points(len(tess), n, 701)
    g = np.random.default_rng(702).standard_normal((2, len(tess), n)).astype(np.float32)
    As, mom, gp = _backward_case(T, theta, pts, g, cuda, nstep=nstep, adaptive=adaptive)
    ref_m, ref_gp = orc.backward(pts, As, g, tess, nstep, adaptive=bool(adaptive))
    assert_adjoint_close(gp, ref_gp)
    assert_grad_close(mom, ref_m, rtol=2e-5)
