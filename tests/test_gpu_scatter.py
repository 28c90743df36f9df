"""The data gradient's LDS box: boxes at and beyond its capacity (10,000 positions),
data of one row or column, partial tiles in both directions, the data gradient
without the grid gradient, the image backward's scatter at odd and thin sizes, more
tiles than one launch holds workgroups, the data gradient without theta's, both
gradients in one launch, and the 1D gradients one by one and together, against the
oracle within the bound of the other data-gradient tests."""
import numpy as np
import pytest
import torch

from cpab import Cpab
from cpab.pytorch._native import native
from oracle import oracle as orc

from helpers import cpab_for, scatter_magnitude, seeded_theta

pytestmark = pytest.mark.gpu


def _dev(a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a)).to(cuda)


@pytest.mark.parametrize("ins,outs", [((100, 100), (32, 32)), ((100, 101), (33, 31)), ((1, 9), (40, 70)),
                                      ((9, 1), (31, 33)), ((20, 20, 25), (32, 2, 32)),
                                      ((20, 21, 25), (33, 3, 5)), ((1, 1, 4), (5, 2, 64))])
def test_scatter_box_limits(cuda, ins, outs):
    nd, B, C = len(ins), 2, 2
    rng = np.random.default_rng(800 + ins[0])
    data = rng.random((B, C, *ins)).astype(np.float32)
    grid = rng.random((B, nd, int(np.prod(outs)))).astype(np.float32)
    grid[:, :, :2] = [0.0, 1.0]            # the box of the first tile reaches both ends
    gout = rng.standard_normal((B, C, *outs)).astype(np.float32)
    gd = torch.full(data.shape, float("nan"), device=cuda)
    native().interp_backward(nd, _dev(data, cuda), _dev(grid, cuda), outs, _dev(gout, cuda), None, gd)
    _, rd = orc.interp_backward(nd, data, grid, outs, gout)
    mag = scatter_magnitude(data.shape, grid, outs, gout)
    err = np.abs(gd.cpu().numpy().astype(np.float64) - rd)
    assert (err <= 1e-4 * mag + 1e-12).all(), float((err / (mag + 1e-30)).max())


@pytest.mark.parametrize("tess,size", [([5, 4], (71, 45)), ([3, 2, 2], (19, 6, 37)), ([7], (1013,))])
def test_image_scatter_odd_sizes(cuda, tess, size):
    # theta and data gradients of the public call against the two-step
    # composition (transform_grid of the meshgrid, then interpolate)
    T = cpab_for(tess)
    rng = np.random.default_rng(810)
    data = _dev(rng.random((2, 3, *size)).astype(np.float32), cuda).requires_grad_()
    theta = _dev(seeded_theta(T, 2, 0.5, 811), cuda).requires_grad_()
    g = _dev(rng.standard_normal((2, 3, *size)).astype(np.float32), cuda)
    got = torch.autograd.grad(T.transform_data(data, theta, list(size)), (data, theta), g)
    grid = T.transform_grid(T.uniform_meshgrid(list(size)), theta)
    ref = torch.autograd.grad(T.interpolate(data, grid, list(size)), (data, theta), g)
    # the same contributions per element in another order: a few float32 ulps
    # of the largest sums
    for a, b in zip(got, ref):
        assert (a - b).abs().max().item() <= 2e-5 * b.abs().max().item()


@pytest.mark.parametrize("size", [(1, (1 << 23) + 11, 1), (3, 50001, 2), (2, 3, 40001), (2050, 3, 5),
                                  (9, 17, 31), (8, 8, 16), (1, 1, 1)])
def test_image_scatter_thin_volumes(cuda, size):
    # volumes whose slices hold few outputs (2^23 slices of one: a workgroup of
    # 512 lanes for each passes the 2^32 lanes of a launch) and partial tiles
    T = cpab_for([2, 1, 1])
    size, ins = list(size), (2, 300, 2)
    rng = np.random.default_rng(820)
    data = rng.random((1, 1, *ins)).astype(np.float32)
    g = rng.standard_normal((1, 1, *size)).astype(np.float32)
    theta = _dev(seeded_theta(T, 1, 0.5, 821), cuda)
    x = _dev(data, cuda).requires_grad_()
    gd = torch.autograd.grad(T.transform_data(x, theta, size), x, _dev(g, cuda))[0]
    with torch.no_grad():
        grid = T.transform_grid(T.uniform_meshgrid(size), theta).cpu().numpy()
    _, rd = orc.interp_backward(3, data, grid, size, g)
    mag = scatter_magnitude(data.shape, grid, size, g)
    assert (np.abs(gd.cpu().numpy() - rd) <= 1e-4 * mag + 1e-12).all()


@pytest.mark.parametrize("size", [(1000, 4), (3, 2049), (33, 31), (32, 32), (1, 1)])
def test_image_scatter_thin_images(cuda, size):
    T = cpab_for([3, 2])
    rng = np.random.default_rng(822)
    data = rng.random((2, 2, 40, 30)).astype(np.float32)
    g = rng.standard_normal((2, 2, *size)).astype(np.float32)
    theta = _dev(seeded_theta(T, 2, 0.5, 823), cuda)
    x = _dev(data, cuda).requires_grad_()
    gd = torch.autograd.grad(T.transform_data(x, theta, list(size)), x, _dev(g, cuda))[0]
    with torch.no_grad():
        grid = T.transform_grid(T.uniform_meshgrid(list(size)), theta).cpu().numpy()
    _, rd = orc.interp_backward(2, data, grid, list(size), g)
    mag = scatter_magnitude(data.shape, grid, size, g)
    assert (np.abs(gd.cpu().numpy() - rd) <= 1e-4 * mag + 1e-12).all()


@pytest.mark.parametrize("tiles", [(1 << 22) - 3, (1 << 22) + 5, (1 << 23) - 16])
def test_scatter_many_tiles(cuda, tiles):
    # grid order: every slice of one output is a tile; a launch holds 2^22
    # workgroups, and interpolate takes fewer than 2^23 tiles
    rng = np.random.default_rng(824)
    data = rng.random((1, 1, 2, 3000, 2)).astype(np.float32)
    grid = rng.random((1, 3, tiles)).astype(np.float32)
    g = rng.standard_normal((1, 1, 1, tiles, 1)).astype(np.float32)
    gd = torch.full(data.shape, float("nan"), device=cuda)
    native().interp_backward(3, _dev(data, cuda), _dev(grid, cuda), (1, tiles, 1), _dev(g, cuda),
                             None, gd)
    _, rd = orc.interp_backward(3, data, grid, (1, tiles, 1), g)
    mag = scatter_magnitude(data.shape, grid, (1, tiles, 1), g)
    assert (np.abs(gd.cpu().numpy() - rd) <= 1e-4 * mag + 1e-12).all()


@pytest.mark.parametrize("tess,size", [([5, 4], (71, 45)), ([3, 2, 2], (19, 6, 37)), ([7], (1013,))])
def test_data_gradient_alone(cuda, tess, size):
    # without theta's gradient no trajectory is replayed: the same data gradient,
    # also in the deterministic mode, which keeps its own passes
    rng = np.random.default_rng(812)
    T = Cpab(tess)
    theta = _dev(seeded_theta(T, 2, 0.5, 813), cuda)
    data = _dev(rng.random((2, 3, *size)).astype(np.float32), cuda).requires_grad_()
    g = _dev(rng.standard_normal((2, 3, *size)).astype(np.float32), cuda)
    both = torch.autograd.grad(T.transform_data(data, theta.clone().requires_grad_(), list(size)),
                               data, g)[0]
    alone = torch.autograd.grad(T.transform_data(data, theta, list(size)), data, g)[0]
    assert (alone - both).abs().max().item() <= 2e-5 * both.abs().max().item()
    T.set_solver_params(deterministic_grad=True)
    runs = [torch.autograd.grad(T.transform_data(data, th, list(size)), data, g)[0]
            for th in (theta, theta, theta.clone().requires_grad_())]
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
    assert (runs[0] - both).abs().max().item() <= 2e-5 * both.abs().max().item()


@pytest.mark.parametrize("ins,outs", [((9, 7), (16, 16)), ((9, 7), (17, 16)), ((30, 40), (1, 1)),
                                      ((30, 40), (3, 300)), ((30, 40), (300, 3)), ((5, 6, 7), (4, 5, 3)),
                                      ((5, 6, 7), (40, 3, 7)), ((5, 6, 7), (33, 2, 9)), ((1, 1), (36, 64)),
                                      ((300, 200), (33, 40)), ((20, 21, 40), (8, 3, 40))])
def test_both_gradients_in_one_launch(cuda, ins, outs):
    # at most and beyond 256 outputs of a tile, partial tiles, boxes beyond their
    # capacity; the grid's gradient as the kernel for it alone gives it
    nd, B, C = len(ins), 3, 2
    rng = np.random.default_rng(840 + outs[0])
    data = rng.random((B, C, *ins)).astype(np.float32)
    grid = (1.2 * rng.random((B, nd, int(np.prod(outs)))) - 0.1).astype(np.float32)
    gout = rng.standard_normal((B, C, *outs)).astype(np.float32)
    gd = torch.full(data.shape, float("nan"), device=cuda)
    gg, alone = (torch.full(grid.shape, float("nan"), device=cuda) for _ in range(2))
    args = (nd, _dev(data, cuda), _dev(grid, cuda), outs, _dev(gout, cuda))
    native().interp_backward(*args, gg, gd)
    native().interp_backward(*args, alone, None)
    assert torch.equal(gg, alone)
    _, rd = orc.interp_backward(nd, data, grid, outs, gout)
    mag = scatter_magnitude(data.shape, grid, outs, gout)
    assert (np.abs(gd.cpu().numpy() - rd) <= 1e-4 * mag + 1e-12).all()


@pytest.mark.parametrize("W,n", [(1, 5), (2, 257), (700, 1000)])
@pytest.mark.parametrize("want", ["grid", "data", "both"])
def test_interp1d_gradients(cuda, W, n, want):
    rng = np.random.default_rng(830 + W)
    data = rng.random((3, 2, W)).astype(np.float32)
    grid = (1.4 * rng.random((3, 1, n)) - 0.2).astype(np.float32)   # some outside
    gout = rng.standard_normal((3, 2, n)).astype(np.float32)
    gg = torch.full(grid.shape, float("nan"), device=cuda) if want != "data" else None
    gd = torch.full(data.shape, float("nan"), device=cuda) if want != "grid" else None
    native().interp_backward(1, _dev(data, cuda), _dev(grid, cuda), (n,), _dev(gout, cuda), gg, gd)
    rg, rd = orc.interp_backward(1, data, grid, (n,), gout)
    if gg is not None:   # two channels' products in order: the same bits
        np.testing.assert_array_equal(gg.cpu().numpy(), rg)
    if gd is not None:
        mag = scatter_magnitude(data.shape, grid, (n,), gout)
        assert (np.abs(gd.cpu().numpy() - rd) <= 1e-4 * mag + 1e-12).all()
