"""The backward at every kind of step count: fewer steps than a group of 8, whole
groups, a partial group, both register capacities (64 and 104 steps) up to the
step cap, with full LDS bins, the LDS cell cache (2D [48, 48]) and rows beyond
the recovery bound, against the oracle at the tolerances of the other backward
tests."""
import numpy as np
import pytest

from oracle import oracle as orc

from helpers import (assert_adjoint_close, assert_grad_close, cpab_for, seeded_theta,
                     uniform_points)
from test_gpu_kernels import _backward_case

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


def _check(tess, nstep, n, scale, cuda):
    T = cpab_for(tess)
    theta = seeded_theta(T, 2, scale, 700 + nstep)
    pts = uniform_points(len(tess), n, 701)
    g = np.random.default_rng(702).standard_normal((2, len(tess), n)).astype(np.float32)
    As, mom, gp = _backward_case(T, theta, pts, g, cuda, nstep=nstep)
    ref_m, ref_gp = orc.backward(pts, As, g, tess, nstep)
    assert_adjoint_close(gp, ref_gp)
    assert_grad_close(mom, ref_m, rtol=2e-5)
