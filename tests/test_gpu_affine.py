"""The fused affine + exponential launch for few and many matrices and for rows of
few and many entries: equal to the oracle's sums and to the separate launches
bit for bit, at counts that do not fill a workgroup and on both sides of the
4096 matrices where the shape changes.  Exponentials of matrices whose norm
overflows.  And the projection over columns of several rounds (128 entries each)
and on both sides of the 32 columns for each of 256 CUs where its form changes."""
import numpy as np
import pytest
import torch

from cpab import Cpab
from cpab.pytorch._native import native
from cpab.pytorch.transformer import basis_tables
from oracle import oracle as orc

from helpers import seeded_theta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tess,n,free", [([3, 3], 1, True), ([5, 3], 3, True), ([8, 8], 16, True),
                                         ([8, 8], 17, True), ([8, 8], 16, False), ([1, 1], 1, False),
                                         ([2, 1, 3], 1, True), ([3, 3, 3], 5, True),
                                         ([4, 3, 2], 35, False), ([7], 3, True)])
def test_affine_expm_shapes(cuda, tess, n, free):
    T = Cpab(tess, zero_boundary=not free)
    nd = len(tess)
    theta = torch.from_numpy(seeded_theta(T, n, 0.3, 950 + n)).to(cuda)
    tab = basis_tables(T.params, cuda)
    As = torch.full((n, T.params.nC, nd, nd + 1), float("nan"), device=cuda)
    Tr, ref_Tr = torch.full_like(As, float("nan")), torch.empty_like(As)
    native().affine_expm(nd, theta, T.params.nC, tab["row_ptr"], tab["col_idx"], tab["vals"],
                         1.0 / 50, As, Tr)
    ref = orc.affine(theta.cpu().numpy(), T.params.basis).reshape(As.shape)
    np.testing.assert_array_equal(As.cpu().numpy(), ref)
    native().expm(nd, As, 1.0 / 50, ref_Tr)
    assert torch.equal(Tr, ref_Tr)


@pytest.mark.parametrize("nd", [2, 3])
def test_expm_of_overflowing_norms(cuda, nd):
    # infinite entries, and finite ones whose squares overflow: the launch ends,
    # and the matrices beside them are what they are alone
    A = torch.rand(64, nd, nd + 1, device=cuda) - 0.5
    ref, out = torch.empty_like(A), torch.empty_like(A)
    native().expm(nd, A, 1.0, ref)
    bad = A.clone()
    for k, v in enumerate([float("inf"), -float("inf"), float("nan"), 3e38, -1e30, 2e19]):
        bad[8 * k + 3, k % nd, k % (nd + 1)] = v
    native().expm(nd, bad, 1.0, out)
    same = (bad == A).all(-1).all(-1)
    assert same.sum() == 64 - 6 and torch.equal(out[same], ref[same])
    # the largest norm that does not overflow (1.8e19) takes the 65 squarings
    # that it always took: the identity's translation by it
    big = torch.zeros(1, nd, nd + 1, device=cuda)
    big[0, 0, nd] = 1.8e19
    native().expm(nd, big, 1.0, out[:1])
    want = torch.eye(nd, nd + 1, device=cuda)
    want[0, nd] = 1.8e19
    torch.testing.assert_close(out[0], want)


@pytest.mark.parametrize("tess,n", [([3, 3], 1), ([8, 8], 3), ([6, 7], 2), ([3, 3, 3], 2), ([2, 1, 3], 5)])
def test_project_long_columns(cuda, tess, n):
    T = Cpab(tess, zero_boundary=False)
    p = T.params
    tab = basis_tables(p, cuda)
    M = np.random.default_rng(960).standard_normal((n, p.D)).astype(np.float32)
    out = torch.full((n, p.d), float("nan"), device=cuda)
    native().project(torch.from_numpy(M).to(cuda), p.D, p.d, tab["col_ptr"], tab["row_idx"],
                     tab["vals_t"], out)
    np.testing.assert_array_equal(out.cpu().numpy(), orc.project(M, p.basis))


@pytest.mark.parametrize("tess,free,n", [([8, 8], True, 28), ([8, 8], True, 29), ([30, 30], False, 2),
                                         ([30, 30], False, 3), ([3, 3, 3], True, 43),
                                         ([8, 8, 8], False, 8), ([50], False, 300)])
def test_project_few_and_many_columns(cuda, tess, free, n):
    T = Cpab(tess, zero_boundary=not free)
    p = T.params
    tab = basis_tables(p, cuda)
    M = np.random.default_rng(961).standard_normal((n, p.D)).astype(np.float32)
    out = torch.full((n, p.d), float("nan"), device=cuda)
    native().project(torch.from_numpy(M).to(cuda), p.D, p.d, tab["col_ptr"], tab["row_idx"],
                     tab["vals_t"], out)
    np.testing.assert_array_equal(out.cpu().numpy(), orc.project(M, p.basis))
