"""The backward's spread launch shapes: short rows, more rows than compute units, odd
row lengths and rounds, on NaN-prefilled outputs against the oracle; a workspace
with room for the unspread shape only; and the size of the workspace asked for."""
import re

import numpy as np
import pytest
import torch

from cpab.pytorch._native import native
from oracle import oracle as orc

from helpers import assert_adjoint_close, assert_grad_close, cpab_for, seeded_theta, uniform_points

pytestmark = pytest.mark.gpu


def _run(cuda, tess, n, nP, T, ws_bytes=None):
    p = cpab_for(tess).params
    nd, ppc = p.ndim, p.ndim * (p.ndim + 1)
    theta = seeded_theta(cpab_for(tess), n, 0.5, 500 + n)
    pts = uniform_points(nd, nP, 501)
    g = np.random.default_rng(502).standard_normal((n, nd, nP)).astype(np.float32)
    As = orc.affine(theta, p.basis).reshape(n, p.nC, nd, nd + 1)
    lib = native()
    mom = torch.full((n, p.nC, ppc), float("nan"), device=cuda)
    gp = torch.full((n, nd, nP), float("nan"), device=cuda)
    size = lib.backward_workspace_size(nd, nP, n, p.nC) if ws_bytes is None else ws_bytes
    ws = torch.empty(size, dtype=torch.uint8, device=cuda)
    lib.backward(nd, torch.tensor(pts, device=cuda), False, n, nP, T, p.nc, 0,
                 torch.tensor(As, device=cuda), torch.tensor(g, device=cuda), mom, gp, ws)
    ref_m, ref_gp = orc.backward(pts, As, g, p.nc, T)
    assert_grad_close(mom.cpu().numpy().reshape(n, -1), ref_m.reshape(n, -1))
    assert_adjoint_close(gp.cpu().numpy(), ref_gp)


@pytest.mark.parametrize("tess,n,nP,T", [([4, 4], 32, 784, 50), ([4, 4], 300, 65, 50), ([4, 4], 1, 63, 20),
                                         ([20, 20], 3, 12501, 50), ([20, 20], 200, 130, 50),
                                         ([5, 5, 5], 8, 5000, 50), ([3, 3, 3], 2, 40001, 70), ([50], 16, 2001, 50),
                                         ([300], 1, 30000, 50), ([10, 10], 1, 30000, 3), ([10, 10], 2, 5000, 90),
                                         ([4, 4, 4], 1, 70000, 8)])
def test_spread_shapes(cuda, tess, n, nP, T):
    _run(cuda, tess, n, nP, T)


def test_unspread_workspace(cuda):
    # the error names the unspread shape's size: a call with exactly that much
    # runs, with the unspread shape
    with pytest.raises(RuntimeError, match="workspace too small") as e:
        _run(cuda, [4, 4], 2, 3000, 50, ws_bytes=16)
    need = int(re.search(r"need (\d+) bytes", str(e.value)).group(1))
    assert need < native().backward_workspace_size(2, 3000, 2, 64)
    _run(cuda, [4, 4], 2, 3000, 50, ws_bytes=need)


@pytest.mark.parametrize("nd,nC,n,nP,per_row", [(2, 1600, 16, 125000, 32), (2, 3600, 16, 262144, 16),
                                               (2, 1024, 1, 262144, 512), (2, 64, 32, 784, 7),
                                               (3, 625, 8, 40000, 64), (1, 50, 16, 10000, 20)])
def test_workspace_holds_the_shapes_that_run(cuda, nd, nC, n, nP, per_row):
    # per_row: the most workgroups that a body takes for a row on 256 CUs, each
    # with a table of nC x ppc floats (the segmented body's 512-lane workgroups,
    # one to four for each CU by their LDS, but no more than cover the row; 7 of
    # 128 lanes, spread, for 784 points).  Beside them the rows' reverse-sweep
    # tables and a few words for each cell.
    ppc = nd * (nd + 1)
    tables = n * per_row * nC * ppc * 4
    rest = n * nC * (4 * {1: 4, 2: 12, 3: 24}[nd] + 16) + 65536
    size = native().backward_workspace_size(nd, nP, n, nC)
    assert tables <= size <= tables + rest
