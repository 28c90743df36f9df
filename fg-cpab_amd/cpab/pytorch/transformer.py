"""Autograd entry point of the CPAB transform on MI355X.

Same interface as the reference's ``cpab/pytorch/transformer.py``:
``CPAB_transformer(points, theta, params, compute_points_grad=False)`` returns
the integrated points ``[n_theta, ndim, nP]`` and differentiates w.r.t. theta
(and the points when asked).  Every numeric step runs in the HIP library
(``libcpab_hip.so``) through its C ABI, called from the native autograd functions
of ``csrc/torch_binding.cpp`` (``_cpab_torch.so``):

  forward   A = B theta and expm(A/T) in one launch (cpab_affine_expm) ->
            integrate (cpab_forward), or A = B theta (cpab_affine) and the 1D
            closed form                                 (transformer.py:72-126)
  backward  fused replay + adjoint + moments, and dtheta = B^T M, in one
            call (cpab_backward_project) [-> sum over theta for shared points]
                                                        (transformer.py:128-168)

``CPAB_chain_transformer`` runs a whole chain of stages (the Python loop of
``Cpab.transform_grid_chain``, cpab/cpab.py:237-280) as one forward launch
(cpab_chain_forward) and one backward launch (cpab_chain_backward).

``CPAB_transform_data`` is ``Cpab.transform_data`` (transform_grid of the
meshgrid, then interpolate; cpab/cpab.py:295-309) as one forward launch
(cpab_transform_data_forward) and one backward launch
(cpab_transform_data_backward): the warped grid never leaves the kernels except
as the saved final points.
"""
import torch

from ._native import torch_binding
from ._tracing import recorded

__all__ = ["CPAB_transformer", "CPAB_chain_transformer", "CPAB_transform_data"]


def CPAB_transformer(points, theta, params, compute_points_grad=False):
    """Transform points through the CPAB velocity field.

    Arguments:
        points: [ndim, n_points] (shared by all thetas) or [n_batch, ndim, n_points]
        theta: [n_batch, d]
        params: parameter object of a ``Cpab`` instance
        compute_points_grad: bool, also return d loss / d points in backward
    Returns:
        transformed points [n_batch, ndim, n_points]
    """
    assert points.is_cuda and theta.is_cuda, "Only GPU tensors supported"
    assert params.ndim in (1, 2, 3), "GPU transformer supports 1D, 2D, and 3D"
    assert type(compute_points_grad) == bool, "compute_points_grad must be bool"
    return recorded(_grid, points, theta, params, compute_points_grad)


def _grid(points, theta, params, compute_points_grad):
    return torch_binding().grid(points, theta, params, basis_tables(params, theta.device),
                                compute_points_grad)


def basis_tables(params, device):
    """Device copies of B as CSR (for A = B theta) and CSC (for B^T M), float32.

    Cached on ``params`` per device.  Replaces the torch sparse COO copies the
    reference keeps in ``params.basis_gpu_sparse(_t)`` (transformer.py:47-66).
    """
    cache = params.__dict__.setdefault("_hip_basis_tables", {})
    key = str(device)
    t = cache.get(key)
    if t is not None:
        return t
    import numpy as np
    B = params.basis.tocsr().astype(np.float64)
    B.sort_indices()
    Bt = B.tocsc()
    Bt.sort_indices()

    def dev(a, dtype):
        return torch.from_numpy(np.ascontiguousarray(a)).to(device=device, dtype=dtype)

    t = {
        "row_ptr": dev(B.indptr.astype(np.int32), torch.int32),
        "col_idx": dev(B.indices.astype(np.int32), torch.int32),
        "vals": dev(B.data.astype(np.float32), torch.float32),
        "col_ptr": dev(Bt.indptr.astype(np.int32), torch.int32),
        "row_idx": dev(Bt.indices.astype(np.int32), torch.int32),
        "vals_t": dev(Bt.data.astype(np.float32), torch.float32),
        "D": int(B.shape[0]),
        "d": int(B.shape[1]),
    }
    cache[key] = t
    return t


def CPAB_chain_transformer(points, theta_stages, params):
    """Chain of CPAB transforms: stage s maps the output of stage s-1 with
    theta_stages[s]; equal, stage by stage, to chaining ``CPAB_transformer``
    (with compute_points_grad=True), as ``Cpab.transform_grid_chain`` does in
    the reference (cpab/cpab.py:270-278).

    Arguments:
        points: [ndim, n_points] (shared) or [n_batch, ndim, n_points]
        theta_stages: [n_stages, n_batch, d] (already scaled by dt if wanted)
    Returns:
        [n_batch, ndim, n_points]
    """
    assert points.is_cuda and theta_stages.is_cuda, "Only GPU tensors supported"
    assert params.ndim in (1, 2, 3), "GPU transformer supports 1D, 2D, and 3D"
    return recorded(_chain, points, theta_stages, params)


def _chain(points, theta_stages, params):
    return torch_binding().chain(points, theta_stages, params,
                                 basis_tables(params, theta_stages.device))


def CPAB_transform_data(data, theta, axes, outsize, params):
    """``interpolate(data, CPAB_transformer(meshgrid, theta, params), outsize)``
    in one fused forward and one fused backward launch.

    Arguments:
        data: [n_batch, n_channels, *in_size]
        theta: [n_batch, d]
        axes: [sum(outsize)] the per-axis coordinates of the uniform grid, axis 0
            first (the ``torch.linspace`` vectors ``Cpab.uniform_meshgrid`` takes the
            Cartesian product of): the kernels look a pixel's start point up
            there instead of reading a meshgrid
        outsize: list of ndim output sizes
    Returns:
        [n_batch, n_channels, *outsize]
    """
    assert data.is_cuda and theta.is_cuda and axes.is_cuda, "Only GPU tensors supported"
    assert params.ndim in (1, 2, 3), "GPU transformer supports 1D, 2D, and 3D"
    return recorded(_image, data, theta, axes, [int(v) for v in outsize], params)


def _image(data, theta, axes, outsize, params):
    return _CPABImageFunction.forward(None, data, theta, axes, outsize, params)


class _CPABImageFunction:
    """The native fused transform_data behind an autograd function's forward:
    its shape checks run before any device work."""

    @staticmethod
    def forward(ctx, data, theta, axes, outsize, params):
        return torch_binding().image(data, theta, axes, outsize, params,
                                     basis_tables(params, theta.device))
