"""``transform_data`` resampling on MI355X.

Same functions and semantics as the reference's
``cpab/pytorch/interpolation.py:3-159``: ``interpolate(ndim, data, grid,
outsize)`` samples ``data [B, C, *in_size]`` at ``grid [B, ndim,
prod(outsize)]`` (coordinate k scaled by ``in_size[k]-1`` and clamped to the
border) and returns ``[B, C, *outsize]``.  Forward and backward (w.r.t. the
grid, and w.r.t. the data when it requires grad) are HIP kernels behind the C
ABI, called from the native autograd function (csrc/torch_binding.cpp); there is
no torch or CPU fallback.  ``deterministic=True`` (an addition to the reference's
arguments; ``Cpab.interpolate`` passes the solver's ``deterministic_grad``) sums
the data gradient as 64-bit integers, the same on every run.
"""
from ._native import torch_binding
from ._tracing import recorded

__all__ = ["interpolate", "interpolate1D", "interpolate2D", "interpolate3D"]


def interpolate(ndim, data, grid, outsize, deterministic=False):
    if ndim == 1:
        return interpolate1D(data, grid, outsize, deterministic)
    elif ndim == 2:
        return interpolate2D(data, grid, outsize, deterministic)
    elif ndim == 3:
        return interpolate3D(data, grid, outsize, deterministic)


def interpolate1D(data, grid, outsize, deterministic=False):
    return _interp(1, data, grid, outsize, deterministic)


def interpolate2D(data, grid, outsize, deterministic=False):
    return _interp(2, data, grid, outsize, deterministic)


def interpolate3D(data, grid, outsize, deterministic=False):
    return _interp(3, data, grid, outsize, deterministic)


def _interp(ndim, data, grid, outsize, deterministic):
    return recorded(_native_interp, ndim, data, grid, [int(v) for v in outsize],
                    bool(deterministic))


def _native_interp(ndim, data, grid, outsize, deterministic):
    return torch_binding().interp(ndim, data, grid, outsize, deterministic)
