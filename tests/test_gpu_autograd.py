"""The native autograd functions as autograd sees them: second derivatives refused,
saved-tensor hooks, in-place changes of a saved input, functional transforms and
forward mode refused, the deterministic setting read when the backward runs,
side streams, traced modules, and a used Cpab object copied and pickled."""
import copy
import pickle

import numpy as np
import pytest
import torch

from cpab import Cpab

from helpers import seeded_theta

pytestmark = pytest.mark.gpu


def _calls(T, cuda):
    """(name, function of theta, tensors it also depends on): every operation."""
    rng = np.random.default_rng(900)
    pts = torch.tensor(rng.random((2, 300)).astype(np.float32), device=cuda, requires_grad=True)
    img = torch.tensor(rng.random((2, 2, 9, 11)).astype(np.float32), device=cuda, requires_grad=True)
    mesh = T.uniform_meshgrid([9, 11])
    return [("grid", lambda th: T.transform_grid(pts, th), pts),
            ("chain", lambda th: T.transform_grid_chain(pts, torch.stack([th, th])), pts),
            ("image", lambda th: T.transform_data(img, th, [9, 11]), img),
            ("interp", lambda th: T.interpolate(img, T.transform_grid(mesh, th), [9, 11]), img)]


def _theta(T, cuda):
    return torch.tensor(seeded_theta(T, 2, 0.5, 901), device=cuda, requires_grad=True)


def test_second_derivative_refused(cuda):
    T = Cpab([3, 4])
    for name, f, x in _calls(T, cuda):
        th = _theta(T, cuda)
        g = torch.autograd.grad(f(th).square().sum(), (th, x), create_graph=True)
        assert all(v.requires_grad for v in g), name
        with pytest.raises(RuntimeError, match="once_differentiable"):
            (g[0].sum() + g[1].sum()).backward()


def test_saved_tensor_hooks_and_versions(cuda):
    T = Cpab([3, 4])
    for name, f, x in _calls(T, cuda):
        th = _theta(T, cuda)
        ref = torch.autograd.grad(f(th).sum(), (th, x))
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(
                lambda t: packed.append(1) or t.cpu(), lambda t: t.to(cuda)):
            out = f(th)
        got = torch.autograd.grad(out.sum(), (th, x))
        assert packed, name
        for a, b in zip(got, ref):
            torch.testing.assert_close(a, b, rtol=2e-5, atol=1e-6 * b.abs().max().item())
        out = f(th)
        with torch.no_grad():
            x.mul_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            out.sum().backward()


def test_functional_transforms_refused(cuda):
    T = Cpab([3, 4])
    th = _theta(T, cuda).detach()
    pts = torch.rand(2, 50, device=cuda)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: T.transform_grid(pts, t[None]))(th)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.jvp(lambda t: T.transform_grid(pts, t), (th,), (th,))


def test_deterministic_read_at_backward_and_copies(cuda):
    T = Cpab([3, 4])
    pts = torch.rand(2, 5000, device=cuda)
    th = _theta(T, cuda)
    out = T.transform_grid(pts, th)
    T.set_solver_params(deterministic_grad=True)
    runs = [torch.autograd.grad(out, th, torch.ones_like(out), retain_graph=True)[0] for _ in range(2)]
    assert torch.equal(*runs)
    for U in (copy.deepcopy(T), pickle.loads(pickle.dumps(T))):
        again = torch.autograd.grad(U.transform_grid(pts, th), th, torch.ones_like(out))[0]
        assert torch.equal(again, runs[0])


def test_side_stream(cuda):
    T = Cpab([20, 20])
    pts = torch.rand(2, 20000, device=cuda)
    th = torch.tensor(seeded_theta(T, 4, 0.5, 902), device=cuda, requires_grad=True)
    ref_out = T.transform_grid(pts, th)
    ref = torch.autograd.grad(ref_out.sum(), th)[0]
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        for _ in range(3):
            out = T.transform_grid(pts, th)
            g = torch.autograd.grad(out.sum(), th)[0]
    s.synchronize()
    assert torch.equal(out, ref_out)
    torch.testing.assert_close(g, ref, rtol=1e-4, atol=1e-5 * ref.abs().max().item())


def test_jit_trace(cuda, tmp_path):
    # a traced module computes with the inputs it is given, and differentiates
    T = Cpab([3, 4])
    for name, f, x in _calls(T, cuda):
        x.requires_grad_(False)   # a trace keeps it as a constant
        th, other = _theta(T, cuda), (0.5 * _theta(T, cuda)).detach().requires_grad_()
        f(th)                     # the first call makes tables that a trace's check would miss
        m = torch.jit.trace(lambda t: f(2 * t).sin(), (th,))
        out, ref = m(other), f(2 * other).sin()
        assert torch.equal(out, ref), name
        for _ in range(2):
            got = torch.autograd.grad(out.sum(), other, retain_graph=True)[0]
            want = torch.autograd.grad(ref.sum(), other, retain_graph=True)[0]
            torch.testing.assert_close(got, want, rtol=2e-5, atol=1e-6 * want.abs().max().item())
        with torch.no_grad():
            assert torch.equal(torch.jit.trace(f, (th,))(other), f(other)), name
        with pytest.raises(RuntimeError, match="export"):
            torch.jit.save(m, str(tmp_path / "m.pt"))


def test_no_grad_keeps_nothing(cuda):
    # evaluating under no_grad with tensors that require gradients allocates what
    # evaluating plain tensors does
    T = Cpab([4, 4])
    img = torch.rand(2, 1, 256, 256, device=cuda)
    th = _theta(T, cuda)

    def peak(x, t):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        with torch.no_grad():
            T.transform_data(x, t, [256, 256])
        return torch.cuda.max_memory_allocated() - before
    T.transform_data(img, th, [256, 256])
    assert peak(img.clone().requires_grad_(), th) == peak(img.clone(), th.detach())
