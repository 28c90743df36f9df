"""Performance cases: the calls a user's program makes of this framework.

Each case is one pass through a public entry point of ``Cpab``
(``transform_grid``, ``transform_grid_chain``, ``transform_data``,
``interpolate``) as a program calls it: the forward and, where the case trains,
the backward for an upstream gradient, returning the output and every gradient
asked for.  The sizes are the benchmark's own configurations and the ranges
around them.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fg-cpab_amd"))

from cpab import Cpab  # noqa: E402

DEV = torch.device("cuda")

# A case's fields.  op: grid | chain | image | interp.  nx, ny, nz: the
# tessellation (0: no such axis).  batch: thetas (chain: thetas per stage).
# points: points per theta (grid, chain), 0 where s0, s1, s2 give a grid of them
# (image, interp: the size).  steps: nstepsolver.  scale: theta ~ N(0, scale^2).
_DEFAULTS = dict(op="grid", nx=1, ny=0, nz=0, batch=1, points=0, s0=0, s1=0, s2=0, channels=1,
                 stages=1, steps=50, scale=0.5, zero_boundary=True, adaptive=False,
                 deterministic=False, batched=False, points_grad=False, data_grad=False, train=True)


def _make(**kw):
    return dict(_DEFAULTS, **kw)


def listed():
    return [
        # Time-series alignment: 16 warps of one 10,000-sample axis, trained.
        _make(name="grid1d", nx=50, batch=16, points=10000),
        # A spatial-transformer layer on 28 x 28 inputs: one field per sample of
        # a small batch, with the point gradient the layer below needs.
        _make(name="grid2d_layer", nx=4, ny=4, batch=32, points=784, batched=True, points_grad=True),
        # The headline registration step: 125,000 scattered points, 16 fields.
        _make(name="grid2d", nx=20, ny=20, batch=16, points=125000),
        # The same work with the solver set coarser than its default (fewer
        # steps for speed), an odd number of points.
        _make(name="grid2d_steps", nx=16, ny=16, batch=16, points=60001, steps=20),
        # A fine field over one large point set: more cells than a workgroup's
        # local memory holds.
        _make(name="grid2d_fine", nx=48, ny=48, batch=2, points=400000),
        # A field that is free at the boundary, integrated with the crossing
        # correction switched on.
        _make(name="grid2d_free", nx=8, ny=8, batch=8, points=50021, scale=0.3,
              zero_boundary=False, adaptive=True),
        # Image warping: a batch of 512 x 512 gray images, gradient to theta.
        _make(name="image2d", op="image", nx=30, ny=30, batch=16, s0=512, s1=512),
        # Warping feature maps inside a network: several channels, an odd size,
        # gradients to theta and to the features.
        _make(name="image2d_features", op="image", nx=8, ny=8, batch=8, s0=225, s1=227, channels=3,
              data_grad=True),
        # Volume registration: one 128^3 volume.
        _make(name="volume3d", op="image", nx=10, ny=10, nz=10, batch=1, s0=128, s1=128, s2=128),
        # Point clouds in 3D, several at a time, with their point gradients.
        _make(name="grid3d", nx=5, ny=5, nz=5, batch=8, points=40000, batched=True, points_grad=True),
        # A composition of 8 fields over a pixel grid.
        _make(name="chain2d", op="chain", nx=16, ny=16, stages=8, batch=1, s0=512, s1=512, scale=0.3),
        # Resampling alone, at a grid the program holds: colour images, gradients
        # to the images and to the grid.
        _make(name="resample2d", op="interp", nx=4, ny=4, batch=8, s0=384, s1=384, channels=3,
              points_grad=True, data_grad=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grid1d", "grid2d", "grid2d", "grid2d", "grid3d", "image2d", "image2d",
                       "image3d", "chain2d", "interp2d"])
    batch = _log(rng, 1, 32)
    steps = rng.choice([50, 50, 50, rng.randint(5, 100)])
    train = rng.random() < 0.8
    if kind == "grid1d":
        return _make(nx=rng.randint(4, 100), batch=batch, points=_log(rng, 300, 40000), steps=steps,
                     train=train, points_grad=rng.random() < 0.3)
    if kind == "grid2d":
        c = _make(nx=rng.randint(3, 40), ny=rng.randint(3, 40), batch=batch, steps=steps, train=train,
                  points=min(_log(rng, 500, 200000), 2000000 // batch), batched=rng.random() < 0.4,
                  points_grad=rng.random() < 0.4, deterministic=rng.random() < 0.15)
        if rng.random() < 0.2:
            c.update(nx=rng.randint(3, 8), ny=rng.randint(3, 8), zero_boundary=False, scale=0.3)
        c["adaptive"] = rng.random() < 0.2
        return c
    if kind == "grid3d":
        n = rng.randint(2, 8)
        return _make(nx=n, ny=rng.randint(2, 8), nz=n, batch=min(batch, 8), steps=steps, train=train,
                     points=min(_log(rng, 500, 100000), 500000 // min(batch, 8)),
                     batched=rng.random() < 0.5, points_grad=rng.random() < 0.5)
    if kind in ("image2d", "interp2d"):
        s = _log(rng, 28, 512)
        c = _make(op="image" if kind == "image2d" else "interp", nx=rng.randint(3, 30),
                  ny=rng.randint(3, 30), batch=max(1, min(batch, 2000000 // (s * s))), s0=s,
                  s1=max(20, min(512, s + rng.randint(-15, 15))), channels=rng.choice([1, 1, 3]),
                  train=train, steps=steps)
        c["data_grad"] = rng.random() < 0.4
        c["points_grad"] = kind == "interp2d" and (not c["data_grad"] or rng.random() < 0.7)
        return c
    if kind == "image3d":
        s = _log(rng, 24, 112)
        n = rng.randint(3, 10)
        return _make(op="image", nx=n, ny=n, nz=n, batch=1, s0=s, s1=s + rng.randint(0, 9),
                     s2=s + rng.randint(0, 9), steps=steps, train=train)
    s = _log(rng, 48, 400)
    return _make(op="chain", nx=rng.randint(4, 24), ny=rng.randint(4, 24), stages=rng.randint(2, 8),
                 batch=rng.choice([1, 1, 2]), s0=s, s1=s + rng.randint(0, 15), scale=0.3, train=train)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

_PLANS = {}


def _plan(c):
    """The program's Cpab object: built once per tessellation and solver setting."""
    tess = [c[k] for k in ("nx", "ny", "nz") if c[k]]
    key = (tuple(tess), c["zero_boundary"], c["steps"], c["adaptive"], c["deterministic"])
    if key not in _PLANS:
        T = Cpab(tess, zero_boundary=c["zero_boundary"])
        T.set_solver_params(c["steps"], c["adaptive"], deterministic_grad=c["deterministic"])
        _PLANS[key] = T
    return _PLANS[key]


def _sizes(c):
    return [c[k] for k in ("s0", "s1", "s2") if c[k]]


def _smooth(shape, gen, cell=8):
    """Smooth random images in [0, 1): coarse uniform noise, enlarged."""
    n = len(shape) - 2
    low = [max(2, s // cell) for s in shape[2:]]
    noise = torch.rand(*shape[:2], *low, device=DEV, generator=gen)
    mode = {1: "linear", 2: "bicubic", 3: "trilinear"}[n]
    return F.interpolate(noise, size=list(shape[2:]), mode=mode, align_corners=True).contiguous()


def _residual(points, batch, gen):
    """An upstream gradient as the mean squared error to smoothly moved targets
    gives it: [batch, ndim, n], 2 / numel times a smooth field plus some noise."""
    nd, n = points.shape[-2:]
    p = points if points.dim() == 3 else points[None]
    k = torch.randint(1, 4, (batch, nd, nd), device=DEV, generator=gen).float()
    phase = torch.rand(batch, nd, 1, device=DEV, generator=gen)
    wave = sum(k[:, :, j:j + 1] * p[:, j:j + 1, :] for j in range(nd)) + phase
    field = 0.05 * torch.sin(2 * math.pi * wave)
    field = field + 0.01 * torch.randn(batch, nd, n, device=DEV, generator=gen)
    return (field * (2.0 / field.numel())).contiguous()


def prepare(case, seed):
    c = dict(_DEFAULTS, **case)
    T = _plan(c)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    nd, n = T.params.ndim, c["batch"]
    rows = n * c["stages"]
    theta = torch.randn(rows, T.params.d, device=DEV, generator=gen) * c["scale"]
    st = {"T": T, "case": c}
    if c["op"] == "chain":
        theta = theta.view(c["stages"], n, -1)
    st["theta"] = theta.requires_grad_(c["train"] and c["op"] != "interp")
    if c["op"] in ("grid", "chain"):
        if c["points"]:
            shape = (n, nd, c["points"]) if c["batched"] else (nd, c["points"])
            pts = torch.rand(shape, device=DEV, generator=gen)
        else:
            pts = T.uniform_meshgrid(_sizes(c))
        st["grad"] = _residual(pts, n, gen)
        st["points"] = pts.requires_grad_(c["train"] and c["points_grad"])
        return st
    size = _sizes(c)
    data = _smooth([n, c["channels"], *size], gen)
    other = _smooth([n, c["channels"], *size], gen)
    st["grad"] = ((data - other) * (2.0 / data.numel())).contiguous()
    st["data"] = data.requires_grad_(c["train"] and c["data_grad"])
    if c["op"] == "interp":
        # A smoothly moved pixel grid, its positions a little away from the
        # pixel centres (where the slope of the interpolant jumps).
        base = T.uniform_meshgrid(size)
        pos = base[None] + 0.5 * n * base.numel() * _residual(base, n, gen)
        for k, s in enumerate(size):
            u = (pos[:, k] * (s - 1)).clamp(0.02, s - 1.02)
            whole = torch.floor(u)
            pos[:, k] = (whole + (u - whole).clamp(0.02, 0.98)) / (s - 1)
        st["points"] = pos.contiguous().requires_grad_(c["train"] and c["points_grad"])
    return st


def _forward(st):
    c, T = st["case"], st["T"]
    if c["op"] == "grid":
        return T.transform_grid(st["points"], st["theta"])
    if c["op"] == "chain":
        return T.transform_grid_chain(st["points"], st["theta"], scale_by_dt=True)
    if c["op"] == "image":
        return T.transform_data(st["data"], st["theta"], _sizes(c))
    return T.interpolate(st["data"], st["points"], _sizes(c))


_INPUTS = ("theta", "points", "data")


def run(st):
    if not st["case"]["train"]:
        with torch.no_grad():
            return {"out": _forward(st)}
    out = _forward(st)
    wanted = [k for k in _INPUTS if k in st and st[k].requires_grad]
    grads = torch.autograd.grad(out, [st[k] for k in wanted], st["grad"])
    return dict({"out": out}, **{"grad_" + k: g for k, g in zip(wanted, grads)})


# --------------------------------------------------------------------------
# work and tolerance
# --------------------------------------------------------------------------

def work(case):
    """Bytes: every input read once, every output written once.  Floating-point
    operations per trajectory and step of the integration scheme (an fma is 2):
    forward 15 (2D) and 43 (3D), backward 83 and 187; 1D 15 per trajectory and
    27 per step backward."""
    c = dict(_DEFAULTS, **case)
    tess = [c[k] for k in ("nx", "ny", "nz") if c[k]]
    nd = len(tess)
    size = _sizes(c)
    n = c["points"] or math.prod(size)
    rows = c["batch"] * c["stages"]
    d = nd * math.prod(t + 1 for t in tess)   # about the size of theta
    train = c["train"]
    traj = float(n) * rows
    if c["op"] == "interp":
        per = c["channels"] * 2.0 ** nd * 3
        values = traj * nd + 2 * traj * c["channels"]
        if train:
            values += traj * c["channels"] * (2 + c["data_grad"]) + traj * nd * (1 + c["points_grad"])
        return {"bytes": 4.0 * values, "flops": traj * per * (3 if train else 1)}
    fwd = {1: 15.0, 2: 15.0 * c["steps"], 3: 43.0 * c["steps"]}[nd]
    bwd = {1: 27.0, 2: 83.0, 3: 187.0}[nd] * c["steps"]
    values = rows * d * (2 if train else 1)
    if c["op"] == "image":
        chan = float(n) * c["batch"] * c["channels"]
        values += 2 * chan + (2 * chan + chan * c["data_grad"] if train else 0)
    else:
        pts = float(n) * nd * (c["batch"] if c["batched"] else 1)
        out = float(n) * nd * c["batch"]
        values += pts + out + (pts + out + (pts if c["points_grad"] else 0) if train else 0)
    return {"bytes": 4.0 * values, "flops": traj * (fwd + (bwd if train else 0))}


def tolerance(case):
    """32-bit sums of many trajectories' contributions, added by atomics in no
    fixed order: the same inputs twice give up to 7e-6 (relative) and 5e-5
    (against the root mean square), resampling alone 1e-7 and 3e-6."""
    c = dict(_DEFAULTS, **case)
    return {"rel": 4e-5, "max": 1e-3} if c["op"] != "interp" else {"rel": 1e-5, "max": 5e-4}


# --------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# --------------------------------------------------------------------------

def _cells(p, tess):
    """Cell of each point p [ndim, N] (float64): intervals; 4 triangles around
    each square's centre (0 low y, 1 high x, 2 high y, 3 low x); 5 tetrahedra per
    cube, mirrored in cubes of odd parity."""
    idx, loc = [], []
    for x, n in zip(p, tess):
        u = x.clamp(0.0, 1.0) * n
        i = torch.floor(u).clamp(max=n - 1)
        idx.append(i.long())
        loc.append(u - i)
    if len(tess) == 1:
        return idx[0]
    if len(tess) == 2:
        nx, ny = tess
        lx, ly = loc
        b3, b1 = lx < ly, (1 - lx) < ly
        t = torch.where(b3, torch.where(b1, 2, 3), torch.where(b1, 1, 0))
        xo, yo = (p[0] <= 0) | (p[0] >= 1), (p[1] <= 0) | (p[1] >= 1)
        side_y = torch.where(p[1] <= 0, 0, 2)
        side_x = torch.where(p[0] <= 0, 3, 1)
        over_x = torch.where(p[0] <= 0, -p[0], p[0] - 1) * nx
        over_y = torch.where(p[1] <= 0, -p[1], p[1] - 1) * ny
        t = torch.where(yo, side_y, t)
        t = torch.where(xo & ~(yo & (over_y > over_x)), side_x, t)
        return 4 * (idx[0] + nx * idx[1]) + t
    i, j, k = idx
    x, y, z = loc
    odd = (i + j + k) % 2 == 1
    x, y = torch.where(odd, y, x), torch.where(odd, 1 - x, y)
    t = torch.where(x - y >= z, 4, 0)
    t = torch.where(y - x >= z, 3, t)
    t = torch.where(x + y + z >= 2, 2, t)
    t = torch.where(z >= x + y, 1, t)
    return 5 * (i + tess[0] * (j + tess[1] * k)) + t


def _apply(M, p):
    """M [N, ndim, ndim + 1] at the points p [ndim, N]."""
    return (M[:, :, :-1] * p.t()[:, None, :]).sum(-1).t() + M[:, :, -1].t()


class _Flow:
    """One integration of rows of points under As [rows, nC, ndim, ndim + 1]."""

    def __init__(self, As, tess, steps, adaptive):
        self.As, self.tess, self.T, self.adaptive = As, tess, steps, adaptive
        rows, nC, nd = As.shape[:3]
        self.rows, self.nC, self.nd = rows, nC, nd
        self.flat = As.reshape(rows * nC, nd, nd + 1)
        sq = torch.zeros(rows * nC, nd + 1, nd + 1, dtype=As.dtype, device=As.device)
        sq[:, :nd] = self.flat / steps
        self.step = torch.matrix_exp(sq)[:, :nd].contiguous()

    def cell(self, p, base):
        return _cells(p, self.tess) + base

    def forward(self, p):
        """p [rows, ndim, n] -> the same shape."""
        if self.nd == 1:
            return self._exact1d(p)
        rows, nd, n = p.shape
        base = (torch.arange(rows, device=p.device) * self.nC).repeat_interleave(n)
        q = p.transpose(0, 1).reshape(nd, -1)
        for _ in range(self.T):
            c = self.cell(q, base)
            e = _apply(self.step[c], q)
            if self.adaptive:
                ce = self.cell(e, base)
                heun = q + (0.5 / self.T) * (_apply(self.flat[c], q) + _apply(self.flat[ce], e))
                e = torch.where(ce == c, e, heun)
            q = e
        return q.reshape(nd, rows, n).transpose(0, 1)

    def _exact1d(self, p):
        n = self.tess[0]
        rows, _, m = p.shape
        base = (torch.arange(rows, device=p.device) * self.nC).repeat_interleave(m)
        x = p.reshape(-1).clone()
        c = _cells(x[None], self.tess)
        left = torch.ones_like(x)
        for _ in range(n + 2):
            a, b = self.flat[base + c, 0, 0], self.flat[base + c, 0, 1]
            v = a * x + b
            nxt = c + torch.sign(v).long()
            wall = torch.where(v > 0, c + 1, c).to(x.dtype) / n
            vw = a * wall + b
            ratio = vw / torch.where(v == 0, torch.ones_like(v), v)
            lin = a.abs() < 1e-12
            hit = torch.where(lin, (wall - x) / torch.where(v == 0, torch.ones_like(v), v),
                              torch.log(ratio.clamp(min=1e-300)) / torch.where(lin, torch.ones_like(a), a))
            stay = (v == 0) | (ratio <= 0) | (nxt < 0) | (nxt >= n) | ~(hit < left) | (left <= 0)
            rel = torch.where(lin, left, torch.expm1(a * left) / torch.where(lin, torch.ones_like(a), a))
            x = torch.where(stay, x + v * rel, wall)
            left = torch.where(stay, torch.zeros_like(left), left - hit)
            c = torch.where(stay, c, nxt)
            if not bool((left > 0).any()):
                break
        return x.reshape(rows, 1, m)

    def _mid(self, q, base, grad_of=None):
        """One explicit-midpoint step (Heun on a crossing when adaptive)."""
        h = 1.0 / self.T
        c = self.cell(q, base)
        A = self.flat[c]
        e = q + h * _apply(A, q + 0.5 * h * _apply(A, q))
        if not self.adaptive:
            return e, c
        ce = self.cell(e, base)
        heun = q + 0.5 * h * (_apply(A, q) + _apply(self.flat[ce], e))
        return torch.where(ce == c, e, heun), c

    def backward(self, p, g):
        """The discrete adjoint of the explicit-midpoint scheme from p: (moments
        [rows, nC, ndim, ndim + 1], gradient of the points)."""
        rows, nd, n = p.shape
        base = (torch.arange(rows, device=p.device) * self.nC).repeat_interleave(n)
        q = p.transpose(0, 1).reshape(nd, -1)
        trail = []
        for _ in range(self.T):
            e, c = self._mid(q, base)
            trail.append((q, c))
            q = e
        h = 1.0 / self.T
        lam = g.to(torch.float64).transpose(0, 1).reshape(nd, -1)
        M = torch.zeros_like(self.flat)
        one = torch.ones(1, q.shape[1], dtype=q.dtype, device=q.device)
        while trail:
            q, c = trail.pop()
            A = self.flat[c]
            At = A[:, :, :nd].transpose(1, 2)
            back = lambda w: (At * w.t()[:, None, :]).sum(-1).t()  # noqa: E731
            mid = q + 0.5 * h * _apply(A, q)
            al = back(lam)
            outer = (h * lam).t()[:, :, None] * torch.cat([mid, one]).t()[:, None, :]
            outer += (0.5 * h * h * al).t()[:, :, None] * torch.cat([q, one]).t()[:, None, :]
            M.index_add_(0, c, outer)
            lam = lam + h * back(lam + 0.5 * h * al)
        return (M.reshape(self.rows, self.nC, nd, nd + 1),
                lam.reshape(nd, rows, n).transpose(0, 1))


def _sample(data, pos, size):
    """Border-clamped linear samples of data [B, C, *in] at pos [B, ndim, n]
    (coordinate 0 fastest), as [B, C, *size], differentiable."""
    B, C = data.shape[:2]
    dims = data.shape[2:]
    nd = len(dims)
    flat = data.reshape(B, C, -1)
    ends, frac = [], []
    for k, s in enumerate(dims):
        # the pixel that a coordinate falls in is the 32-bit product's
        x = pos[:, k] * (s - 1)
        lo = torch.floor(x.detach().float()).double()
        ends.append([lo.clamp(0, s - 1).long(), (lo + 1).clamp(0, s - 1).long()])
        frac.append(x - lo.clamp(0, s - 1))
    out = 0.0
    for corner in range(1 << nd):
        idx, w = 0, 1.0
        for k in range(nd):
            b = (corner >> k) & 1
            idx = idx * dims[k] + ends[k][b]
            w = w * (frac[k] if b else 1 - frac[k])
        out = out + w[:, None] * torch.gather(flat, 2, idx[:, None].expand(B, C, -1))
    out = out.reshape(B, C, *size[::-1])
    return out.permute(0, 1, *range(nd + 1, 1, -1)).contiguous()


def exact(case, seed):
    c = dict(_DEFAULTS, **case)
    st = prepare(case, seed)
    T, nd = st["T"], st["T"].params.ndim
    train = c["train"]
    size = _sizes(c)
    g = st["grad"].double()
    if c["op"] == "interp":
        data = st["data"].detach().double().requires_grad_(st["data"].requires_grad)
        pos = st["points"].detach().double().requires_grad_(st["points"].requires_grad)
        out = _sample(data, pos, size)
        res = {"out": out.detach()}
        if train:
            wanted = [(k, t) for k, t in (("grad_points", pos), ("grad_data", data)) if t.requires_grad]
            res.update(zip([k for k, _ in wanted], torch.autograd.grad(out, [t for _, t in wanted], g)))
        return res
    tess = [c[k] for k in ("nx", "ny", "nz") if c[k]]
    # The basis (part of the program's plan) as the framework's tables hold it.
    coo = T.get_basis().tocoo()
    B = torch.sparse_coo_tensor(
        torch.stack([torch.from_numpy(coo.row).long(), torch.from_numpy(coo.col).long()]),
        torch.from_numpy(coo.data).float().double(), coo.shape).to(DEV).coalesce()
    theta = st["theta"].detach().double().reshape(c["stages"], c["batch"], -1)
    if c["op"] == "chain":
        theta = theta / c["stages"]
    nC = T.params.nC
    flows = [_Flow((B @ th.t()).t().reshape(c["batch"], nC, nd, nd + 1), tess, c["steps"],
                   c["adaptive"]) for th in theta]
    if c["op"] == "image":
        start = T.uniform_meshgrid(size)
    else:
        start = st["points"].detach()
    shared = start.dim() == 2
    p = start.double().expand(c["batch"], nd, -1) if shared else start.double()
    inputs = []
    for f in flows:
        inputs.append(p)
        p = f.forward(p)
    res = {}
    if c["op"] == "image":
        data = st["data"].detach().double().requires_grad_(st["data"].requires_grad)
        p = p.detach().requires_grad_(train)
        out = _sample(data, p, size)
        res["out"] = out.detach()
        if not train:
            return res
        wanted = [p] + ([data] if data.requires_grad else [])
        got = torch.autograd.grad(out, wanted, g)
        lam = got[0]
        if data.requires_grad:
            res["grad_data"] = got[1]
    else:
        res["out"] = p
        if not train:
            return res
        lam = g
    rows = []
    for f, q in zip(flows[::-1], inputs[::-1]):
        M, lam = f.backward(q, lam)
        rows.append((B.t() @ M.reshape(c["batch"], -1).t()).t())
    grad = torch.stack(rows[::-1])
    if c["op"] == "chain":
        grad = grad / c["stages"]
    res["grad_theta"] = grad.reshape(st["theta"].shape)
    if c["points_grad"]:
        res["grad_points"] = lam.sum(0) if shared else lam
    return res
