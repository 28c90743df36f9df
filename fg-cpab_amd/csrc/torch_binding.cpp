// Native autograd functions over the C ABI (include/cpab_hip.h): what
// cpab/pytorch/transformer.py and interpolation.py call.  Each holds the
// checks, allocations, library calls and saved tensors of one differentiable
// operation, and its backward runs on the autograd engine's thread without
// going back through Python (except to read params.deterministic_grad).
//
// Why native: the smallest calls are bound by the host.  One forward + backward
// of 16 x 10,000 1D points (35 us of kernels) took 122 us with the functions as
// torch.autograd.Function over ctypes and takes 67 here; 32 x 784 2D points 132
// and 75, 16 x 60,001 2D points in 20 steps 137 and 90.
#include <torch/extension.h>

#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>

#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "cpab_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

[[noreturn]] void fail(const std::string& msg) { throw std::runtime_error(msg); }

void check(int rc, const char* what) {
  if (rc != 0) fail(std::string(what) + " failed: " + cpab_last_error_string());
}

std::string shape_of(const Tensor& t) {   // as str(tuple(t.shape))
  std::ostringstream s;
  s << "(";
  for (int64_t k = 0; k < t.dim(); ++k) s << (k ? ", " : "") << t.size(k);
  s << (t.dim() == 1 ? ",)" : ")");
  return s.str();
}

std::string dtype_of(const Tensor& t) {
  return std::string("torch.") + c10::getDtypeNames(t.scalar_type()).first;
}

const float* in(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
float* out(Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

Tensor empty(at::IntArrayRef size, const Tensor& like) {
  return at::empty(size, at::TensorOptions().device(like.device()).dtype(at::kFloat));
}

// Device memory used by this call alone: back in torch's caching allocator,
// for work queued behind it on the current stream, when the call returns.
at::DataPtr scratch(int64_t bytes) {
  return c10::hip::HIPCachingAllocator::get()->allocate((size_t)(bytes > 0 ? bytes : 1));
}

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// The tables of basis_tables() (transformer.py) and the solver's parameters as
// they are at the call; kept from forward to backward.
struct Call : torch::CustomClassHolder {
  Tensor row_ptr, col_idx, vals, col_ptr, row_idx, vals_t;
  int d = 0, ndim = 0, nC = 0, T = 0, adaptive = 0;
  int nc[3] = {1, 1, 1};
  int64_t K = 1, n = 0, nP = 0;
  bool batched = false, points_grad = false;
  std::vector<int64_t> outsize;
  PyObject* params = nullptr;

  Call(const py::object& p, const py::dict& tab) {
    auto get = [&](const char* k) { return tab[k].cast<Tensor>(); };
    row_ptr = get("row_ptr");
    col_idx = get("col_idx");
    vals = get("vals");
    col_ptr = get("col_ptr");
    row_idx = get("row_idx");
    vals_t = get("vals_t");
    d = tab["d"].cast<int>();
    ndim = p.attr("ndim").cast<int>();
    nC = py::int_(p.attr("nC")).cast<int>();
    T = py::int_(p.attr("nstepsolver")).cast<int>();
    adaptive = py::hasattr(p, "adaptive_substeps") && py::bool_(p.attr("adaptive_substeps")) ? 1 : 0;
    int k = 0;
    for (const auto& v : p.attr("nc")) {
      if (k == 3) break;
      nc[k++] = py::int_(py::reinterpret_borrow<py::object>(v)).cast<int>();
    }
    params = p.ptr();
    Py_INCREF(params);
  }
  ~Call() override {
    if (!Py_IsInitialized()) return;
    py::gil_scoped_acquire gil;
    Py_XDECREF(params);
  }
  int ppc() const { return ndim * (ndim + 1); }
  // Whether the backward uses the deterministic reduction, read when it runs.
  bool deterministic() const {
    py::gil_scoped_acquire gil;
    const py::handle p(params);
    return py::hasattr(p, "deterministic_grad") && py::bool_(p.attr("deterministic_grad"));
  }
};

// This thread's deterministic setting for the duration of a backward.
struct Deterministic {
  int before;
  explicit Deterministic(bool on) : before(cpab_deterministic()) { cpab_set_deterministic(on ? 1 : 0); }
  ~Deterministic() { cpab_set_deterministic(before); }
};

c10::intrusive_ptr<Call> call_of(AutogradContext* ctx) {
  return c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
}
void keep(AutogradContext* ctx, const c10::intrusive_ptr<Call>& c) {
  ctx->saved_data["call"] =
      c10::IValue::make_capsule(c10::static_intrusive_pointer_cast<torch::CustomClassHolder>(c));
}

// torch.autograd.function.once_differentiable: the gradients cannot be
// differentiated again.
variable_list once(variable_list grads, const Tensor& grad_out) {
  if (!at::GradMode::is_enabled() || !grad_out.requires_grad()) return grads;
  for (Tensor& g : grads)
    if (g.defined()) g = g.detach().set_requires_grad(true);
  torch::autograd::DelayedError err(
      "trying to differentiate twice a function that was marked with @once_differentiable",
      (int64_t)grads.size());
  return err.apply(std::move(grads));
}

Tensor plain(const Tensor& t) { return t.detach().contiguous(); }
Tensor grad_of(const Tensor& g) { return g.detach().to(at::kFloat).contiguous(); }

// Shape and type checks shared by the point transforms; theta of one stage.
void check_inputs(const Tensor& points, const Tensor& theta, Call& c, int64_t d) {
  if (theta.scalar_type() != at::kFloat || points.scalar_type() != at::kFloat)
    fail("expected float32 tensors, got points " + dtype_of(points) + ", theta " + dtype_of(theta));
  if (theta.dim() != 2 || theta.size(1) != d)
    fail("theta must have shape [n_batch, " + std::to_string(d) + "], got " + shape_of(theta));
  if (points.device() != theta.device()) fail("points and theta must be on the same device");
  c.n = theta.size(0);
  c.batched = points.dim() == 3 && points.size(0) == c.n;
  if (points.dim() == 3 && !c.batched)
    fail("batched points have " + std::to_string(points.size(0)) + " entries but theta has " +
         std::to_string(c.n));
  if ((points.dim() != 2 && points.dim() != 3) || points.size(-2) != c.ndim)
    fail("points must be [" + std::to_string(c.ndim) + ", nP] or [n_batch, " +
         std::to_string(c.ndim) + ", nP], got " + shape_of(points));
  c.nP = points.size(-1);
}

// A = B theta and (2D/3D) the one-step maps of `rows` thetas.
Tensor tables(const Call& c, const Tensor& theta, int64_t rows, at::DataPtr& trels, void* s) {
  Tensor As = empty({rows, c.nC, c.ndim, c.ndim + 1}, theta);
  const auto* rp = c.row_ptr.data_ptr<int32_t>();
  const auto* ci = c.col_idx.data_ptr<int32_t>();
  if (c.ndim == 1) {
    check(cpab_affine(1, rows, c.nC, (int)theta.size(-1), in(theta), rp, ci, in(c.vals), out(As), s),
          "cpab_affine");
  } else {
    trels = scratch(As.numel() * 4);
    check(cpab_affine_expm(c.ndim, rows, c.nC, (int)theta.size(-1), in(theta), rp, ci, in(c.vals),
                           (float)(1.0 / (double)c.T), out(As), static_cast<float*>(trels.get()), s),
          "cpab_affine_expm");
  }
  return As;
}

Tensor summed(const Tensor& gp, void* s) {
  Tensor sum = empty({gp.size(1), gp.size(2)}, gp);
  check(cpab_sum_batch(gp.size(0), sum.numel(), in(gp), out(sum), s), "cpab_sum_batch");
  return sum;
}

// One transform, or a chain of K (theta_stages [K, n, d]).
struct Grid : torch::autograd::Function<Grid> {
  static Tensor forward(AutogradContext* ctx, const Tensor& points, const Tensor& theta,
                        const c10::intrusive_ptr<Call>& call, bool chain, bool save_stages) {
    Call& c = *call;
    const c10::OptionalDeviceGuard guard(theta.device());
    void* s = stream_of(theta);
    const Tensor th = plain(theta), pts = plain(points);
    const int64_t rows = c.K * c.n;
    at::DataPtr trels;
    const Tensor As = tables(c, th, rows, trels, s);
    const float* tr = static_cast<const float*>(trels.get());
    Tensor res = empty({c.n, c.ndim, c.nP}, theta), stages;
    if (chain) {
      if (save_stages && c.K > 1) stages = empty({c.K - 1, c.n, c.ndim, c.nP}, theta);
      check(cpab_chain_forward(c.ndim, c.nP, c.n, c.batched, (int)c.K, c.T, c.nc[0], c.nc[1],
                               c.nc[2], c.adaptive, in(pts), tr, in(As), out(res), out(stages), s),
            "cpab_chain_forward");
    } else if (c.ndim == 1) {
      check(cpab_forward_1d_closed_form(c.nP, c.n, c.batched, c.nc[0], in(pts), in(As), out(res), s),
            "cpab_forward_1d_closed_form");
    } else {
      check(cpab_forward(c.ndim, c.nP, c.n, c.batched, c.T, c.nc[0], c.nc[1], c.nc[2], c.adaptive,
                         in(pts), tr, in(As), out(res), s),
            "cpab_forward");
    }
    keep(ctx, call);
    ctx->saved_data["chain"] = chain;
    ctx->save_for_backward({pts, As, stages});
    return res;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    Tensor gp, gtheta;
    {
      const at::NoGradGuard no_grad;
      const auto saved = ctx->get_saved_variables();
      const Tensor &pts = saved[0], &As = saved[1], &stages = saved[2];
      const auto call = call_of(ctx);
      const Call& c = *call;
      const bool chain = ctx->saved_data["chain"].toBool();
      const c10::OptionalDeviceGuard guard(As.device());
      void* s = stream_of(As);
      const Tensor g = grad_of(grads[0]);
      const bool want_points = c.points_grad && ctx->needs_input_grad(0);
      if (want_points) gp = empty({c.n, c.ndim, c.nP}, As);
      gtheta = chain ? empty({c.K, c.n, c.d}, As) : empty({c.n, c.d}, As);
      const at::DataPtr moments = scratch(c.K * c.n * c.nC * c.ppc() * 4);
      const Deterministic det(c.deterministic());
      const int64_t bytes =
          chain ? cpab_chain_backward_workspace_size(c.ndim, c.nP, c.n, (int)c.K, c.nC)
                : cpab_backward_workspace_size(c.ndim, c.nP, c.n, c.nC);
      at::DataPtr ws;
      if (bytes > 0) ws = scratch(bytes);
      const auto* cp = c.col_ptr.data_ptr<int32_t>();
      const auto* ri = c.row_idx.data_ptr<int32_t>();
      auto* m = static_cast<float*>(moments.get());
      if (chain)
        check(cpab_chain_backward(c.ndim, c.nP, c.n, c.batched, (int)c.K, c.T, c.nc[0], c.nc[1],
                                  c.nc[2], c.adaptive, in(pts), in(stages), in(As), in(g), c.d, cp,
                                  ri, in(c.vals_t), m, out(gtheta), out(gp), ws.get(), bytes, s),
              "cpab_chain_backward");
      else
        check(cpab_backward_project(c.ndim, c.nP, c.n, c.batched, c.T, c.nc[0], c.nc[1], c.nc[2],
                                    c.adaptive, in(pts), in(As), in(g), c.d, cp, ri, in(c.vals_t),
                                    m, out(gtheta), out(gp), ws.get(), bytes, s),
              "cpab_backward_project");
      if (want_points && pts.dim() == 2) gp = summed(gp, s);
    }
    return once({gp, gtheta, Tensor(), Tensor(), Tensor()}, grads[0]);
  }
};

Tensor grid(const Tensor& points, const Tensor& theta, const py::object& params,
            const py::dict& tab, bool points_grad) {
  auto c = c10::make_intrusive<Call>(params, tab);
  check_inputs(points, theta, *c, params.attr("d").cast<int64_t>());
  c->points_grad = points_grad;
  py::gil_scoped_release nogil;
  return Grid::apply(points, theta, c, false, false);
}

Tensor chain(const Tensor& points, const Tensor& theta, const py::object& params,
             const py::dict& tab) {
  if (theta.dim() != 3)
    fail("theta_stages must be [n_stages, n_batch, d], got " + shape_of(theta));
  auto c = c10::make_intrusive<Call>(params, tab);
  check_inputs(points, theta.detach().select(0, 0), *c, params.attr("d").cast<int64_t>());
  c->K = theta.size(0);
  c->points_grad = true;
  const bool save =
      at::GradMode::is_enabled() && (points.requires_grad() || theta.requires_grad());
  py::gil_scoped_release nogil;
  return Grid::apply(points, theta, c, true, save);
}

// transform_data: integrate the uniform grid and resample in one pass.
struct Image : torch::autograd::Function<Image> {
  static Tensor forward(AutogradContext* ctx, const Tensor& data, const Tensor& theta,
                        const Tensor& axes, const c10::intrusive_ptr<Call>& call, bool need_data,
                        bool need_theta) {
    Call& c = *call;
    const c10::OptionalDeviceGuard guard(theta.device());
    void* s = stream_of(theta);
    const Tensor d = plain(data), ax = plain(axes), th = plain(theta);
    at::DataPtr trels;
    const Tensor As = tables(c, th, c.n, trels, s);
    // For the backward: with one channel and no grad_data the sample's
    // spatial gradient at each final point (the seed then needs no data
    // reads); the final points themselves when grad_data's scatter or
    // several channels need them.
    const bool one = data.size(1) == 1;
    Tensor seed, fin;
    if (need_theta && one && !need_data) seed = empty({c.n, c.ndim, c.nP}, theta);
    if (need_data || (need_theta && !one)) fin = empty({c.n, c.ndim, c.nP}, theta);
    std::vector<int64_t> size{c.n, data.size(1)};
    size.insert(size.end(), c.outsize.begin(), c.outsize.end());
    Tensor res = empty(size, theta);
    check(cpab_transform_data_forward(c.ndim, c.n, d.size(1), d.sizes().data() + 2,
                                      c.outsize.data(), c.T, c.nc[0], c.nc[1], c.nc[2], c.adaptive,
                                      in(ax), static_cast<const float*>(trels.get()), in(As), in(d),
                                      out(res), out(fin), out(seed), s),
          "cpab_transform_data_forward");
    keep(ctx, call);
    ctx->saved_data["need_data"] = need_data;
    ctx->saved_data["need_theta"] = need_theta;
    ctx->save_for_backward({d, ax, fin, seed, As});
    return res;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    Tensor gdata, gtheta;
    {
      const at::NoGradGuard no_grad;
      const auto saved = ctx->get_saved_variables();
      const Tensor &d = saved[0], &ax = saved[1], &fin = saved[2], &seed = saved[3], &As = saved[4];
      const auto call = call_of(ctx);
      const Call& c = *call;
      const c10::OptionalDeviceGuard guard(As.device());
      void* s = stream_of(As);
      const Tensor g = grad_of(grads[0]);
      if (ctx->saved_data["need_data"].toBool()) gdata = at::empty_like(d);
      if (ctx->saved_data["need_theta"].toBool()) gtheta = empty({c.n, c.d}, As);
      const Deterministic det(c.deterministic());
      // the data's gradient alone needs no trajectories
      const bool alone = gdata.defined() && !gtheta.defined() && cpab_deterministic() == 0 &&
                         c.T >= 1 && c.T <= CPAB_MAX_STEPS;   // other counts are refused below
      if (alone) {
        check(cpab_transform_data_backward_data(c.ndim, c.n, d.size(1), d.sizes().data() + 2,
                                                c.outsize.data(), in(fin), in(g), out(gdata), s),
              "cpab_transform_data_backward_data");
      } else {
        const at::DataPtr moments = scratch(c.n * c.nC * c.ppc() * 4);
        int64_t bytes =
            cpab_transform_data_backward_workspace_size(c.ndim, c.n, c.outsize.data(), c.nC);
        if (gdata.defined())
          bytes += cpab_transform_data_backward_data_workspace_size(c.ndim, c.n, d.size(1),
                                                                    d.sizes().data() + 2);
        at::DataPtr ws;
        if (bytes > 0) ws = scratch(bytes);
        const bool proj = gtheta.defined();
        check(cpab_transform_data_backward(
                  c.ndim, c.n, d.size(1), d.sizes().data() + 2, c.outsize.data(), c.T, c.nc[0],
                  c.nc[1], c.nc[2], c.adaptive, in(ax), in(fin), in(seed), in(As), in(d), in(g),
                  proj ? c.d : 0, proj ? c.col_ptr.data_ptr<int32_t>() : nullptr,
                  proj ? c.row_idx.data_ptr<int32_t>() : nullptr, proj ? in(c.vals_t) : nullptr,
                  static_cast<float*>(moments.get()), out(gtheta), out(gdata), ws.get(), bytes, s),
              "cpab_transform_data_backward");
      }
    }
    return once({gdata, gtheta, Tensor(), Tensor(), Tensor(), Tensor()}, grads[0]);
  }
};

Tensor image(const Tensor& data, const Tensor& theta, const Tensor& axes,
             std::vector<int64_t> outsize, const py::object& params, const py::dict& tab) {
  auto c = c10::make_intrusive<Call>(params, tab);
  const int64_t d = params.attr("d").cast<int64_t>();
  if (data.scalar_type() != at::kFloat || theta.scalar_type() != at::kFloat)
    fail("expected float32 data and theta");
  if (data.dim() != c->ndim + 2)
    fail("data must be [n_batch, n_channels, *in_size] with " + std::to_string(c->ndim) +
         " spatial axes");
  if (theta.dim() != 2 || theta.size(1) != d || theta.size(0) != data.size(0))
    fail("theta must be [n_batch=" + std::to_string(data.size(0)) + ", " + std::to_string(d) +
         "], got " + shape_of(theta));
  int64_t nP = 1, sum = 0;
  for (const int64_t v : outsize) {
    nP *= v;
    sum += v;
  }
  if ((int)outsize.size() != c->ndim || axes.dim() != 1 || axes.size(0) != sum)
    fail("axes must be the [sum(outsize)] per-axis coordinates of the grid");
  c->n = theta.size(0);
  c->nP = nP;
  c->outsize = std::move(outsize);
  const bool grad = at::GradMode::is_enabled();   // without it nothing is kept for a backward
  const bool need_data = grad && data.requires_grad(), need_theta = grad && theta.requires_grad();
  py::gil_scoped_release nogil;
  return Image::apply(data, theta, axes, c, need_data, need_theta);
}

struct Interp : torch::autograd::Function<Interp> {
  static Tensor forward(AutogradContext* ctx, const Tensor& data, const Tensor& grid, int64_t ndim,
                        const std::vector<int64_t>& outsize, bool deterministic, bool need_data,
                        bool need_grid) {
    const c10::OptionalDeviceGuard guard(data.device());
    const Tensor d = plain(data), gr = plain(grid);
    std::vector<int64_t> size{data.size(0), data.size(1)};
    size.insert(size.end(), outsize.begin(), outsize.end());
    Tensor res = empty(size, data);
    check(cpab_interp_forward((int)ndim, d.size(0), d.size(1), d.sizes().data() + 2, outsize.data(),
                              in(d), in(gr), out(res), stream_of(d)),
          "cpab_interp_forward");
    ctx->saved_data["outsize"] = outsize;
    ctx->saved_data["deterministic"] = deterministic;
    ctx->saved_data["need_data"] = need_data;
    ctx->saved_data["need_grid"] = need_grid;
    ctx->save_for_backward({d, gr});
    return res;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    Tensor gdata, ggrid;
    {
      const at::NoGradGuard no_grad;
      const auto saved = ctx->get_saved_variables();
      const Tensor &d = saved[0], &gr = saved[1];
      const c10::OptionalDeviceGuard guard(d.device());
      void* s = stream_of(d);
      const int ndim = (int)d.dim() - 2;
      const int64_t* dims = d.sizes().data() + 2;
      const std::vector<int64_t> outsize = ctx->saved_data["outsize"].toIntVector();
      const Tensor g = grad_of(grads[0]);
      if (ctx->saved_data["need_grid"].toBool()) ggrid = at::empty_like(gr);
      if (ctx->saved_data["need_data"].toBool()) gdata = at::empty_like(d);
      if (ctx->saved_data["deterministic"].toBool() && gdata.defined()) {
        const Deterministic det(true);
        const int64_t bytes =
            cpab_interp_backward_workspace_size(ndim, d.size(0), d.size(1), dims);
        const at::DataPtr ws = scratch(bytes);
        check(cpab_interp_backward_ws(ndim, d.size(0), d.size(1), dims, outsize.data(), in(d),
                                      in(gr), in(g), out(ggrid), out(gdata), ws.get(), bytes, s),
              "cpab_interp_backward_ws");
      } else if (gdata.defined() || ggrid.defined()) {
        check(cpab_interp_backward(ndim, d.size(0), d.size(1), dims, outsize.data(), in(d), in(gr),
                                   in(g), out(ggrid), out(gdata), s),
              "cpab_interp_backward");
      }
    }
    return once({gdata, ggrid, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()}, grads[0]);
  }
};

Tensor interp(int64_t ndim, const Tensor& data, const Tensor& grid, std::vector<int64_t> outsize,
              bool deterministic) {
  if (!(data.is_cuda() && grid.is_cuda())) fail("interpolate: only GPU tensors are supported");
  if (data.scalar_type() != at::kFloat || grid.scalar_type() != at::kFloat)
    fail("interpolate: expected float32, got data " + dtype_of(data) + ", grid " + dtype_of(grid));
  if (data.dim() != ndim + 2 || (int64_t)outsize.size() != ndim)
    fail("interpolate: data must be [B, C, *" + std::to_string(ndim) +
         " sizes] and outsize have " + std::to_string(ndim) + " entries");
  int64_t nP = 1;
  for (const int64_t v : outsize) nP *= v;
  if (grid.dim() != 3 || grid.size(0) != data.size(0) || grid.size(1) != ndim || grid.size(2) != nP)
    fail("interpolate: grid must be [" + std::to_string(data.size(0)) + ", " +
         std::to_string(ndim) + ", " + std::to_string(nP) + "], got " + shape_of(grid));
  const bool need_data = data.requires_grad(), need_grid = grid.requires_grad();
  py::gil_scoped_release nogil;
  return Interp::apply(data, grid, ndim, outsize, deterministic, need_data, need_grid);
}

}  // namespace

PYBIND11_MODULE(_cpab_torch, m) {
  m.def("grid", &grid);
  m.def("chain", &chain);
  m.def("image", &image);
  m.def("interp", &interp);
}
