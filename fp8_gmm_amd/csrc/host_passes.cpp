// The host path of the modules in native code: one call from Python per forward pass, none per backward pass.
//
// A pass of a small layer is bound by its host: its kernels take 50 us, and the Python that allocated its tensors, filled
// the C structures and walked through two autograd functions took 250 - 350 (the backward half of it in the autograd
// engine's thread, where the interpreter's data is cold).  Here a pass is: allocate the results, describe the pass
// (fp8gmm_lay_out_pass), enqueue the kernel that builds its tables, enqueue its launches; the backward pass is a node of
// the autograd graph that does the same without entering the interpreter.
//
// What a pass computes is stated in fp8gmm.h and grouped_linear.py / grouped_mlp.py (reference fp8_gmm/grouped_linear.py:11-183,
// fp8_gmm/grouped_mlp.py:18-325); the Python functions there launch the same kernels with the same tables and serve
// the layouts and options that this file leaves to them.
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>

#include <atomic>

#include "fp8gmm.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

void check(int status) { TORCH_CHECK(status == FP8GMM_OK, "fp8gmm error ", status, ": ", fp8gmm_status_string(status)); }

void* current_stream(const at::Device& device) {
  return c10::hip::getCurrentHIPStream(device.index()).stream();
}

template <class T>
T* ptr(const Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

// Rows per expert, from a CPU tensor or anything that iterates over numbers.
std::vector<int64_t> sizes_of(const py::object& group_sizes) {
  if (THPVariable_Check(group_sizes.ptr())) {
    const Tensor t = THPVariable_Unpack(group_sizes.ptr()).to(at::kCPU, at::kLong).contiguous();
    TORCH_CHECK(t.dim() == 1, "fp8_gmm_amd: group_sizes must be 1-D");
    const int64_t* p = t.const_data_ptr<int64_t>();
    return std::vector<int64_t>(p, p + t.numel());
  }
  std::vector<int64_t> sizes;
  for (const py::handle n : py::iter(group_sizes)) sizes.push_back(py::cast<int64_t>(py::int_(py::reinterpret_borrow<py::object>(n))));
  return sizes;
}

// An exception of Python code that a pass calls - saved-tensor hooks; activation checkpointing ends its recomputation
// with one - reaches the caller as it is.
template <class F>
Tensor with_python_errors(F&& pass) {
  try {
    return pass();
  } catch (python_error& e) {
    e.restore();
    throw py::error_already_set();
  }
}

// How the launches of a module are planned, and its scaling state of both directions.
struct Setup {
  int fwd_fmt = 0, bwd_fmt = 0;
  int grid = 0, stream_k = 0, tile_policy = 0;
  bool two_roundings = false;   // GroupedLinear(cutlass=True)
  Tensor fwd_scale, fwd_scale_inv, fwd_amax, bwd_scale, bwd_scale_inv, bwd_amax;
  at::ScalarType fwd_type() const { return fwd_fmt == FP8GMM_E4M3 ? at::kFloat8_e4m3fn : at::kFloat8_e5m2; }
  at::ScalarType bwd_type() const { return bwd_fmt == FP8GMM_E4M3 ? at::kFloat8_e4m3fn : at::kFloat8_e5m2; }
};

// The scaling update that is due in front of a pass; not any more once it is enqueued.
struct Due {
  bool due = false;
  double fwd_max = 0, bwd_max = 0;
  int margin = 0;
  bool most_recent = false, keep_weights = false;
};

// Whether a block of backend.kernel_timing is open (set_kernel_timing).
std::atomic<bool> kernel_timing{false};

// Enqueues what `launch` does; inside a block of kernel_timing between two events, under what `block` makes of the module
// `backend`: a bracket of that block.  On the current device and stream, as the launch.
template <class Block, class Launch>
void timed(Block&& block, Launch&& launch) {
  if (!kernel_timing.load(std::memory_order_relaxed)) return launch();
  py::gil_scoped_acquire gil;
  const py::object bracket = block(py::module_::import("fp8_gmm_amd.backend"));
  bracket.attr("__enter__")();
  launch();
  bracket.attr("__exit__")(py::none(), py::none(), py::none());
}
// ... that moves `bytes` bytes under a name of its own.
template <class Launch>
void timed(const char* name, int64_t bytes, Launch&& launch) {
  timed([&](const py::module_& backend) { return backend.attr("_timed")(name, py::cpp_function([bytes] { return bytes; })); }, launch);
}

// Builds the tables of a pass and enqueues its launches on the current stream.
void run_pass(int which, const void* desc, const at::Device& device, const Setup* update, Due* due, const Tensor& snapshot_of,
              const Tensor& snapshot, const fp8gmm_routed_rows* routed = nullptr, int64_t rows = 0) {
  fp8gmm_pass_plan plan;
  alignas(16) unsigned char tables[FP8GMM_PASS_TABLES_BYTES];
  check(fp8gmm_lay_out_routed_pass(which, desc, routed, &plan, tables));
  const auto bytes = at::TensorOptions().dtype(at::kByte).device(device);
  const Tensor blob = at::empty({plan.blob_bytes}, bytes);
  void* const stream = current_stream(device);
  fp8gmm_scaling_update updates[2] = {};
  int n = 0;
  if (due != nullptr && due->due) {
    const Tensor* state[2][3] = {{&update->fwd_amax, &update->fwd_scale, &update->fwd_scale_inv},
                                 {&update->bwd_amax, &update->bwd_scale, &update->bwd_scale_inv}};
    for (n = 0; n < 2; ++n) {
      fp8gmm_scaling_update& u = updates[n];
      u.amax_history = ptr<float>(*state[n][0]);
      u.scale = ptr<float>(*state[n][1]);
      u.scale_inv = ptr<float>(*state[n][2]);
      u.history_len = (int32_t)state[n][0]->size(0);
      u.slots = (int32_t)state[n][0]->size(1);
      u.fp8_max = (float)(n == 0 ? due->fwd_max : due->bwd_max);
      u.margin = due->margin;
      u.most_recent = due->most_recent;
      if (n == 0 && due->keep_weights) {   // forward slots: input, weight, output
        u.keep_period = 3;
        u.keep_phase = 1;
      }
    }
  }
  check(fp8gmm_build_pass(tables, blob.data_ptr(), updates, n, ptr<const float>(snapshot_of), ptr<float>(snapshot),
                          snapshot.defined() ? (int)snapshot.numel() : 0, stream));
  if (due != nullptr) due->due = false;
  int slots = 0;
  for (int i = 0; i < plan.n_launches; ++i) slots = std::max(slots, plan.launch[i].plan.n_slots);
  // partial sums of tiles shared along K: from the caching allocator, which hands memory out again in stream order
  Tensor workspace;
  if (slots > 0) workspace = at::empty({(int64_t)slots * FP8GMM_GEMM_SLOT_BYTES}, bytes);
  for (int i = 0; i < plan.n_launches; ++i) {
    const fp8gmm_pass_launch& l = plan.launch[i];
    if (l.kind == FP8GMM_PASS_NOTHING) continue;
    timed([&](const py::module_& backend) {
            return backend.attr("_timed_launch")(py::bytes(reinterpret_cast<const char*>(&l), sizeof(l)));
          },
          [&] {
            check(fp8gmm_run_routed(blob.data_ptr(), &l, routed, rows, ptr<void>(workspace), (size_t)slots * FP8GMM_GEMM_SLOT_BYTES,
                                    stream));
          });
  }
}

// Rows of a pass that come from tokens, go back to tokens, or both: what gather and scatter of a routed layer around the
// module would do (fp8gmm_routed_rows).
struct Route {
  Tensor indices, inverse;   // int32, a permutation of the rows and its inverse, as the sort wrote them
  Tensor weights;            // fp32, of the rows in (token, choice) order: those of scatter
  int64_t top_k = 1;
  bool gathers = false, scatters = false;
};

// `rows`: of the pass.
void check_route(const Route& r, int64_t rows, const Tensor& x) {
  auto list = [&](const Tensor& t, at::ScalarType type) {
    return t.defined() && t.scalar_type() == type && t.dim() == 1 && t.is_contiguous() && t.numel() == rows &&
           t.device() == x.device();
  };
  TORCH_CHECK(r.top_k >= 1 && r.top_k <= FP8GMM_ROUTED_MAX_TOP_K && rows % r.top_k == 0 && rows <= INT32_MAX,
              "fp8_gmm_amd: rows are not top_k of every token");
  TORCH_CHECK(list(r.indices, at::kInt) && list(r.inverse, at::kInt), "fp8_gmm_amd: expected ", rows, " int32 indices");
  TORCH_CHECK(!r.scatters || list(r.weights, at::kFloat), "fp8_gmm_amd: expected ", rows, " fp32 scatter weights");
}

// What a row mover takes: contiguous, on 16 bytes.
Tensor aligned(const Tensor& t) {
  const Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone(at::MemoryFormat::Contiguous);
}

// out[t] = sum of the rows of token t, weighted where `weights` is defined
Tensor scatter_rows(const Tensor& rows, const Tensor& inverse, const Tensor& weights, int64_t top_k) {
  const Tensor out = at::empty({rows.size(0) / top_k, rows.size(1)}, rows.options());
  timed("moe_scatter", 2 * (rows.numel() + out.numel()), [&] {
    check(fp8gmm_moe_scatter(ptr<const void>(rows), ptr<const int32_t>(inverse), ptr<const float>(weights), ptr<void>(out),
                             (int)out.size(0), (int)out.size(1), (int)top_k, current_stream(rows.device())));
  });
  return out;
}

// The part of a route that a backward pass needs.
struct SavedRoute {
  bool gathers = false, scatters = false, want_weights = false;
  int64_t top_k = 1, rows = 0;
  struct Kept {
    SavedVariable indices, inverse, weights, y;
  };
  std::unique_ptr<Kept> kept;   // of a routed pass only
  void save(const Route& r, const Tensor& rows_out, bool dgrad, bool want) {
    gathers = r.gathers;
    scatters = r.scatters;
    want_weights = want;
    top_k = r.top_k;
    rows = r.indices.numel();
    kept = std::make_unique<Kept>();
    if (scatters) {
      kept->weights = SavedVariable(r.weights, false);
      if (want) {
        kept->indices = SavedVariable(r.indices, false);
        kept->y = SavedVariable(rows_out, false);
      }
    }
    if (scatters || (gathers && dgrad)) kept->inverse = SavedVariable(r.inverse, false);
  }
  void reset() {
    if (kept == nullptr) return;
    for (SavedVariable* v : {&kept->indices, &kept->inverse, &kept->weights, &kept->y}) v->reset_data();
  }
  // The kernels follow addresses, and a saved-tensor hook may return anything.
  Tensor list(SavedVariable& v, at::ScalarType type, const at::Device& device) const {
    const Tensor t = v.unpack();
    TORCH_CHECK(t.scalar_type() == type && t.numel() == rows && t.is_contiguous() && t.device() == device,
                "fp8_gmm_amd: a saved-tensor hook returned another tensor than was saved");
    return t;
  }
};

// The gradient of a pass's result as its launches read it: rows, or tokens with what scatter's gradient wants besides.
struct RoutedGradient {
  Tensor dy, inverse, weights, y, grad_weights;
  fp8gmm_routed_rows rows{};
  RoutedGradient(SavedRoute& r, const Tensor& grad, bool want_weights) : dy(grad) {
    if (!r.scatters) return;
    dy = aligned(grad);
    TORCH_CHECK(dy.size(0) * r.top_k == r.rows, "fp8_gmm_amd: a gradient of another size than the result");
    inverse = r.list(r.kept->inverse, at::kInt, dy.device());
    weights = r.list(r.kept->weights, at::kFloat, dy.device());
    if (want_weights) {
      y = r.kept->y.unpack();
      TORCH_CHECK(y.scalar_type() == at::kBFloat16 && y.dim() == 2 && y.size(0) == r.rows && y.size(1) == dy.size(1) &&
                      y.device() == dy.device(),
                  "fp8_gmm_amd: a saved-tensor hook returned another tensor than was saved");
      y = aligned(y);
      grad_weights = at::empty({r.rows}, weights.options());
    }
    rows.inverse = ptr<const int32_t>(inverse);
    rows.weights = ptr<const float>(weights);
    rows.y = ptr<const void>(y);
    rows.grad_weights = ptr<float>(grad_weights);
    rows.top_k = (int32_t)r.top_k;
  }
  const fp8gmm_routed_rows* routed(const SavedRoute& r) const { return r.scatters ? &rows : nullptr; }
  int64_t size(const SavedRoute& r) const { return r.scatters ? r.rows : dy.size(0); }
  // grad_weights alone: nothing upstream of the rows wants a gradient
  void weights_only(SavedRoute& r) const {
    const Tensor indices = r.list(r.kept->indices, at::kInt, dy.device());
    check(fp8gmm_moe_scatter_wgrad(ptr<const void>(y), ptr<const void>(dy), ptr<const int32_t>(indices), rows.grad_weights, (int)r.rows,
                                   (int)dy.size(1), (int)r.top_k, current_stream(dy.device())));
  }
};

// The kernels follow addresses: what they read has to be there.  `w` [experts, out, x's columns].
void check_shapes(const std::vector<int64_t>& sizes, const Tensor& x, const Tensor& w, const Setup& s, int gemms,
                  const Route* route) {
  int64_t rows = 0;
  for (const int64_t n : sizes) rows += n;
  TORCH_CHECK(rows == x.size(0) * (route != nullptr && route->gathers ? route->top_k : 1),
              "group_sizes must sum to the number of input rows");
  if (route != nullptr) check_route(*route, rows, x);
  TORCH_CHECK((int64_t)sizes.size() <= w.size(0), "fp8_gmm_amd: group_sizes has ", sizes.size(), " entries for ", w.size(0),
              " weights");
  TORCH_CHECK(x.size(1) == w.size(2), "fp8_gmm_amd: the input has ", x.size(1), " columns, the weights expect ", w.size(2));
  const int64_t n = (int64_t)sizes.size() * gemms;   // scaling slots: 3 a GEMM forward, 2 backward
  TORCH_CHECK(s.fwd_scale.numel() >= 3 * n && s.fwd_scale_inv.numel() >= 3 * n && s.fwd_amax.size(-1) >= 3 * n &&
                  s.bwd_scale.numel() >= 2 * n && s.bwd_scale_inv.numel() >= 2 * n && s.bwd_amax.size(-1) >= 2 * n,
              "fp8_gmm_amd: the scaling state has too few slots");
}

// Forward-mode differentiation has no rule here and is refused, as the Python functions refuse it: a tangent that is
// silently dropped would be a wrong derivative.
void check_no_tangent(at::TensorList inputs) {
  if (!at::GradMode::is_enabled()) return;
  for (const Tensor& t : inputs)
    TORCH_CHECK(!torch::autograd::isFwGradDefined(t), "fp8_gmm_amd: the grouped modules do not support forward-mode AD");
}

// What a backward pass starts from.  A node behind the pass that returned no gradient stands for zeros, as it does for a
// Python autograd function.
Tensor gradient_of_result(const Node& node, const variable_list& grads) {
  return grads[0].defined() ? grads[0].contiguous() : node.input_metadata(0).zeros_like();
}

// ---- GroupedLinear ------------------------------------------------------------------------------------------------
fp8gmm_linear_pass linear_desc(const Setup& s, const std::vector<int64_t>& sizes, int64_t tokens, int64_t in, int64_t out) {
  fp8gmm_linear_pass d{};
  d.experts = (int32_t)sizes.size();
  d.in_features = (int32_t)in;
  d.out_features = (int32_t)out;
  d.fwd_fmt = s.fwd_fmt;
  d.bwd_fmt = s.bwd_fmt;
  d.grid = s.grid;
  d.stream_k = s.stream_k;
  d.tile_policy = s.tile_policy;
  d.two_roundings = s.two_roundings;
  d.tokens = tokens;
  d.group_sizes = sizes.data();
  return d;
}

struct GroupedLinearBackward : public Node {
  Setup setup;
  std::vector<int64_t> sizes;
  int64_t in = 0, out = 0;
  SavedVariable x_fp8, w_fp8;
  Tensor scale_inv;   // the forward factors as they were
  SavedRoute route;

  std::string name() const override { return "GroupedLinearBackward"; }
  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);   // backward passes of several threads may meet in one graph
    x_fp8.reset_data();
    w_fp8.reset_data();
    route.reset();
  }
  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    at::AutoGradMode no_grad(false);
    variable_list result(route.scatters ? 3 : 2);
    const bool dgrad = task_should_compute_output(0), wgrad = task_should_compute_output(1);
    const bool rgrad = route.want_weights && task_should_compute_output(2);
    const Tensor grad = gradient_of_result(*this, grads);
    const c10::OptionalDeviceGuard guard(grad.device());
    const RoutedGradient from(route, grad, rgrad);
    const Tensor& dy = from.dy;
    if (rgrad) result[2] = from.grad_weights;
    if (!dgrad && !wgrad && route.scatters) {
      if (rgrad) from.weights_only(route);
      return result;
    }
    const int64_t rows = from.size(route);
    const Tensor x = wgrad ? x_fp8.unpack() : Tensor(), w = dgrad ? w_fp8.unpack() : Tensor();
    const Tensor dy_fp8 = at::empty({rows, out}, dy.options().dtype(setup.bwd_type()));
    Tensor dx;
    if (dgrad) dx = at::empty({rows, in}, dy.options());
    if (wgrad) result[1] = at::empty({(int64_t)sizes.size(), out, in}, dy.options());
    fp8gmm_linear_pass d = linear_desc(setup, sizes, rows, in, out);
    d.dgrad = dgrad;
    d.wgrad = wgrad;
    d.dy = ptr<void>(dy);
    d.dy_fp8 = ptr<void>(dy_fp8);
    d.x_fp8 = ptr<void>(x);
    d.w_fp8 = ptr<void>(w);
    d.dx = ptr<void>(dx);
    d.dw = ptr<void>(result[1]);
    d.fwd_scale_inv = ptr<float>(scale_inv);
    d.bwd_scale = ptr<float>(setup.bwd_scale);
    d.bwd_scale_inv = ptr<float>(setup.bwd_scale_inv);
    d.bwd_amax = ptr<float>(setup.bwd_amax);
    run_pass(FP8GMM_LINEAR_BACKWARD, &d, dy.device(), nullptr, nullptr, Tensor(), Tensor(), from.routed(route), rows);
    if (dgrad) result[0] = route.gathers ? scatter_rows(dx, route.list(route.kept->inverse, at::kInt, dx.device()), Tensor(), route.top_k) : dx;
    return result;
  }
};

Tensor linear_step(const Tensor& x, const Tensor& w, const py::object& group_sizes, const std::optional<Tensor>& cached,
                   bool cast_weights, const Setup& setup, Due& due, const Route* route) {
  return with_python_errors([&, sizes = sizes_of(group_sizes)]() mutable {
    py::gil_scoped_release no_gil;
    check_shapes(sizes, x, w, setup, 1, route);
    check_no_tangent({x, w});
    const bool gathers = route != nullptr && route->gathers, scatters = route != nullptr && route->scatters;
    if (scatters) check_no_tangent({route->weights});
    const c10::OptionalDeviceGuard guard(x.device());
    const bool grad = at::GradMode::is_enabled();
    const bool dgrad = grad && x.requires_grad(), wgrad = grad && w.requires_grad();
    const bool rgrad = grad && scatters && route->weights.requires_grad();
    const int64_t tokens = gathers ? x.size(0) * route->top_k : x.size(0);   // rows of the pass
    Tensor y, rows_out, x_fp8, w_fp8, scale_inv;
    {
      at::AutoGradMode no_grad(false);
      const auto fp8 = x.options().dtype(setup.fwd_type());
      x_fp8 = at::empty({tokens, x.size(1)}, fp8);
      w_fp8 = cached.has_value() ? *cached : at::empty(w.sizes(), fp8);
      y = at::empty({tokens, w.size(1)}, x.options());
      if (dgrad || wgrad) scale_inv = at::empty_like(setup.fwd_scale_inv);
      fp8gmm_linear_pass d = linear_desc(setup, sizes, tokens, w.size(2), w.size(1));
      fp8gmm_routed_rows routed{};
      if (gathers) {
        routed.inverse = ptr<const int32_t>(route->inverse);
        routed.top_k = (int32_t)route->top_k;
      }
      d.cast_weights = cast_weights;
      d.x = ptr<void>(x);
      d.x_fp8 = ptr<void>(x_fp8);
      d.w = ptr<void>(w);
      d.w_fp8 = ptr<void>(w_fp8);
      d.y = ptr<void>(y);
      d.fwd_scale = ptr<float>(setup.fwd_scale);
      d.fwd_scale_inv = ptr<float>(setup.fwd_scale_inv);
      d.fwd_amax = ptr<float>(setup.fwd_amax);
      run_pass(FP8GMM_LINEAR_FORWARD, &d, x.device(), &setup, &due, scale_inv.defined() ? setup.fwd_scale_inv : Tensor(),
               scale_inv, gathers ? &routed : nullptr, tokens);
      if (scatters) {
        rows_out = y;
        y = scatter_rows(rows_out, route->inverse, route->weights, route->top_k);
      }
    }
    if (dgrad || wgrad || rgrad) {
      auto node = std::shared_ptr<GroupedLinearBackward>(new GroupedLinearBackward(), torch::autograd::deleteNode);
      if (scatters) node->set_next_edges(torch::autograd::collect_next_edges(x, w, route->weights));
      else node->set_next_edges(torch::autograd::collect_next_edges(x, w));
      if (route != nullptr) node->route.save(*route, rows_out, dgrad, rgrad);
      node->setup = setup;
      node->sizes = std::move(sizes);
      node->in = w.size(2);
      node->out = w.size(1);
      if (wgrad) node->x_fp8 = SavedVariable(x_fp8, false);
      if (dgrad) node->w_fp8 = SavedVariable(w_fp8, false);
      node->scale_inv = scale_inv;
      torch::autograd::set_history(y, node);
    }
    return y;
  });
}

// ---- GroupedMlp ---------------------------------------------------------------------------------------------------
fp8gmm_mlp_pass mlp_desc(const Setup& s, const std::vector<int64_t>& sizes, int64_t tokens, int64_t hidden, int64_t ffn) {
  fp8gmm_mlp_pass d{};
  d.experts = (int32_t)sizes.size();
  d.hidden = (int32_t)hidden;
  d.ffn = (int32_t)ffn;
  d.fwd_fmt = s.fwd_fmt;
  d.bwd_fmt = s.bwd_fmt;
  d.grid = s.grid;
  d.stream_k = s.stream_k;
  d.tile_policy = s.tile_policy;
  d.tokens = tokens;
  d.group_sizes = sizes.data();
  return d;
}

struct GroupedMlpBackward : public Node {
  Setup setup;
  std::vector<int64_t> sizes;
  bool dgrad = false, wgrad = false;
  int64_t hidden = 0, ffn = 0;
  SavedVariable x_fp8, w1_fp8, w2_fp8, pre, act_fp8;
  Tensor scale_inv;
  SavedRoute route;

  std::string name() const override { return "GroupedMlpBackward"; }
  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);   // backward passes of several threads may meet in one graph
    for (SavedVariable* v : {&x_fp8, &w1_fp8, &w2_fp8, &pre, &act_fp8}) v->reset_data();
    route.reset();
  }
  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    at::AutoGradMode no_grad(false);
    variable_list result(route.scatters ? 4 : 3);
    const bool want_x = dgrad && task_should_compute_output(0);
    const bool want_w = wgrad && (task_should_compute_output(1) || task_should_compute_output(2));
    const bool rgrad = route.want_weights && task_should_compute_output(3);
    const Tensor grad = gradient_of_result(*this, grads);
    const c10::OptionalDeviceGuard guard(grad.device());
    const RoutedGradient from(route, grad, rgrad);
    const Tensor& dy = from.dy;
    if (rgrad) result[3] = from.grad_weights;
    if (!want_x && !want_w && route.scatters) {
      if (rgrad) from.weights_only(route);
      return result;
    }
    const int64_t tokens = from.size(route), e = (int64_t)sizes.size();
    const auto bf16 = dy.options(), fp8 = dy.options().dtype(setup.bwd_type());
    const Tensor p = pre.unpack(), w2 = w2_fp8.unpack(), w1 = want_x ? w1_fp8.unpack() : Tensor();
    const Tensor x = want_w ? x_fp8.unpack() : Tensor(), act = want_w ? act_fp8.unpack() : Tensor();
    const Tensor dy_fp8 = at::empty({tokens, hidden}, fp8), dact = at::empty({tokens, ffn}, bf16), dpre = at::empty({tokens, ffn}, fp8);
    Tensor dx;
    if (want_x) dx = at::empty({tokens, hidden}, bf16);
    if (want_w) {
      result[1] = at::empty({e, ffn, hidden}, bf16);
      result[2] = at::empty({e, hidden, ffn}, bf16);
    }
    fp8gmm_mlp_pass d = mlp_desc(setup, sizes, tokens, hidden, ffn);
    d.dgrad = want_x;
    d.wgrad = want_w;
    d.x_fp8 = ptr<void>(x);
    d.w1_fp8 = ptr<void>(w1);
    d.w2_fp8 = ptr<void>(w2);
    d.pre = ptr<void>(p);
    d.act_fp8 = ptr<void>(act);
    d.dy = ptr<void>(dy);
    d.dy_fp8 = ptr<void>(dy_fp8);
    d.dact = ptr<void>(dact);
    d.dpre_fp8 = ptr<void>(dpre);
    d.dx = ptr<void>(dx);
    d.dw1 = ptr<void>(result[1]);
    d.dw2 = ptr<void>(result[2]);
    d.fwd_scale_inv = ptr<float>(scale_inv);
    d.bwd_scale = ptr<float>(setup.bwd_scale);
    d.bwd_scale_inv = ptr<float>(setup.bwd_scale_inv);
    d.bwd_amax = ptr<float>(setup.bwd_amax);
    run_pass(FP8GMM_MLP_BACKWARD, &d, dy.device(), nullptr, nullptr, Tensor(), Tensor(), from.routed(route), tokens);
    if (want_x) result[0] = route.gathers ? scatter_rows(dx, route.list(route.kept->inverse, at::kInt, dx.device()), Tensor(), route.top_k) : dx;
    return result;
  }
};

Tensor mlp_step(const Tensor& x, const Tensor& w1, const Tensor& w2, const py::object& group_sizes,
                const std::optional<Tensor>& cached1, const std::optional<Tensor>& cached2, bool cast_weights,
                const Setup& setup, Due& due, const Route* route) {
  return with_python_errors([&, sizes = sizes_of(group_sizes)]() mutable {
    py::gil_scoped_release no_gil;
    check_shapes(sizes, x, w1, setup, 2, route);
    TORCH_CHECK(w2.size(0) == w1.size(0) && w2.size(1) == w1.size(2) && w2.size(2) == w1.size(1),
                "fp8_gmm_amd: fc2's weights do not follow fc1's");
    check_no_tangent({x, w1, w2});
    const bool gathers = route != nullptr && route->gathers, scatters = route != nullptr && route->scatters;
    if (scatters) check_no_tangent({route->weights});
    const c10::OptionalDeviceGuard guard(x.device());
    const bool grad = at::GradMode::is_enabled();
    const bool dgrad = grad && x.requires_grad(), wgrad = grad && w1.requires_grad();
    const bool rgrad = grad && scatters && route->weights.requires_grad();
    const int64_t tokens = gathers ? x.size(0) * route->top_k : x.size(0), hidden = x.size(1), ffn = w1.size(1);   // rows of the pass
    Tensor y, rows_out, x_fp8, w1_fp8, w2_fp8, pre, act_fp8, scale_inv;
    {
      at::AutoGradMode no_grad(false);
      const auto fp8 = x.options().dtype(setup.fwd_type());
      x_fp8 = at::empty({tokens, hidden}, fp8);
      w1_fp8 = cached1.has_value() ? *cached1 : at::empty(w1.sizes(), fp8);
      w2_fp8 = cached2.has_value() ? *cached2 : at::empty(w2.sizes(), fp8);
      pre = at::empty({tokens, ffn}, x.options());
      act_fp8 = at::empty({tokens, ffn}, fp8);
      y = at::empty({tokens, hidden}, x.options());
      if (dgrad || wgrad) scale_inv = at::empty_like(setup.fwd_scale_inv);
      fp8gmm_mlp_pass d = mlp_desc(setup, sizes, tokens, hidden, ffn);
      fp8gmm_routed_rows routed{};
      if (gathers) {
        routed.inverse = ptr<const int32_t>(route->inverse);
        routed.top_k = (int32_t)route->top_k;
      }
      d.cast_weights = cast_weights;
      d.x = ptr<void>(x);
      d.x_fp8 = ptr<void>(x_fp8);
      d.w1 = ptr<void>(w1);
      d.w1_fp8 = ptr<void>(w1_fp8);
      d.w2 = ptr<void>(w2);
      d.w2_fp8 = ptr<void>(w2_fp8);
      d.pre = ptr<void>(pre);
      d.act_fp8 = ptr<void>(act_fp8);
      d.y = ptr<void>(y);
      d.fwd_scale = ptr<float>(setup.fwd_scale);
      d.fwd_scale_inv = ptr<float>(setup.fwd_scale_inv);
      d.fwd_amax = ptr<float>(setup.fwd_amax);
      run_pass(FP8GMM_MLP_FORWARD, &d, x.device(), &setup, &due, scale_inv.defined() ? setup.fwd_scale_inv : Tensor(),
               scale_inv, gathers ? &routed : nullptr, tokens);
      if (scatters) {
        rows_out = y;
        y = scatter_rows(rows_out, route->inverse, route->weights, route->top_k);
      }
    }
    if (dgrad || wgrad || rgrad) {
      auto node = std::shared_ptr<GroupedMlpBackward>(new GroupedMlpBackward(), torch::autograd::deleteNode);
      if (scatters) node->set_next_edges(torch::autograd::collect_next_edges(x, w1, w2, route->weights));
      else node->set_next_edges(torch::autograd::collect_next_edges(x, w1, w2));
      if (route != nullptr) node->route.save(*route, rows_out, dgrad, rgrad);
      node->setup = setup;
      node->sizes = std::move(sizes);
      node->dgrad = dgrad;
      node->wgrad = wgrad;
      node->hidden = hidden;
      node->ffn = ffn;
      if (dgrad || wgrad) {
        node->pre = SavedVariable(pre, false);
        node->w2_fp8 = SavedVariable(w2_fp8, false);
      }
      if (dgrad) node->w1_fp8 = SavedVariable(w1_fp8, false);
      if (wgrad) {
        node->x_fp8 = SavedVariable(x_fp8, false);
        node->act_fp8 = SavedVariable(act_fp8, false);
      }
      node->scale_inv = scale_inv;
      torch::autograd::set_history(y, node);
    }
    return y;
  });
}

// ---- weights ahead of a pass --------------------------------------------------------------------------------------
// What a forward pass does before its rows are known: a pass without rows, which is the scaling update and the casts of
// one weight stack (GroupedLinear) or two (GroupedMlp) into `fp8`.
void cast_weights(const std::vector<Tensor>& weights, const std::vector<Tensor>& fp8, const Setup& setup, Due& due) {
  py::gil_scoped_release no_gil;
  TORCH_CHECK((weights.size() == 1 || weights.size() == 2) && fp8.size() == weights.size(),
              "fp8_gmm_amd: one or two weight stacks and a result for each");
  const Tensor& w = weights[0];
  for (size_t i = 0; i < weights.size(); ++i)
    TORCH_CHECK(weights[i].dim() == 3 && weights[i].sizes() == fp8[i].sizes() && weights[i].is_contiguous() &&
                    fp8[i].is_contiguous() && weights[i].size(0) == w.size(0) && weights[i].device() == w.device() &&
                    fp8[i].device() == w.device() && weights[i].scalar_type() == at::kBFloat16 &&
                    fp8[i].scalar_type() == setup.fwd_type(),
                "fp8_gmm_amd: weight stacks and results that do not fit together");
  if (weights.size() == 2)
    TORCH_CHECK(weights[1].size(1) == w.size(2) && weights[1].size(2) == w.size(1),
                "fp8_gmm_amd: fc2's weights do not follow fc1's");
  const std::vector<int64_t> sizes((size_t)w.size(0), 0);
  const int64_t slots = 3 * w.size(0) * (int64_t)weights.size();
  TORCH_CHECK(setup.fwd_scale.numel() >= slots && setup.fwd_scale_inv.numel() >= slots && setup.fwd_amax.size(-1) >= slots,
              "fp8_gmm_amd: the scaling state has too few slots");
  const c10::OptionalDeviceGuard guard(w.device());
  auto run = [&](int which, auto& d) {
    d.cast_weights = 1;
    d.fwd_scale = ptr<float>(setup.fwd_scale);
    d.fwd_scale_inv = ptr<float>(setup.fwd_scale_inv);
    d.fwd_amax = ptr<float>(setup.fwd_amax);
    run_pass(which, &d, w.device(), &setup, &due, Tensor(), Tensor());
  };
  if (weights.size() == 1) {
    fp8gmm_linear_pass d = linear_desc(setup, sizes, 0, w.size(2), w.size(1));
    d.w = ptr<void>(w);
    d.w_fp8 = ptr<void>(fp8[0]);
    run(FP8GMM_LINEAR_FORWARD, d);
  } else {
    fp8gmm_mlp_pass d = mlp_desc(setup, sizes, 0, w.size(2), w.size(1));
    d.w1 = ptr<void>(w);
    d.w1_fp8 = ptr<void>(fp8[0]);
    d.w2 = ptr<void>(weights[1]);
    d.w2_fp8 = ptr<void>(fp8[1]);
    run(FP8GMM_MLP_FORWARD, d);
  }
}

// ---- routing around the experts -----------------------------------------------------------------------------------
// What moe_ops._Gating, _TopK and the sort do, without the interpreter: a short batch waits for its host, and a routed layer's
// forward and backward pass through those took 250 of 600 us.

// (x weight^T, x): the logits, and x once more for what follows, so that its two gradients meet here and one kernel adds them.
struct GatingBackward : public Node {
  int64_t hidden = 0;
  SavedVariable x, weight;   // what torch's linear would keep: with a frozen weight the rows may be changed in place afterwards

  std::string name() const override { return "GatingBackward"; }
  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data();
    weight.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    variable_list result(2);
    const Tensor &grad = grads[0], &grad_in = grads[1];
    if (!grad.defined()) {
      result[0] = grad_in;
      return result;
    }
    const c10::OptionalDeviceGuard guard(grad.device());
    const bool want_x = task_should_compute_output(0), want_weight = task_should_compute_output(1);
    const int64_t tokens = grad.size(0), experts = grad.size(1);
    const Tensor rows = want_weight ? x.unpack() : Tensor(), w = want_x ? weight.unpack() : Tensor();
    auto as_saved = [&](const Tensor& t, int64_t n) {
      return t.scalar_type() == at::kBFloat16 && t.device() == grad.device() && t.dim() == 2 && t.size(0) == n && t.size(1) == hidden;
    };
    // a graph of the backward pass is asked for, or a saved-tensor hook returned what the kernels do not read: torch's products
    if (at::GradMode::is_enabled() || (want_weight && !as_saved(rows, tokens)) || (want_x && !as_saved(w, experts))) {
      if (want_x) result[0] = grad_in.defined() ? grad_in + grad.mm(w) : grad.mm(w);
      if (want_weight) result[1] = grad.t().mm(rows);
      return result;
    }
    const Tensor g = aligned(grad), in = grad_in.defined() ? aligned(grad_in) : Tensor();
    const Tensor xs = want_weight ? aligned(rows) : Tensor(), ws = want_x ? w.contiguous() : Tensor();
    if (want_x) result[0] = at::empty({tokens, hidden}, g.options());
    Tensor work;
    if (want_weight) {
      result[1] = at::empty({experts, hidden}, g.options());
      work = at::empty({(int64_t)fp8gmm_gating_workspace_bytes((int)tokens, (int)hidden, (int)experts)}, g.options().dtype(at::kByte));
    }
    timed("gating_backward", 2 * tokens * hidden * (want_weight + 2 * want_x), [&] {
      check(fp8gmm_gating_backward(ptr<void>(g), ptr<void>(xs), ptr<void>(ws), ptr<void>(in), ptr<void>(result[0]),
                                   ptr<void>(result[1]), (int)tokens, (int)hidden, (int)experts, ptr<void>(work),
                                   current_stream(g.device())));
    });
    return result;
  }
};

std::pair<Tensor, Tensor> gating(const Tensor& x, const Tensor& weight) {
  py::gil_scoped_release no_gil;
  TORCH_CHECK(x.dim() == 2 && weight.dim() == 2 && x.size(1) == weight.size(1) && x.scalar_type() == at::kBFloat16 &&
                  weight.scalar_type() == at::kBFloat16 && x.is_contiguous() && weight.is_contiguous(),
              "fp8_gmm_amd: rows and gate that do not fit together");
  check_no_tangent({x, weight});
  Tensor logits, rows;
  {
    at::AutoGradMode no_grad(false);
    logits = at::linear(x, weight);
    rows = x.detach();
  }
  auto node = std::shared_ptr<GatingBackward>(new GatingBackward(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(x, weight));
  node->hidden = x.size(1);
  if (weight.requires_grad()) node->x = SavedVariable(x, false);
  if (x.requires_grad()) node->weight = SavedVariable(weight, false);
  torch::autograd::set_history(logits, node);
  torch::autograd::set_history(rows, node);
  return {logits, rows};
}

// The chain from the weights of the chosen experts back to the scores.
struct RouteTopKBackward : public Node {
  SavedVariable probs, selected;
  int64_t tokens = 0, experts = 0, top_k = 0;
  at::ScalarType type = at::kBFloat16;

  std::string name() const override { return "RouteTopKBackward"; }
  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    probs.reset_data();
    selected.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    at::AutoGradMode no_grad(false);
    const Tensor grad = gradient_of_result(*this, grads), p = probs.unpack(), s = selected.unpack();
    TORCH_CHECK(p.scalar_type() == at::kFloat && p.numel() == tokens * experts && p.is_contiguous() && p.device() == grad.device() &&
                    s.scalar_type() == at::kLong && s.numel() == tokens * top_k && s.is_contiguous() && s.device() == grad.device(),
                "fp8_gmm_amd: a saved-tensor hook returned another tensor than was saved");
    const c10::OptionalDeviceGuard guard(grad.device());
    const Tensor result = at::empty({tokens, experts}, grad.options().dtype(type));
    check(fp8gmm_route_topk_backward(ptr<float>(p), ptr<int64_t>(s), ptr<float>(grad), (int)tokens, (int)experts, (int)top_k,
                                     ptr<void>(result), type == at::kBFloat16, current_stream(grad.device())));
    return {result};
  }
};

// Rows per expert on their way to the host.
struct Counts {
  Tensor host;   // page-locked
  c10::Event event;
  std::vector<int64_t> wait() {
    event.synchronize();
    const int32_t* p = host.const_data_ptr<int32_t>();
    return std::vector<int64_t>(p, p + host.numel());
  }
};

// The router's choice, the sort of its (token, choice) pairs by expert and the copy of the experts' row counts to the host:
// (weights fp32 [tokens * top_k], indices, bin_ids, bins, tokens_per_expert, inverse, Counts).
py::tuple route(const Tensor& scores, int64_t top_k) {
  Tensor weights, indices, bin_ids, bins, counts, inverse;
  std::unique_ptr<Counts> copy;
  {
    py::gil_scoped_release no_gil;
    TORCH_CHECK(scores.is_cuda() && scores.dim() == 2 && scores.is_contiguous() &&
                    (scores.scalar_type() == at::kBFloat16 || scores.scalar_type() == at::kFloat) &&
                    scores.size(0) * top_k <= INT32_MAX,
                "fp8_gmm_amd: scores that the routing kernels do not take");
    check_no_tangent({scores});
    const c10::OptionalDeviceGuard guard(scores.device());
    const int64_t tokens = scores.size(0), experts = scores.size(1), rows = tokens * top_k;
    const bool grad = at::GradMode::is_enabled() && scores.requires_grad();
    void* const stream = current_stream(scores.device());
    Tensor probs, selected;
    {
      at::AutoGradMode no_grad(false);
      const auto ints = scores.options().dtype(at::kInt);
      probs = at::empty({tokens, experts}, scores.options().dtype(at::kFloat));
      weights = at::empty({rows}, probs.options());
      selected = at::empty({tokens, top_k}, scores.options().dtype(at::kLong));
      check(fp8gmm_route_topk(ptr<void>(scores), scores.scalar_type() == at::kBFloat16, (int)tokens, (int)experts, (int)top_k,
                              ptr<float>(probs), ptr<float>(weights), ptr<int64_t>(selected), stream));
      indices = at::empty({rows}, ints);
      bin_ids = at::empty({rows}, ints);
      inverse = at::empty({rows}, ints);
      counts = at::empty({experts}, ints);
      bins = at::empty({experts}, ints);
      const Tensor work = at::empty({(int64_t)fp8gmm_route_workspace_bytes((int)rows, (int)experts)}, ints.dtype(at::kByte));
      check(fp8gmm_route_sort_selected(ptr<int64_t>(selected), (int)rows, (int)experts, ptr<int32_t>(bin_ids), ptr<int32_t>(indices),
                                       ptr<int32_t>(inverse), ptr<int32_t>(counts), ptr<int32_t>(bins), ptr<void>(work), stream));
      copy.reset(new Counts{at::empty({experts}, at::TensorOptions().dtype(at::kInt).pinned_memory(true)),
                            c10::Event(scores.device().type())});
      copy->host.copy_(counts, /*non_blocking=*/true);
      copy->event.record(c10::impl::VirtualGuardImpl(scores.device().type()).getStream(scores.device()));
    }
    if (grad) {
      auto node = std::shared_ptr<RouteTopKBackward>(new RouteTopKBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(scores));
      node->probs = SavedVariable(probs, false);
      node->selected = SavedVariable(selected, false);
      node->tokens = tokens;
      node->experts = experts;
      node->top_k = top_k;
      node->type = scores.scalar_type();
      torch::autograd::set_history(weights, node);
    }
  }
  return py::make_tuple(weights, indices, bin_ids, bins, counts, inverse, std::move(copy));
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.doc() = "Host path of the grouped modules in native code (see host_passes.cpp).";
  py::class_<Setup>(m, "Setup")
      .def(py::init([](int fwd_fmt, int bwd_fmt, int grid, const Tensor& fs, const Tensor& fsi, const Tensor& fa,
                       const Tensor& bs, const Tensor& bsi, const Tensor& ba) {
        Setup s;
        s.fwd_fmt = fwd_fmt;
        s.bwd_fmt = bwd_fmt;
        s.grid = grid;
        s.fwd_scale = fs;
        s.fwd_scale_inv = fsi;
        s.fwd_amax = fa;
        s.bwd_scale = bs;
        s.bwd_scale_inv = bsi;
        s.bwd_amax = ba;
        return s;
      }))
      .def_readonly("fwd_fmt", &Setup::fwd_fmt)
      .def_readwrite("stream_k", &Setup::stream_k)
      .def_readwrite("two_roundings", &Setup::two_roundings)
      .def_readwrite("tile_policy", &Setup::tile_policy);
  py::class_<Due>(m, "Due")
      .def(py::init<>())
      .def(py::init([](double fwd_max, double bwd_max, int margin, bool most_recent, bool keep_weights) {
        return Due{true, fwd_max, bwd_max, margin, most_recent, keep_weights};
      }))
      .def_readonly("due", &Due::due);
  py::class_<Route>(m, "Route")
      .def(py::init([](const Tensor& indices, const Tensor& inverse, const std::optional<Tensor>& weights, int64_t top_k,
                       bool gathers, bool scatters) {
        return Route{indices, inverse, weights.value_or(Tensor()), top_k, gathers, scatters};
      }));
  m.def("linear_step", &linear_step, py::arg("x"), py::arg("w"), py::arg("group_sizes"), py::arg("cached"), py::arg("cast_weights"),
        py::arg("setup"), py::arg("due"), py::arg("route") = nullptr);
  m.def("mlp_step", &mlp_step, py::arg("x"), py::arg("w1"), py::arg("w2"), py::arg("group_sizes"), py::arg("cached1"),
        py::arg("cached2"), py::arg("cast_weights"), py::arg("setup"), py::arg("due"), py::arg("route") = nullptr);
  m.def("cast_weights", &cast_weights);
  py::class_<Counts>(m, "Counts").def("wait", &Counts::wait, py::call_guard<py::gil_scoped_release>());
  m.def("gating", &gating);
  m.def("route", &route);
  m.def("set_kernel_timing", [](bool on) { kernel_timing.store(on, std::memory_order_relaxed); });
}
