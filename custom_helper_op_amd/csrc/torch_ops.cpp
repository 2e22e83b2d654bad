// The host path between torch and the C ABI, in C++: argument checks, output allocation, the
// launches and the autograd nodes of the five operators, as the extension module `_chop_torch`.
//
// What bounds a small call is this path, not the GPU: in Python (checks, ctypes, one
// torch.autograd.Function each way) a tiny forward cost 22 us of host time against 8 us on the
// GPU and a small training pass 77 us against 33 us.  Here a call parses its arguments once with
// the interpreter's fast calling convention, releases the interpreter lock, and the backward
// pass takes it for nothing of its own (saved-tensor hooks and errors do).
//
// A node hung on the result does not take part in everything that an autograd function of Python
// does: while torch.jit records a trace, under the transforms of torch.func and where an input
// carries a forward-mode tangent the call goes through one (ops._Operator), which is recorded, or
// refused with torch's own message.
//
// The checks and their order (types, then shapes) are those of CostVolumeOp::Compute and its siblings
// (custom_helper_op/cc/kernels/cost_volume_kernels.cc:91-106, :220-243;
// cost_volume_kernels_v2.cc:93-110; cost_volume_kernels_v3.cc:94-115, :231-255;
// cost_aggregate_kernels.cc:85-106, :196-226; feature_aggregate_kernels.cc:69-92, :176-210).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <mutex>
#include <string>

#include "../../include/chop_costvol.h"

namespace {

using at::Tensor;

// the operators, numbered as ops.py passes them
enum Op { V1 = 0, V2 = 1, AGGREGATE = 2, V3 = 3, FEATURE = 4 };

PyObject *g_invalid_argument = nullptr;  // ops.InvalidArgumentError
PyObject *g_chop_error = nullptr;        // _lib.ChopError
PyObject *g_recorded = nullptr;          // ops._recorded

struct InvalidArgument : std::runtime_error {
  using std::runtime_error::runtime_error;
};
struct LibraryError : std::runtime_error {
  int code;
  LibraryError(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};
struct PythonError {};  // the interpreter's error indicator is set

inline void require(bool ok, const char *message) {
  if (!ok) throw InvalidArgument(message);
}
inline void check(int rc) {
  if (rc != CHOP_OK) throw LibraryError(rc, chop_last_error_string());
}

// One call of an operator.
struct Call {
  Op op = V1;
  int reduce = 0, half = 1;
  int64_t groups = 1;
  bool grid = false;  // per-voxel hypotheses in `depth` (V2 always; V1 in 16-bit storage by choice)
  Tensor ref, src, depth, offsets, Rs, Ts, default_cost;
  // set by checked()
  int64_t B = 0, H = 0, W = 0, C = 0, D = 0, N = 0, srcH = 0, srcW = 0;
};

inline int storage16(at::ScalarType t) {
  return t == at::kHalf ? CHOP_STORAGE_F16 : t == at::kBFloat16 ? CHOP_STORAGE_BF16 : 0;
}

const char *dtype_name(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return "torch.float32";
    case at::kDouble: return "torch.float64";
    case at::kHalf: return "torch.float16";
    case at::kBFloat16: return "torch.bfloat16";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    default: return c10::toString(t);
  }
}

Tensor prepared(const Tensor &t, at::ScalarType dtype, at::Device device, const char *name) {
  if (t.scalar_type() != dtype)
    throw InvalidArgument(std::string(name) + " must have dtype " + dtype_name(dtype) + ", got " +
                          dtype_name(t.scalar_type()));
  if (t.device() != device) throw InvalidArgument(std::string(name) + " must live on " + device.str());
  return t.is_contiguous() ? t : t.contiguous();
}

inline bool shaped(const Tensor &t, at::IntArrayRef want) { return t.sizes() == want; }

// Types, devices and shapes of a call's inputs and, for a gradient, of what flows back and of the
// mask; makes them contiguous and fills in the sizes.
void check_inputs(Call &c, Tensor *cost_grad = nullptr, Tensor *mask = nullptr) {
  const Tensor &lead = c.op == FEATURE ? c.src : c.ref;
  const at::ScalarType dt = lead.scalar_type();
  const at::Device dev = lead.device();
  at::ScalarType real = dt;
  if (c.op == V1 || c.op == V2) {
    require(dt == at::kFloat || dt == at::kDouble || storage16(dt),
            "dtype must be float32 or float64 (float16/bfloat16 storage as an extension)");
    if (storage16(dt)) real = at::kFloat;
  } else {
    require(dt == at::kFloat || dt == at::kDouble, "dtype must be float32 or float64");
  }
  if (c.op != FEATURE) c.ref = prepared(c.ref, dt, dev, "ref_image");
  c.src = prepared(c.src, dt, dev, "src_images");
  auto depth_inputs = [&] {
    c.depth = prepared(c.depth, real, dev, c.grid ? "depth_grid" : "base_plane");
    if (!c.grid) c.offsets = prepared(c.offsets, real, dev, "offsets");
  };
  auto cameras = [&] {
    c.Rs = prepared(c.Rs, real, dev, "Rs");
    c.Ts = prepared(c.Ts, real, dev, "Ts");
  };
  if (c.op != V1) depth_inputs();
  cameras();
  if (cost_grad != nullptr) {
    *cost_grad = prepared(*cost_grad, dt, dev, c.op == FEATURE ? "mapped_feature_grad" : "cost_grad");
    *mask = prepared(*mask, at::kInt, dev, c.op == FEATURE ? "mapped_mask" : "cost_mask");
  }
  if (c.op == V1) depth_inputs();
  if (c.op == FEATURE) {
    require(c.src.dim() == 5, "src_images must have rank 5");
    c.B = c.src.size(0), c.N = c.src.size(1), c.srcH = c.src.size(2), c.srcW = c.src.size(3);
    c.C = c.src.size(4);
    require(c.depth.dim() == 4 && c.depth.size(0) == c.B && c.depth.size(3) == 1,
            "base_plane must have rank 4, and must compate to ref_image");
    c.H = c.depth.size(1), c.W = c.depth.size(2);
    require(c.offsets.dim() == 2 && c.offsets.size(0) == c.B,
            "offsets must have rank 2, and must compate to ref_image");
  } else {
    if (c.op == V1 && c.grid)
      require(storage16(dt), "depth_grid with the squared-difference op needs float16 or bfloat16 features");
    require(c.ref.dim() == 4, "ref image must have rank 4");
    c.B = c.ref.size(0), c.H = c.ref.size(1), c.W = c.ref.size(2), c.C = c.ref.size(3);
    require(c.src.dim() == 5 && c.src.size(0) == c.B && c.src.size(2) == c.H && c.src.size(3) == c.W &&
                c.src.size(4) == c.C,
            "src_images must have rank 5, and must compate to ref_image");
    c.N = c.src.size(1), c.srcH = c.H, c.srcW = c.W;
  }
  require(shaped(c.Rs, {c.B, c.N, 3, 3}), "Rs must have rank 2, and must compate to ref_image");
  require(shaped(c.Ts, {c.B, c.N, 3}), "Ts must have rank 2, and must compate to ref_image");
  if (c.grid) {
    require(c.depth.dim() == 4 && c.depth.size(0) == c.B && c.depth.size(1) == c.H && c.depth.size(2) == c.W,
            "depth_grid must have rank 4, and must compate to ref_image");
    c.D = c.depth.size(3);
  } else {
    if (c.op != FEATURE) {
      require(shaped(c.depth, {c.B, c.H, c.W, 1}), "base_plane must have rank 4, and must compate to ref_image");
      require(c.offsets.dim() == 2 && c.offsets.size(0) == c.B,
              "offsets must have rank 2, and must compate to ref_image");
    }
    c.D = c.offsets.size(1);
  }
  if (c.op == V2)
    require(c.groups > 0 && c.C % c.groups == 0, "image_channels must be divisible by groups");
  if (c.op == V3) {
    require(c.groups > 0 && c.C % c.groups == 0, "image_channels and groups_ must match");
    require(c.C / c.groups <= 8, "image_channels / groups_ less than MAX_SUBCHANNELS_SIZE(8)");
  }
}

// values per voxel in the cost and in the mask, and the tensors' shapes
at::DimVector cost_shape(const Call &c) {
  at::DimVector s{c.B, c.H, c.W, c.D};
  if (c.op == V1) s.push_back(c.C);
  if (c.op == V2) s.push_back(c.groups);
  if (c.op == V3) s.push_back(1);
  if (c.op == FEATURE) s.push_back(c.N), s.push_back(c.C);
  return s;
}
at::DimVector mask_shape(const Call &c) {
  at::DimVector s{c.B, c.H, c.W, c.D};
  if (c.op == V1) s.push_back(c.reduce == 0 ? 1 : c.C);
  if (c.op == V2) s.push_back(c.reduce == 0 ? 1 : c.groups);
  if (c.op == V3) s.push_back(c.reduce == 0 ? 1 : 3);
  if (c.op == FEATURE) s.push_back(c.N), s.push_back(1);
  return s;
}

inline void *current_stream(const Tensor &t) {
  return static_cast<void *>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}
inline void on_gpu(const Tensor &t) {
  if (!t.is_cuda()) throw InvalidArgument("Expected a cuda device, but got: " + t.device().str());
}

template <typename T>
inline T *ptr(const Tensor &t) {
  return t.defined() ? static_cast<T *>(t.data_ptr()) : nullptr;
}

#define CHOP_DIMS c.B, c.H, c.W, c.C, c.D, c.N, c.srcH, c.srcW
#define CHOP_BY_TYPE(STEM, ...)                                            \
  (dt == at::kFloat ? [&] { using T = float; return STEM##_f32(__VA_ARGS__); }() \
                    : [&] { using T = double; return STEM##_f64(__VA_ARGS__); }())

// Forward: allocates and launches.  The inputs have been checked.
void forward(const Call &c, Tensor &cost, Tensor &mask) {
  const Tensor &lead = c.op == FEATURE ? c.src : c.ref;
  on_gpu(lead);
  const c10::DeviceGuard guard(lead.device());
  const at::ScalarType dt = lead.scalar_type();
  const auto options = lead.options().requires_grad(false);
  cost = at::empty(cost_shape(c), options);
  mask = at::empty(mask_shape(c), options.dtype(at::kInt));
  void *s = current_stream(lead);
  int32_t *m = ptr<int32_t>(mask);
  const int groups = (int)c.groups, r = c.reduce, h = c.half;
  const bool fill = c.default_cost.defined();
  if (const int st = storage16(dt)) {
    void *ref = ptr<void>(c.ref), *src = ptr<void>(c.src), *out = ptr<void>(cost);
    const float *depth = ptr<float>(c.depth), *Rs = ptr<float>(c.Rs), *Ts = ptr<float>(c.Ts);
    if (c.op == V1)
      check(chop_cost_volume_fwd_16(s, st, r, h, CHOP_DIMS, ref, src, c.grid ? nullptr : depth,
                                    ptr<float>(c.offsets), c.grid ? depth : nullptr, Rs, Ts, out, m));
    else if (fill)
      check(chop_cost_volume_v2_fwd_fill_16(s, st, r, h, CHOP_DIMS, groups, ref, src, depth, Rs, Ts,
                                            ptr<float>(c.default_cost), out, m));
    else
      check(chop_cost_volume_v2_fwd_16(s, st, r, h, CHOP_DIMS, groups, ref, src, depth, Rs, Ts, out, m));
    return;
  }
#define CHOP_PLANE ptr<T>(c.depth), ptr<T>(c.offsets), ptr<T>(c.Rs), ptr<T>(c.Ts)
  switch (c.op) {
    case V1:
      check(CHOP_BY_TYPE(chop_cost_volume_fwd, s, r, h, CHOP_DIMS, ptr<T>(c.ref), ptr<T>(c.src), CHOP_PLANE,
                         ptr<T>(cost), m));
      break;
    case V2:
      if (fill)
        check(CHOP_BY_TYPE(chop_cost_volume_v2_fwd_fill, s, r, h, CHOP_DIMS, groups, ptr<T>(c.ref),
                           ptr<T>(c.src), ptr<T>(c.depth), ptr<T>(c.Rs), ptr<T>(c.Ts),
                           ptr<T>(c.default_cost), ptr<T>(cost), m));
      else
        check(CHOP_BY_TYPE(chop_cost_volume_v2_fwd, s, r, h, CHOP_DIMS, groups, ptr<T>(c.ref), ptr<T>(c.src),
                           ptr<T>(c.depth), ptr<T>(c.Rs), ptr<T>(c.Ts), ptr<T>(cost), m));
      break;
    case AGGREGATE:
      if (fill)
        check(CHOP_BY_TYPE(chop_cost_aggregate_fwd_fill, s, r, h, CHOP_DIMS, ptr<T>(c.ref), ptr<T>(c.src),
                           CHOP_PLANE, ptr<T>(c.default_cost), ptr<T>(cost), m));
      else
        check(CHOP_BY_TYPE(chop_cost_aggregate_fwd, s, r, h, CHOP_DIMS, ptr<T>(c.ref), ptr<T>(c.src),
                           CHOP_PLANE, ptr<T>(cost), m));
      break;
    case V3:
      check(CHOP_BY_TYPE(chop_cost_volume_v3_fwd, s, r, h, CHOP_DIMS, groups, ptr<T>(c.ref), ptr<T>(c.src),
                         CHOP_PLANE, ptr<T>(cost), m));
      break;
    case FEATURE:
      check(CHOP_BY_TYPE(chop_feature_aggregate_fwd, s, h, CHOP_DIMS, ptr<T>(c.src), CHOP_PLANE,
                         ptr<T>(cost), m));
      break;
  }
}

// Gradient: `depth_grad` stays undefined when it is not wanted (V3 and FeatureAggregate always
// compute it).  Everything has been checked but the shapes of the upstream gradient and the mask.
void backward(const Call &c, const Tensor &cost_grad, const Tensor &mask, bool want_depth, Tensor &ref_grad, Tensor &src_grad,
              Tensor &depth_grad) {
  const Tensor &lead = c.op == FEATURE ? c.src : c.ref;
  const at::ScalarType dt = lead.scalar_type();
  const char *mis_grad[] = {"cost_grad must have rank 5, and must compate to ref_image",
                            "cost_grad must have rank 5, and must compate to ref_image",
                            "cost_grad must have rank 4, and must compate to ref_image",
                            "cost_grad must have rank 5, and must compate to ref_image",
                            "mapped_feature_grad must have rank 6, and must compate to src_images"};
  const char *mis_mask[] = {"cost_mask must have rank 5, and must compate to ref_image",
                            "cost_mask must have rank 5, and must compate to ref_image",
                            "cost_mask must have rank 4, and must compate to ref_image",
                            "cost_mask must have rank 5, and must compate to ref_image",
                            "mapped_mask must have rank 6, and must compate to src_images"};
  require(shaped(cost_grad, cost_shape(c)), mis_grad[c.op]);
  require(shaped(mask, mask_shape(c)), mis_mask[c.op]);
  on_gpu(lead);
  const c10::DeviceGuard guard(lead.device());
  const auto options = lead.options().requires_grad(false);
  if (c.op != FEATURE) ref_grad = at::empty(c.ref.sizes(), options);
  src_grad = at::empty(c.src.sizes(), options);
  if (want_depth || c.op == V3 || c.op == FEATURE)
    depth_grad = at::empty(c.depth.sizes(), c.depth.options().requires_grad(false));
  void *s = current_stream(lead);
  const int32_t *m = ptr<int32_t>(mask);
  const int groups = (int)c.groups, r = c.reduce, h = c.half;
  if (const int st = storage16(dt)) {
    const size_t need = chop_cost_volume_bwd16_workspace_bytes(c.B, c.H, c.W, c.C, c.N, c.srcH, c.srcW);
    const Tensor ws = at::empty({(int64_t)(need > 0 ? need : 1)}, options.dtype(at::kByte));
    void *ref = ptr<void>(c.ref), *src = ptr<void>(c.src), *cg = ptr<void>(cost_grad);
    const float *depth = ptr<float>(c.depth), *Rs = ptr<float>(c.Rs), *Ts = ptr<float>(c.Ts);
    if (c.op == V1)
      check(chop_cost_volume_bwd_16(s, st, r, h, CHOP_DIMS, ref, src, c.grid ? nullptr : depth,
                                    ptr<float>(c.offsets), c.grid ? depth : nullptr, Rs, Ts, cg, m,
                                    ptr<void>(ref_grad), ptr<void>(src_grad), ptr<float>(depth_grad),
                                    ptr<void>(ws), need));
    else
      check(chop_cost_volume_v2_bwd_16(s, st, r, h, CHOP_DIMS, groups, ref, src, depth, Rs, Ts, cg, m,
                                       ptr<void>(ref_grad), ptr<void>(src_grad), ptr<float>(depth_grad),
                                       ptr<void>(ws), need));
    return;
  }
#define CHOP_GRADS ptr<T>(cost_grad), m, ptr<T>(ref_grad), ptr<T>(src_grad), ptr<T>(depth_grad)
  switch (c.op) {
    case V1:
      check(CHOP_BY_TYPE(chop_cost_volume_bwd, s, r, h, CHOP_DIMS, ptr<T>(c.ref), ptr<T>(c.src), CHOP_PLANE,
                         CHOP_GRADS));
      break;
    case V2:
      check(CHOP_BY_TYPE(chop_cost_volume_v2_bwd, s, r, h, CHOP_DIMS, groups, ptr<T>(c.ref), ptr<T>(c.src),
                         ptr<T>(c.depth), ptr<T>(c.Rs), ptr<T>(c.Ts), CHOP_GRADS));
      break;
    case AGGREGATE:
      check(CHOP_BY_TYPE(chop_cost_aggregate_bwd, s, r, h, CHOP_DIMS, ptr<T>(c.ref), ptr<T>(c.src), CHOP_PLANE,
                         CHOP_GRADS));
      break;
    case V3:
      check(CHOP_BY_TYPE(chop_cost_volume_v3_bwd, s, r, h, CHOP_DIMS, groups, ptr<T>(c.ref), ptr<T>(c.src),
                         CHOP_PLANE, CHOP_GRADS));
      break;
    case FEATURE:
      check(CHOP_BY_TYPE(chop_feature_aggregate_bwd, s, h, CHOP_DIMS, ptr<T>(c.src), CHOP_PLANE,
                         ptr<T>(cost_grad), m, ptr<T>(src_grad), ptr<T>(depth_grad)));
      break;
  }
}

// Gradient of the layers' scalar default: the upstream gradient summed over the voxels that
// received it (16-bit storage is read as stored and summed in float).
Tensor default_gradient(int reduce, const Tensor &g, const Tensor &mask, const Tensor &like) {
  require(like.numel() == 1, "default_cost must be a scalar");
  const c10::DeviceGuard guard(g.device());
  const at::ScalarType dt = g.scalar_type();
  const int64_t n_mask = mask.numel(), inner = n_mask ? g.numel() / n_mask : 1;
  Tensor out = at::empty(like.sizes(), g.options().requires_grad(false).dtype(storage16(dt) ? at::kFloat : dt));
  void *s = current_stream(g);
  const int32_t *m = ptr<int32_t>(mask);
  if (const int st = storage16(dt))
    check(chop_cost_default_fill_grad_16(s, st, reduce, n_mask, inner, ptr<void>(g), m, nullptr, ptr<float>(out)));
  else
    check(CHOP_BY_TYPE(chop_cost_default_fill_grad, s, reduce, n_mask, inner, ptr<T>(g), m, nullptr, ptr<T>(out)));
  return out.scalar_type() == like.scalar_type() ? out : out.to(like.scalar_type());
}

// The exception in flight as the interpreter's error; its lock is held.
void set_error() {
  try {
    throw;
  } catch (const PythonError &) {
  } catch (const InvalidArgument &e) {
    PyErr_SetString(g_invalid_argument, e.what());
  } catch (const LibraryError &e) {
    PyObject *args = Py_BuildValue("(is)", e.code, e.what());
    if (args != nullptr) {
      PyErr_SetObject(g_chop_error, args);
      Py_DECREF(args);
    }
  } catch (...) {
    // torch's own, and what Python code called from here raised: a saved-tensor hook may end the
    // call with an exception of its own, as checkpointing does where it has recomputed enough
    torch::translate_exception_to_python(std::current_exception());
  }
}

// The exception in flight as one of Python, for threads that do not hold the lock.
python_error as_python_error() {
  const PyGILState_STATE lock = PyGILState_Ensure();
  set_error();
  python_error e;
  e.persist();
  PyGILState_Release(lock);
  return e;
}

// ---- autograd -------------------------------------------------------------------------------
// The gradient registered for an operator (custom_helper_ops.py:41-61, :74-94, :107-131,
// :141-161, :174-195): the Grad op is fed the forward's mask; offsets, Rs and Ts receive no
// gradient.  Edges: ref, src, depth, offsets, Rs, Ts, default.
struct OpBackward : public torch::autograd::Node {
  Op op = V1;
  int reduce = 0, half = 1;
  int64_t groups = 1;
  bool grid = false;
  torch::autograd::SavedVariable ref, src, depth, offsets, Rs, Ts, default_cost, mask;

  std::string name() const override { return "CostVolumeBackward"; }
  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    for (auto *v : {&ref, &src, &depth, &offsets, &Rs, &Ts, &default_cost, &mask}) v->reset_data();
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    // The engine knows the types of torch's exceptions and of those that come from Python; any other
    // it raises as a bare RuntimeError.
    try {
      return gradients(std::move(grads));
    } catch (const InvalidArgument &) {
      throw as_python_error();
    } catch (const LibraryError &) {
      throw as_python_error();
    }
  }
  torch::autograd::variable_list gradients(torch::autograd::variable_list &&grads) {
    const std::lock_guard<std::mutex> lock(mutex_);
    const c10::AutoGradMode no_grad(false);
    Call c;
    c.op = op, c.reduce = reduce, c.half = half, c.groups = groups, c.grid = grid;
    c.ref = ref.unpack(), c.src = src.unpack(), c.depth = depth.unpack(), c.offsets = offsets.unpack();
    c.Rs = Rs.unpack(), c.Ts = Ts.unpack(), c.default_cost = default_cost.unpack();
    Tensor m = mask.unpack();
    Tensor g = grads[0].defined() ? grads[0] : input_metadata(0).zeros_like();
    // all of them again: a saved-tensor hook may have given back something else
    check_inputs(c, &g, &m);
    torch::autograd::variable_list out(7);
    backward(c, g, m, task_should_compute_output(2), out[0], out[1], out[2]);
    if (c.default_cost.defined() && task_should_compute_output(6))
      out[6] = default_gradient(reduce, g, m, c.default_cost);
    return out;
  }
};

inline bool wants_grad(const Tensor &t) { return t.defined() && t.requires_grad(); }

// Runs a checked call's forward and, where an input requires a gradient, hangs the node on it.
// `given` holds the inputs as the caller passed them (not made contiguous): they are what the
// graph continues from and what is saved.
void differentiable_forward(const Call &given, Call &c, Tensor &cost, Tensor &mask) {
  const bool any = c10::GradMode::is_enabled() &&
                   (wants_grad(given.ref) || wants_grad(given.src) || wants_grad(given.depth) ||
                    wants_grad(given.offsets) || wants_grad(given.Rs) || wants_grad(given.Ts) ||
                    wants_grad(given.default_cost));
  {
    const c10::AutoGradMode no_grad(false);
    check_inputs(c);
    if (c.default_cost.defined()) {
      const Tensor &lead = c.ref;
      const at::ScalarType dt = lead.scalar_type();
      c.default_cost = prepared(c.default_cost, storage16(dt) ? at::kFloat : dt, lead.device(), "default_cost");
      require(c.default_cost.numel() == 1, "default_cost must be a scalar");
    }
    forward(c, cost, mask);
  }
  if (!any) return;
  std::shared_ptr<OpBackward> node(new OpBackward(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(given.ref, given.src, given.depth, given.offsets,
                                                           given.Rs, given.Ts, given.default_cost));
  node->op = c.op, node->reduce = c.reduce, node->half = c.half, node->groups = c.groups, node->grid = c.grid;
  using torch::autograd::SavedVariable;
  auto save = [](const Tensor &t) { return t.defined() ? SavedVariable(t, false) : SavedVariable(); };
  node->ref = save(given.ref), node->src = save(given.src), node->depth = save(given.depth);
  node->offsets = save(given.offsets), node->Rs = save(given.Rs), node->Ts = save(given.Ts);
  node->default_cost = save(given.default_cost), node->mask = save(mask);
  torch::autograd::set_history(cost, node);
}

// ---- Python ---------------------------------------------------------------------------------
struct WithoutLock {  // the interpreter lock, released for the scope
  PyThreadState *state = PyEval_SaveThread();
  ~WithoutLock() { PyEval_RestoreThread(state); }
};

// A tensor argument.  Anything else (arrays, lists) goes through torch.as_tensor, on `device`
// where one is given, as does a tensor that lives elsewhere.
Tensor tensor_arg(PyObject *o, const at::Device *device = nullptr) {
  if (o == Py_None) return Tensor();
  if (THPVariable_Check(o)) {
    const Tensor &t = THPVariable_Unpack(o);
    return device != nullptr && t.device() != *device ? t.to(*device) : t;
  }
  PyObject *torch = PyImport_ImportModule("torch");
  PyObject *made = torch ? PyObject_CallMethod(torch, "as_tensor", "O", o) : nullptr;
  Py_XDECREF(torch);
  if (made == nullptr) throw PythonError();
  if (!THPVariable_Check(made)) {
    Py_DECREF(made);
    throw InvalidArgument("a tensor is wanted");
  }
  Tensor t = THPVariable_Unpack(made);
  Py_DECREF(made);
  return device != nullptr && t.device() != *device ? t.to(*device) : t;
}

int reduce_arg(PyObject *o) {
  if (PyUnicode_Check(o)) {
    if (PyUnicode_CompareWithASCIIString(o, "MEAN") == 0) return CHOP_REDUCE_MEAN;
    if (PyUnicode_CompareWithASCIIString(o, "MIN") == 0) return CHOP_REDUCE_MIN;
  }
  // the reference aborts the process here (LOG(FATAL), cost_volume_kernels.cc:71)
  PyObject *repr = PyObject_Repr(o);
  if (repr == nullptr) throw PythonError();
  const char *text = PyUnicode_AsUTF8(repr);
  const std::string message =
      std::string("Invalid reduce method ") + (text ? text : "?") + ". Supported types: MEAN, MIN";
  Py_DECREF(repr);
  throw InvalidArgument(message);
}

int64_t groups_arg(PyObject *o) {  // not an int: 0, which every check of the groups rejects
  if (!PyLong_Check(o)) return 0;
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v > 0 && v <= INT32_MAX ? v : 0;
}

bool truth(PyObject *o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PythonError();
  return v != 0;
}

// half_centor: what int() takes, so that None or a word are refused
bool half_arg(PyObject *o) {
  if (PyBool_Check(o)) return o == Py_True;
  PyObject *number = PyNumber_Long(o);
  if (number == nullptr) throw PythonError();
  const int v = PyObject_IsTrue(number);
  Py_DECREF(number);
  return v != 0;
}

PyObject *wrap(const Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject *wrap_tuple(std::initializer_list<const Tensor *> ts) {
  PyObject *out = PyTuple_New((Py_ssize_t)ts.size());
  if (out == nullptr) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor *t : ts) {
    PyObject *o = wrap(*t);
    if (o == nullptr) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i++, o);
  }
  return out;
}

template <typename F>
PyObject *guarded(F &&body) {
  try {
    return body();
  } catch (...) {
    set_error();
  }
  return nullptr;
}

bool count_is(Py_ssize_t n, Py_ssize_t want, const char *name) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, n);
  return false;
}

// The arguments both directions begin with:
//   op, ref | None, src, base_plane or depth_grid, offsets | None, Rs, Ts, reduce, groups, half, grid
constexpr Py_ssize_t kCallArgs = 11;
Call call_args(PyObject *const *a, bool move_small) {
  Call c;
  c.op = (Op)PyLong_AsLong(a[0]);
  c.reduce = reduce_arg(a[7]);
  c.ref = tensor_arg(a[1]);
  c.src = tensor_arg(a[2]);
  const at::Device device = (c.op == FEATURE ? c.src : c.ref).device();
  const at::Device *small = move_small ? &device : nullptr;
  c.depth = tensor_arg(a[3], c.op == V2 ? small : nullptr);
  c.offsets = tensor_arg(a[4], small);
  c.Rs = tensor_arg(a[5], small);
  c.Ts = tensor_arg(a[6], small);
  c.groups = groups_arg(a[8]);
  c.half = half_arg(a[9]);
  c.grid = truth(a[10]);
  return c;
}

// Whether a transform of torch.func (grad, vmap, jvp, ...) is active on this thread.
bool in_functional_transform() {
  return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// Whether an input carries a tangent of forward-mode differentiation.
bool has_tangent(const Call &c) {
  for (const Tensor *t : {&c.ref, &c.src, &c.depth, &c.offsets, &c.Rs, &c.Ts, &c.default_cost})
    if (t->defined() && t->_fw_grad(0).defined()) return true;
  return false;
}

// forward(<call>, default | None, differentiable) -> (cost, mask)
PyObject *py_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!count_is(n, kCallArgs + 2, "forward")) return nullptr;
  return guarded([&] {
    const bool differentiable = truth(a[kCallArgs + 1]);
    // A trace can hold an autograd function of Python; of a call from here it would only hold the
    // allocations.  Under the transforms of torch.func such a function says what it lacks.
    if (differentiable && (torch::jit::tracer::isTracing() || in_functional_transform()))
      return PyObject_Vectorcall(g_recorded, a, kCallArgs + 1, nullptr);
    Call given = call_args(a, differentiable);
    given.default_cost = tensor_arg(a[kCallArgs]);
    // The operators have no forward derivative: Python's autograd function refuses a tangent, which
    // would be lost on the way through here.
    if (differentiable && has_tangent(given)) return PyObject_Vectorcall(g_recorded, a, kCallArgs + 1, nullptr);
    Call c = given;
    Tensor cost, mask;
    {
      const WithoutLock unlocked;
      if (differentiable) {
        differentiable_forward(given, c, cost, mask);
      } else {
        const c10::AutoGradMode no_grad(false);
        differentiable_forward(given, c, cost, mask);
      }
    }
    return wrap_tuple({&cost, &mask});
  });
}

// backward(<call>, cost_grad, cost_mask, want_depth) -> (ref_grad | None, src_grad, depth_grad | None)
PyObject *py_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!count_is(n, kCallArgs + 3, "backward")) return nullptr;
  return guarded([&] {
    Call c = call_args(a, false);
    Tensor cg = tensor_arg(a[kCallArgs]), mask = tensor_arg(a[kCallArgs + 1]);
    const bool want_depth = truth(a[kCallArgs + 2]);
    Tensor rg, sg, dg;
    {
      const WithoutLock unlocked;
      const c10::AutoGradMode no_grad(false);
      check_inputs(c, &cg, &mask);
      backward(c, cg, mask, want_depth, rg, sg, dg);
    }
    return wrap_tuple({&rg, &sg, &dg});
  });
}

// default_gradient(reduce, cost_grad, cost_mask, default) -> the gradient of the filled forms' scalar
PyObject *py_default_gradient(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!count_is(n, 4, "default_gradient")) return nullptr;
  return guarded([&] {
    const int reduce = reduce_arg(a[0]);
    const Tensor g = tensor_arg(a[1]).contiguous(), like = tensor_arg(a[3]);
    const Tensor mask = prepared(tensor_arg(a[2]), at::kInt, g.device(), "cost_mask");
    Tensor out;
    {
      const WithoutLock unlocked;
      const c10::AutoGradMode no_grad(false);
      out = default_gradient(reduce, g, mask, like);
    }
    return wrap(out);
  });
}

// combine_projection(ref_cam [B,2,4,4], src_cam [B,N,2,4,4], scale [3]) -> (Rs, Ts)
PyObject *py_combine_projection(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!count_is(n, 3, "combine_projection")) return nullptr;
  return guarded([&] {
    Tensor ref = tensor_arg(a[0]), src = tensor_arg(a[1]), scale = tensor_arg(a[2]);
    Tensor Rs, Ts;
    {
      const WithoutLock unlocked;
      const c10::AutoGradMode no_grad(false);
      const at::ScalarType dt = ref.scalar_type();
      require(dt == at::kFloat || dt == at::kDouble, "dtype must be float32 or float64");
      const at::Device dev = ref.device();
      ref = prepared(ref, dt, dev, "ref_cam");
      src = prepared(src, dt, dev, "src_cam");
      scale = prepared(scale, dt, dev, "scale");
      require(ref.dim() == 4 && ref.size(1) == 2 && ref.size(2) == 4 && ref.size(3) == 4, "ref_cam must be [B,2,4,4]");
      const int64_t B = ref.size(0);
      require(src.dim() == 5 && src.size(0) == B && src.size(2) == 2 && src.size(3) == 4 && src.size(4) == 4,
              "src_cam must be [B,N,2,4,4]");
      require(scale.dim() == 1 && scale.size(0) == 3, "scale must have 3 entries");
      const int64_t N = src.size(1);
      on_gpu(ref);
      const c10::DeviceGuard guard(dev);
      const auto options = ref.options().requires_grad(false);
      Rs = at::empty({B, N, 3, 3}, options);
      Ts = at::empty({B, N, 3}, options);
      void *s = current_stream(ref);
      check(CHOP_BY_TYPE(chop_combine_projection, s, B, N, ptr<T>(ref), ptr<T>(src), ptr<T>(scale), ptr<T>(Rs),
                         ptr<T>(Ts)));
    }
    return wrap_tuple({&Rs, &Ts});
  });
}

// python_side(InvalidArgumentError, ChopError, recorded): the exception classes to raise and what
// forward() hands a call to in the modes that only an autograd function of Python takes part in
PyObject *py_python_side(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!count_is(n, 3, "python_side")) return nullptr;
  Py_INCREF(a[0]), Py_INCREF(a[1]), Py_INCREF(a[2]);
  g_invalid_argument = a[0], g_chop_error = a[1], g_recorded = a[2];
  Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"forward", (PyCFunction)(void (*)(void))py_forward, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)(void))py_backward, METH_FASTCALL, nullptr},
    {"combine_projection", (PyCFunction)(void (*)(void))py_combine_projection, METH_FASTCALL, nullptr},
    {"default_gradient", (PyCFunction)(void (*)(void))py_default_gradient, METH_FASTCALL, nullptr},
    {"python_side", (PyCFunction)(void (*)(void))py_python_side, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_chop_torch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__chop_torch(void) { return PyModule_Create(&g_module); }
