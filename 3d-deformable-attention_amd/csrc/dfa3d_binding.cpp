// Calls of the operator from Python without the interpreter's share of the work: operand checks, output tensors and the C-ABI call of
// dfa3d_hip in one step.  On 2 x 100 queries a forward spends 6 us in its kernel; checks, allocations and the call through ctypes
// took 10 of the 17 us that it cost.
//
// Every function takes the operands only where all of them are what its kernels read: plain tensors (no subclass, no transform's
// wrapper) of the right shapes and types, contiguous, on the device that is current, under no dispatch mode, with something to do.  Anything else
// is declined (None), and the Python form of the call, which says what is wrong, takes it from there.  The library's entry points come as addresses
// (bind), so this module serves whichever build of the library is loaded.
#include <Python.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <initializer_list>
#include <limits>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../include/dfa3d.h"

namespace {

struct Api {
  decltype(&dfa3d_last_error) last_error;
  decltype(&dfa3d_packed_dist_bytes) packed_dist_bytes;
  decltype(&dfa3d_fused_forward) fused_forward;
  decltype(&dfa3d_fused_backward_workspace_bytes) fused_backward_workspace_bytes;
  decltype(&dfa3d_fused_backward) fused_backward;
  decltype(&dfa3d_wms_deform_attn_forward) attention_forward;
  decltype(&dfa3d_wms_deform_attn_backward_workspace_bytes) attention_backward_workspace_bytes;
  decltype(&dfa3d_wms_deform_attn_backward) attention_backward;
  decltype(&dfa3d_ms_depth_score_sample_forward) score_forward;
  decltype(&dfa3d_ms_depth_score_sample_backward_workspace_bytes) score_backward_workspace_bytes;
  decltype(&dfa3d_ms_depth_score_sample_backward_into) score_backward;
  decltype(&dfa3d_pack_dist) pack_dist;
  decltype(&dfa3d_linear_add) linear_add;
  decltype(&dfa3d_linear_sum) linear_sum;
} api;

using at::Tensor;

// strided, with storage of its own, on `device`
bool is_plain(const Tensor &t, int64_t device) {
  return t.defined() && t.is_cuda() && t.get_device() == device && t.layout() == at::kStrided && t.has_storage() && !t.is_neg() && !t.is_conj();
}
// the operands of one call; `ok` says whether all of them can be read as they are
struct Operands {
  int64_t device;
  bool ok = true;
  bool locked = true;          // this thread holds the interpreter's lock
  // a tensor that is no wrapper: on this device, contiguous, with storage of its own
  const Tensor &need(PyObject *o) {
    static const Tensor none;
    if (!THPVariable_CheckExact(o)) { ok = false; return none; }
    return need(THPVariable_Unpack(o));
  }
  const Tensor &need(const Tensor &t) {
    if (!is_plain(t, device) || !t.is_contiguous() || t.unsafeGetTensorImpl()->is_python_dispatch()) ok = false;
    return t;
  }
  const Tensor &may_have(PyObject *o) {
    static const Tensor none;
    return o == Py_None ? none : need(o);
  }
};

bool shape_is(const Tensor &t, std::initializer_list<int64_t> want) { return t.sizes() == at::IntArrayRef(want); }
bool fits_int(std::initializer_list<int64_t> dims) {
  for (int64_t d : dims)
    if (d <= 0 || d > std::numeric_limits<int>::max()) return false;
  return true;
}
// code of a storage type, -1 for any other; type of locations, weights and float sums that goes with it
int code_of(at::ScalarType t) { return t == at::kFloat ? DFA3D_F32 : t == at::kDouble ? DFA3D_F64 : t == at::kBFloat16 ? DFA3D_BF16 : -1; }
at::ScalarType aux_of(at::ScalarType t) { return t == at::kBFloat16 ? at::kFloat : t; }
void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const int64_t *keys(const Tensor &t) { return static_cast<const int64_t *>(t.data_ptr()); }

PyObject *declined() { Py_RETURN_NONE; }
// What became of a call: taken, declined, or refused by the library, whose entry point is then named.
struct Outcome {
  bool taken;
  const char *refused_by = nullptr;
  int rc = 0;
  std::string message() const { return std::string(refused_by) + " failed with code " + std::to_string(rc) + ": " + api.last_error(); }
};
constexpr Outcome kDeclined{false};
Outcome outcome(const char *name, int rc) { return rc == 0 ? Outcome{true} : Outcome{false, name, rc}; }
// the Python answer where there are no results
PyObject *without_results(const Outcome &o) {
  if (o.refused_by == nullptr) return declined();
  PyErr_SetString(PyExc_RuntimeError, o.message().c_str());
  return nullptr;
}
// a tuple that owns the tensors; an undefined one is None
PyObject *tuple_of(std::initializer_list<Tensor> tensors) {
  PyObject *out = PyTuple_New((Py_ssize_t)tensors.size());
  if (out == nullptr) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor &t : tensors) PyTuple_SET_ITEM(out, i++, t.defined() ? THPVariable_Wrap(t) : Py_NewRef(Py_None));
  return out;
}
// im2col_step as the reference checks it
bool step_ok(int64_t batch, int64_t given) {
  const int64_t step = given < batch ? given : batch;
  return step > 0 && batch % step == 0;
}
// an im2col_step that is no number is one that no batch has
int64_t step_of(PyObject *o) {
  if (!PyLong_CheckExact(o)) return 0;
  const long long given = PyLong_AsLongLong(o);
  if (given == -1 && PyErr_Occurred()) { PyErr_Clear(); return 0; }
  return given;
}
// without the interpreter's lock, where this thread holds it
struct NoGil {
  PyThreadState *state;
  explicit NoGil(bool locked) : state(locked ? PyEval_SaveThread() : nullptr) {}
  ~NoGil() {
    if (state != nullptr) PyEval_RestoreThread(state);
  }
};

// options of a backward into tensors of its own
dfa3d_launch_options own_gradients(bool clear) {
  dfa3d_launch_options o{};
  o.direct = DFA3D_FEW_POINTS;
  o.clear = clear ? 1 : 0;
  return o;
}

// shapes of a one-stage call
struct FusedDims {
  int64_t B, S, M, C, D, L, Q, P, heads;
  int code;
  at::ScalarType type, aux;
};
bool fused_dims(const Tensor &value, const Tensor &dist, const Tensor &shapes, const Tensor &starts, const Tensor &loc, const Tensor &attn,
                FusedDims &d) {
  if (value.dim() != 4 || dist.dim() != 4 || loc.dim() != 6) return false;
  d.B = value.size(0); d.S = value.size(1); d.M = value.size(2); d.C = value.size(3);
  d.heads = dist.size(2); d.D = dist.size(3);
  d.Q = loc.size(1); d.L = loc.size(3); d.P = loc.size(4);
  d.type = value.scalar_type(); d.aux = aux_of(d.type); d.code = code_of(d.type);
  return d.code >= 0 && fits_int({d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P}) && (d.heads == d.M || d.heads == 1) &&
         shape_is(dist, {d.B, d.S, d.heads, d.D}) && shape_is(loc, {d.B, d.Q, d.M, d.L, d.P, 3}) && shape_is(attn, {d.B, d.Q, d.M, d.L, d.P}) &&
         shape_is(shapes, {d.L, 3}) && shape_is(starts, {d.L}) && dist.scalar_type() == d.type && loc.scalar_type() == d.aux &&
         attn.scalar_type() == d.aux && shapes.scalar_type() == at::kLong && starts.scalar_type() == at::kLong;
}

bool numbers(PyObject *const *args, int64_t &device, void *&stream) {
  device = PyLong_AsLongLong(args[0]);
  stream = PyLong_AsVoidPtr(args[1]);
  return !PyErr_Occurred();
}
// a dispatch mode (fake tensors, tracing) or a function transform would give the outputs that are allocated here another form
bool plain_dispatch() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
// a tracer, a functorch transform, a profiler or another observer sees what this thread calls
bool observed() {
  const c10::DispatchKeySet modes = c10::impl::tls_local_dispatch_key_set().included_;
  return at::hasCallbacks() || torch::jit::tracer::isTracing() || modes.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         modes.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}
#define TAKES(n)                                                                            \
  if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; } \
  Operands in; void *stream;                                                                \
  if (!numbers(args, in.device, stream)) return nullptr;                                    \
  if (!plain_dispatch()) return declined();

struct FusedResults { Tensor out, score, wu; };
Outcome fused_forward(const Operands &in, void *stream, const Tensor &value, const Tensor &dist, const Tensor &shapes, const Tensor &starts,
                      const Tensor &loc, const Tensor &attn, int64_t step, bool need_score, bool need_wu, const Tensor &packed, FusedResults &to) {
  FusedDims d;
  if (!in.ok || !fused_dims(value, dist, shapes, starts, loc, attn, d) || !step_ok(d.B, step)) return kDeclined;
  if (packed.defined()) {
    const size_t least = d.heads == 1 ? api.packed_dist_bytes(d.B, d.S, d.D, d.L, d.code) : 0;
    if (least == 0 || packed.nbytes() < least) return kDeclined;
  }
  const auto store = value.options(), aux = store.dtype(d.aux);
  to.out = at::empty({d.B, d.Q, d.M * d.C}, store);
  if (need_score) to.score = at::empty({d.B, d.Q, d.M, d.L, d.P, 4}, store);
  if (need_wu) to.wu = at::empty({d.B, d.Q, d.M, 1}, aux);
  NoGil no_gil(in.locked);
  return outcome("dfa3d_fused_forward",
                 api.fused_forward(ptr(value), ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(attn), ptr(to.out), ptr(to.score), ptr(to.wu),
                                   ptr(packed), d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, d.code, nullptr, stream));
}
// fused_forward(device, stream, value, dist, shapes, starts, loc, attn, im2col_step, need_score, need_weight_update, packed)
// -> (out, score or None, weight_update or None), or None
PyObject *fused_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(12)
  const Tensor &value = in.need(args[2]), &dist = in.need(args[3]), &shapes = in.need(args[4]), &starts = in.need(args[5]),
               &loc = in.need(args[6]), &attn = in.need(args[7]), &packed = in.may_have(args[11]);
  FusedResults r;
  const Outcome o = fused_forward(in, stream, value, dist, shapes, starts, loc, attn, step_of(args[8]), args[9] == Py_True, args[10] == Py_True,
                                  packed, r);
  return o.taken ? tuple_of({r.out, r.score, r.wu}) : without_results(o);
  END_HANDLE_TH_ERRORS
}

struct FusedGradients { Tensor value, dist, loc, attn; };
Outcome fused_gradients(const Operands &in, void *stream, const Tensor &value, const Tensor &dist, const Tensor &shapes, const Tensor &starts,
                        const Tensor &loc, const Tensor &attn, const Tensor &grad_out, const Tensor &grad_score, const Tensor &grad_wu, int64_t step,
                        FusedGradients &to) {
  FusedDims d;
  if (!in.ok || !fused_dims(value, dist, shapes, starts, loc, attn, d) || !step_ok(d.B, step)) return kDeclined;
  if (grad_out.numel() != d.B * d.Q * d.M * d.C || grad_out.scalar_type() != d.type) return kDeclined;
  if (grad_score.defined() && (!shape_is(grad_score, {d.B, d.Q, d.M, d.L, d.P, 4}) || grad_score.scalar_type() != d.type)) return kDeclined;
  if (grad_wu.defined() && (grad_wu.numel() != d.B * d.Q * d.M || grad_wu.scalar_type() != d.aux)) return kDeclined;
  // bfloat16 gradients are written as such where that is offered
  const dfa3d_launch_options clear = own_gradients(true);
  const bool g16 = d.type == at::kBFloat16 &&
                   api.fused_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, DFA3D_BF16G, &clear) > 0;
  const int code = g16 ? DFA3D_BF16G : d.code;
  const size_t bytes = api.fused_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, code, &clear);
  const auto aux = value.options().dtype(d.aux), sums = g16 ? value.options() : aux;
  to = FusedGradients{at::empty(value.sizes(), sums), at::empty(dist.sizes(), sums), at::empty(loc.sizes(), aux), at::empty(attn.sizes(), aux)};
  Tensor workspace;
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, value.options().dtype(at::kByte));
  Outcome o{false};
  {
    NoGil no_gil(in.locked);
    o = outcome("dfa3d_fused_backward",
                api.fused_backward(ptr(value), ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(attn), ptr(grad_out), ptr(grad_score), ptr(grad_wu),
                                   ptr(to.value), ptr(to.dist), ptr(to.loc), ptr(to.attn), ptr(workspace), bytes, d.B, d.S, d.M, d.C, d.D, d.L, d.Q,
                                   d.P, d.heads, code, &clear, stream));
  }
  if (!o.taken) return o;
  to.value = to.value.to(d.type);
  to.dist = to.dist.to(d.type);
  return o;
}
// fused_gradients(device, stream, value, dist, shapes, starts, loc, attn, grad_out, grad_score, grad_weight_update, im2col_step)
// -> gradients of value, dist, loc and attn in their types, or None
PyObject *fused_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(12)
  const Tensor &value = in.need(args[2]), &dist = in.need(args[3]), &shapes = in.need(args[4]), &starts = in.need(args[5]),
               &loc = in.need(args[6]), &attn = in.need(args[7]), &grad_out = in.need(args[8]), &grad_score = in.may_have(args[9]),
               &grad_wu = in.may_have(args[10]);
  FusedGradients g;
  const Outcome o = fused_gradients(in, stream, value, dist, shapes, starts, loc, attn, grad_out, grad_score, grad_wu, step_of(args[11]), g);
  return o.taken ? tuple_of({g.value, g.dist, g.loc, g.attn}) : without_results(o);
  END_HANDLE_TH_ERRORS
}

// shapes of a call of stage 2 alone
struct AttentionDims {
  int64_t B, S, M, C, L, Q, P, shape_width, loc_width;
  int code;
  at::ScalarType type, aux;
};
bool attention_dims(const Tensor &value, const Tensor &shapes, const Tensor &starts, const Tensor &loc, const Tensor &attn, const Tensor &score,
                    AttentionDims &d) {
  if (value.dim() != 4 || shapes.dim() != 2 || loc.dim() != 6) return false;
  d.B = value.size(0); d.S = value.size(1); d.M = value.size(2); d.C = value.size(3);
  d.L = shapes.size(0); d.shape_width = shapes.size(1);
  d.Q = loc.size(1); d.P = loc.size(4); d.loc_width = loc.size(5);
  d.type = value.scalar_type(); d.aux = aux_of(d.type); d.code = code_of(d.type);
  return d.code >= 0 && fits_int({d.B, d.S, d.M, d.C, d.L, d.Q, d.P}) && (d.shape_width == 2 || d.shape_width == 3) &&
         (d.loc_width == 2 || d.loc_width == 3) && shape_is(loc, {d.B, d.Q, d.M, d.L, d.P, d.loc_width}) &&
         shape_is(attn, {d.B, d.Q, d.M, d.L, d.P}) && shape_is(starts, {d.L}) && loc.scalar_type() == d.aux && attn.scalar_type() == d.aux &&
         shapes.scalar_type() == at::kLong && starts.scalar_type() == at::kLong &&
         (!score.defined() || (shape_is(score, {d.B, d.Q, d.M, d.L, d.P, 4}) && score.scalar_type() == d.type));
}

Outcome attention_forward(const Operands &in, void *stream, const Tensor &value, const Tensor &shapes, const Tensor &starts, const Tensor &loc,
                          const Tensor &attn, const Tensor &score, int64_t step, Tensor &out) {
  AttentionDims d;
  if (!in.ok || !attention_dims(value, shapes, starts, loc, attn, score, d) || !step_ok(d.B, step)) return kDeclined;
  out = at::empty({d.B, d.Q, d.M * d.C}, value.options());
  NoGil no_gil(in.locked);
  return outcome("dfa3d_wms_deform_attn_forward",
                 api.attention_forward(ptr(value), keys(shapes), d.shape_width, keys(starts), ptr(loc), d.loc_width, ptr(attn), ptr(score), ptr(out),
                                       d.B, d.S, d.M, d.C, d.L, d.Q, d.P, d.code, nullptr, stream));
}
// attention_forward(device, stream, value, shapes, starts, loc, attn, score or None, im2col_step) -> out, or None
PyObject *attention_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(9)
  const Tensor &value = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &attn = in.need(args[6]), &score = in.may_have(args[7]);
  Tensor out;
  const Outcome o = attention_forward(in, stream, value, shapes, starts, loc, attn, score, step_of(args[8]), out);
  return o.taken ? THPVariable_Wrap(out) : without_results(o);
  END_HANDLE_TH_ERRORS
}

struct AttentionGradients { Tensor value, loc, attn, score; };
Outcome attention_gradients(const Operands &in, void *stream, const Tensor &value, const Tensor &shapes, const Tensor &starts, const Tensor &loc,
                            const Tensor &attn, const Tensor &score, const Tensor &grad_out, int64_t step, AttentionGradients &to) {
  AttentionDims d;
  if (!in.ok || !attention_dims(value, shapes, starts, loc, attn, score, d) || d.loc_width != 2 || !step_ok(d.B, step)) return kDeclined;
  if (grad_out.numel() != d.B * d.Q * d.M * d.C || grad_out.scalar_type() != d.type) return kDeclined;
  const dfa3d_launch_options clear = own_gradients(true);
  const size_t bytes = api.attention_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.L, d.Q, d.P, d.code, &clear);
  const auto aux = value.options().dtype(d.aux);
  to = AttentionGradients{at::empty(value.sizes(), aux), at::empty(loc.sizes(), aux), at::empty(attn.sizes(), aux), Tensor()};
  Tensor workspace;
  if (score.defined()) to.score = at::empty(score.sizes(), aux);
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, value.options().dtype(at::kByte));
  Outcome o{false};
  {
    NoGil no_gil(in.locked);
    o = outcome("dfa3d_wms_deform_attn_backward",
                api.attention_backward(ptr(value), keys(shapes), d.shape_width, keys(starts), ptr(loc), d.loc_width, ptr(attn), ptr(score), ptr(grad_out),
                                       ptr(to.value), ptr(to.loc), d.loc_width, ptr(to.attn), ptr(to.score), ptr(workspace), bytes, d.B, d.S, d.M, d.C,
                                       d.L, d.Q, d.P, d.code, &clear, stream));
  }
  if (!o.taken) return o;
  to.value = to.value.to(d.type);
  if (score.defined()) to.score = to.score.to(d.type);
  return o;
}
// attention_gradients(device, stream, value, shapes, starts, loc (2 wide), attn, score or None, grad_out, im2col_step)
// -> gradients of value, loc, attn and score (None without one) in their types, or None
PyObject *attention_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(10)
  const Tensor &value = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &attn = in.need(args[6]), &score = in.may_have(args[7]), &grad_out = in.need(args[8]);
  AttentionGradients g;
  const Outcome o = attention_gradients(in, stream, value, shapes, starts, loc, attn, score, grad_out, step_of(args[9]), g);
  return o.taken ? tuple_of({g.value, g.loc, g.attn, g.score}) : without_results(o);
  END_HANDLE_TH_ERRORS
}

// shapes of a call of stage 1 alone
struct ScoreDims {
  int64_t B, S, M, D, L, Q, P;
  int code;
  at::ScalarType type, aux;
};
bool score_dims(const Tensor &dist, const Tensor &shapes, const Tensor &starts, const Tensor &loc, ScoreDims &d) {
  if (dist.dim() != 4 || shapes.dim() != 2 || loc.dim() != 6) return false;
  d.B = dist.size(0); d.S = dist.size(1); d.M = dist.size(2); d.D = dist.size(3);
  d.L = shapes.size(0); d.Q = loc.size(1); d.P = loc.size(4);
  d.type = dist.scalar_type(); d.aux = aux_of(d.type); d.code = code_of(d.type);
  return d.code >= 0 && fits_int({d.B, d.S, d.M, d.D, d.L, d.Q, d.P}) && shape_is(loc, {d.B, d.Q, d.M, d.L, d.P, 3}) &&
         shape_is(shapes, {d.L, 3}) && shape_is(starts, {d.L}) && loc.scalar_type() == d.aux && shapes.scalar_type() == at::kLong &&
         starts.scalar_type() == at::kLong;
}

Outcome score_forward(const Operands &in, void *stream, const Tensor &dist, const Tensor &shapes, const Tensor &starts, const Tensor &loc, int64_t step,
                      Tensor &score) {
  ScoreDims d;
  if (!in.ok || !score_dims(dist, shapes, starts, loc, d) || !step_ok(d.B, step)) return kDeclined;
  score = at::empty({d.B, d.Q, d.M, d.L, d.P, 4}, dist.options());
  NoGil no_gil(in.locked);
  return outcome("dfa3d_ms_depth_score_sample_forward", api.score_forward(ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(score), d.B, d.S, d.M,
                                                                          d.D, d.L, d.Q, d.P, d.code, nullptr, stream));
}
// score_forward(device, stream, dist, shapes, starts, loc, im2col_step) -> score, or None
PyObject *score_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(7)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]);
  Tensor score;
  const Outcome o = score_forward(in, stream, dist, shapes, starts, loc, step_of(args[6]), score);
  return o.taken ? THPVariable_Wrap(score) : without_results(o);
  END_HANDLE_TH_ERRORS
}

struct ScoreGradients { Tensor dist, loc; };
Outcome score_gradients(const Operands &in, void *stream, const Tensor &dist, const Tensor &shapes, const Tensor &starts, const Tensor &loc,
                        const Tensor &grad_score, int64_t step, ScoreGradients &to) {
  ScoreDims d;
  if (!in.ok || !score_dims(dist, shapes, starts, loc, d) || !step_ok(d.B, step)) return kDeclined;
  if (!shape_is(grad_score, {d.B, d.Q, d.M, d.L, d.P, 4}) || grad_score.scalar_type() != d.type) return kDeclined;
  const dfa3d_launch_options options = own_gradients(false);      // (this entry point clears by itself)
  const size_t bytes = api.score_backward_workspace_bytes(d.B, d.S, d.M, d.D, d.L, d.Q, d.P, d.code, &options);
  const auto aux = dist.options().dtype(d.aux);
  to = ScoreGradients{at::empty(dist.sizes(), aux), at::empty(loc.sizes(), aux)};
  Tensor workspace;
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, dist.options().dtype(at::kByte));
  Outcome o{false};
  {
    NoGil no_gil(in.locked);
    o = outcome("dfa3d_ms_depth_score_sample_backward",
                api.score_backward(ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(grad_score), ptr(to.dist), ptr(to.loc), ptr(workspace), bytes, d.B,
                                   d.S, d.M, d.D, d.L, d.Q, d.P, d.code, &options, stream));
  }
  if (!o.taken) return o;
  to.dist = to.dist.to(d.type);
  return o;
}
// score_gradients(device, stream, dist, shapes, starts, loc, grad_score, im2col_step) -> gradients of dist and loc in their types, or None
PyObject *score_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(8)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &grad_score = in.need(args[6]);
  ScoreGradients g;
  const Outcome o = score_gradients(in, stream, dist, shapes, starts, loc, grad_score, step_of(args[7]), g);
  return o.taken ? tuple_of({g.dist, g.loc}) : without_results(o);
  END_HANDLE_TH_ERRORS
}

Outcome pack_dist(const Operands &in, void *stream, const Tensor &dist, const Tensor &shapes, const Tensor &starts, Tensor &packed) {
  if (!in.ok || dist.dim() != 4 || dist.size(2) != 1 || shapes.dim() != 2 || shapes.size(1) != 3 || !shape_is(starts, {shapes.size(0)}) ||
      shapes.scalar_type() != at::kLong || starts.scalar_type() != at::kLong)
    return kDeclined;
  const int64_t B = dist.size(0), S = dist.size(1), D = dist.size(3), L = shapes.size(0);
  const int code = code_of(dist.scalar_type());
  if (!(code == DFA3D_F32 || code == DFA3D_BF16) || !fits_int({B, S, D, L})) return kDeclined;
  const size_t bytes = api.packed_dist_bytes(B, S, D, L, code);
  if (bytes == 0) return kDeclined;
  packed = at::empty({(int64_t)bytes}, dist.options().dtype(at::kByte));
  NoGil no_gil(in.locked);
  return outcome("dfa3d_pack_dist", api.pack_dist(ptr(dist), keys(shapes), keys(starts), ptr(packed), bytes, B, S, D, L, code, stream));
}
// pack_dist(device, stream, dist (bs, keys, 1, D), shapes, starts) -> packed distribution, or None
PyObject *pack_dist(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(5)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]);
  Tensor packed;
  const Outcome o = pack_dist(in, stream, dist, shapes, starts, packed);
  return o.taken ? THPVariable_Wrap(packed) : without_results(o);
  END_HANDLE_TH_ERRORS
}

// Calls of the Functions as a whole: forward, and the node of the graph where one is recorded, whose backward runs without the interpreter.  A
// node of Python's needs the interpreter's lock on the engine's thread, which is handed over twice a backward, and costs its context and two
// wrappers: 1 x 50 queries on 15 x 25 maps, passes in a row, six measurements on one card, node in Python and native: a training pass 49 to 109
// and 41 to 78 us (the hand-over to the engine's thread takes next to nothing or most of that, from run to run), the forward 11.9 to 12.7 and
// 9.4 to 10.2 recorded, 10.1 and 8.0 not.
enum Kind { kScore, kStage2, kPlain, kFused, kWeightUpdate };      // numbered as in recording.py
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// (kind, im2col_step, saved tensors, gradients of the outputs) -> gradients of the saved tensors: a Function's own backward, for what is not as the
// kernels read it, and for a backward that is recorded itself
PyObject *python_backward = nullptr;

struct WithGil {
  PyGILState_STATE state = PyGILState_Ensure();
  ~WithGil() { PyGILState_Release(state); }
};
PyObject *python_tuple(const variable_list &t) {
  PyObject *to = PyTuple_New((Py_ssize_t)t.size());
  for (size_t i = 0; to != nullptr && i < t.size(); ++i)
    PyTuple_SET_ITEM(to, (Py_ssize_t)i, t[i].defined() ? THPVariable_Wrap(t[i]) : Py_NewRef(Py_None));
  return to;
}
variable_list gradients_by_python(Kind kind, int64_t step, const variable_list &t, const variable_list &grads) {
  WithGil gil;
  PyObject *saved = python_tuple(t), *incoming = python_tuple(grads), *got = nullptr;
  if (saved != nullptr && incoming != nullptr && python_backward != nullptr)
    got = PyObject_CallFunction(python_backward, "iLOO", (int)kind, (long long)step, saved, incoming);
  Py_XDECREF(saved);
  Py_XDECREF(incoming);
  variable_list to(t.size());
  if (got != nullptr && PyTuple_CheckExact(got) && (size_t)PyTuple_GET_SIZE(got) == t.size()) {
    for (size_t i = 0; i < t.size(); ++i)
      if (PyObject *g = PyTuple_GET_ITEM(got, (Py_ssize_t)i); THPVariable_Check(g)) to[i] = THPVariable_Unpack(g);
    Py_DECREF(got);
    return to;
  }
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "no gradients");
  Py_XDECREF(got);
  python_error e;
  e.persist();
  throw e;
}
// an incoming gradient as a contiguous tensor of the output's type
Tensor incoming(const Tensor &g, at::ScalarType like, int64_t device, bool &ok) {
  if (!g.defined()) return g;
  if (!is_plain(g, device) || g.unsafeGetTensorImpl()->is_python_dispatch()) { ok = false; return g; }
  return g.contiguous().to(like);
}
// the saved tensors' gradients, or false
bool gradients_of(Kind kind, int64_t step, const variable_list &t, const variable_list &grads, variable_list &to) {
  if (c10::GradMode::is_enabled() || !plain_dispatch() || observed() || !t[0].defined() || !t[0].is_cuda()) return false;
  Operands in{t[0].get_device()};
  in.locked = false;
  if (c10::hip::current_device() != in.device) return false;
  for (const Tensor &x : t) in.need(x);
  const Tensor &loc = t[kind == kFused || kind == kWeightUpdate ? 4 : 3];
  if (!in.ok || loc.dim() != 6 || t[0].dim() != 4) return false;
  const at::ScalarType type = t[0].scalar_type();
  Tensor g = incoming(grads[0], type, in.device, in.ok), score, wu;
  if (kind == kFused) score = incoming(grads[1], type, in.device, in.ok);
  if (kind == kWeightUpdate) wu = incoming(grads[1], aux_of(type), in.device, in.ok);
  if (!in.ok) return false;
  if (!g.defined()) {
    g = kind == kScore ? at::zeros({t[0].size(0), loc.size(1), t[0].size(2), loc.size(3), loc.size(4), 4}, t[0].options())
                       : at::zeros({t[0].size(0), loc.size(1), t[0].size(2) * t[0].size(3)}, t[0].options());
  }
  void *stream = c10::hip::getCurrentHIPStream(in.device).stream();
  Outcome o{false};
  if (kind == kScore) {
    ScoreGradients r;
    o = score_gradients(in, stream, t[0], t[1], t[2], t[3], g, step, r);
    to = {r.dist, Tensor(), Tensor(), r.loc};
  } else if (kind == kStage2 || kind == kPlain) {
    AttentionGradients r;
    o = attention_gradients(in, stream, t[0], t[1], t[2], t[3], t[4], kind == kStage2 ? t[5] : Tensor(), g, step, r);
    to = {r.value, Tensor(), Tensor(), r.loc, r.attn};
    if (kind == kStage2) to.push_back(r.score);
  } else {
    FusedGradients r;
    o = fused_gradients(in, stream, t[0], t[1], t[2], t[3], t[4], t[5], g, score, wu, step, r);
    to = {r.value, r.dist, Tensor(), Tensor(), r.loc, r.attn};
  }
  if (o.refused_by != nullptr) throw std::runtime_error(o.message());
  return o.taken;
}

// The nodes, which hand out outputs that are there already.
template <typename Self, Kind KIND> struct Recorded : torch::autograd::Function<Self> {
  template <typename... Tensors>
  static variable_list forward(AutogradContext *ctx, int64_t step, const variable_list *outputs, const Tensors &...saved) {
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({saved...});
    ctx->saved_data["step"] = step;
    return *outputs;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const int64_t step = ctx->saved_data["step"].toInt();
    const variable_list saved = ctx->get_saved_variables();
    variable_list to;
    if (!gradients_of(KIND, step, saved, grads, to)) to = gradients_by_python(KIND, step, saved, grads);
    to.insert(to.begin(), 2, Tensor());                      // of the step and the outputs
    return to;
  }
};
}  // namespace
namespace dfa3d {      // (their names are what a graph shows)
struct MultiScaleDepthScoreSampleFunction : Recorded<MultiScaleDepthScoreSampleFunction, kScore> {};
struct WeightedMultiScaleDeformableAttnFunction : Recorded<WeightedMultiScaleDeformableAttnFunction, kStage2> {};
struct MultiScaleDeformableAttnFunction : Recorded<MultiScaleDeformableAttnFunction, kPlain> {};
struct MultiScale3DDeformableAttnFunction : Recorded<MultiScale3DDeformableAttnFunction, kFused> {};
struct MultiScale3DDeformableAttnWeightUpdateFunction : Recorded<MultiScale3DDeformableAttnWeightUpdateFunction, kWeightUpdate> {};
}  // namespace dfa3d
namespace {
// What Python sees of a node: the name of its class and what a node made in Python has of its context.
template <typename F> torch::autograd::CppNode<F> &node_of(PyObject *o) {
  return *static_cast<torch::autograd::CppNode<F> *>(reinterpret_cast<torch::autograd::THPCppFunction *>(o)->cdata.get());
}
template <typename F> PyObject *saved_tensors(PyObject *o, void *) {
  HANDLE_TH_ERRORS
  return python_tuple(node_of<F>(o).ctx_.get_saved_variables());
  END_HANDLE_TH_ERRORS
}
template <typename F> PyObject *im2col_step(PyObject *o, void *) {
  HANDLE_TH_ERRORS
  return PyLong_FromLongLong(node_of<F>(o).ctx_.saved_data.at("step").toInt());
  END_HANDLE_TH_ERRORS
}
// of the tensors and the step
template <typename F> PyObject *needs_input_grad(PyObject *o, void *) {
  HANDLE_TH_ERRORS
  const auto &edges = node_of<F>(o).next_edges();
  PyObject *to = PyTuple_New((Py_ssize_t)edges.size() + 1);
  if (to == nullptr) return nullptr;
  for (size_t i = 0; i <= edges.size(); ++i) PyTuple_SET_ITEM(to, (Py_ssize_t)i, PyBool_FromLong(i < edges.size() && edges[i].is_valid()));
  return to;
  END_HANDLE_TH_ERRORS
}
template <typename F> void show_as(const char *name) {
  using namespace torch::autograd;
  static PyGetSetDef properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                     {"saved_tensors", saved_tensors<F>, nullptr, nullptr, nullptr},
                                     {"im2col_step", im2col_step<F>, nullptr, nullptr, nullptr},
                                     {"needs_input_grad", needs_input_grad<F>, nullptr, nullptr, nullptr},
                                     {nullptr, nullptr, nullptr, nullptr, nullptr}};
  static PyTypeObject type;
  if (type.tp_name != nullptr) return;                       // (already)
  torch::autograd::_initFunctionPyTypeObject(type, name, properties, nullptr);
  Py_INCREF(&type);
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<F>), &type);
}

// the outputs with a node behind them, where one is to be made
template <typename F, typename... Tensors> variable_list recorded_outputs(variable_list outputs, int64_t step, const Tensors &...inputs) {
  if (!c10::GradMode::is_enabled() || !(inputs.requires_grad() || ...)) return outputs;
  return F::apply(step, (const variable_list *)&outputs, inputs...);
}

// call(device, stream, kind, arguments of a Function's apply) -> what apply returns, or None
PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(4)
  const long kind = PyLong_AsLong(args[2]);
  if (kind == -1 && PyErr_Occurred()) return nullptr;
  if (!PyTuple_CheckExact(args[3]) || at::autocast::is_autocast_enabled(at::kCUDA)) return declined();
  const Py_ssize_t given = PyTuple_GET_SIZE(args[3]);
  const auto arg = [&](Py_ssize_t i) { return PyTuple_GET_ITEM(args[3], i); };
  if (kind == kScore && given == 5) {
    const Tensor &dist = in.need(arg(0)), &shapes = in.need(arg(1)), &starts = in.need(arg(2)), &loc = in.need(arg(3));
    const int64_t step = step_of(arg(4));
    Tensor score;
    const Outcome o = score_forward(in, stream, dist, shapes, starts, loc, step, score);
    if (!o.taken) return without_results(o);
    return THPVariable_Wrap(recorded_outputs<dfa3d::MultiScaleDepthScoreSampleFunction>({score}, step, dist, shapes, starts, loc)[0]);
  }
  if ((kind == kStage2 && given == 7) || (kind == kPlain && given == 6)) {
    const Tensor &value = in.need(arg(0)), &shapes = in.need(arg(1)), &starts = in.need(arg(2)), &loc = in.need(arg(3)), &attn = in.need(arg(4));
    const Tensor score = kind == kStage2 ? in.need(arg(5)) : Tensor();
    const int64_t step = step_of(arg(given - 1));
    Tensor out;
    const Outcome o = attention_forward(in, stream, value, shapes, starts, loc, attn, score, step, out);
    if (!o.taken) return without_results(o);
    return THPVariable_Wrap(
        (kind == kStage2 ? recorded_outputs<dfa3d::WeightedMultiScaleDeformableAttnFunction>({out}, step, value, shapes, starts, loc, attn, score)
                         : recorded_outputs<dfa3d::MultiScaleDeformableAttnFunction>({out}, step, value, shapes, starts, loc, attn))[0]);
  }
  if ((kind == kFused && given == 7) || (kind == kWeightUpdate && (given == 7 || given == 8))) {
    const Tensor &value = in.need(arg(0)), &dist = in.need(arg(1)), &shapes = in.need(arg(2)), &starts = in.need(arg(3)), &loc = in.need(arg(4)),
                 &attn = in.need(arg(5));
    const int64_t step = step_of(arg(6));
    Tensor packed = given == 8 ? in.may_have(arg(7)) : Tensor();
    if (!in.ok) return declined();
    // the packed form of a distribution shared by all heads, where making it pays: functional._packed_for_forward
    if (!packed.defined() && dist.dim() == 4 && dist.size(2) == 1 && loc.numel() / 3 >= dist.size(0) * dist.size(1) * dist.size(3)) {
      const Outcome o = pack_dist(in, stream, dist, shapes, starts, packed);
      if (o.refused_by != nullptr) return without_results(o);
    }
    FusedResults r;
    const Outcome o = fused_forward(in, stream, value, dist, shapes, starts, loc, attn, step, kind == kFused, kind == kWeightUpdate, packed, r);
    if (!o.taken) return without_results(o);
    const variable_list out =
        kind == kFused ? recorded_outputs<dfa3d::MultiScale3DDeformableAttnFunction>({r.out, r.score}, step, value, dist, shapes, starts, loc, attn)
                       : recorded_outputs<dfa3d::MultiScale3DDeformableAttnWeightUpdateFunction>({r.out, r.wu}, step, value, dist, shapes, starts, loc, attn);
    return tuple_of({out[0], out[1]});
  }
  return declined();
  END_HANDLE_TH_ERRORS
}
PyObject *set_python_backward(PyObject *, PyObject *f) {
  Py_INCREF(f);
  PyObject *before = std::exchange(python_backward, f);
  Py_XDECREF(before);
  Py_RETURN_NONE;
}

// Where the kernels form a product of rows x width elements, sums of depth terms, in the library's place: they read four neighbours of a
// row at a time; not where few rows meet a deep sum of one layer; where several layers' terms are summed (of_several), for which the
// library takes a call each and their sums, with up to 1024 terms in all whatever the rows.  Library and kernels, us:
//   a call after the other   4096 rows of 256 by 256 20, 8     of 256 by 64 20, 8     20000 of 512 by 512 98, 70     100000 of 256 by 256 123, 93
//     deep sums of one layer, 4096 rows: of 512 by 256 19, 22     of 2048 by 256 41, 51 to 89     of 1024 by 1024 72, 58
//   The library's 20 are its host's time, which bounds it up to some 5000 rows.  On the device alone (captured in a graph)
//     256 by 256   16 rows 9.6, 5.5   100 31, 5.9   625 6.3, 6.1   1500 6.4, 8.1   4096 10.7, 9.2
//     512 by 256   16 rows 4.5, 5.4   100 6.1, 5.9   625 6.6, 8.0   2500 10.8, 11.4
//     256 by 64    100 11.7, 5.8   2500 6.1, 6.2   6600 6.4, 8.4   10000 8.4, 8.7
//     512, 256 and 256 terms   16 rows 30, 9.1   1000 22, 12   4000 41, 29   16000 100, 74     512 and 512   1000 16, 12   8000 48, 49
//     256, 128 and 128         1000 18, 9.2   4000 33, 22     128, 64 and 64   1000 17, 8.5   8000 39, 17
//   So the device alone is up to 2 us slower with the kernels for one layer of some rows and widths; the host's 12 weigh more.
bool product_applies(int64_t rows, int64_t width, int64_t depth, bool of_several = false) {
  return width > 0 && depth > 0 && width <= 4096 && depth <= 4096 && width % 2 == 0 && depth % 4 == 0 && rows > 0 && rows <= (int64_t(1) << 31) &&
         (depth <= 256 || of_several || rows * width >= (int64_t(1) << 22));
}
// pairs of a flat tuple, 0 where it is none of 1 to as many pairs as a call takes
Py_ssize_t pairs_of(PyObject *o) {
  const Py_ssize_t n = PyTuple_CheckExact(o) ? PyTuple_GET_SIZE(o) : 0;
  return n % 2 == 0 && n / 2 <= DFA3D_MAX_LINEAR_SETS ? n / 2 : 0;
}
bool is_float_matrix(const Tensor &t) { return t.scalar_type() == at::kFloat && t.dim() == 2; }
bool recorded(const Tensor &t) { return t.defined() && t.requires_grad() && c10::GradMode::is_enabled(); }

// linear(device, stream, x (..., K), weight (O, K), bias (O) or None, addend (..., O) or None) -> F.linear + addend, not recorded, or None
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(6)
  const Tensor &x = in.need(args[2]), &w = in.need(args[3]), &b = in.may_have(args[4]), &addend = in.may_have(args[5]);
  if (!in.ok || x.scalar_type() != at::kFloat || x.dim() < 2 || !is_float_matrix(w) || x.size(-1) != w.size(1) || w.size(1) == 0 ||
      (b.defined() && (b.scalar_type() != at::kFloat || !shape_is(b, {w.size(0)}))) || recorded(x) || recorded(w) || recorded(b) ||
      (addend.defined() && (addend.scalar_type() != at::kFloat || recorded(addend))) ||
      at::autocast::is_autocast_enabled(at::kCUDA) || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer))
    return declined();
  const int64_t O = w.size(0), K = w.size(1), rows = x.numel() / K;
  if (!product_applies(rows, O, K)) return declined();
  auto sizes = x.sizes().vec();
  sizes.back() = O;
  if (addend.defined() && addend.sizes() != at::IntArrayRef(sizes)) return declined();
  Tensor y = at::empty(sizes, x.options());
  int rc;
  {
    NoGil no_gil(in.locked);
    rc = api.linear_add(static_cast<const float *>(ptr(x)), static_cast<const float *>(ptr(w)), static_cast<const float *>(ptr(b)),
                        static_cast<const float *>(ptr(addend)), static_cast<float *>(ptr(y)), rows, (int)O, (int)K, stream);
  }
  if (rc != 0) return without_results(outcome("dfa3d_linear_add", rc));
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// linear_sum(device, stream, (rows (..., O), weight (O, K), ...)) -> sum of rows times weight (..., K), not recorded, or None
PyObject *linear_sum(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(3)
  const Py_ssize_t n = pairs_of(args[2]);
  if (n == 0 || at::autocast::is_autocast_enabled(at::kCUDA) || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer)) return declined();
  dfa3d_linear_set sets[DFA3D_MAX_LINEAR_SETS];
  int64_t K = 0, rows = 0, depth = 0, deepest = 0;
  std::vector<int64_t> sizes;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor &g = in.need(PyTuple_GET_ITEM(args[2], 2 * i)), &w = in.need(PyTuple_GET_ITEM(args[2], 2 * i + 1));
    if (!in.ok || g.scalar_type() != at::kFloat || g.dim() < 2 || !is_float_matrix(w) || g.size(-1) != w.size(0) || w.size(0) == 0 || recorded(g) ||
        recorded(w))
      return declined();
    auto shape = g.sizes().vec();
    shape.back() = w.size(1);
    if (i == 0) { sizes = shape; K = w.size(1); rows = g.numel() / w.size(0); }
    if (shape != sizes) return declined();
    depth += w.size(0);
    deepest = std::max(deepest, w.size(0));
    if (w.size(0) % 4 != 0) return declined();
    sets[i] = dfa3d_linear_set{static_cast<const float *>(ptr(w)), static_cast<const float *>(ptr(g)), static_cast<int>(w.size(0))};
  }
  if (!product_applies(rows, K, deepest, n > 1 && depth <= 1024)) return declined();
  Tensor y = at::empty(sizes, THPVariable_Unpack(PyTuple_GET_ITEM(args[2], 0)).options());
  int rc;
  {
    NoGil no_gil(in.locked);
    rc = api.linear_sum(sets, (int)n, static_cast<float *>(ptr(y)), rows, (int)K, stream);
  }
  if (rc != 0) return without_results(outcome("dfa3d_linear_sum", rc));
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// built_for() -> (version of the torch that this module was compiled against, version of the library's interface).  It touches no
// tensor and nothing of torch's: another torch's module says so before anything of it runs.
PyObject *built_for(PyObject *, PyObject *) { return Py_BuildValue("(si)", DFA3D_BUILT_FOR, DFA3D_ABI_VERSION); }

// seen() -> whether a tracer, a functorch transform, a profiler or another observer sees what this thread calls
PyObject *seen(PyObject *, PyObject *) { return PyBool_FromLong(observed()); }

// bind(dict of entry point -> address)
PyObject *bind(PyObject *, PyObject *table) {
  HANDLE_TH_ERRORS
  auto address = [&](const char *name, auto &to) {
    PyObject *o = PyDict_Check(table) ? PyDict_GetItemString(table, name) : nullptr;
    void *p = o != nullptr ? PyLong_AsVoidPtr(o) : nullptr;
    if (p == nullptr) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "no address of %s", name);
      return false;
    }
    to = reinterpret_cast<std::decay_t<decltype(to)>>(p);
    return true;
  };
  Api a;
  if (!address("dfa3d_last_error", a.last_error) || !address("dfa3d_packed_dist_bytes", a.packed_dist_bytes) ||
      !address("dfa3d_fused_forward", a.fused_forward) ||
      !address("dfa3d_fused_backward_workspace_bytes", a.fused_backward_workspace_bytes) ||
      !address("dfa3d_fused_backward", a.fused_backward) || !address("dfa3d_wms_deform_attn_forward", a.attention_forward) ||
      !address("dfa3d_wms_deform_attn_backward_workspace_bytes", a.attention_backward_workspace_bytes) ||
      !address("dfa3d_wms_deform_attn_backward", a.attention_backward) ||
      !address("dfa3d_ms_depth_score_sample_forward", a.score_forward) ||
      !address("dfa3d_ms_depth_score_sample_backward_workspace_bytes", a.score_backward_workspace_bytes) ||
      !address("dfa3d_ms_depth_score_sample_backward_into", a.score_backward) || !address("dfa3d_pack_dist", a.pack_dist) ||
      !address("dfa3d_linear_add", a.linear_add) || !address("dfa3d_linear_sum", a.linear_sum))
    return nullptr;
  api = a;
  show_as<dfa3d::MultiScaleDepthScoreSampleFunction>("MultiScaleDepthScoreSampleFunctionBackward");
  show_as<dfa3d::WeightedMultiScaleDeformableAttnFunction>("WeightedMultiScaleDeformableAttnFunctionBackward");
  show_as<dfa3d::MultiScaleDeformableAttnFunction>("MultiScaleDeformableAttnFunctionBackward");
  show_as<dfa3d::MultiScale3DDeformableAttnFunction>("MultiScale3DDeformableAttnFunctionBackward");
  show_as<dfa3d::MultiScale3DDeformableAttnWeightUpdateFunction>("MultiScale3DDeformableAttnWeightUpdateFunctionBackward");
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

typedef PyObject *(*Fast)(PyObject *, PyObject *const *, Py_ssize_t);
PyCFunction as_method(Fast f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }
PyMethodDef methods[] = {
    {"built_for", built_for, METH_NOARGS, nullptr},
    {"bind", bind, METH_O, nullptr},
    {"seen", seen, METH_NOARGS, nullptr},
    {"fused_forward", as_method(fused_forward), METH_FASTCALL, nullptr},
    {"fused_gradients", as_method(fused_gradients), METH_FASTCALL, nullptr},
    {"attention_forward", as_method(attention_forward), METH_FASTCALL, nullptr},
    {"attention_gradients", as_method(attention_gradients), METH_FASTCALL, nullptr},
    {"score_forward", as_method(score_forward), METH_FASTCALL, nullptr},
    {"score_gradients", as_method(score_gradients), METH_FASTCALL, nullptr},
    {"pack_dist", as_method(pack_dist), METH_FASTCALL, nullptr},
    {"call", as_method(call), METH_FASTCALL, nullptr},
    {"set_python_backward", set_python_backward, METH_O, nullptr},
    {"linear", as_method(linear), METH_FASTCALL, nullptr},
    {"linear_sum", as_method(linear_sum), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
