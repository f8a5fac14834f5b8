// Calls of the operator from Python without the interpreter's share of the work: operand checks, output tensors and the C-ABI call of
// dfa3d_hip in one step.  On 2 x 100 queries a forward spends 6 us in its kernel; checks, allocations and the call through ctypes
// took 10 of the 17 us that it cost.
//
// Every function takes the operands only where all of them are what its kernels read: plain tensors (no subclass, no transform's
// wrapper) of the right shapes and types, contiguous, on the device that is current, under no dispatch mode, with something to do.  Anything else is declined
// (None), and the Python form of the call, which says what is wrong, takes it from there.  The library's entry points come as
// addresses (bind), so this module serves whichever build of the library is loaded.
#include <Python.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <initializer_list>
#include <limits>
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
  decltype(&dfa3d_linear) linear;
  decltype(&dfa3d_linear_sum) linear_sum;
} api;

using at::Tensor;

// the operands of one call; `ok` says whether all of them can be read as they are
struct Operands {
  int64_t device;
  bool ok = true;
  // a tensor that is no wrapper: on this device, contiguous, with storage of its own
  const Tensor &need(PyObject *o) {
    static const Tensor none;
    if (!THPVariable_CheckExact(o)) { ok = false; return none; }
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || !t.has_storage() || !t.is_contiguous() ||
        t.is_neg() || t.is_conj())
      ok = false;
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
PyObject *failed(const char *name, int rc) {
  PyErr_Format(PyExc_RuntimeError, "%s failed with code %d: %s", name, rc, api.last_error());
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
bool step_ok(int64_t batch, PyObject *o) {
  if (!PyLong_CheckExact(o)) return false;
  const long long given = PyLong_AsLongLong(o), step = given < batch ? given : batch;
  if (given == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  return step > 0 && batch % step == 0;
}
struct NoGil {
  PyThreadState *state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
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
#define TAKES(n)                                                                            \
  if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; } \
  Operands in; void *stream;                                                                \
  if (!numbers(args, in.device, stream)) return nullptr;                                    \
  if (!plain_dispatch()) return declined();

// fused_forward(device, stream, value, dist, shapes, starts, loc, attn, im2col_step, need_score, need_weight_update, packed)
// -> (out, score or None, weight_update or None), or None
PyObject *fused_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(12)
  const Tensor &value = in.need(args[2]), &dist = in.need(args[3]), &shapes = in.need(args[4]), &starts = in.need(args[5]),
               &loc = in.need(args[6]), &attn = in.need(args[7]), &packed = in.may_have(args[11]);
  FusedDims d;
  if (!in.ok || !fused_dims(value, dist, shapes, starts, loc, attn, d) || !step_ok(d.B, args[8])) return declined();
  if (packed.defined()) {
    const size_t least = d.heads == 1 ? api.packed_dist_bytes(d.B, d.S, d.D, d.L, d.code) : 0;
    if (least == 0 || packed.nbytes() < least) return declined();
  }
  const auto store = value.options(), aux = store.dtype(d.aux);
  Tensor out = at::empty({d.B, d.Q, d.M * d.C}, store), score, wu;
  if (args[9] == Py_True) score = at::empty({d.B, d.Q, d.M, d.L, d.P, 4}, store);
  if (args[10] == Py_True) wu = at::empty({d.B, d.Q, d.M, 1}, aux);
  int rc;
  {
    NoGil no_gil;
    rc = api.fused_forward(ptr(value), ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(attn), ptr(out), ptr(score), ptr(wu), ptr(packed),
                           d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, d.code, nullptr, stream);
  }
  if (rc != 0) return failed("dfa3d_fused_forward", rc);
  return tuple_of({out, score, wu});
  END_HANDLE_TH_ERRORS
}

// fused_gradients(device, stream, value, dist, shapes, starts, loc, attn, grad_out, grad_score, grad_weight_update, im2col_step)
// -> gradients of value, dist, loc and attn in their types, or None
PyObject *fused_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(12)
  const Tensor &value = in.need(args[2]), &dist = in.need(args[3]), &shapes = in.need(args[4]), &starts = in.need(args[5]),
               &loc = in.need(args[6]), &attn = in.need(args[7]), &grad_out = in.need(args[8]), &grad_score = in.may_have(args[9]),
               &grad_wu = in.may_have(args[10]);
  FusedDims d;
  if (!in.ok || !fused_dims(value, dist, shapes, starts, loc, attn, d) || !step_ok(d.B, args[11])) return declined();
  if (grad_out.numel() != d.B * d.Q * d.M * d.C || grad_out.scalar_type() != d.type) return declined();
  if (grad_score.defined() && (!shape_is(grad_score, {d.B, d.Q, d.M, d.L, d.P, 4}) || grad_score.scalar_type() != d.type)) return declined();
  if (grad_wu.defined() && (grad_wu.numel() != d.B * d.Q * d.M || grad_wu.scalar_type() != d.aux)) return declined();
  // bfloat16 gradients are written as such where that is offered
  const dfa3d_launch_options clear = own_gradients(true);
  const bool g16 = d.type == at::kBFloat16 &&
                   api.fused_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, DFA3D_BF16G, &clear) > 0;
  const int code = g16 ? DFA3D_BF16G : d.code;
  const size_t bytes = api.fused_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.D, d.L, d.Q, d.P, d.heads, code, &clear);
  const auto aux = value.options().dtype(d.aux), sums = g16 ? value.options() : aux;
  Tensor grad_value = at::empty(value.sizes(), sums), grad_dist = at::empty(dist.sizes(), sums), grad_loc = at::empty(loc.sizes(), aux),
         grad_attn = at::empty(attn.sizes(), aux), workspace;
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, value.options().dtype(at::kByte));
  int rc;
  {
    NoGil no_gil;
    rc = api.fused_backward(ptr(value), ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(attn), ptr(grad_out), ptr(grad_score), ptr(grad_wu),
                            ptr(grad_value), ptr(grad_dist), ptr(grad_loc), ptr(grad_attn), ptr(workspace), bytes, d.B, d.S, d.M, d.C, d.D, d.L,
                            d.Q, d.P, d.heads, code, &clear, stream);
  }
  if (rc != 0) return failed("dfa3d_fused_backward", rc);
  return tuple_of({grad_value.to(d.type), grad_dist.to(d.type), grad_loc, grad_attn});
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

// attention_forward(device, stream, value, shapes, starts, loc, attn, score or None, im2col_step) -> out, or None
PyObject *attention_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(9)
  const Tensor &value = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &attn = in.need(args[6]), &score = in.may_have(args[7]);
  AttentionDims d;
  if (!in.ok || !attention_dims(value, shapes, starts, loc, attn, score, d) || !step_ok(d.B, args[8])) return declined();
  Tensor out = at::empty({d.B, d.Q, d.M * d.C}, value.options());
  int rc;
  {
    NoGil no_gil;
    rc = api.attention_forward(ptr(value), keys(shapes), d.shape_width, keys(starts), ptr(loc), d.loc_width, ptr(attn), ptr(score), ptr(out),
                               d.B, d.S, d.M, d.C, d.L, d.Q, d.P, d.code, nullptr, stream);
  }
  if (rc != 0) return failed("dfa3d_wms_deform_attn_forward", rc);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// attention_gradients(device, stream, value, shapes, starts, loc (2 wide), attn, score or None, grad_out, im2col_step)
// -> gradients of value, loc, attn and score (None without one) in their types, or None
PyObject *attention_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(10)
  const Tensor &value = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &attn = in.need(args[6]), &score = in.may_have(args[7]), &grad_out = in.need(args[8]);
  AttentionDims d;
  if (!in.ok || !attention_dims(value, shapes, starts, loc, attn, score, d) || d.loc_width != 2 || !step_ok(d.B, args[9])) return declined();
  if (grad_out.numel() != d.B * d.Q * d.M * d.C || grad_out.scalar_type() != d.type) return declined();
  const dfa3d_launch_options clear = own_gradients(true);
  const size_t bytes = api.attention_backward_workspace_bytes(d.B, d.S, d.M, d.C, d.L, d.Q, d.P, d.code, &clear);
  const auto aux = value.options().dtype(d.aux);
  Tensor grad_value = at::empty(value.sizes(), aux), grad_loc = at::empty(loc.sizes(), aux), grad_attn = at::empty(attn.sizes(), aux), grad_score,
         workspace;
  if (score.defined()) grad_score = at::empty(score.sizes(), aux);
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, value.options().dtype(at::kByte));
  int rc;
  {
    NoGil no_gil;
    rc = api.attention_backward(ptr(value), keys(shapes), d.shape_width, keys(starts), ptr(loc), d.loc_width, ptr(attn), ptr(score), ptr(grad_out),
                                ptr(grad_value), ptr(grad_loc), d.loc_width, ptr(grad_attn), ptr(grad_score), ptr(workspace), bytes, d.B, d.S,
                                d.M, d.C, d.L, d.Q, d.P, d.code, &clear, stream);
  }
  if (rc != 0) return failed("dfa3d_wms_deform_attn_backward", rc);
  return tuple_of({grad_value.to(d.type), grad_loc, grad_attn, grad_score.defined() ? grad_score.to(d.type) : grad_score});
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

// score_forward(device, stream, dist, shapes, starts, loc, im2col_step) -> score, or None
PyObject *score_forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(7)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]);
  ScoreDims d;
  if (!in.ok || !score_dims(dist, shapes, starts, loc, d) || !step_ok(d.B, args[6])) return declined();
  Tensor score = at::empty({d.B, d.Q, d.M, d.L, d.P, 4}, dist.options());
  int rc;
  {
    NoGil no_gil;
    rc = api.score_forward(ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(score), d.B, d.S, d.M, d.D, d.L, d.Q, d.P, d.code, nullptr, stream);
  }
  if (rc != 0) return failed("dfa3d_ms_depth_score_sample_forward", rc);
  return THPVariable_Wrap(score);
  END_HANDLE_TH_ERRORS
}

// score_gradients(device, stream, dist, shapes, starts, loc, grad_score, im2col_step) -> gradients of dist and loc in their types, or None
PyObject *score_gradients(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(8)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]), &loc = in.need(args[5]),
               &grad_score = in.need(args[6]);
  ScoreDims d;
  if (!in.ok || !score_dims(dist, shapes, starts, loc, d) || !step_ok(d.B, args[7])) return declined();
  if (!shape_is(grad_score, {d.B, d.Q, d.M, d.L, d.P, 4}) || grad_score.scalar_type() != d.type) return declined();
  const dfa3d_launch_options options = own_gradients(false);      // (this entry point clears by itself)
  const size_t bytes = api.score_backward_workspace_bytes(d.B, d.S, d.M, d.D, d.L, d.Q, d.P, d.code, &options);
  const auto aux = dist.options().dtype(d.aux);
  Tensor grad_dist = at::empty(dist.sizes(), aux), grad_loc = at::empty(loc.sizes(), aux), workspace;
  if (bytes > 0) workspace = at::empty({(int64_t)bytes}, dist.options().dtype(at::kByte));
  int rc;
  {
    NoGil no_gil;
    rc = api.score_backward(ptr(dist), keys(shapes), keys(starts), ptr(loc), ptr(grad_score), ptr(grad_dist), ptr(grad_loc), ptr(workspace), bytes,
                            d.B, d.S, d.M, d.D, d.L, d.Q, d.P, d.code, &options, stream);
  }
  if (rc != 0) return failed("dfa3d_ms_depth_score_sample_backward", rc);
  return tuple_of({grad_dist.to(d.type), grad_loc});
  END_HANDLE_TH_ERRORS
}

// pack_dist(device, stream, dist (bs, keys, 1, D), shapes, starts) -> packed distribution, or None
PyObject *pack_dist(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(5)
  const Tensor &dist = in.need(args[2]), &shapes = in.need(args[3]), &starts = in.need(args[4]);
  if (!in.ok || dist.dim() != 4 || dist.size(2) != 1 || shapes.dim() != 2 || shapes.size(1) != 3 || !shape_is(starts, {shapes.size(0)}) ||
      shapes.scalar_type() != at::kLong || starts.scalar_type() != at::kLong)
    return declined();
  const int64_t B = dist.size(0), S = dist.size(1), D = dist.size(3), L = shapes.size(0);
  const int code = code_of(dist.scalar_type());
  if (!(code == DFA3D_F32 || code == DFA3D_BF16) || !fits_int({B, S, D, L})) return declined();
  const size_t bytes = api.packed_dist_bytes(B, S, D, L, code);
  if (bytes == 0) return declined();
  Tensor packed = at::empty({(int64_t)bytes}, dist.options().dtype(at::kByte));
  int rc;
  {
    NoGil no_gil;
    rc = api.pack_dist(ptr(dist), keys(shapes), keys(starts), ptr(packed), bytes, B, S, D, L, code, stream);
  }
  if (rc != 0) return failed("dfa3d_pack_dist", rc);
  return THPVariable_Wrap(packed);
  END_HANDLE_TH_ERRORS
}

// Where the kernels form a product of rows x width elements, sums of depth terms.  They read four neighbours of a row at a time, and take the
// library's place except where few rows meet a deep sum.  Library and kernel, us a call one after the other: 4096 rows of 256 by 256 19, 9; 256 by 64
// 19, 8; sums of 512 by 256 19, 22; of 2048 by 256 41, 51 to 89; of 1024 by 1024 72, 58; 20000 rows of 512 by 512 98, 70; of 2048 by 256 165, 145; 100000 of
// 256 by 256 123, 93.  The 18 to 19 are the library call's host time, which bounds it up to some 5000 rows; on the device alone (captured in a graph)
// 100 rows of 256 by 256 30, 8, 625 rows 5.5, 8.0, 1500 rows 5.6, 8.2, 4096 rows 10, 9; of 256 by 64 4096 rows 5.4, 7.8, 10000 rows 7.3, 8.2.
bool product_applies(int64_t rows, int64_t width, int64_t depth) {
  return width > 0 && depth > 0 && width <= 4096 && depth <= 4096 && width % 2 == 0 && depth % 4 == 0 && rows > 0 && rows <= (int64_t(1) << 31) &&
         (depth <= 256 || rows * width >= (int64_t(1) << 22));
}
// pairs of a flat tuple, 0 where it is none of 1 to as many pairs as a call takes
Py_ssize_t pairs_of(PyObject *o) {
  const Py_ssize_t n = PyTuple_CheckExact(o) ? PyTuple_GET_SIZE(o) : 0;
  return n % 2 == 0 && n / 2 <= DFA3D_MAX_LINEAR_SETS ? n / 2 : 0;
}
bool is_float_matrix(const Tensor &t) { return t.scalar_type() == at::kFloat && t.dim() == 2; }
bool recorded(const Tensor &t) { return t.defined() && t.requires_grad() && c10::GradMode::is_enabled(); }

// linear(device, stream, x (..., K), weight (O, K), bias (O) or None) -> F.linear, not recorded, or None
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TAKES(5)
  const Tensor &x = in.need(args[2]), &w = in.need(args[3]), &b = in.may_have(args[4]);
  if (!in.ok || x.scalar_type() != at::kFloat || x.dim() < 2 || !is_float_matrix(w) || x.size(-1) != w.size(1) || w.size(1) == 0 ||
      (b.defined() && (b.scalar_type() != at::kFloat || !shape_is(b, {w.size(0)}))) || recorded(x) || recorded(w) || recorded(b) ||
      at::autocast::is_autocast_enabled(at::kCUDA) || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer))
    return declined();
  const int64_t O = w.size(0), K = w.size(1), rows = x.numel() / K;
  if (!product_applies(rows, O, K)) return declined();
  auto sizes = x.sizes().vec();
  sizes.back() = O;
  Tensor y = at::empty(sizes, x.options());
  int rc;
  {
    NoGil no_gil;
    rc = api.linear(static_cast<const float *>(ptr(x)), static_cast<const float *>(ptr(w)), static_cast<const float *>(ptr(b)),
                    static_cast<float *>(ptr(y)), rows, (int)O, (int)K, stream);
  }
  if (rc != 0) return failed("dfa3d_linear", rc);
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
  int64_t K = 0, rows = 0;
  std::vector<int64_t> sizes;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor &g = in.need(PyTuple_GET_ITEM(args[2], 2 * i)), &w = in.need(PyTuple_GET_ITEM(args[2], 2 * i + 1));
    if (!in.ok || g.scalar_type() != at::kFloat || g.dim() < 2 || !is_float_matrix(w) || g.size(-1) != w.size(0) || w.size(0) == 0 || recorded(g) ||
        recorded(w))
      return declined();
    auto shape = g.sizes().vec();
    shape.back() = w.size(1);
    if (i == 0) { sizes = shape; K = w.size(1); rows = g.numel() / w.size(0); }
    if (shape != sizes || !product_applies(rows, K, w.size(0))) return declined();
    sets[i] = dfa3d_linear_set{static_cast<const float *>(ptr(w)), static_cast<const float *>(ptr(g)), static_cast<int>(w.size(0))};
  }
  Tensor y = at::empty(sizes, THPVariable_Unpack(PyTuple_GET_ITEM(args[2], 0)).options());
  int rc;
  {
    NoGil no_gil;
    rc = api.linear_sum(sets, (int)n, static_cast<float *>(ptr(y)), rows, (int)K, stream);
  }
  if (rc != 0) return failed("dfa3d_linear_sum", rc);
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// built_for() -> (version of the torch that this module was compiled against, version of the library's interface).  It touches no
// tensor and nothing of torch's: another torch's module says so before anything of it runs.
PyObject *built_for(PyObject *, PyObject *) { return Py_BuildValue("(si)", DFA3D_BUILT_FOR, DFA3D_ABI_VERSION); }

// seen() -> whether a tracer, a functorch transform, a profiler or another observer sees what this thread calls
PyObject *seen(PyObject *, PyObject *) {
  const c10::DispatchKeySet modes = c10::impl::tls_local_dispatch_key_set().included_;
  return PyBool_FromLong(at::hasCallbacks() || torch::jit::tracer::isTracing() || modes.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
                         modes.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode));
}

// bind(dict of entry point -> address)
PyObject *bind(PyObject *, PyObject *table) {
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
      !address("dfa3d_linear", a.linear) || !address("dfa3d_linear_sum", a.linear_sum))
    return nullptr;
  api = a;
  Py_RETURN_NONE;
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
    {"linear", as_method(linear), METH_FASTCALL, nullptr},
    {"linear_sum", as_method(linear_sum), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
