// The class surface's calls in one piece of native code each: checks, workspace look-ups and the C ABI call.
//
// A job of a few tokens is bound by what a call costs on the host. A launch takes 3.4 us there whoever makes it;
// checking tensors from Python, collecting their addresses and crossing into the library came to 2 to 4 us more per
// call, and to 20 us for the two launches and eight results of a job of eight ranks. Measured on the host per pass, us,
// before / with these: a one-GPU job of 16 tokens 25.9 / 15.9, a rank's five calls for 125 tokens 29.4 / 19.7, all eight
// ranks of a job of 16 tokens each 38.3 / 17.4; per pass among others, where the kernels now count as well: 26.4 / 19.7,
// 28.8 / 21.6, 35.5 / 15.1.
//
// Every function does a call in full or refuses it: None means that nothing has been launched, and the Python code,
// which accepts every form and raises for the rest, has the call. Only plain forms are taken: exact tensors without
// wrappers of any kind, of the expected type, device and shape, dense; exact ints in range. A refused status of the C
// ABI is left to the Python code as well. So nothing that was accepted is refused and nothing that was refused accepted.
//
// What is kept between calls are the workspace tensors that the rank object owns anyway (it calls forget() when it
// replaces one), never an address and nothing about a caller's tensor. The interpreter's lock is released around the
// C ABI call, as ctypes does; the workspace in use is held by the call, and arguments by the caller's frame.

#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <algorithm>
#include <memory>
#include <vector>

#include "moe_a2a.h"

namespace host_calls {

using at::ScalarType;
using at::Tensor;

// the tensor behind `o` if its memory can be handed on as it is
const Tensor* plain(PyObject* o) {
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                            c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::FuncTorchBatched,
                                            c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched});
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.key_set().has_any(wrapped) || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  return &t;
}

bool dense(const Tensor& t, ScalarType dt, int64_t device) {
  return t.scalar_type() == dt && t.is_cuda() && t.get_device() == device && t.is_contiguous();
}

bool shaped(const Tensor& t, int64_t a, int64_t b) { return t.dim() == 2 && t.size(0) == a && t.size(1) == b; }
bool shaped(const Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}

int32_t* ints(const Tensor& t) { return t.defined() ? static_cast<int32_t*>(t.data_ptr()) : nullptr; }

bool row_type(ScalarType dt) { return dt == at::kHalf || dt == at::kBFloat16; }
int32_t code(ScalarType dt) { return dt == at::kBFloat16 ? MOE_A2A_BF16 : MOE_A2A_F16; }

// an exact int from 0 to the largest int32
bool count(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && *v >= 0 && *v <= INT32_MAX;
}

bool same_address(PyObject* o, const Tensor& t) {
  return PyLong_CheckExact(o) && PyLong_AsVoidPtr(o) == t.data_ptr();
}

struct Names {
  PyObject *num_experts, *experts_per_token, *hidden_dim, *max_num_tokens, *in_dtype, *out_dtype, *x, *indices, *weights;
};
Names names;

bool type_of(PyObject* cfg, PyObject* name, ScalarType* dt) {
  PyObject* o = PyObject_GetAttr(cfg, name);
  if (!o) {
    PyErr_Clear();
    return false;
  }
  const bool ok = THPDtype_Check(o);
  if (ok) *dt = reinterpret_cast<THPDtype*>(o)->scalar_type;
  Py_DECREF(o);
  return ok;
}

// the current stream of a device; false with an exception set
bool stream_of(PyObject* raw_stream, PyObject* device, void** stream) {
  PyObject* r = PyObject_CallFunctionObjArgs(raw_stream, device, nullptr);
  if (!r) return false;
  *stream = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return !PyErr_Occurred();
}

// The C ABI call with the interpreter's lock released. Its arguments are worked out before that, by the caller: the
// address of a tensor that gives none (a lazily cloned one that cannot be copied, one that must not be written) is an
// exception, which needs the lock on its way out.
template <typename... Params, typename... Args>
bool launched(int (*entry)(Params...), Args... args) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = entry(args...);
  Py_END_ALLOW_THREADS
  return rc == MOE_A2A_OK;
}

// ------------------------------------------------------------------ one rank's calls

struct GemmOut {
  int64_t out_dim;
  bool second;  // (a layer that reads the first buffer of its width)
  Tensor out;
};

struct Workspace {
  Tensor send_counts, send_buf, send_meta;
  Tensor num, expert_x, expert_meta, offsets, plan;
  int64_t long_rows = 0;  // longer streams take the entry points with a planning launch
  Tensor row_position, entry_row;  // what those launches work out (stages 2 and 4)
  Tensor expert_y;
  Tensor back_counts, back_buf, back_meta, back_plan;
  Tensor where, direct_num, direct_x, direct_meta, direct_offsets;
  std::vector<GemmOut> gemm;
};

struct State {
  moe_a2a_shape shape;
  int64_t nle, max_recv, hidden, topk, device;
  ScalarType in, out;
  std::shared_ptr<Workspace> ws = std::make_shared<Workspace>();
  PyObject *raw_stream = nullptr, *device_index = nullptr;
  PyObject* cfg = nullptr;  // where the row types come from, if the rank object has said so
};

struct RankCalls {
  PyObject_HEAD
  State* s;
};

State& state(PyObject* self) { return *reinterpret_cast<RankCalls*>(self)->s; }

PyObject* rank_new(PyTypeObject* type, PyObject* args, PyObject*) {
  HANDLE_TH_ERRORS
  int32_t f[6];
  PyObject *in, *out, *device, *raw, *cfg = nullptr;
  if (!PyArg_ParseTuple(args, "(iiiiii)OOOO|O", &f[0], &f[1], &f[2], &f[3], &f[4], &f[5], &in, &out, &device, &raw, &cfg)) return nullptr;
  if (!THPDtype_Check(in) || !THPDtype_Check(out) || !PyLong_CheckExact(device) || f[0] < 1) {
    PyErr_SetString(PyExc_TypeError, "RankCalls((world_size, rank, num_experts, experts_per_token, hidden_dim, "
                                     "max_num_tokens), in_dtype, out_dtype, device_index, raw_stream, cfg=None)");
    return nullptr;
  }
  PyObject* self = type->tp_alloc(type, 0);
  if (!self) return nullptr;
  auto* s = new State();
  reinterpret_cast<RankCalls*>(self)->s = s;
  s->shape = moe_a2a_shape{f[0], f[1], f[2], f[3], f[4], f[5]};
  s->nle = f[2] / f[0];
  s->topk = f[3];
  s->hidden = f[4];
  s->max_recv = (int64_t)f[5] * f[0];
  s->in = reinterpret_cast<THPDtype*>(in)->scalar_type;
  s->out = reinterpret_cast<THPDtype*>(out)->scalar_type;
  s->device = PyLong_AsLongLong(device);
  Py_INCREF(raw);
  s->raw_stream = raw;
  Py_INCREF(device);
  s->device_index = device;
  if (cfg && cfg != Py_None) {
    Py_INCREF(cfg);
    s->cfg = cfg;
  }
  return self;
  END_HANDLE_TH_ERRORS
}

void rank_dealloc(PyObject* self) {
  State* s = reinterpret_cast<RankCalls*>(self)->s;
  if (s) {
    Py_XDECREF(s->raw_stream);
    Py_XDECREF(s->device_index);
    Py_XDECREF(s->cfg);
    delete s;
  }
  PyTypeObject* type = Py_TYPE(self);
  type->tp_free(self);
  Py_DECREF(type);
}

PyObject* rank_forget(PyObject* self, PyObject*) {
  state(self).ws = std::make_shared<Workspace>();
  Py_RETURN_NONE;
}

// Whether rows are there (`t`, a workspace buffer or an argument) and of the type that these calls were made for, which the
// config still names: a caller may set its types between two calls, and the Python code then makes the buffers anew.
bool known(const State& s, const Tensor& t, PyObject* name, ScalarType made_for) {
  ScalarType now;
  return t.defined() && t.scalar_type() == made_for && (!s.cfg || (type_of(s.cfg, name, &now) && now == made_for));
}
bool known_in(const State& s, const Tensor& t) { return known(s, t, names.in_dtype, s.in); }
bool known_out(const State& s, const Tensor& t) { return known(s, t, names.out_dtype, s.out); }

#define REFUSE Py_RETURN_NONE
#define TAKES(N)                                                          \
  if (n != N) {                                                           \
    PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n); \
    return nullptr;                                                       \
  }

// the workspace to change: a copy where a call in another thread is using it (calls come and go under the interpreter's lock)
std::shared_ptr<Workspace> own(State& s) { return s.ws.use_count() == 1 ? s.ws : std::make_shared<Workspace>(*s.ws); }

// The tensors of one method filled in; arguments: tensors or None, in the order of `to`.
PyObject* learn(State& s, PyObject* const* a, std::initializer_list<Tensor Workspace::*> to, int64_t long_rows = -1) {
  for (size_t i = 0; i < to.size(); ++i)
    if (a[i] != Py_None && !plain(a[i])) REFUSE;
  auto next = own(s);
  for (auto field : to) {
    if (*a == Py_None) {
      (*next).*field = Tensor();
    } else {
      (*next).*field = *plain(*a);
    }
    ++a;
  }
  if (long_rows >= 0) next->long_rows = long_rows;
  s.ws = std::move(next);
  Py_RETURN_TRUE;
}

PyObject* learn_send(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(3)
  return learn(state(self), a, {&Workspace::send_counts, &Workspace::send_buf, &Workspace::send_meta});
  END_HANDLE_TH_ERRORS
}

// (x, indices) -> tokens
PyObject* dispatch_send(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(2)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *x = plain(a[0]), *idx = plain(a[1]);
  if (!known_in(s, ws->send_buf) || !x || !idx || idx->dim() != 2) REFUSE;
  const int64_t T = idx->size(0);
  if (T > s.shape.max_num_tokens || idx->size(1) != s.topk || !shaped(*x, T, s.hidden) || !dense(*x, s.in, s.device) ||
      !dense(*idx, at::kInt, s.device))
    REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  if (!launched(moe_a2a_dispatch_send, &s.shape, x->data_ptr(), ints(*idx), (int32_t)T, ws->send_buf.data_ptr(),
                ints(ws->send_meta), ints(ws->send_counts), nullptr, stream))
    REFUSE;
  return PyLong_FromLongLong(T);
  END_HANDLE_TH_ERRORS
}

// (num, expert_x, expert_meta, offsets or None, plan or None, long_rows); offsets: the compact layout
PyObject* learn_recv(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(6)
  int64_t long_rows;
  if (!count(a[5], &long_rows)) REFUSE;
  return learn(state(self), a, {&Workspace::num, &Workspace::expert_x, &Workspace::expert_meta, &Workspace::offsets, &Workspace::plan}, long_rows);
  END_HANDLE_TH_ERRORS
}

// (row_position)
PyObject* learn_positions(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(1)
  return learn(state(self), a, {&Workspace::row_position});
  END_HANDLE_TH_ERRORS
}

// (counts, buf, meta, rows) -> rows that sized the launch
PyObject* dispatch_recv(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(4)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *counts = plain(a[0]), *buf = plain(a[1]), *meta = plain(a[2]);
  int64_t rows;
  if (!known_in(s, ws->expert_x) || !counts || !buf || !meta || !count(a[3], &rows)) REFUSE;
  if (buf->dim() != 2 || buf->size(1) != s.hidden || meta->dim() != 2 || meta->size(1) != MOE_A2A_META_DIM ||
      counts->numel() < s.shape.world_size || !dense(*counts, at::kInt, s.device) || !dense(*buf, s.in, s.device) ||
      !dense(*meta, at::kInt, s.device))
    REFUSE;
  const int64_t capacity = std::min(buf->size(0), meta->size(0));
  if (capacity > INT32_MAX) REFUSE;
  rows = std::min(rows, capacity);
  const bool compact = ws->offsets.defined();
  const bool planned = rows > ws->long_rows;
  if (planned && (!ws->row_position.defined() || ws->row_position.numel() < capacity)) REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const int32_t hint = (int32_t)rows, room = (int32_t)capacity, compact_room = compact ? (int32_t)ws->expert_x.size(0) : 0;
  void *const from = buf->data_ptr(), *const to = ws->expert_x.data_ptr();
  int32_t *const m = ints(*meta), *const c = ints(*counts), *const num = ints(ws->num), *const to_meta = ints(ws->expert_meta);
  int32_t *const plan = ints(ws->plan), *const offsets = ints(ws->offsets);
  int32_t* const position = planned ? ints(ws->row_position) : nullptr;
  const bool ok =
      compact && planned ? launched(moe_a2a_dispatch_recv_compact_long, &s.shape, from, m, c, hint, room, num, offsets, to, to_meta,
                                    compact_room, plan, position, stream)
      : compact ? launched(moe_a2a_dispatch_recv_compact, &s.shape, from, m, c, hint, room, num, offsets, to, to_meta, compact_room,
                           plan, stream)
      : planned ? launched(moe_a2a_dispatch_recv_long, &s.shape, from, m, c, hint, room, num, to, to_meta, plan, position, stream)
                : launched(moe_a2a_dispatch_recv, &s.shape, from, m, c, hint, room, num, to, to_meta, plan, stream);
  if (!ok) REFUSE;
  return PyLong_FromLongLong(rows);
  END_HANDLE_TH_ERRORS
}

PyObject* learn_scale(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(1)
  return learn(state(self), a, {&Workspace::expert_y});
  END_HANDLE_TH_ERRORS
}

// rows of an expert buffer in this rank's layouts, padded [nle, max_recv, width] or compact [rows, width]
bool expert_rows(const State& s, const Tensor& t, int64_t width) {
  return shaped(t, s.nle, s.max_recv, width) || (t.dim() == 2 && t.size(1) == width && t.size(0) <= INT32_MAX);
}

// (expert_x, num, rows) -> expert_y
PyObject* expert_scale(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(3)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *x = plain(a[0]), *num = plain(a[1]);
  int64_t rows;
  if (!x || !known_in(s, *x) || !known_out(s, ws->expert_y) || !num || !count(a[2], &rows)) REFUSE;
  if (!row_type(s.in) || !row_type(s.out) || !expert_rows(s, *x, s.hidden) || x->sizes() != ws->expert_y.sizes() ||
      num->numel() < s.nle || !dense(*x, s.in, s.device) || !dense(*num, at::kInt, s.device))
    REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const bool ok =
      x->dim() == 2 ? launched(moe_a2a_expert_scale_compact, &s.shape, x->data_ptr(), ints(*num), (int32_t)rows,
                               (int32_t)x->size(0), code(s.in), code(s.out), ws->expert_y.data_ptr(), stream)
                    : launched(moe_a2a_expert_scale, &s.shape, x->data_ptr(), ints(*num), (int32_t)rows, code(s.in), code(s.out),
                               ws->expert_y.data_ptr(), stream);
  if (!ok) REFUSE;
  return THPVariable_Wrap(ws->expert_y);
  END_HANDLE_TH_ERRORS
}

// (out, out is the second buffer of its width)
PyObject* learn_gemm(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(2)
  State& s = state(self);
  const Tensor* out = plain(a[0]);
  if (!out || out->dim() < 2) REFUSE;
  auto next = own(s);
  // (one per width and place, as the rank object owns them: its names are these two)
  const GemmOut made{out->size(-1), a[1] == Py_True, *out};
  auto known = std::find_if(next->gemm.begin(), next->gemm.end(),
                            [&](const GemmOut& g) { return g.out_dim == made.out_dim && g.second == made.second; });
  if (known == next->gemm.end()) next->gemm.push_back(made);
  else *known = made;
  s.ws = std::move(next);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (expert_x, num, weights, bias or None, rows) -> the product, in the rank's buffer of that width
PyObject* expert_gemm(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(5)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *x = plain(a[0]), *num = plain(a[1]), *w = plain(a[2]), *bias = a[3] == Py_None ? nullptr : plain(a[3]);
  int64_t rows;
  if (ws->gemm.empty() || !x || !num || !w || (!bias && a[3] != Py_None) || !count(a[4], &rows)) REFUSE;
  const ScalarType dt = x->scalar_type();
  if (!row_type(dt) || w->dim() != 3 || x->dim() < 2) REFUSE;
  const int64_t in_dim = x->size(-1), out_dim = w->size(1);
  if (in_dim > INT32_MAX || out_dim > INT32_MAX || !expert_rows(s, *x, in_dim) || !shaped(*w, s.nle, out_dim, in_dim) ||
      (bias && !(shaped(*bias, s.nle, out_dim) && dense(*bias, dt, s.device))) || num->numel() < s.nle ||
      !dense(*x, dt, s.device) || !dense(*w, dt, s.device) || !dense(*num, at::kInt, s.device))
    REFUSE;
  const Tensor *first = nullptr, *second = nullptr;
  for (const GemmOut& g : ws->gemm)
    if (g.out_dim == out_dim && g.out.scalar_type() == dt && g.out.dim() == x->dim() && g.out.size(0) == x->size(0) &&
        (x->dim() == 2 || g.out.size(1) == x->size(1)))
      (g.second ? second : first) = &g.out;
  if (!first) REFUSE;
  const Tensor* out = first->data_ptr() == x->data_ptr() ? second : first;
  if (!out || out->data_ptr() == x->data_ptr()) REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const void* b = bias ? bias->data_ptr() : nullptr;
  const bool ok =
      x->dim() == 2 ? launched(moe_a2a_expert_gemm_compact, &s.shape, x->data_ptr(), ints(*num), (int32_t)rows,
                               (int32_t)x->size(0), w->data_ptr(), b, (int32_t)in_dim, (int32_t)out_dim, code(dt),
                               out->data_ptr(), stream)
                    : launched(moe_a2a_expert_gemm, &s.shape, x->data_ptr(), ints(*num), (int32_t)rows, w->data_ptr(), b,
                               (int32_t)in_dim, (int32_t)out_dim, code(dt), out->data_ptr(), stream);
  if (!ok) REFUSE;
  return THPVariable_Wrap(*out);
  END_HANDLE_TH_ERRORS
}

// (counts, buf, meta, plan or None)
PyObject* learn_back(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(4)
  return learn(state(self), a, {&Workspace::back_counts, &Workspace::back_buf, &Workspace::back_meta, &Workspace::back_plan});
  END_HANDLE_TH_ERRORS
}

// (expert_meta, expert_y, num, rows, (addresses that the plan is for) or None) -> True
PyObject* combine_send(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(5)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *meta = plain(a[0]), *y = plain(a[1]), *num = plain(a[2]);
  int64_t rows;
  if (!known_out(s, ws->back_buf) || !meta || !y || !num || !count(a[3], &rows)) REFUSE;
  const bool compact = y->dim() == 2;
  if (!row_type(s.out) || !expert_rows(s, *y, s.hidden) || num->numel() < s.nle || !dense(*y, s.out, s.device) ||
      !dense(*meta, at::kInt, s.device) || !dense(*num, at::kInt, s.device) ||
      (compact ? meta->dim() != 2 || meta->size(1) != MOE_A2A_META_DIM : meta->numel() < s.nle * s.max_recv * MOE_A2A_META_DIM))
    REFUSE;
  const bool planned = PyTuple_CheckExact(a[4]) && PyTuple_GET_SIZE(a[4]) == 2 && same_address(PyTuple_GET_ITEM(a[4], 0), *meta) &&
                       same_address(PyTuple_GET_ITEM(a[4], 1), *num);
  if (planned && !ws->back_plan.defined()) REFUSE;
  const int64_t capacity = std::min(ws->back_buf.size(0), ws->back_meta.size(0));
  rows = std::min(rows, capacity);
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const int32_t* plan = planned ? ints(ws->back_plan) : nullptr;
  const bool ok =
      compact ? launched(moe_a2a_combine_send_compact, &s.shape, y->data_ptr(), ints(*meta), ints(*num), (int32_t)rows,
                         (int32_t)std::min(y->size(0), meta->size(0)), (int32_t)capacity, ws->back_buf.data_ptr(),
                         ints(ws->back_meta), ints(ws->back_counts), plan, stream)
              : launched(moe_a2a_combine_send, &s.shape, y->data_ptr(), ints(*meta), ints(*num), (int32_t)rows, (int32_t)capacity,
                         ws->back_buf.data_ptr(), ints(ws->back_meta), ints(ws->back_counts), plan, stream);
  if (!ok) REFUSE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// rows of a result that the weights address: [>= T, hidden] of the out type, and [T, K] weights
bool takes_results(const State& s, const Tensor& out, const Tensor& weights) {
  return weights.dim() == 2 && weights.size(1) == s.topk && weights.size(0) <= INT32_MAX && out.dim() == 2 &&
         out.size(0) >= weights.size(0) && out.size(1) == s.hidden && row_type(s.out) && dense(out, s.out, s.device) &&
         dense(weights, at::kFloat, s.device);
}

// (entry_row)
PyObject* learn_table(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(1)
  return learn(state(self), a, {&Workspace::entry_row});
  END_HANDLE_TH_ERRORS
}

// (out, weights, counts, buf, meta, accumulate, rows from which streams are long) -> True
PyObject* combine_recv(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(7)
  State& s = state(self);
  const Tensor *out = plain(a[0]), *weights = plain(a[1]), *counts = plain(a[2]), *buf = plain(a[3]), *meta = plain(a[4]);
  int64_t long_rows;
  if (!out || !known_out(s, *out) || !weights || !counts || !buf || !meta || !PyBool_Check(a[5]) || !count(a[6], &long_rows)) REFUSE;
  if (!takes_results(s, *out, *weights) || buf->dim() != 2 || buf->size(1) != s.hidden || meta->dim() != 2 ||
      meta->size(1) != MOE_A2A_META_DIM || counts->numel() < s.shape.world_size || !dense(*counts, at::kInt, s.device) ||
      !dense(*buf, s.out, s.device) || !dense(*meta, at::kInt, s.device))
    REFUSE;
  const int64_t T = weights->size(0), capacity = std::min(buf->size(0), meta->size(0)), rows = std::min(capacity, T * s.topk);
  const auto ws = s.ws;
  const bool mapped = rows > long_rows;
  if (capacity > INT32_MAX || (mapped && (!ws->entry_row.defined() || ws->entry_row.numel() < T * s.topk))) REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const int32_t accumulate = a[5] == Py_True;
  void *const from = buf->data_ptr(), *const to = out->data_ptr();
  int32_t *const m = ints(*meta), *const c = ints(*counts);
  const float* const w = static_cast<const float*>(weights->data_ptr());
  int32_t* const table = mapped ? ints(ws->entry_row) : nullptr;
  const bool ok = mapped ? launched(moe_a2a_combine_recv_long, &s.shape, from, m, c, (int32_t)rows, (int32_t)capacity, w, (int32_t)T, to,
                                    accumulate, code(s.out), table, stream)
                         : launched(moe_a2a_combine_recv, &s.shape, from, m, c, (int32_t)rows, (int32_t)capacity, w, (int32_t)T, to,
                                    accumulate, code(s.out), stream);
  if (!ok) REFUSE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// A job of one rank: (num, expert_x, expert_meta, where, offsets or None)
PyObject* learn_direct(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(5)
  return learn(state(self), a, {&Workspace::direct_num, &Workspace::direct_x, &Workspace::direct_meta, &Workspace::where, &Workspace::direct_offsets});
  END_HANDLE_TH_ERRORS
}

// (x, indices) -> tokens
PyObject* direct_dispatch(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(2)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *x = plain(a[0]), *idx = plain(a[1]);
  if (!ws->where.defined() || !known_in(s, ws->direct_x) || !x || !idx || idx->dim() != 2) REFUSE;
  const int64_t T = idx->size(0);
  const bool compact = ws->direct_offsets.defined();
  if (T > s.shape.max_num_tokens || idx->size(1) != s.topk || !shaped(*x, T, s.hidden) || !dense(*x, s.in, s.device) ||
      !dense(*idx, at::kInt, s.device) || (compact && T * s.topk > ws->direct_x.size(0)))
    REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const void* xs[1] = {x->data_ptr()};
  const int32_t* ids[1] = {ints(*idx)};
  const int32_t tokens[1] = {(int32_t)T};
  if (!launched(moe_a2a_local_dispatch, &s.shape, xs, ids, tokens, compact ? (int32_t)ws->direct_x.size(0) : 0, -1, -1,
                ints(ws->where), ints(ws->direct_num), ints(ws->direct_offsets), ws->direct_x.data_ptr(), ints(ws->direct_meta),
                stream))
    REFUSE;
  return PyLong_FromLongLong(T);
  END_HANDLE_TH_ERRORS
}

// (out, weights, expert_meta, expert_y, num, (address of expert_meta, of num, tokens) of the dispatch) -> True
PyObject* direct_combine(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(6)
  State& s = state(self);
  const auto ws = s.ws;
  const Tensor *out = plain(a[0]), *weights = plain(a[1]), *meta = plain(a[2]), *y = plain(a[3]), *num = plain(a[4]);
  if (!ws->where.defined() || !out || !known_out(s, *out) || !weights || !meta || !y || !num || !PyTuple_CheckExact(a[5]) || PyTuple_GET_SIZE(a[5]) != 3) REFUSE;
  if (!takes_results(s, *out, *weights) || !dense(*y, s.out, s.device)) REFUSE;
  const int64_t T = weights->size(0);
  int64_t tokens_dispatched;
  if (!same_address(PyTuple_GET_ITEM(a[5], 0), *meta) || !same_address(PyTuple_GET_ITEM(a[5], 1), *num) ||
      !count(PyTuple_GET_ITEM(a[5], 2), &tokens_dispatched) || tokens_dispatched != T)
    REFUSE;
  const bool compact = ws->direct_offsets.defined();
  if (compact ? y->dim() != 2 || y->size(0) < T * s.topk || y->size(1) != s.hidden : !shaped(*y, s.nle, s.max_recv, s.hidden)) REFUSE;
  void* stream;
  if (!stream_of(s.raw_stream, s.device_index, &stream)) return nullptr;
  const float* ws_of[1] = {static_cast<const float*>(weights->data_ptr())};
  void* outs[1] = {out->data_ptr()};
  const int32_t tokens[1] = {(int32_t)T};
  if (!launched(moe_a2a_local_combine, &s.shape, y->data_ptr(), ints(ws->where), ws_of, tokens, outs, -1, 1, code(s.out), stream))
    REFUSE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ calls without a rank object

bool can_allocate() { return !c10::impl::TorchDispatchModeTLS::any_modes_set(); }

// (raw_stream, input, weight, bias or None) -> [M, N]
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(4)
  const Tensor *x = plain(a[1]), *w = plain(a[2]), *bias = a[3] == Py_None ? nullptr : plain(a[3]);
  if (!x || !w || (!bias && a[3] != Py_None) || !x->is_cuda() || !can_allocate()) REFUSE;
  const ScalarType dt = x->scalar_type();
  const int64_t device = x->get_device();
  if (!row_type(dt) || x->dim() != 2 || w->dim() != 2 || w->size(1) != x->size(1) || !dense(*x, dt, device) || !dense(*w, dt, device) ||
      (bias && (bias->dim() != 1 || bias->size(0) != w->size(0) || !dense(*bias, dt, device))))
    REFUSE;
  const int64_t m = x->size(0), cols = w->size(0), k = x->size(1);
  if (m > INT32_MAX || cols > INT32_MAX || k > INT32_MAX) REFUSE;
  PyObject* index = PyLong_FromLongLong(device);
  if (!index) return nullptr;
  void* stream;
  const bool have_stream = stream_of(a[0], index, &stream);
  Py_DECREF(index);
  if (!have_stream) return nullptr;
  const Tensor out = at::empty({m, cols}, at::TensorOptions().dtype(dt).device(x->device()));
  if (!launched(moe_a2a_linear, x->data_ptr(), w->data_ptr(), bias ? bias->data_ptr() : nullptr, (int32_t)m, (int32_t)cols,
                (int32_t)k, code(dt), out.data_ptr(), stream))
    REFUSE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

bool number_of(PyObject* cfg, PyObject* name, int64_t* v) {  // false without an exception: not a plain count
  PyObject* o = PyObject_GetAttr(cfg, name);
  if (!o) {
    PyErr_Clear();
    return false;
  }
  const bool ok = count(o, v);
  Py_DECREF(o);
  return ok;
}

bool tensor_of(PyObject* data, PyObject* name, Tensor* t) {
  PyObject* o = PyObject_GetAttr(data, name);
  if (!o) {
    PyErr_Clear();
    return false;
  }
  const Tensor* p = plain(o);
  if (p) *t = *p;
  Py_DECREF(o);
  return p != nullptr;
}

// (raw_stream, cfg, world_size, inputs of the ranks, own rank data or None, own rank, every rank's result): one
// step of a job whose ranks share this GPU, as `submission._run_direct` does it -> a list of every rank's result, or
// the own rank's. `inputs[r][1]` is rank r's data; the own rank's comes with the call where only its result is asked for.
PyObject* job(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TAKES(7)
  constexpr int MAX_RANKS = 64, MAX_EXPERTS = 1024, MAX_TOPK = 64;  // of moe_a2a_local_dispatch
  PyObject *cfg = a[1], *inputs = a[3], *own = a[4];
  int64_t W, own_rank, E, K, H, max_tokens;
  ScalarType in, out;
  const bool everyone = a[6] == Py_True;
  if (!count(a[2], &W) || W < 1 || W > MAX_RANKS || !count(a[5], &own_rank) || own_rank >= W || !can_allocate()) REFUSE;
  if (!(PyList_CheckExact(inputs) || PyTuple_CheckExact(inputs)) || PySequence_Fast_GET_SIZE(inputs) != W) REFUSE;
  if (!number_of(cfg, names.num_experts, &E) || !number_of(cfg, names.experts_per_token, &K) || !number_of(cfg, names.hidden_dim, &H) ||
      !number_of(cfg, names.max_num_tokens, &max_tokens) || !type_of(cfg, names.in_dtype, &in) || !type_of(cfg, names.out_dtype, &out) ||
      !row_type(in) || !row_type(out) ||
      E > MAX_EXPERTS || K > MAX_TOPK || E % W != 0)
    REFUSE;
  Tensor x[MAX_RANKS], ids[MAX_RANKS], weights[MAX_RANKS];
  const void* xs[MAX_RANKS];
  const int32_t* is[MAX_RANKS];
  const float* wts[MAX_RANKS];
  int32_t tokens[MAX_RANKS];
  int64_t entries = 0, device = -1;
  for (int64_t r = 0; r < W; ++r) {
    PyObject* d = own;
    if (own == Py_None || r != own_rank) {
      PyObject* item = PySequence_Fast_GET_ITEM(inputs, r);
      if (!PyTuple_CheckExact(item) || PyTuple_GET_SIZE(item) != 4) REFUSE;
      d = PyTuple_GET_ITEM(item, 1);
    }
    Py_INCREF(d);  // (reading an attribute may run code that changes `inputs`)
    const bool there = tensor_of(d, names.x, &x[r]) && tensor_of(d, names.indices, &ids[r]) && tensor_of(d, names.weights, &weights[r]);
    Py_DECREF(d);
    if (!there || (PySequence_Fast_GET_SIZE(inputs) != W)) REFUSE;
    if (r == 0) {
      if (!x[0].is_cuda()) REFUSE;
      device = x[0].get_device();
    }
    const int64_t T = ids[r].dim() == 2 ? ids[r].size(0) : -1;
    if (T < 0 || T > INT32_MAX || ids[r].size(1) != K || !shaped(x[r], T, H) || !shaped(weights[r], T, K) || !dense(x[r], in, device) ||
        !dense(ids[r], at::kInt, device) || !dense(weights[r], at::kFloat, device))
      REFUSE;
    xs[r] = x[r].data_ptr();
    is[r] = ints(ids[r]);
    wts[r] = static_cast<const float*>(weights[r].data_ptr());
    tokens[r] = (int32_t)T;
    entries += T * K;
  }
  if (entries > INT32_MAX || c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA)->getDevice().index() != device) REFUSE;
  PyObject* index = PyLong_FromLongLong(device);
  if (!index) return nullptr;
  void* stream;
  const bool have_stream = stream_of(a[0], index, &stream);
  Py_DECREF(index);
  if (!have_stream) return nullptr;
  const moe_a2a_shape shape{(int32_t)W, 0, (int32_t)E, (int32_t)K, (int32_t)H, (int32_t)max_tokens};
  const auto options = at::TensorOptions().device(x[0].device());
  const Tensor rows = at::empty({std::max<int64_t>(entries, 1), H}, options.dtype(out));
  const Tensor where = at::empty({std::max<int64_t>(entries, 1)}, options.dtype(at::kInt));
  if (!launched(moe_a2a_local_dispatch, &shape, xs, is, tokens, (int32_t)rows.size(0), code(in), code(out), ints(where), nullptr,
                nullptr, rows.data_ptr(), nullptr, stream))
    REFUSE;
  // (a tensor of its own for each rank: views of one would keep all results as long as any of them)
  Tensor y[MAX_RANKS];
  void* outs[MAX_RANKS] = {};
  for (int64_t r = 0; r < W; ++r) {
    if (!everyone && r != own_rank) continue;
    y[r] = at::empty({tokens[r], H}, options.dtype(out));
    outs[r] = y[r].data_ptr();
  }
  if (!launched(moe_a2a_local_combine, &shape, rows.data_ptr(), ints(where), wts, tokens, outs, everyone ? -1 : (int32_t)own_rank,
                0, code(out), stream))
    REFUSE;
  if (!everyone) return THPVariable_Wrap(y[own_rank]);
  PyObject* list = PyList_New(W);
  if (!list) return nullptr;
  for (int64_t r = 0; r < W; ++r) {
    PyObject* o = THPVariable_Wrap(y[r]);
    if (!o) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, r, o);
  }
  return list;
  END_HANDLE_TH_ERRORS
}

#define FAST(NAME, DOC) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, DOC}
PyMethodDef rank_methods[] = {
    {"forget", rank_forget, METH_NOARGS, "the rank object has replaced a workspace buffer"},
    FAST(learn_send, "(counts, buf, meta)"),
    FAST(dispatch_send, "(x, indices) -> tokens or None"),
    FAST(learn_recv, "(num, expert_x, expert_meta, offsets, plan, long_rows)"),
    FAST(learn_positions, "(row_position)"),
    FAST(dispatch_recv, "(counts, buf, meta, rows) -> rows or None"),
    FAST(learn_scale, "(expert_y)"),
    FAST(expert_scale, "(expert_x, num, rows) -> expert_y or None"),
    FAST(learn_gemm, "(out, second)"),
    FAST(expert_gemm, "(expert_x, num, weights, bias, rows) -> out or None"),
    FAST(learn_back, "(counts, buf, meta, plan)"),
    FAST(combine_send, "(expert_meta, expert_y, num, rows, planned_for) -> True or None"),
    FAST(learn_table, "(entry_row)"),
    FAST(combine_recv, "(out, weights, counts, buf, meta, accumulate, long_rows) -> True or None"),
    FAST(learn_direct, "(num, expert_x, expert_meta, where, offsets)"),
    FAST(direct_dispatch, "(x, indices) -> tokens or None"),
    FAST(direct_combine, "(out, weights, expert_meta, expert_y, num, dispatched_for) -> True or None"),
    {nullptr, nullptr, 0, nullptr}};
PyMethodDef functions[] = {
    FAST(linear, "(raw_stream, input, weight, bias) -> output or None"),
    FAST(job, "(raw_stream, cfg, world_size, inputs, own, own_rank, everyone) -> results or None"),
};
#undef FAST

PyType_Slot rank_slots[] = {{Py_tp_new, reinterpret_cast<void*>(rank_new)},
                            {Py_tp_dealloc, reinterpret_cast<void*>(rank_dealloc)},
                            {Py_tp_methods, rank_methods},
                            {0, nullptr}};
PyType_Spec rank_spec = {"moe_a2a_torch.RankCalls", sizeof(RankCalls), 0, Py_TPFLAGS_DEFAULT, rank_slots};

}  // namespace host_calls

// what the extension was built from (build.extension_id): the Python code and these calls have to be of one state
std::string a2a_extension_id() { return A2A_EXTENSION_ID; }

// {"RankCalls": type, "linear": function, "job": function}
py::dict a2a_host_calls() {
  using namespace host_calls;
  auto intern = [](const char* s) { return PyUnicode_InternFromString(s); };
  if (!names.x)
    names = Names{intern("num_experts"), intern("experts_per_token"), intern("hidden_dim"), intern("max_num_tokens"),
                  intern("in_dtype"),    intern("out_dtype"),         intern("x"),          intern("indices"),
                  intern("weights")};
  py::dict d;
  d["RankCalls"] = py::reinterpret_steal<py::object>(PyType_FromSpec(&rank_spec));
  for (PyMethodDef& f : functions) d[f.ml_name] = py::reinterpret_steal<py::object>(PyCFunction_New(&f, nullptr));
  return d;
}
