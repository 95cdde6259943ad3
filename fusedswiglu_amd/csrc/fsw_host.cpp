// The host path of the public entry points in native code: argument checks, allocations, the library calls and the autograd
// nodes of calls that nothing watches.  A training step of a small model is bound by its host time: in Python the launchers'
// checks, torch.autograd.Function and the custom operators took 100 of the 150 us of a step of 8192 x 256 x 768, whose kernels
// take 60.  All arithmetic stays in libfusedswiglu.
//
// Every function here answers None for a call that is not plain - other types, devices, orders or sizes than the kernels take
// as they are, tensor subclasses, autocast, a transform, tracer, mode, profiler or forward-mode AD at work - and the Python
// path behind it then does what it always did, its errors included.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/version.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include "../../include/fusedswiglu.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// From Python, at import: (check(status) raises, swiglu backward and down projection backward for calls that are not plain)
PyObject* g_check = nullptr;
PyObject* g_swiglu_backward = nullptr;
PyObject* g_down_backward = nullptr;
// the rule for padded copies (pads_rows in _launch.py)
int64_t g_pad_min_work = 0, g_pad_min_steps = 0, g_max_ld = 0;

// A failed library call: the Python exception that the launchers raise.
void check(int status) {
  if (status == FSW_OK) return;
  py::gil_scoped_acquire gil;
  PyObject* r = PyObject_CallFunction(g_check, "i", status);  // raises; the message is this thread's
  Py_XDECREF(r);
  if (r) throw std::runtime_error("libfusedswiglu call failed");
  python_error err;
  err.persist();
  throw err;
}

// Whether something watches the dispatcher or changes what a call means, on this thread and now.
bool watched() {
  using c10::DispatchKey;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  const c10::DispatchKeySet usual({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView});
  return !(tls.included_ - usual).empty() || c10::impl::TorchDispatchModeTLS::stack_len() > 0 ||
         at::impl::PythonTorchFunctionTLS::stack_len() > 0 || at::autocast::is_autocast_enabled(at::kCUDA) ||
         torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr || at::hasCallbacks();
}

bool plain(const Tensor& t, const Tensor& like) {
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::FuncTorchBatched,
                                         DispatchKey::FuncTorchGradWrapper, DispatchKey::Negative, DispatchKey::Conjugate,
                                         DispatchKey::ZeroTensor});
  return t.defined() && t.is_cuda() && t.device() == like.device() && t.scalar_type() == like.scalar_type() &&
         t.layout() == at::kStrided && !t.key_set().has_any(wrapped);
}
bool computes(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }

uintptr_t addr(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); }
int64_t pad8(int64_t n) { return (n + 7) & ~int64_t(7); }

// t seen as rows of its last dimension with one pitch and unit inner stride, without a copy.
struct Rows {
  int64_t rows = 0, cols = 0, ld = 0;
  uintptr_t p = 0;
  bool ok = false;
};
Rows rows_of(const Tensor& t) {
  Rows r;
  if (t.dim() < 2) return r;
  r.cols = t.size(-1);
  if (t.numel() == 0) return r;
  r.rows = t.numel() / r.cols;
  r.p = addr(t);
  if (t.is_contiguous()) r.ld = r.cols;
  else if (t.dim() == 2 && t.stride(1) == 1 && (t.size(0) == 1 || t.stride(0) >= r.cols)) r.ld = t.size(0) > 1 ? t.stride(0) : r.cols;
  else return r;
  r.ok = true;
  return r;
}
bool whole_chunks(const Rows& r) { return !((r.cols | r.ld) & 7 || r.p & 15); }

int64_t steps_of(int64_t m, int64_t n, int64_t k) {
  return (k + 31) / 32 * std::max<int64_t>((m + 63) / 64 * ((n + 63) / 64), 320);
}
// pads_rows of _launch.py for a forward (one product) or a backward (two)
bool pads_rows(int64_t T, int64_t D, int64_t I, bool backward) {
  if (T * D * I < g_pad_min_work || D > g_max_ld - 8 || I > g_max_ld - 8) return false;
  if (!backward) return steps_of(T, I, D) >= g_pad_min_steps;
  return steps_of(T, D, 2 * I) + steps_of(D, I, T + T / 2) >= 2 * g_pad_min_steps;
}

// The gate and up weights of a call, one parameter each or the halves of one.
struct Weights {
  Tensor gate, up;   // packed: up is undefined, gate holds both
  bool packed, out_in;
  int64_t D = 0, I = 0, ld = 0;
  uintptr_t pg = 0, pu = 0;
  bool ok = false;
  Weights(const Tensor& g, const Tensor& u, bool packed, bool out_in) : gate(g), up(u), packed(packed), out_in(out_in) {
    if (g.dim() != 2) return;
    const Rows r = rows_of(g);
    if (!r.ok) return;
    if (packed) {
      if (r.rows != g.size(0) || (out_in ? g.size(0) : g.size(1)) % 2) return;
      D = out_in ? g.size(1) : g.size(0);
      I = (out_in ? g.size(0) : g.size(1)) / 2;
      ld = r.ld;
      pg = r.p;
      pu = pg + 2 * static_cast<uintptr_t>(out_in ? I * ld : I);
    } else {
      const Rows ru = rows_of(u);
      if (!ru.ok || u.dim() != 2 || u.sizes() != g.sizes() || ru.ld != r.ld) return;
      D = out_in ? g.size(1) : g.size(0);
      I = out_in ? g.size(0) : g.size(1);
      ld = r.ld;
      pg = r.p;
      pu = ru.p;
    }
    ok = D > 0 && I > 0;
  }
  int64_t rows() const { return out_in ? I : D; }
  int64_t cols() const { return out_in ? D : I; }
  bool whole() const { return !((cols() | ld) & 7 || (pg | pu) & 15); }
};

struct Call {  // what every library call of one pass shares
  int dtype;
  void* stream;
  at::TensorOptions options;
  Call(const Tensor& like, bool out_in, bool padded)
      : dtype((like.scalar_type() == at::kHalf ? FSW_DTYPE_FP16 : FSW_DTYPE_BF16) | (out_in ? FSW_WEIGHTS_OUT_IN : 0) | (padded ? FSW_ROWS_PADDED : 0)),
        stream(c10::hip::getCurrentHIPStream(like.device().index()).stream()),
        options(like.options().requires_grad(false).memory_format(std::nullopt)) {}
  Tensor empty(at::IntArrayRef sizes) const { return at::empty(sizes, options); }
  // scratch of a step; holds the tensor
  Tensor scratch(int step, int64_t T, int64_t D, int64_t I, int64_t* bytes) const {
    *bytes = fsw_workspace_bytes(step | (dtype & FSW_WEIGHTS_OUT_IN), T, D, I);
    return *bytes > 0 ? at::empty({*bytes}, options.dtype(at::kByte)) : Tensor();
  }
};
void* ptr(uintptr_t p) { return reinterpret_cast<void*>(p); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// Copies between row pitches that go into one launch; the arrays outlive it.
struct Copies {
  fsw_row_copy copy[FSW_MAX_ROW_COPIES];
  int count = 0;
  void add(uintptr_t src, uintptr_t dst, int64_t rows, int64_t cols, int64_t ld_src, int64_t ld_dst, bool pad) {
    TORCH_INTERNAL_ASSERT(count < FSW_MAX_ROW_COPIES);
    copy[count++] = {ptr(src), ptr(dst), rows, cols, ld_src, ld_dst, pad};
  }
  void run(const Call& c) {
    if (count > 0) check(fsw_repack_group(copy, count, c.stream));
    count = 0;
  }
};

// Padded copies of rows the tiled kernels cannot read as they are (`keep` holds them), and of the two weights together.
void pad_rows(const Call& c, Rows& r, Tensor& keep, Copies& todo) {
  if (whole_chunks(r) && r.ld < g_max_ld) return;
  keep = c.empty({r.rows, pad8(r.cols)});
  todo.add(r.p, addr(keep), r.rows, r.cols, r.ld, pad8(r.cols), true);
  r.p = addr(keep);
  r.ld = pad8(r.cols);
}
void pad_weights(const Call& c, Weights& w, Tensor (&keep)[2], Copies& todo) {
  if (w.whole() && w.ld < g_max_ld) return;
  for (auto& k : keep) k = c.empty({w.rows(), pad8(w.cols())});
  todo.add(w.pg, addr(keep[0]), w.rows(), w.cols(), w.ld, pad8(w.cols()), true);
  todo.add(w.pu, addr(keep[1]), w.rows(), w.cols(), w.ld, pad8(w.cols()), true);
  w.pg = addr(keep[0]);
  w.pu = addr(keep[1]);
  w.ld = pad8(w.cols());
}
// The dense array of the given shape from a result whose rows are padded (as it is if they are not).
Tensor dense(const Call& c, const Tensor& padded, int64_t cols, at::IntArrayRef shape, Copies& todo) {
  if (padded.size(-1) == cols) return padded;
  Tensor out = c.empty(shape);
  todo.add(addr(padded), addr(out), padded.size(0), cols, padded.size(1), cols, false);
  return out;
}

c10::SmallVector<int64_t, 6> with_last(const Tensor& t, int64_t last) {
  c10::SmallVector<int64_t, 6> s(t.sizes().begin(), t.sizes().end());
  s.back() = last;
  return s;
}

// Whether run_forward can take the call.
bool forward_ok(const Tensor& x, const Weights& w) {
  const Rows r = rows_of(x);
  return w.ok && r.ok && r.cols == w.D;
}

// out, and if `save` the pre-activations: dense, or [T, I rounded up to 8] where the call runs on padded copies.
void run_forward(const Tensor& x, Weights w, bool save, Tensor& out, Tensor& g, Tensor& u) {
  const c10::DeviceGuard guard(x.device());
  Rows rx = rows_of(x);
  const int64_t T = rx.rows, D = w.D, I = w.I;
  const bool padded = ((D | I | rx.ld | w.ld) & 7 || (rx.p | w.pg | w.pu) & 15) && pads_rows(T, D, I, false);
  const Call c(x, w.out_in, padded);
  Tensor keep_x, keep_w[2];
  if (padded) {
    Copies todo;
    pad_rows(c, rx, keep_x, todo);
    pad_weights(c, w, keep_w, todo);
    todo.run(c);
  }
  const int64_t ldo = padded ? pad8(I) : I;
  const auto shape = with_last(x, I);
  const std::array<int64_t, 2> wide{T, ldo};
  const at::IntArrayRef result = ldo != I ? at::IntArrayRef(wide) : at::IntArrayRef(shape);
  out = c.empty(result);
  if (save) {
    g = c.empty(result);
    u = c.empty(result);
  }
  check(fsw_swiglu_forward(ptr(rx.p), ptr(w.pg), ptr(w.pu), ptr(out), ptr(g), ptr(u), T, D, I, rx.ld, w.ld, ldo, c.dtype, c.stream));
  if (padded) {
    Copies todo;
    const Tensor result_rows = out;
    out = dense(c, result_rows, I, shape, todo);
    todo.run(c);
  }
}

// The gradients that are asked for, or false for a call that is not plain.  Without g and u the pre-activations are recomputed.
bool run_backward(const Tensor& grad, const Tensor& x, Weights w, const Tensor& g, const Tensor& u, bool need_x, bool need_w, Tensor& dx,
                  Tensor& dw_gate, Tensor& dw_up) {
  Rows rx = rows_of(x);
  if (!w.ok || !rx.ok || rx.cols != w.D) return false;
  const int64_t T = rx.rows, D = w.D, I = w.I;
  const bool recompute = !g.defined() || g.numel() == 0;
  const bool padded = ((D | I | rx.ld | w.ld) & 7 || (rx.p | w.pg | w.pu) & 15) && pads_rows(T, D, I, true);
  const int64_t ldi = padded ? pad8(I) : I;
  if (grad.dim() != x.dim() || grad.size(-1) != I || grad.numel() != T * I) return false;
  if (!recompute && (g.numel() != T * ldi || u.numel() != T * ldi || !g.is_contiguous() || !u.is_contiguous() || (addr(g) | addr(u)) & 15))
    return false;
  // (on the edge kernel each step by itself weighs padded copies)
  if ((recompute || w.packed) && !padded && ((D | I | rx.ld | w.ld) & 7 || (rx.p | w.pg | w.pu | addr(grad)) & 15)) return false;
  const c10::DeviceGuard guard(x.device());
  const Call c(x, w.out_in, padded);
  const Tensor dout = grad.contiguous();
  Tensor keep_x, keep_w[2], keep_d;
  Copies todo;  // (what the gradients read: goes with the gating gradient)
  if (padded && (need_w || recompute)) pad_rows(c, rx, keep_x, todo);
  if (padded && (need_x || recompute)) pad_weights(c, w, keep_w, todo);
  const Tensor dG = c.empty({T, ldi}), dU = c.empty({T, ldi});
  const int64_t rows = w.rows(), cols = w.cols(), ldx = padded ? pad8(D) : D;
  // results: dense, or padded and made dense at the end; the halves of a packed gradient lie in one array
  Tensor pg, pu;
  int64_t ld_dw = padded ? pad8(cols) : cols;
  uintptr_t p_dwg = 0, p_dwu = 0;
  if (need_w) {
    if (w.packed) {
      dw_gate = c.empty({w.out_in ? 2 * I : D, w.out_in ? D : 2 * I});
      p_dwg = addr(dw_gate);
      p_dwu = p_dwg + 2 * static_cast<uintptr_t>(w.out_in ? I * D : I);
      if (!padded) ld_dw = dw_gate.size(1);
    }
    if (!w.packed || padded) {
      pg = c.empty({rows, ld_dw});
      pu = c.empty({rows, ld_dw});
    }
  }
  void* dwg = pg.defined() ? ptr(pg) : ptr(p_dwg);
  void* dwu = pu.defined() ? ptr(pu) : ptr(p_dwu);
  if (need_x) dx = ldx == D ? c.empty(x.sizes()) : c.empty({T, ldx});
  int64_t bytes = 0;
  Tensor ws;
  if (need_x || need_w) ws = c.scratch(need_x && need_w ? 7 : need_x ? 1 : 2, T, D, I, &bytes);
  if (!recompute && !padded) {
    check(fsw_swiglu_backward(ptr(dout), ptr(g), ptr(u), ptr(rx.p), ptr(w.pg), ptr(w.pu), ptr(dG), ptr(dU), ptr(dx), dwg, dwu, T, D, I,
                              rx.ld, w.ld, ldx, ld_dw, ptr(ws), bytes, c.dtype, c.stream));
  } else {
    if (recompute) {
      Rows rd;
      rd.rows = T, rd.cols = rd.ld = I, rd.p = addr(dout);
      if (padded) pad_rows(c, rd, keep_d, todo);
      todo.run(c);
      check(fsw_gating_grad_recompute(ptr(rx.p), ptr(w.pg), ptr(w.pu), ptr(rd.p), ptr(dU), ptr(dG), T, D, I, rx.ld, w.ld, ldi, c.dtype, c.stream));
    } else {
      check(fsw_elementwise_backward_group(ptr(dout), ptr(g), ptr(u), ptr(dU), ptr(dG), T, I, I, ldi, ldi, todo.copy, todo.count,
                                           c.dtype & ~(FSW_WEIGHTS_OUT_IN | FSW_ROWS_PADDED), c.stream));
      todo.count = 0;
    }
    if (need_x && need_w)
      check(fsw_swiglu_gradients(ptr(rx.p), ptr(w.pg), ptr(w.pu), ptr(dG), ptr(dU), ptr(dx), dwg, dwu, T, D, I, rx.ld, w.ld, ldi, ldx, ld_dw,
                                 ptr(ws), bytes, c.dtype, c.stream));
    else if (need_w)
      check(fsw_weight_grad(ptr(rx.p), ptr(dU), ptr(dG), dwu, dwg, T, D, I, rx.ld, ldi, ld_dw, ptr(ws), bytes, c.dtype, c.stream));
    else if (need_x)
      check(fsw_input_grad(ptr(dG), ptr(dU), ptr(w.pg), ptr(w.pu), ptr(dx), T, D, I, ldi, w.ld, ldx, ptr(ws), bytes, c.dtype, c.stream));
  }
  const Tensor dx_rows = dx;  // (held until the copies are enqueued)
  if (need_x) dx = dense(c, dx_rows, D, x.sizes(), todo);
  if (need_w) {
    if (w.packed && padded) {
      todo.add(addr(pg), p_dwg, rows, cols, ld_dw, dw_gate.size(1), false);
      todo.add(addr(pu), p_dwu, rows, cols, ld_dw, dw_gate.size(1), false);
    } else if (!w.packed && ld_dw != cols) {
      dw_gate = dense(c, pg, cols, {rows, cols}, todo);
      dw_up = dense(c, pu, cols, {rows, cols}, todo);
    } else if (!w.packed) {
      dw_gate = pg;
      dw_up = pu;
    }
  }
  todo.run(c);
  return true;
}

Tensor unpack(PyObject* o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }

// A backward pass that is not plain, in Python: a tuple of tensors or None.
variable_list in_python(PyObject* fn, std::initializer_list<Tensor> tensors, std::initializer_list<bool> flags, size_t results) {
  py::gil_scoped_acquire gil;
  py::tuple args(tensors.size() + flags.size());
  size_t i = 0;
  for (const Tensor& t : tensors) args[i++] = py::reinterpret_steal<py::object>(THPVariable_Wrap(t));
  for (bool f : flags) args[i++] = py::bool_(f);
  py::object r = py::reinterpret_steal<py::object>(PyObject_CallObject(fn, args.ptr()));
  if (!r) {
    python_error err;
    err.persist();
    throw err;
  }
  py::tuple t = py::reinterpret_borrow<py::tuple>(r);
  variable_list out(results);
  for (size_t k = 0; k < results; k++) out[k] = unpack(py::object(t[k]).ptr());
  return out;
}

enum { kPacked = 1, kOutIn = 2, kRecompute = 4, kOperator = 8 };  // kOperator: the module's entry points, whose operator is
                                                                  // what a recorded or watched backward pass goes through

Tensor swiglu_node_forward(AutogradContext* ctx, const Tensor& x, const Tensor& wg, const Tensor& wu, int64_t flags) {
  Tensor out, g, u;
  {
    const at::AutoDispatchBelowADInplaceOrView below;  // (nothing in here is recorded)
    run_forward(x, Weights(wg, wu, flags & kPacked, flags & kOutIn), !(flags & kRecompute), out, g, u);
  }
  ctx->save_for_backward({x, wg, wu, g, u});
  ctx->saved_data["flags"] = flags;
  return out;
}

variable_list swiglu_node_backward(AutogradContext* ctx, Tensor grad) {
  const auto saved = ctx->get_saved_variables();
  const Tensor &x = saved[0], &wg = saved[1], &wu = saved[2], &g = saved[3], &u = saved[4];
  const int64_t flags = ctx->saved_data["flags"].toInt();
  const bool packed = flags & kPacked, out_in = flags & kOutIn, need_x = ctx->needs_input_grad(0), need_g = ctx->needs_input_grad(1);
  const bool need_u = !packed && ctx->needs_input_grad(2);
  if (grad.scalar_type() != x.scalar_type()) grad = grad.to(x.scalar_type());
  Tensor dx, dwg, dwu;
  bool done = !((flags & kOperator) && (c10::GradMode::is_enabled() || watched())) && plain(grad, x) && plain(x, x) && plain(wg, x) &&
              (packed || plain(wu, x)) && (!g.defined() || (plain(g, x) && plain(u, x)));
  if (done) {
    const at::AutoDispatchBelowADInplaceOrView below;
    done = run_backward(grad, x, Weights(wg, wu, packed, out_in), g, u, need_x, need_g || need_u, dx, dwg, dwu);
  }
  if (!done) {
    const variable_list r = in_python(g_swiglu_backward, {grad, x, wg, wu, g, u}, {need_x, need_g, need_u, packed, out_in, bool(flags & kOperator)}, 3);
    dx = r[0], dwg = r[1], dwu = r[2];
  }
  return {need_x ? dx : Tensor(), need_g ? dwg : Tensor(), need_u ? dwu : Tensor()};
}

enum { kBF16Function, kHalfFunction, kOperatorCall };  // FusedSwiGLU, FastAccumFusedSwiGLU, ops.swiglu: what grad_fn is called
template <int KIND>
struct SwigluNode : torch::autograd::Function<SwigluNode<KIND>> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& wg, const Tensor& wu, int64_t flags) {
    return swiglu_node_forward(ctx, x, wg, wu, flags);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list r = swiglu_node_backward(ctx, grads[0]);
    r.emplace_back();
    return r;
  }
};
struct PackedNode : torch::autograd::Function<PackedNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, int64_t flags) {
    return swiglu_node_forward(ctx, x, w, Tensor(), flags);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) { return swiglu_node_backward(ctx, grads[0]); }
};

// ---- the down projection -------------------------------------------------------------------------------------------------
bool down_ok(const Tensor& a, const Tensor& w, bool out_in) {
  const Rows ra = rows_of(a), rw = rows_of(w);
  const int64_t I = w.dim() == 2 ? w.size(out_in ? 1 : 0) : 0, D = w.dim() == 2 ? w.size(out_in ? 0 : 1) : 0;
  // (others may run on padded copies: left to Python)
  return ra.ok && rw.ok && I > 0 && D > 0 && ra.cols == I && whole_chunks(ra) && whole_chunks(rw) && !((D | I) & 7);
}

Tensor run_down(const Tensor& a, const Tensor& w, bool out_in) {
  const c10::DeviceGuard guard(a.device());
  const Call c(a, out_in, false);
  const Rows ra = rows_of(a), rw = rows_of(w);
  const int64_t T = ra.rows, I = ra.cols, D = w.size(out_in ? 0 : 1);
  Tensor y = c.empty(with_last(a, D));
  int64_t bytes;
  const Tensor ws = c.scratch(4, T, D, I, &bytes);
  check(fsw_down_proj_forward(ptr(ra.p), ptr(rw.p), ptr(y), T, I, D, ra.ld, rw.ld, D, ptr(ws), bytes, c.dtype, c.stream));
  return y;
}

struct DownNode : torch::autograd::Function<DownNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& w, bool out_in) {
    ctx->save_for_backward({a, w});
    ctx->saved_data["out_in"] = out_in;
    const at::AutoDispatchBelowADInplaceOrView below;
    return run_down(a, w, out_in);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &a = saved[0], &w = saved[1];
    const bool out_in = ctx->saved_data["out_in"].toBool(), need_a = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
    Tensor grad = grads[0];
    if (grad.scalar_type() != a.scalar_type()) grad = grad.to(a.scalar_type());
    const Tensor gy = grad.contiguous();
    const Rows ra = rows_of(a), rg = rows_of(gy), rw = rows_of(w);
    const int64_t I = a.size(-1), D = gy.size(-1), T = rg.rows;
    Tensor da, dw;
    if (!c10::GradMode::is_enabled() && !watched() && plain(gy, a) && plain(a, a) && plain(w, a) && down_ok(a, w, out_in) && rg.ok &&
        T == ra.rows && D == w.size(out_in ? 0 : 1) && whole_chunks(rg)) {
      const at::AutoDispatchBelowADInplaceOrView below;
      const c10::DeviceGuard guard(a.device());
      const Call c(a, out_in, false);
      if (need_a) da = c.empty(a.sizes());
      if (need_w) dw = c.empty(w.sizes());
      int64_t bytes;
      const Tensor ws = c.scratch(need_a && need_w ? 8 : need_a ? 5 : 6, T, D, I, &bytes);
      if (need_a && need_w)
        check(fsw_down_proj_backward(ptr(ra.p), ptr(rg.p), ptr(rw.p), ptr(da), ptr(dw), T, I, D, ra.ld, rg.ld, rw.ld, I, w.size(1), ptr(ws),
                                     bytes, c.dtype, c.stream));
      else if (need_a)
        check(fsw_down_proj_input_grad(ptr(rg.p), ptr(rw.p), ptr(da), T, I, D, rg.ld, rw.ld, I, ptr(ws), bytes, c.dtype, c.stream));
      else if (need_w)
        check(fsw_down_proj_weight_grad(ptr(ra.p), ptr(rg.p), ptr(dw), T, I, D, ra.ld, rg.ld, w.size(1), ptr(ws), bytes, c.dtype, c.stream));
    } else {
      const variable_list r = in_python(g_down_backward, {gy, a, w}, {need_a, need_w, out_in}, 2);
      da = r[0], dw = r[1];
    }
    return {need_a ? da : Tensor(), need_w ? dw : Tensor(), Tensor()};
  }
};

// ---- the nodes as grad_fn --------------------------------------------------------------------------------------------------
// What the Python nodes of the general path show of themselves: their name, saved_tensors and needs_input_grad.
template <typename T>
torch::autograd::CppNode<T>* node_of(PyObject* self) {
  return static_cast<torch::autograd::CppNode<T>*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get());
}
// weights: 2; 1 packed; 0 for the down projection, which saves its two arguments
template <typename T, int WEIGHTS>
PyObject* node_saved_tensors(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  variable_list v = node_of<T>(self)->ctx_.get_saved_variables();
  if (WEIGHTS == 1) v.erase(v.begin() + 2);
  if (WEIGHTS > 0) {  // pre-activations: none where they are recomputed, else in x's shape, without the padding of their rows
    const bool out_in = node_of<T>(self)->ctx_.saved_data["flags"].toInt() & kOutIn;
    const Tensor x = v[0], w = v[1];
    const int64_t I = (out_in ? w.size(0) : w.size(1)) / (WEIGHTS == 1 ? 2 : 1);
    for (size_t i = v.size() - 2; i < v.size(); i++)
      v[i] = v[i].defined() ? v[i].reshape(with_last(x, v[i].size(-1))).narrow(-1, 0, I) : at::empty({0}, x.options().requires_grad(false));
  }
  py::tuple t(v.size());
  for (size_t i = 0; i < v.size(); i++) t[i] = py::reinterpret_steal<py::object>(THPVariable_Wrap(v[i]));
  return t.release().ptr();
  END_HANDLE_TH_ERRORS
}
// (of the tensors; the flags behind them never do)
template <typename T, int TENSORS>
PyObject* node_needs_input_grad(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  py::tuple t(TENSORS);
  for (int i = 0; i < TENSORS; i++) t[i] = py::bool_(node_of<T>(self)->ctx_.needs_input_grad(i));
  return t.release().ptr();
  END_HANDLE_TH_ERRORS
}
PyObject* node_set_sequence_nr(PyObject* self, PyObject* n) {
  HANDLE_TH_ERRORS
  const unsigned long long value = PyLong_AsUnsignedLongLong(n);
  if (PyErr_Occurred()) return nullptr;
  reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata->set_sequence_nr(value);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}
PyObject* node_name(PyObject* self, PyObject*) { return PyObject_GetAttrString(reinterpret_cast<PyObject*>(Py_TYPE(self)), "__name__"); }

template <typename T, int WEIGHTS, int TENSORS>
bool show_node(const char* name) {
  using namespace torch::autograd;  // (THPCppFunction_*)
  static PyGetSetDef properties[] = {{"saved_tensors", node_saved_tensors<T, WEIGHTS>, nullptr, nullptr, nullptr},
                                     {"needs_input_grad", node_needs_input_grad<T, TENSORS>, nullptr, nullptr, nullptr},
                                     THP_FUNCTION_DEFAULT_PROPERTIES,
                                     {nullptr, nullptr, nullptr, nullptr, nullptr}};
  static PyMethodDef node_methods[] = {{"name", node_name, METH_NOARGS, nullptr},
                                       {"register_hook", THPCppFunction_register_hook, METH_O, nullptr},
                                       {"register_prehook", THPCppFunction_register_prehook, METH_O, nullptr},
                                       {"_register_hook_dict", THPCppFunction_register_hook_dict, METH_O, nullptr},
                                       {"_sequence_nr", THPCppFunction_sequence_nr, METH_NOARGS, nullptr},
                                       {"_set_sequence_nr", node_set_sequence_nr, METH_O, nullptr},
                                       {nullptr, nullptr, 0, nullptr}};
  static PyTypeObject type;
  if (!torch::autograd::_initFunctionPyTypeObject(type, name, properties, node_methods)) return false;
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<T>), &type);
  return true;
}

// ---- Python ------------------------------------------------------------------------------------------------------------------
bool exact(PyObject* o) { return THPVariable_CheckExact(o) || reinterpret_cast<PyObject*>(Py_TYPE(o)) == ParameterClass; }

bool records(std::initializer_list<const Tensor*> ts) {
  if (!c10::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
bool inference(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && t->is_inference()) return true;
  return false;
}

// swiglu(x, w_gate, w_up or None (packed), dtype code or -1 (any), recompute, weights_out_in, operator) -> out or None
PyObject* py_swiglu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "swiglu takes 7 arguments");
    return nullptr;
  }
  const bool packed = args[2] == Py_None;
  if (!exact(args[0]) || !exact(args[1]) || !(packed || exact(args[2])) || watched()) Py_RETURN_NONE;
  const Tensor x = THPVariable_Unpack(args[0]), wg = THPVariable_Unpack(args[1]), wu = unpack(args[2]);
  const long want = PyLong_AsLong(args[3]);
  const bool recompute = args[4] == Py_True, out_in = args[5] == Py_True, op = args[6] == Py_True;
  if (!plain(x, x) || !computes(x) || (want >= 0 && want != (x.scalar_type() == at::kHalf ? FSW_DTYPE_FP16 : FSW_DTYPE_BF16)) ||
      !plain(wg, x) || !(packed || plain(wu, x)) || !forward_ok(x, Weights(wg, wu, packed, out_in)))
    Py_RETURN_NONE;
  Tensor out;
  if (records({&x, &wg, &wu})) {
    if (inference({&x, &wg, &wu})) Py_RETURN_NONE;
    const int64_t flags = (packed ? kPacked : 0) | (out_in ? kOutIn : 0) | (recompute ? kRecompute : 0) | (op ? kOperator : 0);
    const py::gil_scoped_release unlocked;
    out = packed ? PackedNode::apply(x, wg, flags)
          : op   ? SwigluNode<kOperatorCall>::apply(x, wg, wu, flags)
          : x.scalar_type() == at::kHalf ? SwigluNode<kHalfFunction>::apply(x, wg, wu, flags)
                                         : SwigluNode<kBF16Function>::apply(x, wg, wu, flags);
  } else {
    const py::gil_scoped_release unlocked;
    const at::AutoDispatchBelowADInplaceOrView below;
    Tensor g, u;
    run_forward(x, Weights(wg, wu, packed, out_in), false, out, g, u);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// down_proj(act, w_down, weights_out_in) -> y or None
PyObject* py_down_proj(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "down_proj takes 3 arguments");
    return nullptr;
  }
  if (!exact(args[0]) || !exact(args[1]) || watched()) Py_RETURN_NONE;
  const Tensor a = THPVariable_Unpack(args[0]), w = THPVariable_Unpack(args[1]);
  const bool out_in = args[2] == Py_True;
  if (!plain(a, a) || !computes(a) || !plain(w, a) || !down_ok(a, w, out_in)) Py_RETURN_NONE;
  Tensor y;
  if (records({&a, &w})) {
    if (inference({&a, &w})) Py_RETURN_NONE;
    const py::gil_scoped_release unlocked;
    y = DownNode::apply(a, w, out_in);
  } else {
    const py::gil_scoped_release unlocked;
    const at::AutoDispatchBelowADInplaceOrView below;
    y = run_down(a, w, out_in);
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// setup(check, swiglu_backward, down_backward, least work and steps for padded copies, longest rows of the tiled kernels)
PyObject* py_setup(PyObject*, PyObject* args) {
  PyObject *a, *b, *c;
  long long work, steps, ld;
  if (!PyArg_ParseTuple(args, "OOOLLL", &a, &b, &c, &work, &steps, &ld)) return nullptr;
  Py_INCREF(a), Py_INCREF(b), Py_INCREF(c);
  g_check = a, g_swiglu_backward = b, g_down_backward = c;
  g_pad_min_work = work, g_pad_min_steps = steps, g_max_ld = ld;
  Py_RETURN_NONE;
}

// pads_rows(T, D, I, backward) -> bool, for the test that holds it against the rule in Python
PyObject* py_pads_rows(PyObject*, PyObject* args) {
  long long T, D, I;
  int backward;
  if (!PyArg_ParseTuple(args, "LLLp", &T, &D, &I, &backward)) return nullptr;
  return PyBool_FromLong(pads_rows(T, D, I, backward));
}

PyMethodDef methods[] = {
    {"swiglu", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_swiglu)), METH_FASTCALL, nullptr},
    {"down_proj", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_down_proj)), METH_FASTCALL, nullptr},
    {"setup", py_setup, METH_VARARGS, nullptr},
    {"pads_rows", py_pads_rows, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fsw_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fsw_host() {
  static const bool shown = [] {  // (once per process)
#define FSW_NODE(name) "torch.autograd.function." name "Backward"
    return show_node<SwigluNode<kBF16Function>, 2, 3>(FSW_NODE("FusedSwiGLU")) &&
           show_node<SwigluNode<kHalfFunction>, 2, 3>(FSW_NODE("FastAccumFusedSwiGLU")) &&
           show_node<SwigluNode<kOperatorCall>, 2, 3>(FSW_NODE("GeneratedBackwardFor_fusedswiglu_amd_swiglu_forward_default")) &&
           show_node<PackedNode, 1, 2>(FSW_NODE("_PackedSwiGLU")) &&
           show_node<DownNode, 0, 2>(FSW_NODE("GeneratedBackwardFor_fusedswiglu_amd_down_proj_forward_default"));
#undef FSW_NODE
  }();
  if (!shown) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
