// host_calls.cpp - the Python calls of the kernels, prepared natively: a CPython
// extension (lib/bd3_host.so) that takes torch tensors, makes them readable for
// the kernels, allocates outputs and workspaces and calls the C ABI of
// libbd3attn.so on the tensors' current stream.
//
// Why: prepared in Python (attribute reads, torch.empty, slices of the cache and
// of the modulation vectors, ctypes argument conversion) a call cost more host
// time than most of the kernels it launches take. Host time per call, launches
// included: attention_inputs with a cache 16.0 -> 7.7 us, decode of a 16-token
// block (two launches) 16.4 -> 8.2, ln_modulate 12.9 -> 5.0, with the residual
// 17.8 -> 6.2, gate_residual 11.4 -> 4.7, the sampling draw 10.8 -> 5.5 (now two
// launches), training forward + backward 128 -> 87 (67 of it autograd's own).
//
// The C ABI's addresses come from the caller (bind), which loads the library, so
// the library path and a missing library behave as there. Argument errors raise
// AssertionError with the same texts as the Python checks and the library's
// messages, runtime errors RuntimeError. Every function drops the GIL once its
// arguments are unpacked: a launch can wait for a full queue.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <string>
#include <type_traits>

#include "bd3attn.h"

namespace {

using at::Tensor;

constexpr int kHeadDim = 64;
const float kScale = 1.0f / std::sqrt((float)kHeadDim);

// The C ABI, bound by name.
struct Library {
  decltype(&bd3_last_error) last_error;
  decltype(&bd3_attn_fwd) attn_fwd;
  decltype(&bd3_attn_bwd_workspace_bytes) attn_bwd_workspace_bytes;
  decltype(&bd3_attn_bwd) attn_bwd;
  decltype(&bd3_decode) decode;
  decltype(&bd3_decode_splitkv) decode_splitkv;
  decltype(&bd3_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&bd3_qkv_rope) qkv_rope;
  decltype(&bd3_subs_sample_ws) subs_sample_ws;
  decltype(&bd3_subs_sample_workspace_bytes) subs_sample_workspace_bytes;
  decltype(&bd3_ln_modulate) ln_modulate;
  decltype(&bd3_gate_residual) gate_residual;
  decltype(&bd3_gate_residual_ln_modulate) gate_residual_ln_modulate;
} g_lib = {};

// A Python exception to raise: its type (PyExc_...) and text.
struct Refused {
  PyObject* type;
  std::string text;
};

void require(bool ok, const char* text) {
  if (!ok) throw Refused{PyExc_AssertionError, text};
}

// Status of a C-ABI call, as kernels._native.check maps it.
void check(int status) {
  if (status == BD3_OK) return;
  const char* m = g_lib.last_error();
  const std::string text = m ? m : "";
  if (status == BD3_EINVAL) throw Refused{PyExc_AssertionError, text};
  throw Refused{PyExc_RuntimeError, "libbd3attn: " + text};
}

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// Runs f and turns what it throws into a Python exception.
template <class F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const Refused& r) {
    PyErr_SetString(r.type, r.text.c_str());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// Argument readers: positional only, in the order of the Python wrappers.
struct Args {
  PyObject* const* a;
  Py_ssize_t n, at = 0;
  Args(PyObject* const* args, Py_ssize_t count, Py_ssize_t want) : a(args), n(count) {
    if (count != want) throw Refused{PyExc_TypeError, "wrong number of arguments"};
  }
  Tensor tensor() {
    PyObject* o = a[at++];
    if (!THPVariable_Check(o)) throw Refused{PyExc_TypeError, "expected a tensor"};
    return THPVariable_Unpack(o);
  }
  Tensor maybe_tensor() {  // undefined for None
    if (a[at] == Py_None) {
      ++at;
      return Tensor();
    }
    return tensor();
  }
  int64_t integer() {
    const long long v = PyLong_AsLongLong(a[at++]);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  int32_t int32() {
    const int64_t v = integer();
    if (v < INT32_MIN || v > INT32_MAX) throw Refused{PyExc_OverflowError, "argument does not fit 32 bits"};
    return (int32_t)v;
  }
  uint64_t unsigned64() {  // modulo 2^64, any integer, as ctypes takes it (a seed or counter set by the caller)
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(a[at++]);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  double real() {
    const double v = PyFloat_AsDouble(a[at++]);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
  }
};

template <class... T>
PyObject* pack(const T&... t) {
  PyObject* r = PyTuple_New(sizeof...(T));
  if (r == nullptr) return nullptr;
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t)), ...);
  return r;
}

// The kernels read 16-byte vectors of rows in place: 16-byte aligned base,
// last stride 1, other strides multiples of 8 elements. Anything else is
// copied (kernels._native.as_kernel_input).
bool vec_ready(const Tensor& t) {
  if (t.dim() == 0 || t.stride(-1) != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if (t.stride(i) % 8 != 0) return false;
  return true;
}

Tensor ready(const Tensor& t) { return vec_ready(t) ? t : t.contiguous(); }

// (b, h, s) element strides of 4-D tensors, in order.
template <class... T>
std::array<int64_t, 3 * sizeof...(T)> strides(const T&... ts) {
  std::array<int64_t, 3 * sizeof...(T)> s;
  size_t i = 0;
  auto add = [&](const Tensor& t) {
    require(t.dim() == 4 && t.stride(-1) == 1, "tensors must be 4-D with last stride 1");
    for (int d = 0; d < 3; ++d) s[i++] = t.stride(d);
  };
  (add(ts), ...);
  return s;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The kernels read the operands' addresses as they are: refuses any that is not
// on the first one's GPU (an undefined one is an absent optional argument).
template <class... T>
void on_one_gpu(const Tensor& first, const T&... others) {
  require(first.is_cuda(), "inputs must be on CUDA");
  require((... && (!others.defined() || others.device() == first.device())), "inputs must be on one device");
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(bytes, 1)}, like.options().dtype(at::kByte));
}

int32_t dim32(const Tensor& t, int64_t d) { return (int32_t)t.size(d); }

// attn_fwd(q, k, v, block_size) -> (q, k, v, O, L): the tensors as the kernel read them.
PyObject* attn_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 4);
    Tensor q = a.tensor(), k = a.tensor(), v = a.tensor();
    const int32_t bs = a.int32();
    Tensor o, lse;
    on_one_gpu(q, k, v);
    {
      NoGil nogil;
      const c10::DeviceGuard device(q.device());
      q = ready(q);
      k = ready(k);
      v = ready(v);
      o = at::empty(q.sizes(), q.options());
      lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
      const auto st = strides(q, k, v, o);
      check(g_lib.attn_fwd(ptr(q), ptr(k), ptr(v), ptr(o), static_cast<float*>(ptr(lse)), dim32(q, 0), dim32(q, 1),
                           dim32(q, 2) / 2, dim32(q, 3), bs, st.data(), kScale, stream_of(q)));
    }
    return pack(q, k, v, o, lse);
  });
}

// attn_bwd(q, k, v, O, L, dO, block_size) -> (dQ, dK, dV)
PyObject* attn_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 7);
    Tensor q = a.tensor(), k = a.tensor(), v = a.tensor(), o = a.tensor(), lse = a.tensor(), dout = a.tensor();
    const int32_t bs = a.int32();
    Tensor dq, dk, dv;
    on_one_gpu(q, k, v, o, lse, dout);
    {
      NoGil nogil;
      const c10::DeviceGuard device(q.device());
      q = ready(q);
      k = ready(k);
      v = ready(v);
      o = ready(o);
      lse = lse.contiguous();
      dout = ready(dout.to(q.scalar_type()));
      dq = at::empty(q.sizes(), q.options());
      dk = at::empty(q.sizes(), q.options());
      dv = at::empty(q.sizes(), q.options());
      const int32_t B = dim32(q, 0), H = dim32(q, 1), half = dim32(q, 2) / 2, D = dim32(q, 3);
      const size_t bytes = g_lib.attn_bwd_workspace_bytes(B, H, half, D);
      const Tensor ws = workspace(bytes, q);
      const auto st = strides(q, k, v, o, dout, dq, dk, dv);
      check(g_lib.attn_bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr(dout), static_cast<const float*>(ptr(lse)), ptr(dq),
                           ptr(dk), ptr(dv), ptr(ws), bytes, B, H, half, D, bs, st.data(), kScale, stream_of(q)));
    }
    return pack(dq, dk, dv);
  });
}

// decode(q, k, v, block_size, n_splits[, token_major]) -> O; n_splits 0:
// bd3_decode's own count; token_major: O is a (b, h, s, d) view of (b, s, h, d)
// memory, so that a caller's transpose + reshape to (b, s, h * d) copies nothing
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, n == 6 ? 6 : 5);
    Tensor q = a.tensor(), k = a.tensor(), v = a.tensor();
    const int32_t bs = a.int32(), splits = a.int32();
    const bool token_major = n == 6 && a.int32() != 0;
    Tensor o;
    on_one_gpu(q, k, v);
    {
      NoGil nogil;
      const c10::DeviceGuard device(q.device());
      q = ready(q);
      k = ready(k);
      v = ready(v);
      const int32_t B = dim32(q, 0), H = dim32(q, 1), L = dim32(q, 2), D = dim32(q, 3), kv = dim32(k, 2);
      o = token_major ? at::empty({B, L, H, D}, q.options()).transpose(1, 2) : at::empty(q.sizes(), q.options());
      const size_t bytes = g_lib.decode_workspace_bytes(B, H, L, kv, D, splits);
      const Tensor ws = bytes ? workspace(bytes, q) : Tensor();
      const auto st = strides(q, k, v, o);
      if (splits == 0)
        check(g_lib.decode(ptr(q), ptr(k), ptr(v), ptr(o), B, H, L, kv, D, bs, st.data(), kScale, ptr(ws), bytes,
                           stream_of(q)));
      else
        check(g_lib.decode_splitkv(ptr(q), ptr(k), ptr(v), ptr(o), B, H, L, kv, D, bs, splits, st.data(), kScale,
                                   ptr(ws), bytes, stream_of(q)));
    }
    return THPVariable_Wrap(o);
  });
}

// qkv_rope(qkv, heads, sin, cos, positions or None, pos0, k_buf, v_buf, len) -> (q, k_all, v_all):
// k and v go to slots len .. len + seq - 1 of the buffers (batch, heads, capacity,
// 64), k_all / v_all are their first len + seq tokens; without buffers
// (None) to new tensors.
PyObject* qkv_rope(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 9);
    Tensor qkv = a.tensor();
    const int64_t heads = a.integer();
    Tensor sin = a.tensor(), cos = a.tensor(), positions = a.maybe_tensor();
    const int32_t pos0 = a.int32();
    Tensor k = a.maybe_tensor(), v = a.maybe_tensor();
    const int64_t len = a.integer();
    Tensor q, k_all, v_all;
    on_one_gpu(qkv, sin, cos, k, v);
    {
      NoGil nogil;
      const c10::DeviceGuard device(qkv.device());
      qkv = ready(qkv);
      sin = sin.contiguous();
      cos = cos.contiguous();
      if (positions.defined()) positions = positions.to(qkv.device(), at::kLong).contiguous();
      const int64_t B = qkv.size(0), S = qkv.size(1);
      q = at::empty({B, heads, S, kHeadDim}, qkv.options());
      Tensor k_out, v_out;
      if (k.defined()) {
        k_out = k.narrow(2, len, S);
        v_out = v.narrow(2, len, S);
      } else {
        k_out = at::empty_like(q);
        v_out = at::empty_like(q);
      }
      const int64_t xs[2] = {qkv.stride(0), qkv.stride(1)};
      const auto st = strides(q, k_out, v_out);
      check(g_lib.qkv_rope(ptr(qkv), xs, (int32_t)B, (int32_t)S, (int32_t)heads, kHeadDim,
                           static_cast<const int64_t*>(ptr(positions)), pos0, static_cast<const float*>(ptr(sin)),
                           static_cast<const float*>(ptr(cos)), dim32(sin, 0), ptr(q), ptr(k_out), ptr(v_out),
                           st.data(), stream_of(qkv)));
      k_all = k.defined() ? k.narrow(2, 0, len + S) : k_out;
      v_all = v.defined() ? v.narrow(2, 0, len + S) : v_out;
    }
    return pack(q, k_all, v_all);
  });
}

// subs_sample(logits, block, mask_index, keep, u or None, seed, offset) -> the next block
PyObject* subs_sample(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 7);
    const Tensor logits = a.tensor(), block = a.tensor();
    const int32_t mask = a.int32();
    const double keep = a.real();
    Tensor u = a.maybe_tensor();
    const uint64_t seed = a.unsigned64(), offset = a.unsigned64();
    Tensor out;
    on_one_gpu(logits, u);
    {
      NoGil nogil;
      const c10::DeviceGuard device(logits.device());
      const int64_t rows = block.numel(), vocab = logits.size(-1);
      Tensor lg = logits.reshape({rows, vocab});
      if (lg.stride(-1) != 1) lg = lg.contiguous();
      const Tensor xt = block.reshape({rows}).to(logits.device(), at::kLong).contiguous();
      out = at::empty_like(xt);
      if (u.defined()) u = u.reshape({rows, vocab}).contiguous();
      const size_t bytes = g_lib.subs_sample_workspace_bytes((int32_t)rows, (int32_t)vocab);
      const Tensor ws = bytes ? workspace(bytes, lg) : Tensor();
      check(g_lib.subs_sample_ws(ptr(lg), lg.stride(0), lg.scalar_type() == at::kFloat, static_cast<int64_t*>(ptr(xt)),
                                 static_cast<int64_t*>(ptr(out)), (int32_t)rows, (int32_t)vocab, mask, keep,
                                 static_cast<const double*>(ptr(u)), seed, offset, ptr(ws), bytes, stream_of(lg)));
      out = out.view(block.sizes());
    }
    return THPVariable_Wrap(out);
  });
}

int32_t is_f32(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return 1;
  if (t.scalar_type() == at::kBFloat16) return 0;
  throw Refused{PyExc_KeyError, std::string("bf16 or fp32 tensors only, got ") + c10::toString(t.scalar_type())};
}

// A (batch, d) or (batch, 1, d) modulation vector as (batch, d).
Tensor vec(Tensor t) {
  if (t.dim() == 3) {
    require(t.size(1) == 1, "modulation vectors broadcast over the sequence");
    t = t.select(1, 0);
  }
  return ready(t);
}

bool is_bd(const Tensor& t, int64_t B, int64_t D) { return t.dim() == 2 && t.size(0) == B && t.size(1) == D; }

at::ScalarType float_type(bool f32) { return f32 ? at::kFloat : at::kBFloat16; }

// ln_modulate(x, weight, shift, scale, eps, out_fp32): out_fp32 -1 keeps the eager dtype
PyObject* ln_modulate(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 6);
    Tensor x = a.tensor(), w = a.tensor(), shift = a.tensor(), scale = a.tensor();
    const double eps = a.real();
    const int64_t want = a.integer();
    Tensor out;
    on_one_gpu(x, w, shift, scale);
    {
      NoGil nogil;
      const c10::DeviceGuard device(x.device());
      const int64_t B = x.size(0), S = x.size(1), D = x.size(2);
      x = ready(x);
      w = ready(w);
      shift = vec(shift);
      scale = vec(scale);
      require(shift.scalar_type() == scale.scalar_type() && is_bd(shift, B, D) && is_bd(scale, B, D),
              "shift and scale must be (batch, d_model) of one dtype");
      const int32_t xf = is_f32(x), mf = is_f32(shift);
      out = at::empty({B, S, D}, x.options().dtype(float_type(want < 0 ? xf || mf : want != 0)));
      const int64_t st[5] = {x.stride(0), x.stride(1), shift.stride(0), out.stride(0), out.stride(1)};
      check(g_lib.ln_modulate(ptr(x), xf, ptr(w), is_f32(w), ptr(shift), ptr(scale), mf, ptr(out), is_f32(out),
                              (int32_t)B, (int32_t)S, (int32_t)D, st, (float)eps, stream_of(x)));
    }
    return THPVariable_Wrap(out);
  });
}

// gate_residual(x, gate, y, out or None)
PyObject* gate_residual(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 4);
    Tensor x = a.tensor(), gate = a.tensor(), y = a.tensor(), out = a.maybe_tensor();
    on_one_gpu(x, gate, y, out);
    {
      NoGil nogil;
      const c10::DeviceGuard device(x.device());
      const int64_t B = x.size(0), S = x.size(1), D = x.size(2);
      x = ready(x);
      y = ready(y);
      gate = vec(gate);
      const int32_t xf = is_f32(x), gf = is_f32(gate), yf = is_f32(y);
      const at::ScalarType type = float_type(xf || gf || yf);
      if (!out.defined()) out = at::empty({B, S, D}, x.options().dtype(type));
      require(out.scalar_type() == type && out.sizes() == x.sizes(), "out must have the result's shape and dtype");
      const int64_t st[7] = {x.stride(0), x.stride(1),   gate.stride(0), y.stride(0),
                             y.stride(1), out.stride(0), out.stride(1)};
      check(g_lib.gate_residual(ptr(x), xf, ptr(gate), gf, ptr(y), yf, ptr(out), (int32_t)B, (int32_t)S, (int32_t)D,
                                st, stream_of(x)));
    }
    return THPVariable_Wrap(out);
  });
}

// gate_residual_ln_modulate(x, gate, y, weight, shift, scale, eps, out_fp32, x_out or None) -> (x_out, out)
PyObject* gate_residual_ln_modulate(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&] {
    Args a(args, n, 9);
    Tensor x = a.tensor(), gate = a.tensor(), y = a.tensor(), w = a.tensor(), shift = a.tensor(), scale = a.tensor();
    const double eps = a.real();
    const int64_t want = a.integer();
    Tensor x_out = a.maybe_tensor(), out;
    on_one_gpu(x, gate, y, w, shift, scale, x_out);
    {
      NoGil nogil;
      const c10::DeviceGuard device(x.device());
      const int64_t B = x.size(0), S = x.size(1), D = x.size(2);
      x = ready(x);
      y = ready(y);
      w = ready(w);
      gate = vec(gate);
      shift = vec(shift);
      scale = vec(scale);
      require(gate.scalar_type() == shift.scalar_type() && shift.scalar_type() == scale.scalar_type() &&
                  is_bd(gate, B, D) && is_bd(shift, B, D) && is_bd(scale, B, D),
              "gate, shift and scale must be (batch, d_model) of one dtype");
      if (gate.stride(0) != shift.stride(0) || shift.stride(0) != scale.stride(0)) {  // one batch stride for the three
        gate = gate.contiguous();
        shift = shift.contiguous();
        scale = scale.contiguous();
      }
      const int32_t xf = is_f32(x), mf = is_f32(gate), yf = is_f32(y);
      const bool rf = xf || mf || yf;
      if (!x_out.defined()) x_out = at::empty({B, S, D}, x.options().dtype(float_type(rf)));
      require(x_out.scalar_type() == float_type(rf) && x_out.sizes() == x.sizes(),
              "x_out must have the residual's shape and dtype");
      out = at::empty({B, S, D}, x.options().dtype(float_type(want < 0 ? rf || mf : want != 0)));
      const int64_t st[9] = {x.stride(0),     x.stride(1),     gate.stride(0), y.stride(0),  y.stride(1),
                             x_out.stride(0), x_out.stride(1), out.stride(0),  out.stride(1)};
      check(g_lib.gate_residual_ln_modulate(ptr(x), xf, ptr(gate), ptr(y), yf, ptr(x_out), ptr(w), is_f32(w),
                                            ptr(shift), ptr(scale), mf, ptr(out), is_f32(out), (int32_t)B, (int32_t)S,
                                            (int32_t)D, st, (float)eps, stream_of(x)));
    }
    return pack(x_out, out);
  });
}

// bind({"bd3_...": address}): the C ABI of the loaded library.
PyObject* bind(PyObject*, PyObject* dict) {
  return guarded([&]() -> PyObject* {
    if (!PyDict_Check(dict)) throw Refused{PyExc_TypeError, "bind takes a dict of addresses"};
    auto set = [&](const char* name, auto& fn) {
      PyObject* o = PyDict_GetItemString(dict, name);
      void* p = o ? PyLong_AsVoidPtr(o) : nullptr;
      if (p == nullptr) throw Refused{PyExc_KeyError, std::string("no address for ") + name};
      fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(p);
    };
    Library l = {};
    set("bd3_last_error", l.last_error);
    set("bd3_attn_fwd", l.attn_fwd);
    set("bd3_attn_bwd_workspace_bytes", l.attn_bwd_workspace_bytes);
    set("bd3_attn_bwd", l.attn_bwd);
    set("bd3_decode", l.decode);
    set("bd3_decode_splitkv", l.decode_splitkv);
    set("bd3_decode_workspace_bytes", l.decode_workspace_bytes);
    set("bd3_qkv_rope", l.qkv_rope);
    set("bd3_subs_sample_ws", l.subs_sample_ws);
    set("bd3_subs_sample_workspace_bytes", l.subs_sample_workspace_bytes);
    set("bd3_ln_modulate", l.ln_modulate);
    set("bd3_gate_residual", l.gate_residual);
    set("bd3_gate_residual_ln_modulate", l.gate_residual_ln_modulate);
    g_lib = l;
    Py_RETURN_NONE;
  });
}

#define BD3_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    BD3_FAST(attn_fwd),
    BD3_FAST(attn_bwd),
    BD3_FAST(decode),
    BD3_FAST(qkv_rope),
    BD3_FAST(subs_sample),
    BD3_FAST(ln_modulate),
    BD3_FAST(gate_residual),
    BD3_FAST(gate_residual_ln_modulate),
    {nullptr, nullptr, 0, nullptr},
};
#undef BD3_FAST

PyModuleDef module = {PyModuleDef_HEAD_INIT, "bd3_host", "Native preparation of the kernels' Python calls.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_bd3_host(void) { return PyModule_Create(&module); }
