// Native half of the pulsar_cuda op surface: output allocation, the current stream and the
// library call of each op, for the Python wrappers in pulsar_cuda/__init__.py, which have
// checked the operands (device, dtype, shape, contiguity) before they come here.
//
// A call through ctypes with its outputs from torch.empty costs 5 us of Python beside the
// 3.4 us of the launch itself (output tensors 2.6, torch.cuda.current_stream 2.0, argument
// conversion 0.5); from here it is 1.5.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/pulsar_hip.h"

namespace {

using at::Tensor;

// Positional arguments of one call.
struct Args {
  PyObject* const* a;
  Py_ssize_t n;
  const Tensor& t(int i) const {
    TORCH_CHECK_TYPE(i < n && THPVariable_Check(a[i]), "argument ", i, " must be a tensor");
    return THPVariable_Unpack(a[i]);
  }
  Tensor opt(int i) const { return a[i] == Py_None ? Tensor() : t(i); }
  int64_t i64(int i) const {
    const long long v = PyLong_AsLongLong(a[i]);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  float f32(int i) const {
    const double v = PyFloat_AsDouble(a[i]);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return (float)v;
  }
};

struct Unlocked {  // the interpreter lock given up for a scope
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// The library call, without the interpreter lock (as through ctypes): a launch can wait for
// room in the queue.
template <typename F, typename... A>
void run(F f, A... args) {
  int rc;
  {
    Unlocked scope;
    rc = f(args...);
  }
  if (rc != PULSAR_OK) {
    const char* m = pulsar_last_error();
    throw std::runtime_error(m && *m ? m : "pulsar_hip error " + std::to_string(rc));
  }
}

int code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? PULSAR_BF16 : PULSAR_F32; }

hipStream_t stream(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// A tensor with elements but without memory (a fake one, while a program is traced) is an error
// here: the kernels would read and write address 0. Out of line: a call takes 3 to 8 pointers.
[[gnu::noinline, gnu::cold]] void* no_memory(const Tensor& t) {
  TORCH_CHECK(t.numel() == 0, "the tensor has no memory to read or write");
  return nullptr;
}
void* q(const Tensor& t) {
  void* d = t.data_ptr();
  return d ? d : no_memory(t);
}
const void* p(const Tensor& t) { return t.defined() ? q(t) : nullptr; }
template <typename X>
const X* p(const Tensor& t) { return reinterpret_cast<const X*>(p(t)); }
template <typename X>
X* q(const Tensor& t) { return reinterpret_cast<X*>(q(t)); }

// An output of the layout of argument i. A subclass of torch.Tensor allocates it by its own
// empty_like, so that it is of the subclass's type.
Tensor like(const Args& a, int i) {
  const Tensor& t = a.t(i);
  if (THPVariable_CheckExact(a.a[i])) return at::empty_like(t);
  THPObjectPtr torch(PyImport_ImportModule("torch"));
  if (!torch) throw python_error();
  THPObjectPtr r(PyObject_CallMethod(torch.get(), "empty_like", "O", a.a[i]));
  if (!r) throw python_error();
  TORCH_CHECK_TYPE(THPVariable_Check(r.get()), "empty_like of a tensor subclass gave no tensor");
  return THPVariable_Unpack(r.get());
}
// The gradient of weight argument i. The library zeroes the used entries that it adds to; a
// longer weight's others are zero too.
Tensor like_weight(const Args& a, int i, int64_t used) {
  Tensor dw = like(a, i);
  if (dw.numel() != used) dw.zero_();
  return dw;
}
Tensor make(const Tensor& on, at::IntArrayRef shape, at::ScalarType dt) {
  return at::empty(shape, on.options().dtype(dt).requires_grad(false));
}
Tensor make(const Tensor& on, at::IntArrayRef shape) { return make(on, shape, on.scalar_type()); }

PyObject* out(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* pair(const Tensor& a, const Tensor& b, bool list) {
  THPObjectPtr x(out(a)), y(out(b));
  if (!x || !y) throw python_error();
  PyObject* r = list ? PyList_New(2) : PyTuple_New(2);
  if (!r) throw python_error();
  if (list) {
    PyList_SET_ITEM(r, 0, x.release());
    PyList_SET_ITEM(r, 1, y.release());
  } else {
    PyTuple_SET_ITEM(r, 0, x.release());
    PyTuple_SET_ITEM(r, 1, y.release());
  }
  return r;
}

// (x, weight, eps) -> (y, rsqrt)
PyObject* rmsnorm_forward(const Args& a) {
  const Tensor &x = a.t(0), &w = a.t(1);
  const int64_t dim = x.size(-1), rows = dim ? x.numel() / dim : 0;
  Tensor y = like(a, 0), rs = make(x, {rows}, at::kFloat);
  if (rows)
    run(pulsar_rmsnorm_forward, p(x), p<float>(w), q(y), q<float>(rs), rows, dim, a.f32(2), code(x),
                                 stream(x));
  return pair(y, rs, false);
}

// (x, weight, cos, sin, B, H, T, sB, sH, sT, eps) -> (y, rsqrt)
PyObject* qk_rmsnorm_rope_forward(const Args& a) {
  const Tensor &x = a.t(0), &w = a.t(1), &c = a.t(2), &s = a.t(3);
  Tensor y = make(x, x.sizes()), rs = make(x, {x.numel() / 64}, at::kFloat);
  run(pulsar_qk_rmsnorm_rope_forward, p(x), a.i64(7), a.i64(8), a.i64(9), a.i64(4), a.i64(5),
                                       a.i64(6), 64, p<float>(w), p<float>(c), p<float>(s), q(y),
                                       q<float>(rs), a.f32(10), code(x), stream(x));
  return pair(y, rs, false);
}

// (attn, gate) -> out
PyObject* fused_attn_gate_forward(const Args& a) {
  const Tensor &x = a.t(0), &g = a.t(1);
  const int64_t B = x.size(0), H = x.size(1), T = x.size(2), D = x.size(3);
  Tensor o = make(x, {B, T, H * D});
  run(pulsar_fused_attn_gate_forward, p(x), p<float>(g), q(o), B, H, T, D, code(x), stream(x));
  return out(o);
}

// (x, weight) -> y
PyObject* causal_conv1d_k4_forward(const Args& a) {
  const Tensor &x = a.t(0), &w = a.t(1);
  Tensor y = like(a, 0);
  run(pulsar_causal_conv1d_k4_forward, p(x), p<float>(w), q(y), x.size(0), x.size(1), x.size(2),
                                        code(x), stream(x));
  return out(y);
}

// (gu, d_ff) -> out
PyObject* fused_swiglu_forward(const Args& a) {
  const Tensor& gu = a.t(0);
  TORCH_CHECK(gu.dim() > 0, "gu must have at least one dimension");
  const int64_t d = a.i64(1), rows = d ? gu.numel() / (2 * d) : 0;
  std::vector<int64_t> shape = gu.sizes().vec();
  shape.back() = d;
  Tensor o = make(gu, shape);
  if (rows) run(pulsar_fused_swiglu_forward, p(gu), q(o), rows, d, code(gu), stream(gu));
  return out(o);
}

// (logits, bias, top_k, z_loss_weight) -> (idx, weights, z_loss, probs_mean)
PyObject* moe_router_topk_forward(const Args& a) {
  const Tensor &l = a.t(0), &b = a.t(1);
  const int64_t N = l.size(0), E = l.size(1), K = a.i64(2);
  Tensor idx = make(l, {N, K}, at::kLong), w = make(l, {N, K}, at::kBFloat16);
  Tensor z = make(l, {}, at::kFloat), pm = make(l, {E}, at::kFloat);
  // per-workgroup partial statistics (merged in a fixed order inside the library)
  Tensor ws = make(l, {std::max<int64_t>(1, pulsar_moe_router_workspace_bytes(N, E) / 4)}, at::kFloat);
  run(pulsar_moe_router_topk_forward_ws, p(l), code(l), p<float>(b), q<int64_t>(idx),
                                          q<uint16_t>(w), q<float>(z), q<float>(pm), N, E, K,
                                          a.f32(3), q<float>(ws), stream(l));
  THPObjectPtr r(PyTuple_New(4));
  if (!r) throw python_error();
  const Tensor* o[4] = {&idx, &w, &z, &pm};
  for (int i = 0; i < 4; ++i) {
    PyObject* t = out(*o[i]);
    if (!t) throw python_error();
    PyTuple_SET_ITEM(r.get(), i, t);
  }
  return r.release();
}

// (x, topk_idx, slots, E, C, counts) -> expert_inputs
PyObject* moe_dispatch_forward(const Args& a) {
  const Tensor &x = a.t(0), &ti = a.t(1), &ts = a.t(2);
  const int64_t E = a.i64(3), C = a.i64(4);
  const Tensor n = a.opt(5);
  Tensor o = make(x, {E, C, x.size(1)});
  run(pulsar_moe_dispatch_forward, p(x), p<int64_t>(ti), p<int32_t>(ts), p<int64_t>(n), q(o),
                                    x.size(0), x.size(1), ti.size(1), E, C, code(x), stream(x));
  return out(o);
}

// (expert_outputs, topk_idx, weights, slots, shared) -> out
PyObject* moe_combine_forward(const Args& a) {
  const Tensor &eo = a.t(0), &ti = a.t(1), &w = a.t(2), &ts = a.t(3);
  const Tensor sh = a.opt(4);
  const int64_t N = ti.size(0), D = eo.size(2);
  Tensor o = make(eo, {N, D});
  if (N)
    run(pulsar_moe_combine_forward, p(eo), p<int64_t>(ti), p<uint16_t>(w), p<int32_t>(ts), p(sh),
                                     q(o), N, D, ti.size(1), eo.size(0), eo.size(1), code(eo),
                                     stream(eo));
  return out(o);
}

// (flat_e, order, E, C) -> (slots, counts)
PyObject* moe_slots_from_order(const Args& a) {
  const Tensor &f = a.t(0), &o = a.t(1);
  const int64_t M = f.numel(), E = a.i64(2);
  Tensor s = make(f, {M}, at::kInt), n = make(f, {E}, at::kLong);
  run(pulsar_moe_slots_from_order, p<int64_t>(f), p<int64_t>(o), q<int32_t>(s), q<int64_t>(n), M, E,
                                    a.i64(3), stream(f));
  return pair(s, n, false);
}

// (dy, x, weight, rsqrt, dw's layout) -> [dx, dw]
PyObject* rmsnorm_backward(const Args& a) {
  const Tensor &dy = a.t(0), &x = a.t(1), &w = a.t(2), &rs = a.t(3);
  const int64_t dim = x.size(-1);
  Tensor dx = like(a, 1), dw = like_weight(a, 4, dim);
  run(pulsar_rmsnorm_backward, p(dy), p(x), p<float>(w), p<float>(rs), q(dx), q<float>(dw),
                                x.numel() / dim, dim, code(x), stream(x));
  return pair(dx, dw, true);
}

// (dy, x, weight, rsqrt, cos, sin, dx, B, H, T, sB, sH, sT, dB, dH, dT) -> [dx, dw]
PyObject* qk_rmsnorm_rope_backward(const Args& a) {
  const Tensor &dy = a.t(0), &x = a.t(1), &w = a.t(2), &rs = a.t(3), &c = a.t(4), &s = a.t(5);
  const Tensor& dx = a.t(6);
  Tensor dw = like_weight(a, 2, 64 * a.i64(8));
  run(pulsar_qk_rmsnorm_rope_backward, p(dy), p(x), a.i64(10), a.i64(11), a.i64(12), q(dx),
                                        a.i64(13), a.i64(14), a.i64(15), a.i64(7), a.i64(8), a.i64(9),
                                        64, p<float>(w), p<float>(rs), p<float>(c), p<float>(s),
                                        q<float>(dw), code(x), stream(x));
  return pair(dx, dw, true);
}

// (grad_out, attn, gate) -> [d_attn, d_gate]
PyObject* fused_attn_gate_backward(const Args& a) {
  const Tensor &go = a.t(0), &x = a.t(1), &g = a.t(2);
  const int64_t B = x.size(0), H = x.size(1), T = x.size(2);
  Tensor da = like(a, 1), dg = make(x, {B, T, H}, at::kFloat);
  if (da.numel())
    run(pulsar_fused_attn_gate_backward, p(go), p(x), p<float>(g), q(da), q<float>(dg), B, H, T, 64,
                                          code(x), stream(x));
  return pair(da, dg, true);
}

// (dout, gu, d_ff) -> dgu
PyObject* fused_swiglu_backward(const Args& a) {
  const Tensor &d = a.t(0), &gu = a.t(1);
  const int64_t f = a.i64(2), rows = f ? gu.numel() / (2 * f) : 0;
  Tensor o = like(a, 1);
  if (rows) run(pulsar_fused_swiglu_backward, p(d), p(gu), q(o), rows, f, code(gu), stream(gu));
  return out(o);
}

// (dout, x, weight) -> [dx, dw]
PyObject* causal_conv1d_k4_backward(const Args& a) {
  const Tensor &d = a.t(0), &x = a.t(1), &w = a.t(2);
  Tensor dx = like(a, 1), dw = like_weight(a, 2, 4 * x.size(2));
  run(pulsar_causal_conv1d_k4_backward, p(d), p(x), p<float>(w), q(dx), q<float>(dw), x.size(0),
                                         x.size(1), x.size(2), code(x), stream(x));
  return pair(dx, dw, true);
}

// (d_weights, logits, topk_idx, z_loss_weight, d_z_loss, d_probs_mean) -> d_logits
PyObject* moe_router_topk_backward(const Args& a) {
  const Tensor &dw = a.t(0), &l = a.t(1), &ti = a.t(2);
  const Tensor dz = a.opt(4), dp = a.opt(5);
  Tensor o = like(a, 1);
  if (l.size(0))
    run(pulsar_moe_router_topk_backward, p<uint16_t>(dw), p(l), code(l), p<int64_t>(ti), a.f32(3),
                                          p<float>(dz), p<float>(dp), q(o), l.size(0), l.size(1),
                                          ti.size(1), stream(l));
  return out(o);
}

// (d_expert_inputs, topk_idx, slots, N, D) -> dx
PyObject* moe_dispatch_backward(const Args& a) {
  const Tensor &d = a.t(0), &ti = a.t(1), &ts = a.t(2);
  const int64_t N = a.i64(3), D = a.i64(4);
  Tensor o = make(d, {N, D});
  if (N)
    run(pulsar_moe_dispatch_backward, p(d), p<int64_t>(ti), p<int32_t>(ts), q(o), N, D, ti.size(1),
                                       d.size(0), d.size(1), code(d), stream(d));
  return out(o);
}

// (d_out, expert_outputs, topk_idx, weights, slots) -> [d_expert_outputs, d_weights]
PyObject* moe_combine_backward(const Args& a) {
  const Tensor &d = a.t(0), &eo = a.t(1), &ti = a.t(2), &w = a.t(3), &ts = a.t(4);
  const int64_t N = ti.size(0), K = ti.size(1);
  Tensor de = like(a, 1), dw = make(eo, {N, K}, at::kBFloat16);
  run(pulsar_moe_combine_backward, p(d), p(eo), p<int64_t>(ti), p<uint16_t>(w), p<int32_t>(ts),
                                    q(de), q<uint16_t>(dw), N, eo.size(2), K, eo.size(0), eo.size(1),
                                    code(eo), stream(eo));
  return pair(de, dw, true);
}

template <PyObject* (*F)(const Args&), int N>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == N, "expected ", N, " arguments, got ", n);
  return F(Args{args, n});
  END_HANDLE_TH_ERRORS
}

#define OP(name, n) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call<name, n>)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    OP(rmsnorm_forward, 3),          OP(qk_rmsnorm_rope_forward, 11),
    OP(fused_attn_gate_forward, 2),  OP(causal_conv1d_k4_forward, 2),
    OP(fused_swiglu_forward, 2),     OP(moe_router_topk_forward, 4),
    OP(moe_dispatch_forward, 6),     OP(moe_combine_forward, 5),
    OP(moe_slots_from_order, 4),     OP(rmsnorm_backward, 5),
    OP(qk_rmsnorm_rope_backward, 16), OP(fused_attn_gate_backward, 3),
    OP(fused_swiglu_backward, 3),    OP(causal_conv1d_k4_backward, 3),
    OP(moe_router_topk_backward, 6), OP(moe_dispatch_backward, 5),
    OP(moe_combine_backward, 5),     {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__ops(void) { return PyModule_Create(&module); }
