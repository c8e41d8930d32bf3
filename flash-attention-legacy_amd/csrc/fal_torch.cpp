// Tensor binding of libfal_hip.so for Python (module _fal_torch, used by hip_ext.py).
//
// One call per entry point: argument checks, output and workspace allocation on the
// input's device, and the launch on the current stream.  Through ctypes the same steps took
// 14 us (forward) to 28 us (backward) of interpreter time per call, more than the kernels of
// a decode step or a small training step; here 6 and 10 us (one decoded token, 32/8 heads over
// 1000 cache rows, 23.5 -> 11.4 us per call, training step of 2x8x128 rows 142 -> 64 us).  The
// library itself is reached through function pointers that hip_ext.py resolves, so it can be
// another build of it.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/fal_api.h"

namespace {

using at::Tensor;
using Strides = std::array<int64_t, 3>;

struct Api {
  decltype(&fal_last_error) last_error;
  decltype(&fal_fwd_workspace_size) fwd_ws;
  decltype(&fal_fwd_varlen_workspace_size) fwd_varlen_ws;
  decltype(&fal_bwd_workspace_best) bwd_ws;
  decltype(&fal_bwd_varlen_workspace_size) bwd_varlen_ws;
  decltype(&fal_decode_workspace_size) decode_ws;
  // fp16, bf16
  decltype(&fal_fwd) fwd[2];
  decltype(&fal_fwd_varlen) fwd_varlen[2];
  decltype(&fal_bwd) bwd[2];
  decltype(&fal_bwd_varlen) bwd_varlen[2];
  decltype(&fal_decode) decode[2];
} api;

[[noreturn]] void fail(const std::string& msg) { throw std::runtime_error(msg); }

void require(bool ok, const char* msg) {
  if (!ok) fail(msg);
}

void check_status(int rc) {
  if (rc == 0) return;
  const char* msg = api.last_error();
  fail(msg && *msg ? std::string(msg) : "flash_attn_legacy error " + std::to_string(rc));
}

bool half_type(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

// t is a CUDA tensor of `like` (or, without it, of float16 or bfloat16)
void check_half_cuda(const char* name, const Tensor& t, const Tensor* like = nullptr) {
  if (!t.is_cuda()) fail(std::string(name) + " must be on CUDA");
  if (!like) {
    if (!half_type(t.scalar_type())) fail(std::string(name) + " must be float16 or bfloat16");
  } else if (t.scalar_type() != like->scalar_type()) {
    fail(std::string(name) + " must be " + (like->scalar_type() == at::kHalf ? "float16" : "bfloat16") + " like Q");
  }
}

std::string shape_str(at::IntArrayRef s) {
  std::string r = "[";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + "]";
}

// L is the forward's fp32 log-sum-exp of `shape` on Q's device (the kernels index it by the
// problem's sizes, so a smaller tensor would be read out of bounds)
void check_lse(const Tensor& l, at::IntArrayRef shape, const Tensor& q) {
  if (l.scalar_type() == at::kFloat && l.sizes() == shape && l.device() == q.device()) return;
  const std::string type = torch::getTHPDtype(l.scalar_type())->name;   // (torch's own: "float16")
  fail("L must be float32 " + shape_str(shape) + " on " + q.device().str() + ", got torch." + type + " " +
       shape_str(l.sizes()) + " on " + l.device().str());
}

// Keep strided views the kernels can address directly (unit last stride, other strides
// multiples of 8 elements, 16-byte aligned base, and along `seq`, if given, rows no closer than
// a row is long: a gradient broadcast over the sequence has stride 0 there, which only the
// forward's Q and the backward's O may); copy anything else.
Tensor usable(const Tensor& t, int64_t seq = -1) {
  const auto s = t.strides();
  bool ok = s.back() == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
            (seq < 0 || t.size(seq) <= 1 || s[seq] >= t.size(-1));
  for (size_t i = 0; ok && i + 1 < s.size(); ++i) ok = s[i] % 8 == 0;
  return ok ? t : t.contiguous();
}

// (batch, head, sequence) strides; of packed [total, H, d] tensors (unused, head, token)
Strides batched(const Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }
Strides packed(const Tensor& t) { return {0, t.stride(1), t.stride(0)}; }

Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(bytes, 1)}, like.options().dtype(at::kByte));
}

Tensor cu_on(const Tensor& cu, const Tensor& like) {
  return cu.device() == like.device() && cu.is_contiguous() ? cu : cu.to(like.device()).contiguous();
}

int bf16(const Tensor& t) { return t.scalar_type() == at::kBFloat16; }
void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
const int32_t* ints(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }
float* floats(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

std::vector<Tensor> forward(Tensor q, Tensor k, Tensor v, double scale, bool causal) {
  check_half_cuda("Q", q);
  require(q.dim() == 4, "Q must be [B, H_q, N, d]");
  require(k.dim() == 4 && v.dim() == 4, "K,V must be 4D");
  check_half_cuda("K", k, &q);
  check_half_cuda("V", v, &q);
  const int64_t b = q.size(0), hq = q.size(1), n = q.size(2), d = q.size(3), hkv = k.size(1), nk = k.size(2);
  require(k.size(0) == b && k.size(3) == d, "K shape mismatch");
  require(v.sizes() == at::IntArrayRef({b, hkv, nk, d}), "V shape mismatch");
  q = usable(q), k = usable(k, 2), v = usable(v, 2);
  const c10::DeviceGuard guard(q.device());
  Tensor o = at::empty({b, hq, n, d}, q.options()), l = at::empty({b, hq, n}, q.options().dtype(at::kFloat));
  // non-zero only for grids smaller than the GPU (split-KV partials)
  const size_t nws = api.fwd_ws(b, hq, n, nk, d, causal);
  Tensor ws;
  if (nws) ws = workspace(nws, q);
  const Strides qs = batched(q), ks = batched(k), vs = batched(v), os = batched(o);
  check_status(api.fwd[bf16(q)](q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), floats(l), b, hq, hkv, n, nk, d,
                                qs.data(), ks.data(), vs.data(), os.data(), (float)scale, causal,
                                nws ? ws.data_ptr() : nullptr, nws, stream(q)));
  return {o, l};
}

std::vector<Tensor> forward_varlen(Tensor q, Tensor k, Tensor v, Tensor cu_q, Tensor cu_k, int64_t max_q, int64_t max_k,
                                   double scale, bool causal) {
  check_half_cuda("Q", q);
  require(q.dim() == 3, "Q must be [total_q, H_q, d]");
  require(k.dim() == 3 && v.dim() == 3, "K,V must be 3D");
  check_half_cuda("K", k, &q);
  check_half_cuda("V", v, &q);
  require(cu_q.scalar_type() == at::kInt, "cu_seqlens_q must be int32");
  require(cu_k.scalar_type() == at::kInt, "cu_seqlens_k must be int32");
  const int64_t tq = q.size(0), hq = q.size(1), d = q.size(2), tk = k.size(0), hkv = k.size(1);
  const int64_t seqs = cu_q.size(0) - 1;
  require(k.size(2) == d && v.size(2) == d, "K,V head_dim mismatch");
  require(v.size(1) == hkv, "V num_heads mismatch");
  require(cu_k.size(0) == seqs + 1, "cu_seqlens_k length mismatch");
  q = usable(q), k = usable(k, 0), v = usable(v, 0);
  const c10::DeviceGuard guard(q.device());
  cu_q = cu_on(cu_q, q), cu_k = cu_on(cu_k, q);
  Tensor o = at::empty({tq, hq, d}, q.options()), l = at::empty({tq, hq}, q.options().dtype(at::kFloat));
  // zero for up to 64 sequences (the kernel derives its work items from cu_seqlens)
  const size_t nws = api.fwd_varlen_ws(seqs, tq, max_q, d);
  Tensor ws;
  if (nws) ws = workspace(nws, q);
  const Strides qs = packed(q), ks = packed(k), vs = packed(v), os = packed(o);
  check_status(api.fwd_varlen[bf16(q)](q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), floats(l), ints(cu_q),
                                       ints(cu_k), seqs, tq, tk, hq, hkv, d, max_q, max_k, qs.data(), ks.data(),
                                       vs.data(), os.data(), (float)scale, causal, nws ? ws.data_ptr() : nullptr, nws,
                                       stream(q)));
  return {o, l};
}

// The checks that both backward forms share, in order, up to the shapes of Q and K.
void check_grad_types(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o) {
  check_half_cuda("dO", dout, &q);
  check_half_cuda("K", k, &q);
  check_half_cuda("V", v, &q);
  check_half_cuda("O", o, &q);
}

std::vector<Tensor> backward(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor l, double scale, bool causal) {
  require(q.is_cuda() && half_type(q.scalar_type()), "Q must be CUDA float16 or bfloat16");
  require(q.dim() == 4 && k.dim() == 4, "Q, K must be 4D");
  require(dout.sizes() == q.sizes(), "dO shape must match Q");
  const int64_t b = q.size(0), hq = q.size(1), n = q.size(2), d = q.size(3), hkv = k.size(1), nk = k.size(2);
  require(hkv != 0 && hq % hkv == 0, "H_q must be divisible by H_kv for GQA");
  check_grad_types(dout, q, k, v, o);
  require(k.size(0) == b && k.size(3) == d, "K shape mismatch");
  require(v.sizes() == k.sizes(), "V shape must match K");
  require(o.sizes() == q.sizes(), "O shape must match Q");
  check_lse(l, {b, hq, n}, q);
  dout = usable(dout, 2), q = usable(q, 2), k = usable(k, 2), v = usable(v, 2), o = usable(o), l = l.contiguous();
  const c10::DeviceGuard guard(q.device());
  Tensor dq = at::empty({b, hq, n, d}, q.options());
  Tensor dk = at::empty({b, hkv, nk, d}, q.options()), dv = at::empty({b, hkv, nk, d}, q.options());
  const Tensor ws = workspace(api.bwd_ws(b, hq, hkv, n, nk, d, causal), q);
  const Strides dos = batched(dout), qs = batched(q), ks = batched(k), vs = batched(v), os = batched(o),
                dqs = batched(dq), dks = batched(dk), dvs = batched(dv);
  check_status(api.bwd[bf16(q)](dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), floats(l),
                                dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), b, hq, hkv, n, nk, d, dos.data(), qs.data(),
                                ks.data(), vs.data(), os.data(), dqs.data(), dks.data(), dvs.data(), (float)scale, causal,
                                ws.data_ptr(), (size_t)ws.numel(), stream(q)));
  return {dq, dk, dv};
}

std::vector<Tensor> backward_varlen(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor l, Tensor cu_q, Tensor cu_k,
                                    int64_t max_q, int64_t max_k, double scale, bool causal) {
  require(q.is_cuda() && half_type(q.scalar_type()), "Q must be CUDA float16 or bfloat16");
  check_grad_types(dout, q, k, v, o);
  require(q.dim() == 3 && k.dim() == 3, "Q, K must be 3D");
  require(dout.sizes() == q.sizes(), "dO shape must match Q");
  const int64_t tq = q.size(0), hq = q.size(1), d = q.size(2), tk = k.size(0), hkv = k.size(1);
  require(hkv != 0 && hq % hkv == 0, "H_q must be divisible by H_kv for GQA");
  require(k.size(2) == d, "K,V head_dim mismatch");
  require(v.sizes() == k.sizes(), "V shape must match K");
  require(o.sizes() == q.sizes(), "O shape must match Q");
  check_lse(l, {tq, hq}, q);
  require(cu_q.dim() == 1 && cu_q.size(0) >= 1, "cu_seqlens_q must be a 1-D tensor of num_seqs + 1 offsets");
  const int64_t seqs = cu_q.size(0) - 1;
  require(cu_k.dim() == 1 && cu_k.size(0) == seqs + 1, "cu_seqlens_k length mismatch");
  require(cu_q.scalar_type() == at::kInt, "cu_seqlens_q must be int32");
  require(cu_k.scalar_type() == at::kInt, "cu_seqlens_k must be int32");
  dout = usable(dout, 0), q = usable(q, 0), k = usable(k, 0), v = usable(v, 0), o = usable(o), l = l.contiguous();
  const c10::DeviceGuard guard(q.device());
  cu_q = cu_on(cu_q, q), cu_k = cu_on(cu_k, q);
  // rows outside every segment come back zero (written by the library's schedule kernels)
  Tensor dq = at::empty({tq, hq, d}, q.options());
  Tensor dk = at::empty({tk, hkv, d}, q.options()), dv = at::empty({tk, hkv, d}, q.options());
  const Tensor ws = workspace(api.bwd_varlen_ws(seqs, tq, tk, hq, d), q);
  const Strides dos = packed(dout), qs = packed(q), ks = packed(k), vs = packed(v), os = packed(o), dqs = packed(dq),
                dks = packed(dk), dvs = packed(dv);
  check_status(api.bwd_varlen[bf16(q)](
      dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), floats(l), dq.data_ptr(), dk.data_ptr(),
      dv.data_ptr(), ints(cu_q), ints(cu_k), seqs, tq, tk, hq, hkv, d, max_q, max_k, dos.data(), qs.data(), ks.data(),
      vs.data(), os.data(), dqs.data(), dks.data(), dvs.data(), (float)scale, causal, ws.data_ptr(), (size_t)ws.numel(),
      stream(q)));
  return {dq, dk, dv};
}

// head_axis: 1 for caches [B, Hkv, S, d], 2 for [B, S, Hkv, d].  bias may be undefined.
std::vector<Tensor> decode(Tensor q, Tensor k, Tensor v, Tensor lens, double scale, Tensor bias, int64_t head_axis,
                           bool want_lse) {
  check_half_cuda("q", q);
  check_half_cuda("k_cache", k, &q);
  check_half_cuda("v_cache", v, &q);
  require(q.dim() == 3 && k.dim() == 4 && v.dim() == 4, "decode expects q [B,Hq,d] and 4-D caches");
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(head_axis), s = k.size(3 - head_axis);
  require(k.sizes() == v.sizes() && k.size(0) == b && k.size(3) == d, "k_cache / v_cache shape mismatch");
  if (lens.numel() != b)
    fail("cache_seqlens must hold " + std::to_string(b) + " lengths, got " + std::to_string(lens.numel()));
  if (bias.defined() && (bias.dim() != 2 || bias.size(0) != b || bias.size(1) < s)) {
    std::string sh = shape_str(bias.sizes());
    sh = "(" + sh.substr(1, sh.size() - 2) + (bias.dim() == 1 ? ",)" : ")");
    fail("mask_bias must be [B=" + std::to_string(b) + ", >= S=" + std::to_string(s) + "], got " + sh);
  }
  q = usable(q), k = usable(k, 3 - head_axis), v = usable(v, 3 - head_axis);
  const c10::DeviceGuard guard(q.device());
  if (lens.scalar_type() != at::kInt || lens.device() != q.device() || lens.dim() != 1 || !lens.is_contiguous())
    lens = lens.reshape({-1}).to(q.device(), at::kInt).contiguous();
  if (bias.defined()) {
    bias = bias.to(q.device(), at::kFloat);
    if (bias.stride(-1) != 1) bias = bias.contiguous();
  }
  Tensor o = at::empty({b, hq, d}, q.options()), l;
  if (want_lse) l = at::empty({b, hq}, q.options().dtype(at::kFloat));
  const Tensor ws = workspace(api.decode_ws(b, hq, hkv, s, d), q);
  const Strides qs = {q.stride(0), q.stride(1), 0}, os = {o.stride(0), o.stride(1), 0};
  const Strides ks = {k.stride(0), k.stride(head_axis), k.stride(3 - head_axis)};
  const Strides vs = {v.stride(0), v.stride(head_axis), v.stride(3 - head_axis)};
  check_status(api.decode[bf16(q)](q.data_ptr(), k.data_ptr(), v.data_ptr(), ints(lens),
                                   bias.defined() ? floats(bias) : nullptr, bias.defined() ? bias.stride(0) : 0,
                                   o.data_ptr(), want_lse ? floats(l) : nullptr, b, hq, hkv, d, s, qs.data(), ks.data(),
                                   vs.data(), os.data(), (float)scale, ws.data_ptr(), (size_t)ws.numel(), stream(q)));
  if (want_lse) return {o, l};
  return {o};
}

// ---------------------------------------------------------------------------
// Python side: positional arguments only (hip_ext.py has the signatures).  The GIL is
// released while the call runs, as ctypes does.
// ---------------------------------------------------------------------------
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

struct Args {
  PyObject* const* a;
  Py_ssize_t n;
  Tensor tensor(int i) const {
    if (i >= n || !THPVariable_Check(a[i])) throw torch::TypeError("argument " + std::to_string(i + 1) + " must be a tensor");
    return THPVariable_Unpack(a[i]);
  }
  Tensor optional(int i) const { return i < n && a[i] == Py_None ? Tensor() : tensor(i); }
  double number(int i) const {
    const double x = PyFloat_AsDouble(a[i]);
    if (x == -1.0 && PyErr_Occurred()) throw python_error();
    return x;
  }
  int64_t integer(int i) const {
    const long long x = PyLong_AsLongLong(a[i]);
    if (x == -1 && PyErr_Occurred()) throw python_error();
    return x;
  }
  void count(Py_ssize_t want) const {
    if (n != want) throw torch::TypeError("expected " + std::to_string(want) + " arguments, got " + std::to_string(n));
  }
};

PyObject* to_list(const std::vector<Tensor>& ts) {
  PyObject* list = PyList_New((Py_ssize_t)ts.size());
  if (!list) throw python_error();
  for (size_t i = 0; i < ts.size(); ++i) PyList_SET_ITEM(list, (Py_ssize_t)i, THPVariable_Wrap(ts[i]));
  return list;
}

PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args x{a, n};
  x.count(5);
  Tensor q = x.tensor(0), k = x.tensor(1), v = x.tensor(2);
  const double scale = x.number(3);
  const bool causal = x.integer(4) != 0;
  std::vector<Tensor> r;
  {
    NoGil nogil;
    r = forward(std::move(q), std::move(k), std::move(v), scale, causal);
  }
  return to_list(r);
  END_HANDLE_TH_ERRORS
}

PyObject* py_forward_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args x{a, n};
  x.count(9);
  Tensor q = x.tensor(0), k = x.tensor(1), v = x.tensor(2), cu_q = x.tensor(3), cu_k = x.tensor(4);
  const int64_t max_q = x.integer(5), max_k = x.integer(6);
  const double scale = x.number(7);
  const bool causal = x.integer(8) != 0;
  std::vector<Tensor> r;
  {
    NoGil nogil;
    r = forward_varlen(std::move(q), std::move(k), std::move(v), std::move(cu_q), std::move(cu_k), max_q, max_k, scale,
                       causal);
  }
  return to_list(r);
  END_HANDLE_TH_ERRORS
}

PyObject* py_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args x{a, n};
  x.count(8);
  Tensor dout = x.tensor(0), q = x.tensor(1), k = x.tensor(2), v = x.tensor(3), o = x.tensor(4), l = x.tensor(5);
  const double scale = x.number(6);
  const bool causal = x.integer(7) != 0;
  std::vector<Tensor> r;
  {
    NoGil nogil;
    r = backward(std::move(dout), std::move(q), std::move(k), std::move(v), std::move(o), std::move(l), scale, causal);
  }
  return to_list(r);
  END_HANDLE_TH_ERRORS
}

PyObject* py_backward_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args x{a, n};
  x.count(12);
  Tensor dout = x.tensor(0), q = x.tensor(1), k = x.tensor(2), v = x.tensor(3), o = x.tensor(4), l = x.tensor(5),
         cu_q = x.tensor(6), cu_k = x.tensor(7);
  const int64_t max_q = x.integer(8), max_k = x.integer(9);
  const double scale = x.number(10);
  const bool causal = x.integer(11) != 0;
  std::vector<Tensor> r;
  {
    NoGil nogil;
    r = backward_varlen(std::move(dout), std::move(q), std::move(k), std::move(v), std::move(o), std::move(l),
                        std::move(cu_q), std::move(cu_k), max_q, max_k, scale, causal);
  }
  return to_list(r);
  END_HANDLE_TH_ERRORS
}

PyObject* py_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Args x{a, n};
  x.count(8);
  Tensor q = x.tensor(0), k = x.tensor(1), v = x.tensor(2), lens = x.tensor(3);
  const double scale = x.number(4);
  Tensor bias = x.optional(5);
  const int64_t head_axis = x.integer(6);
  require(head_axis == 1 || head_axis == 2, "head axis must be 1 or 2");
  const bool want_lse = x.integer(7) != 0;
  std::vector<Tensor> r;
  {
    NoGil nogil;
    r = decode(std::move(q), std::move(k), std::move(v), std::move(lens), scale, std::move(bias), head_axis, want_lse);
  }
  return to_list(r);
  END_HANDLE_TH_ERRORS
}

// bind({name: address}): the library's entry points
PyObject* py_bind(PyObject*, PyObject* table) {
  HANDLE_TH_ERRORS
  auto set = [&](auto& fn, const char* name) {
    PyObject* v = PyDict_Check(table) ? PyDict_GetItemString(table, name) : nullptr;
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (PyErr_Occurred()) throw python_error();
    if (!p) throw torch::TypeError(std::string("bind: no address for ") + name);
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(p);
  };
  set(api.last_error, "fal_last_error");
  set(api.fwd_ws, "fal_fwd_workspace_size");
  set(api.fwd_varlen_ws, "fal_fwd_varlen_workspace_size");
  set(api.bwd_ws, "fal_bwd_workspace_best");
  set(api.bwd_varlen_ws, "fal_bwd_varlen_workspace_size");
  set(api.decode_ws, "fal_decode_workspace_size");
  set(api.fwd[0], "fal_fwd"), set(api.fwd[1], "fal_fwd_bf16");
  set(api.fwd_varlen[0], "fal_fwd_varlen"), set(api.fwd_varlen[1], "fal_fwd_varlen_bf16");
  set(api.bwd[0], "fal_bwd"), set(api.bwd[1], "fal_bwd_bf16");
  set(api.bwd_varlen[0], "fal_bwd_varlen"), set(api.bwd_varlen[1], "fal_bwd_varlen_bf16");
  set(api.decode[0], "fal_decode"), set(api.decode[1], "fal_decode_bf16");
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)py_bind, METH_O, nullptr},
    {"forward", (PyCFunction)(void*)py_forward, METH_FASTCALL, nullptr},
    {"forward_varlen", (PyCFunction)(void*)py_forward_varlen, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void*)py_backward, METH_FASTCALL, nullptr},
    {"backward_varlen", (PyCFunction)(void*)py_backward_varlen, METH_FASTCALL, nullptr},
    {"decode", (PyCFunction)(void*)py_decode, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fal_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__fal_torch() { return PyModule_Create(&module); }
