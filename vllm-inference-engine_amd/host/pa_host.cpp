// The decode attention calls from torch tensors to the C ABI in native code.
//
// A decode layer's launch takes 5-7 us on the GPU for small batches; checking
// nine tensors, reading their strides and building a forty-argument ctypes call
// in Python took about 12 us of host time per call, so a loop over layers ran
// at the host's pace. With this path it runs at the GPU's, measured on MI355X as
// back-to-back calls: one sequence of 300 tokens 12.2 -> 5.6 us per call (head_dim
// 64, 14 / 2 heads, rotary form), 8 of up to 512 12.6 -> 6.3 (write form), 128 of
// up to 1088 12.3 -> 11.4.
//
// Each function launches the call it is given, or returns None without having
// done anything when something about it is not plain: another device than the
// current one, a type, shape, alignment or stride the Python entry point
// refuses or copies, a tensor subclass, a functorch wrapper, an active
// __torch_function__ or dispatch mode, or a workspace too small. The Python entry
// point then runs its own checks, with its own errors, and its own call. Where the
// library reports a HIP error, the status is returned for the caller to raise: the
// call was made, or the error is an earlier one that only this report tells of.
//
// The module is not linked against the library: bind() is given the addresses
// of the library the process has loaded, whatever file that is.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "paged_attention.h"

namespace {

using at::Tensor;
using Obj = py::handle;

#define PA_HOST_CALLS(X)                    \
  X(pa_decode_batched_workspace_bytes)      \
  X(pa_decode_rope_batched_workspace_bytes) \
  X(pa_decode_batched_f16)                  \
  X(pa_decode_kv_write_batched_f16)         \
  X(pa_decode_rope_batched_f16)

// The loaded library's entry points (bind).
struct Api {
#define PA_HOST_MEMBER(name) decltype(&::name) name;
  PA_HOST_CALLS(PA_HOST_MEMBER)
#undef PA_HOST_MEMBER
} api;

void bind(const py::dict& addresses) {
#define PA_HOST_BIND(name) \
  api.name = reinterpret_cast<decltype(&::name)>(addresses[#name].cast<uintptr_t>());
  PA_HOST_CALLS(PA_HOST_BIND)
#undef PA_HOST_BIND
}

// The tensors of plain torch.Tensor (or Parameter) objects, with no mode active
// that intercepts torch calls.
template <size_t N>
bool unpack(const Obj (&objects)[N], const Tensor* (&tensors)[N]) {
  if (at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set())
    return false;
  for (size_t i = 0; i < N; ++i) {
    if (!THPVariable_CheckExact(objects[i].ptr())) return false;
    tensors[i] = &THPVariable_Unpack(objects[i].ptr());
  }
  return true;
}

// Plain strided CUDA tensors of one type on one device.
bool plain(const Tensor& t, c10::ScalarType type, c10::Device dev) {
  constexpr c10::DispatchKeySet wrappers({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper,
                                          c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return t.defined() && t.is_cuda() && t.device() == dev && t.scalar_type() == type &&
         t.layout() == c10::kStrided && !t.key_set().has_any(wrappers) && !t.is_nested();
}

bool current(c10::Device dev) {
  return c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA)->getDevice() == dev;
}

// Rows [rows, heads, dim] of a [rows, heads, dim] or [rows, heads, 1, dim]
// tensor: whether it is one, and its strides.
bool rows3(const Tensor& t, int64_t rows, int64_t heads, int64_t dim, int64_t (&st)[3]) {
  const int last = t.dim() - 1;
  if (last != 2 && !(last == 3 && t.size(2) == 1)) return false;
  if (t.size(0) != rows || t.size(1) != heads || t.size(last) != dim) return false;
  st[0] = t.stride(0);
  st[1] = t.stride(1);
  st[2] = t.stride(last);
  return true;
}

bool rows2(const Tensor& t, int64_t rows, int64_t dim, int64_t (&st)[2]) {
  const int last = t.dim() - 1;
  if (last != 1 && !(last == 2 && t.size(1) == 1)) return false;
  if (t.size(0) != rows || t.size(last) != dim) return false;
  st[0] = t.stride(0);
  st[1] = t.stride(last);
  return true;
}

// Unit head_dim stride, 8-element aligned strides and a 16-byte aligned base.
bool rows16(const Tensor& t, const int64_t (&st)[3]) {
  return st[2] == 1 && st[0] % 8 == 0 && st[1] % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0;
}

// What the three calls share: pools, tables, lengths and the sizes.
struct Call {
  int64_t n, hq, hkv, d, bs, blocks, width;
  int64_t ks[4], vs[4], bts[2];

  bool fill(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& bt,
            const Tensor& lens) {
    const c10::Device dev = q.device();
    if (!plain(q, at::kHalf, dev) || !plain(k, at::kHalf, dev) || !plain(v, at::kHalf, dev) ||
        !plain(bt, at::kInt, dev) || !plain(lens, at::kInt, dev) || !current(dev))
      return false;
    if (k.dim() != 4 || k.sizes() != v.sizes() || bt.dim() != 2 || lens.dim() != 1 || q.dim() < 3)
      return false;
    n = q.size(0);
    hq = q.size(1);
    blocks = k.size(0);
    bs = k.size(1);
    hkv = k.size(2);
    d = k.size(3);
    width = bt.size(1);
    // Sizes the C ABI takes as int.
    for (int64_t x : {n, hq, hkv, d, bs, blocks, width})
      if (x <= 0 || x > 0x7fffffff) return false;
    // The C ABI reads lengths at unit stride, as the Python call passes them.
    if (hq % hkv || bt.size(0) != n || lens.size(0) != n) return false;
    for (int i = 0; i < 4; ++i) {
      ks[i] = k.stride(i);
      vs[i] = v.stride(i);
    }
    bts[0] = bt.stride(0);
    bts[1] = bt.stride(1);
    return true;
  }
};

// The caller's zero-initialised workspace of this (device, stream), if large enough.
bool workspace(const Tensor& ws, c10::Device dev, size_t need, void*& ptr) {
  ptr = nullptr;
  if (need == 0) return true;
  if (!ws.defined() || ws.device() != dev || ws.nbytes() < need) return false;
  ptr = ws.data_ptr();
  return true;
}

py::object done(int status, const Tensor& out) {
  if (status == PA_OK) return py::cast(out);
  return status == PA_ERR_HIP ? py::object(py::int_(status)) : py::object(py::none());
}

py::object decode(Obj q_, Obj k_, Obj v_, Obj bt_, Obj lens_, double scale, Obj ws_,
                  int64_t stream) {
  const Tensor* t[6];
  if (!unpack({q_, k_, v_, bt_, lens_, ws_}, t)) return py::none();
  const Tensor &q = *t[0], &k = *t[1], &v = *t[2], &bt = *t[3], &lens = *t[4], &ws = *t[5];
  Call c;
  int64_t qs[3];
  if (!c.fill(q, k, v, bt, lens) || q.dim() != 3 || !rows3(q, c.n, c.hq, c.d, qs) || !rows16(q, qs))
    return py::none();
  const size_t need = api.pa_decode_batched_workspace_bytes(c.n, c.hq, c.hkv, c.d, c.bs, c.width);
  void* wp;
  if (!workspace(ws, q.device(), need, wp)) return py::none();
  const Tensor out = at::empty_like(q);
  const int64_t os[3] = {out.stride(0), out.stride(1), out.stride(2)};
  int status;
  {
    py::gil_scoped_release release;
    status = api.pa_decode_batched_f16(q.data_ptr(), qs, k.data_ptr(), c.ks, v.data_ptr(), c.vs,
                                   (const int32_t*)bt.data_ptr(), c.bts,
                                   (const int32_t*)lens.data_ptr(), out.data_ptr(), os, c.n, c.hq,
                                   c.hkv, c.d, c.bs, c.blocks, c.width, (float)scale, wp, need,
                                   (void*)stream);
  }
  return done(status, out);
}

py::object kv_write_decode(Obj q_, Obj key_, Obj value_, Obj k_, Obj v_, Obj bt_, Obj lens_,
                           double scale, Obj ws_, int64_t stream) {
  const Tensor* t[8];
  if (!unpack({q_, key_, value_, k_, v_, bt_, lens_, ws_}, t)) return py::none();
  const Tensor &q = *t[0], &key = *t[1], &value = *t[2], &k = *t[3], &v = *t[4], &bt = *t[5],
               &lens = *t[6], &ws = *t[7];
  Call c;
  int64_t qs[3], ys[3], zs[3];
  if (!c.fill(q, k, v, bt, lens) || !plain(key, at::kHalf, q.device()) ||
      !plain(value, at::kHalf, q.device()) || !rows3(q, c.n, c.hq, c.d, qs) || !rows16(q, qs) ||
      !rows3(key, c.n, c.hkv, c.d, ys) || !rows16(key, ys) || !rows3(value, c.n, c.hkv, c.d, zs) ||
      !rows16(value, zs))
    return py::none();
  const size_t need = api.pa_decode_batched_workspace_bytes(c.n, c.hq, c.hkv, c.d, c.bs, c.width);
  void* wp;
  if (!workspace(ws, q.device(), need, wp)) return py::none();
  const Tensor out = at::empty({c.n, c.hq, c.d}, q.options());
  const int64_t os[3] = {c.hq * c.d, c.d, 1};
  int status;
  {
    py::gil_scoped_release release;
    status = api.pa_decode_kv_write_batched_f16(
        q.data_ptr(), qs, key.data_ptr(), ys, value.data_ptr(), zs, k.data_ptr(), c.ks,
        v.data_ptr(), c.vs, (const int32_t*)bt.data_ptr(), c.bts, (const int32_t*)lens.data_ptr(),
        out.data_ptr(), os, c.n, c.hq, c.hkv, c.d, c.bs, c.blocks, c.width, (float)scale, wp, need,
        (void*)stream);
  }
  return done(status, out);
}

py::object rope_decode(Obj q_, Obj key_, Obj value_, Obj cos_, Obj sin_, Obj k_, Obj v_, Obj bt_,
                       Obj lens_, double scale, Obj ws_, int64_t stream) {
  const Tensor* t[10];
  if (!unpack({q_, key_, value_, cos_, sin_, k_, v_, bt_, lens_, ws_}, t)) return py::none();
  const Tensor &q = *t[0], &key = *t[1], &value = *t[2], &cos = *t[3], &sin = *t[4], &k = *t[5],
               &v = *t[6], &bt = *t[7], &lens = *t[8], &ws = *t[9];
  Call c;
  int64_t qs[3], ys[3], zs[3], cs[2], ss[2];
  if (!c.fill(q, k, v, bt, lens) || !plain(key, at::kHalf, q.device()) ||
      !plain(value, at::kHalf, q.device()) || !plain(cos, at::kHalf, q.device()) ||
      !plain(sin, at::kHalf, q.device()) || c.d % 2 || !rows3(q, c.n, c.hq, c.d, qs) ||
      !rows3(key, c.n, c.hkv, c.d, ys) || !rows3(value, c.n, c.hkv, c.d, zs) ||
      !rows2(cos, c.n, c.d, cs) || !rows2(sin, c.n, c.d, ss))
    return py::none();
  const size_t need =
      api.pa_decode_rope_batched_workspace_bytes(c.n, c.hq, c.hkv, c.d, c.bs, c.width);
  void* wp;
  if (!workspace(ws, q.device(), need, wp)) return py::none();
  const Tensor out = at::empty({c.n, c.hq, c.d}, q.options());
  const int64_t os[3] = {c.hq * c.d, c.d, 1};
  int status;
  {
    py::gil_scoped_release release;
    status = api.pa_decode_rope_batched_f16(
        q.data_ptr(), qs, key.data_ptr(), ys, value.data_ptr(), zs, cos.data_ptr(), cs,
        sin.data_ptr(), ss, k.data_ptr(), c.ks, v.data_ptr(), c.vs, (const int32_t*)bt.data_ptr(),
        c.bts, (const int32_t*)lens.data_ptr(), out.data_ptr(), os, c.n, c.hq, c.hkv, c.d, c.bs,
        c.blocks, c.width, (float)scale, wp, need, (void*)stream);
  }
  return done(status, out);
}

}  // namespace

PYBIND11_MODULE(_pa_host, m) {
  py::list calls;
#define PA_HOST_NAME(name) calls.append(#name);
  PA_HOST_CALLS(PA_HOST_NAME)
#undef PA_HOST_NAME
  m.attr("ABI_VERSION") = PA_ABI_VERSION;  // of the argument lists compiled in here
  m.attr("CALLS") = py::tuple(calls);
  m.def("bind", &bind);
  m.def("decode", &decode);
  m.def("kv_write_decode", &kv_write_decode);
  m.def("rope_decode", &rope_decode);
}
