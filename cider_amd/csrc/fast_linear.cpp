// Python extension `_cider_fast`: the common case of a linear call in native
// code.  One call checks the operands, allocates the result and the workspace
// from torch's allocator and enqueues the library call on the current stream.
//
// It replaces host work only.  Through ctypes an eager decode linear
// (M=1 N=10240 K=2560) took 12.3 us per call on the host for a 5.2-6.0 us
// kernel, per-group and int4 layers 19-21 us for 9.4-12.5 us of kernels: their
// Python checks, device and stream contexts, allocations and argument
// conversions were the bound.
//
// linear(op, x, w, scale, bias, group_size, any_dim) -> Tensor, or None for
// every call it does not take (another dtype, layout, shape, device, tensor
// subclass, a functorch or fake tensor, an empty operand, an M the library has
// no bf16 path for): the caller then takes the general Python path, which
// raises what there is to raise.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "cider_hip.h"
#include "cider_hip_ext.h"

namespace {

// A plain dense CUDA tensor with memory of its own (no subclass, wrapper,
// lazy negation or conjugation).
bool plain(PyObject* o) { return THPVariable_CheckExact(o); }
bool dense(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
         !t.is_neg() && !t.is_conj() && !t.key_set().has(c10::DispatchKey::Python) &&
         t.is_contiguous();
}

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "linear takes 7 arguments");
    return nullptr;
  }
  const long op = PyLong_AsLong(args[0]), gs = PyLong_AsLong(args[5]);
  const int any_dim = PyObject_IsTrue(args[6]);
  if (PyErr_Occurred()) return nullptr;
  const bool has_bias = args[4] != Py_None;
  if (!plain(args[1]) || !plain(args[2]) || !plain(args[3]) || (has_bias && !plain(args[4])))
    Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(args[1]);
  const at::Tensor& w = THPVariable_Unpack(args[2]);
  const at::Tensor& s = THPVariable_Unpack(args[3]);
  const at::Tensor bias_in = has_bias ? THPVariable_Unpack(args[4]) : at::Tensor();
  if (!dense(x) || !dense(w) || !dense(s) || (has_bias && !dense(bias_in))) Py_RETURN_NONE;

  const bool w4 = op == CIDER_OP_W4A8 || op == CIDER_OP_W4A8_PERGROUP;
  const bool grouped = op == CIDER_OP_PERGROUP || op == CIDER_OP_W4A8_PERGROUP;
  if (!(w4 || grouped || op == CIDER_OP_PERCHANNEL)) Py_RETURN_NONE;
  const auto xt = x.scalar_type();
  const bool bf = xt == at::kBFloat16;
  if ((!bf && xt != at::kHalf) || w.dim() != 2 || x.dim() < 1 || (!any_dim && x.dim() != 2) ||
      w.scalar_type() != (w4 ? at::kByte : at::kChar))
    Py_RETURN_NONE;
  const int64_t N = w.size(0), K = w.size(1) * (w4 ? 2 : 1);
  if (N == 0 || K == 0 || x.size(-1) != K || x.numel() == 0) Py_RETURN_NONE;
  const int64_t M = x.numel() / K;
  if (s.scalar_type() != (op == CIDER_OP_W4A8_PERGROUP ? at::kHalf : at::kFloat)) Py_RETURN_NONE;
  if (grouped) {
    const bool gs_ok = gs == 64 || gs == 128 || (gs == 256 && !w4);
    if (!gs_ok || K % gs != 0 || s.dim() != 2 || s.size(0) != K / gs || s.size(1) != N)
      Py_RETURN_NONE;
  } else if (s.numel() != N) {
    Py_RETURN_NONE;
  }
  if (has_bias && (op == CIDER_OP_W4A8 || bias_in.scalar_type() != at::kHalf ||
                   bias_in.numel() != N))
    Py_RETURN_NONE;
  const c10::Device dev = x.device();
  if (w.device() != dev || s.device() != dev || (has_bias && bias_in.device() != dev))
    Py_RETURN_NONE;

  // before anything is allocated (and a zero bias filled) for a call that the
  // library would turn down
  if (bf && !cider_linear_bf16_supported((int)op, x.const_data_ptr(), w.const_data_ptr(),
                                         s.const_data_ptr(), M, K, (int)gs))
    Py_RETURN_NONE;

  at::Tensor y;
  int rc = CIDER_OK;
  bool taken = true;
  Py_BEGIN_ALLOW_THREADS
  try {
    const c10::DeviceGuard guard(dev);
    const auto opt = at::TensorOptions().device(dev);
    at::DimVector shape(x.sizes());
    shape.back() = N;
    y = at::empty(shape, opt.dtype(xt));
    const size_t nb =
        cider_workspace_bytes((int)op, M, N, K, grouped ? (int)gs : 0);
    at::Tensor ws, bias = bias_in;
    if (nb) ws = at::empty({(int64_t)nb}, opt.dtype(at::kByte));
    // without a bias the int8 linears add zeros, as their Python functions do
    if (!has_bias && !w4) bias = at::zeros({N}, opt.dtype(at::kHalf));
    if (!dense(y) || (nb && !dense(ws)) || (bias.defined() && !dense(bias))) {
      taken = false;  // a dispatch mode made another kind of tensor
    } else {
      void* const st = (void*)c10::hip::getCurrentHIPStream(dev.index()).stream();
      const void* const xp = x.const_data_ptr();
      const void* const wp = w.const_data_ptr();
      const void* const sp = s.const_data_ptr();
      const void* const bp = bias.defined() ? bias.const_data_ptr() : nullptr;
      void* const yp = y.mutable_data_ptr();
      void* const wsp = nb ? ws.mutable_data_ptr() : nullptr;
      const float* const sf = (const float*)sp;
      if (bf)
        rc = cider_linear_bf16((int)op, xp, wp, sp, bp, yp, wsp, nb, M, N, K, (int)gs, st);
      else if (op == CIDER_OP_PERCHANNEL)
        rc = cider_perchannel_linear(xp, (const int8_t*)wp, sf, bp, yp, wsp, nb, M, N, K, st);
      else if (op == CIDER_OP_PERGROUP)
        rc = cider_pergroup_linear(xp, (const int8_t*)wp, sf, bp, yp, wsp, nb, M, N, K, (int)gs,
                                   st);
      else if (op == CIDER_OP_W4A8)
        rc = cider_w4a8_linear(xp, (const uint8_t*)wp, sf, yp, wsp, nb, M, N, K, st);
      else
        rc = cider_w4a8_pergroup_linear(xp, (const uint8_t*)wp, sp, bp, yp, wsp, nb, M, N, K,
                                        (int)gs, st);
    }
  } catch (...) {
    Py_BLOCK_THREADS
    throw;
  }
  Py_END_ALLOW_THREADS
  if (!taken || rc == CIDER_E_UNSUPPORTED) Py_RETURN_NONE;
  if (rc != CIDER_OK) {
    PyErr_SetString(rc == CIDER_E_INVALID ? PyExc_ValueError : PyExc_RuntimeError,
                    cider_last_error());
    return nullptr;
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL,
     "linear(op, x, w, scale, bias, group_size, any_dim) -> Tensor or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cider_fast", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__cider_fast() { return PyModule_Create(&module); }
