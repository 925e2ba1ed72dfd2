// The Python wrappers' ordinary calls without their host work: argument checks, allocations and args structs of lq_zoo_simple_gla,
// lq_zoo_chunk_forward, lq_zoo_rotate_qkv, lq_split_rotate_quant_xBC and lq_ssd_combined in native code.  Each function serves the
// ordinary form of its call (plain tensors on the current GPU, fp32 scales, shapes that need no padding) and returns None for any other,
// and for what is to be refused: the caller then takes the wrapper's general path, which converts, pads, copies or raises.  Nothing is
// kept from one call for the next.
//
// Host time of a call on one machine, general path -> here (the C entry with its launches in brackets): Mamba-2 cell B1 T2048 H8 26.5 ->
// 10.1 us (7.3 for two launches), KDA B1 T2048 H8 26.6 -> 10.3 (6.6), SSD layer B1 L512 H80, prologue and forward, 56 -> 25.3 (20.6 for
// five).  That was longer than the kernels of the first and the last (17 and 30 us): a ctypes struct of 30 to 60 fields, their conversions
// and attribute reads of tensors.  Whole calls 24.1 -> 16.7 and 52.3 -> 28.0.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include <climits>
#include <cmath>

#include "../../include/linquant_hip.h"

namespace {

// set once, while the module is loaded: entry points of liblinquant_hip.so and the function that raises for a failed call
decltype(&lq_zoo_simple_gla) simple_gla_entry;
decltype(&lq_zoo_simple_gla_workspace_bytes) simple_gla_bytes;
decltype(&lq_zoo_chunk_forward) chunk_forward_entry;
decltype(&lq_zoo_chunk_forward_workspace_bytes) chunk_forward_bytes;
decltype(&lq_zoo_rotate_qkv) rotate_entry;
decltype(&lq_split_rotate_quant_xBC) split_rotate_entry;
decltype(&lq_ssd_combined) ssd_entry;
decltype(&lq_ssd_combined_workspace_bytes) ssd_bytes;
PyObject* raise_failed;

using at::ScalarType;
using at::Tensor;

// a plain tensor with memory of its own on the GPU of the call
bool plain(PyObject* o, const c10::Device& dev, Tensor& t) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return t.defined() && t.layout() == at::kStrided && t.unsafeGetTensorImpl()->has_storage() && t.device() == dev;
}
bool optional(PyObject* o, const c10::Device& dev, Tensor& t) { return o == Py_None || plain(o, dev, t); }

bool aligned(const Tensor& t, uintptr_t n = 16) { return (uintptr_t)t.const_data_ptr() % n == 0; }

// dense fp32 with `numel` entries
bool table(const Tensor& t, int64_t numel, uintptr_t align = 4) {
  return t.scalar_type() == ScalarType::Float && t.is_contiguous() && t.numel() == numel && aligned(t, align);
}
const float* f32(const Tensor& t) { return t.defined() ? (const float*)t.const_data_ptr() : nullptr; }

bool number(PyObject* o, double& x) {
  if (PyFloat_CheckExact(o)) return x = PyFloat_AS_DOUBLE(o), true;
  if (!PyLong_CheckExact(o)) return false;
  x = PyLong_AsDouble(o);
  return !(x == -1.0 && PyErr_Occurred() && (PyErr_Clear(), true));
}
bool integer(PyObject* o, int64_t& x) {
  if (!PyLong_CheckExact(o)) return false;
  x = PyLong_AsLongLong(o);
  return !(x == -1 && PyErr_Occurred() && (PyErr_Clear(), true)) && x >= 0 && x <= INT_MAX;
}
bool fits(at::IntArrayRef s) {
  for (const int64_t n : s)
    if (n <= 0 || n > INT_MAX) return false;
  return true;
}

// the GPU of the first tensor, if it is the current one and nothing watches the operators of this thread
bool device_of(PyObject* o, c10::Device& dev) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.get_device() != c10::hip::current_device()) return false;
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0) return false;
  dev = t.device();
  return true;
}
hipStream_t stream_of(const c10::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

Tensor empty(at::IntArrayRef size, ScalarType dt, const c10::Device& dev) { return at::empty(size, at::TensorOptions().dtype(dt).device(dev)); }

PyObject* failed(const char* entry, int rc) {
  PyObject* r = PyObject_CallFunction(raise_failed, "si", entry, rc);  // raises
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, entry);
  return nullptr;
}

// q, k, v of a zoo call: dense, one 16-bit type, whole 64-token chunks, widths that need no padding
bool operands(const Tensor& q, const Tensor& k, const Tensor& v) {
  const ScalarType act = v.scalar_type();
  if ((act != ScalarType::Half && act != ScalarType::BFloat16) || q.scalar_type() != act || k.scalar_type() != act) return false;
  if (q.dim() != 4 || v.dim() != 4 || k.sizes() != q.sizes() || !fits(q.sizes()) || !fits(v.sizes())) return false;
  for (int i = 0; i < 3; ++i)
    if (v.size(i) != q.size(i)) return false;
  if (q.size(1) % 64 != 0 || (q.size(3) != 64 && q.size(3) != 128) || v.size(3) % 64 != 0) return false;
  return q.is_contiguous() && k.is_contiguous() && v.is_contiguous();
}
// `n` scales of a call's dict by role; their entries
bool scales(PyObject* dict, const c10::Device& dev, const char* const* names, const int64_t* sizes, int n, int unaligned, Tensor* sc) {
  if (!PyDict_CheckExact(dict)) return false;
  for (int i = 0; i < n; ++i) {
    PyObject* o = PyDict_GetItemString(dict, names[i]);
    if (!o || !plain(o, dev, sc[i]) || !table(sc[i], sizes[i], i < unaligned ? 4 : 16)) return false;
  }
  return true;
}
bool output_type(PyObject* o, ScalarType act, ScalarType& ot) {
  ot = act;
  if (o == Py_None) return true;
  if (!THPDtype_Check(o)) return false;
  ot = ((THPDtype*)o)->scalar_type;
  return ot == act || ot == ScalarType::Float;
}

// ---- simple_gla(q, k, v, g, scales, eta, scale, final_state, bits, out_dtype, prologue): chunk_simple_gla_int8, chunks of 64 tokens
PyObject* simple_gla(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) Py_RETURN_NONE;
  c10::Device dev(c10::DeviceType::CPU);
  Tensor q, k, v, g, sc[6], sg_qk, sg_v;
  if (!device_of(arg[0], dev) || !plain(arg[0], dev, q) || !plain(arg[1], dev, k) || !plain(arg[2], dev, v) || !optional(arg[3], dev, g)) Py_RETURN_NONE;
  if (!operands(q, k, v)) Py_RETURN_NONE;
  const ScalarType act = v.scalar_type();
  const int64_t B = q.size(0), T = q.size(1), H = q.size(2), K = q.size(3), V = v.size(3);
  if (g.defined() && (g.dim() != 3 || g.size(0) != B || g.size(1) != T || g.size(2) != H || !table(g, B * T * H))) Py_RETURN_NONE;
  static const char* const names[6] = {"q", "k", "kw", "vw", "vl", "state"};
  const int64_t sizes[6] = {H, H, H * K, H * V, H * V, H * V};
  if (!scales(arg[4], dev, names, sizes, 6, 2, sc)) Py_RETURN_NONE;
  double eta, scale = 0.0;
  int64_t bits;
  if (!number(arg[5], eta) || !(arg[6] == Py_None || number(arg[6], scale)) || !integer(arg[8], bits) || bits < 2 || bits > 8) Py_RETURN_NONE;
  if (arg[6] == Py_None) scale = std::pow((double)K, -0.5);
  const int final_state = PyObject_IsTrue(arg[7]);
  if (final_state < 0) return nullptr;
  ScalarType ot;
  if (!output_type(arg[9], act, ot)) Py_RETURN_NONE;
  if (arg[10] != Py_None) {  // the rotations; with D_QK (whose reciprocals are a tensor operation) the general path
    if (!PyDict_CheckExact(arg[10]) || (V != 64 && V != 128)) Py_RETURN_NONE;
    PyObject *key, *value;
    for (Py_ssize_t at = 0; PyDict_Next(arg[10], &at, &key, &value);) {
      if (!PyUnicode_CheckExact(key)) Py_RETURN_NONE;
      const bool qk = PyUnicode_CompareWithASCIIString(key, "signs_qk") == 0;
      if (!qk && PyUnicode_CompareWithASCIIString(key, "signs_v") != 0) Py_RETURN_NONE;
      Tensor& t = qk ? sg_qk : sg_v;
      if (!optional(value, dev, t) || (t.defined() && !table(t, qk ? K : V, 16))) Py_RETURN_NONE;
    }
  }
  lq_zoo_simple_gla_args a = {};
  a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr(), a.g = f32(g);
  a.sq = f32(sc[0]), a.sk = f32(sc[1]), a.skw = f32(sc[2]), a.svw = f32(sc[3]), a.svl = f32(sc[4]), a.ss = f32(sc[5]);
  a.eta = (float)eta, a.scale = (float)scale, a.qmax = (1 << (bits - 1)) - 1;
  a.batch = (int)B, a.seqlen = (int)T, a.nheads = (int)H, a.kdim = (int)K, a.vdim = (int)V, a.chunk_size = 64;
  a.act_dtype = act == ScalarType::BFloat16 ? LQ_DT_BF16 : LQ_DT_F16;
  a.signs_qk = f32(sg_qk), a.signs_v = f32(sg_v);
  int64_t bytes = 0;
  if (simple_gla_bytes(&a, &bytes) != 0) Py_RETURN_NONE;
  Tensor o, ht;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    Tensor ws = empty({bytes}, ScalarType::Byte, dev);
    o = empty(v.sizes(), ot, dev);
    if (final_state) ht = empty({B, H, K, V}, ScalarType::Float, dev);
    a.o = o.data_ptr(), a.o_is_f32 = ot == ScalarType::Float, a.ht = final_state ? (float*)ht.data_ptr() : nullptr;
    a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
    rc = simple_gla_entry(&a, stream_of(dev));
  }
  if (rc != 0) return failed("lq_zoo_simple_gla", rc);
  PyObject* po = THPVariable_Wrap(o);
  PyObject* ph = final_state ? THPVariable_Wrap(ht) : (Py_INCREF(Py_None), Py_None);
  return Py_BuildValue("(NN)", po, ph);
  END_HANDLE_TH_ERRORS
}

// ---- chunk_forward(q, k, v, g, beta, scales, sigma, tau, eta, scale, final_state, bits, out_dtype, rot, dqk): chunk_gla_int8 (beta None),
// chunk_delta_int8 and chunk_kda_int8, chunks of 64 tokens
PyObject* chunk_forward(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) Py_RETURN_NONE;
  c10::Device dev(c10::DeviceType::CPU);
  Tensor q, k, v, g, beta, sc[7], rot, dqk;
  if (!device_of(arg[0], dev) || !plain(arg[0], dev, q) || !plain(arg[1], dev, k) || !plain(arg[2], dev, v) || !optional(arg[3], dev, g) ||
      !optional(arg[4], dev, beta) || !optional(arg[13], dev, rot) || !optional(arg[14], dev, dqk))
    Py_RETURN_NONE;
  if (!operands(q, k, v)) Py_RETURN_NONE;
  const ScalarType act = v.scalar_type();
  const int64_t B = q.size(0), T = q.size(1), H = q.size(2), K = q.size(3), V = v.size(3);
  const bool delta = beta.defined(), diag = g.defined() && g.dim() == 4;
  if (delta && (beta.dim() != 3 || beta.size(0) != B || beta.size(1) != T || !table(beta, B * T * H))) Py_RETURN_NONE;
  if (diag ? g.sizes() != q.sizes() || !table(g, B * T * H * K, 16)
           : !delta || (g.defined() && (g.dim() != 3 || g.size(0) != B || g.size(1) != T || !table(g, B * T * H))))
    Py_RETURN_NONE;
  if (rot.defined() && (!diag || rot.dim() != 2 || rot.size(0) != K || rot.size(1) != K || !rot.is_contiguous() || !aligned(rot) ||
                        (rot.scalar_type() != ScalarType::Float && rot.scalar_type() != ScalarType::Half)))
    Py_RETURN_NONE;
  if (dqk.defined() && (!delta || !diag || dqk.dim() != 2 || dqk.size(0) != H || !table(dqk, H * K, 16))) Py_RETURN_NONE;
  static const char* const linear_names[] = {"q", "k", "vw", "kw", "vl", "state"};
  static const char* const delta_names[] = {"q", "k", "ew", "kw", "el", "state", "w"};
  const int64_t sizes[7] = {H, H, H * V, H * K, H * V, H * V, H};
  if (!scales(arg[5], dev, delta ? delta_names : linear_names, sizes, 6, 3, sc)) Py_RETURN_NONE;
  if (delta && !scales(arg[5], dev, delta_names + 6, sizes + 6, 1, 1, sc + 6)) Py_RETURN_NONE;
  double sigma, tau, eta, scale = 0.0;
  int64_t bits;
  if (!number(arg[6], sigma) || !number(arg[7], tau) || !number(arg[8], eta) || !(arg[9] == Py_None || number(arg[9], scale)) || !integer(arg[11], bits) ||
      bits < 2 || bits > 8)
    Py_RETURN_NONE;
  if (arg[9] == Py_None) scale = std::pow((double)K, -0.5);
  const int final_state = PyObject_IsTrue(arg[10]);
  if (final_state < 0) return nullptr;
  ScalarType ot;
  if (!output_type(arg[12], act, ot)) Py_RETURN_NONE;
  lq_zoo_chunk_forward_args a = {};
  a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr(), a.g = f32(g), a.beta = f32(beta);
  a.sq = f32(sc[0]), a.sk = f32(sc[1]), a.svw = f32(sc[2]), a.skw = f32(sc[3]), a.svl = f32(sc[4]), a.ss = f32(sc[5]), a.sw = f32(sc[6]);
  if (rot.defined() && rot.scalar_type() == ScalarType::Float) a.rot_f32 = f32(rot);
  else if (rot.defined()) a.rot = rot.const_data_ptr();
  a.dqk = f32(dqk);
  a.sigma = (float)sigma, a.tau = (float)tau, a.eta = (float)eta, a.scale = (float)scale, a.qmax = (1 << (bits - 1)) - 1;
  a.family = delta ? LQ_FAMILY_DELTA : LQ_FAMILY_LINEAR, a.decay = diag ? LQ_DECAY_DIAGONAL : (g.defined() ? LQ_DECAY_SCALAR : LQ_DECAY_NONE);
  a.batch = (int)B, a.seqlen = (int)T, a.nheads = (int)H, a.kdim = (int)K, a.vdim = (int)V, a.chunk_size = 64;
  a.act_dtype = act == ScalarType::BFloat16 ? LQ_DT_BF16 : LQ_DT_F16;
  int64_t bytes = 0;
  if (chunk_forward_bytes(&a, &bytes) != 0) Py_RETURN_NONE;
  Tensor o, ht;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    Tensor ws = empty({bytes + (rot.defined() ? 2 * K * K : 0)}, ScalarType::Byte, dev);
    o = empty(v.sizes(), ot, dev);
    if (final_state) ht = empty({B, H, K, V}, ScalarType::Float, dev);
    a.o = o.data_ptr(), a.o_is_f32 = ot == ScalarType::Float, a.ht = final_state ? (float*)ht.data_ptr() : nullptr;
    a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
    if (rot.defined()) a.rot_ws = (char*)ws.data_ptr() + bytes;
    rc = chunk_forward_entry(&a, stream_of(dev));
  }
  if (rc != 0) return failed("lq_zoo_chunk_forward", rc);
  PyObject* po = THPVariable_Wrap(o);
  PyObject* ph = final_state ? THPVariable_Wrap(ht) : (Py_INCREF(Py_None), Py_None);
  return Py_BuildValue("(NN)", po, ph);
  END_HANDLE_TH_ERRORS
}

// ---- rotate_qkv(q, k, v, signs_qk, signs_v): rotate_qkv into new tensors, without D_QK
PyObject* rotate_qkv(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  c10::Device dev(c10::DeviceType::CPU);
  Tensor in[3], sg_qk, sg_v, out[3];
  PyObject* first = arg[0] != Py_None ? arg[0] : (arg[1] != Py_None ? arg[1] : arg[2]);
  if (!device_of(first, dev) || !optional(arg[3], dev, sg_qk) || !optional(arg[4], dev, sg_v)) Py_RETURN_NONE;
  const Tensor& ref = THPVariable_Unpack(first);
  if (ref.dim() != 4 || (ref.scalar_type() != ScalarType::Half && ref.scalar_type() != ScalarType::BFloat16)) Py_RETURN_NONE;
  for (int i = 0; i < 3; ++i) {
    if (!optional(arg[i], dev, in[i])) Py_RETURN_NONE;
    const Tensor& t = in[i];
    if (!t.defined()) continue;
    if (t.dim() != 4 || t.scalar_type() != ref.scalar_type() || !t.is_contiguous() || !fits(t.sizes()) || (t.size(3) != 64 && t.size(3) != 128)) Py_RETURN_NONE;
    for (int d = 0; d < 3; ++d)
      if (t.size(d) != ref.size(d)) Py_RETURN_NONE;
  }
  if (in[0].defined() && in[1].defined() && in[0].size(3) != in[1].size(3)) Py_RETURN_NONE;
  const int64_t K = in[0].defined() ? in[0].size(3) : (in[1].defined() ? in[1].size(3) : 0), V = in[2].defined() ? in[2].size(3) : 0;
  if ((sg_qk.defined() && !table(sg_qk, K, 16)) || (sg_v.defined() && !table(sg_v, V, 16))) Py_RETURN_NONE;
  lq_zoo_rotate_qkv_args a = {};
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    for (int i = 0; i < 3; ++i)
      if (in[i].defined()) out[i] = empty(in[i].sizes(), in[i].scalar_type(), dev);
    auto at = [](const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; };
    a.q = at(in[0]), a.k = at(in[1]), a.v = at(in[2]);
    a.q_out = const_cast<void*>(at(out[0])), a.k_out = const_cast<void*>(at(out[1])), a.v_out = const_cast<void*>(at(out[2]));
    a.signs_qk = f32(sg_qk), a.signs_v = f32(sg_v);
    a.batch = (int)ref.size(0), a.seqlen = (int)ref.size(1), a.nheads = (int)ref.size(2), a.kdim = (int)K, a.vdim = (int)V;
    a.act_dtype = ref.scalar_type() == ScalarType::BFloat16 ? LQ_DT_BF16 : LQ_DT_F16;
    rc = rotate_entry(&a, stream_of(dev));
  }
  if (rc != 0) return failed("lq_zoo_rotate_qkv", rc);
  PyObject* o[3];
  for (int i = 0; i < 3; ++i) o[i] = in[i].defined() ? THPVariable_Wrap(out[i]) : (Py_INCREF(Py_None), Py_None);
  return Py_BuildValue("(NNN)", o[0], o[1], o[2]);
  END_HANDLE_TH_ERRORS
}

// ---- split_rotate(xBC, r_signs, nheads, ngroups, d_state, headdim, B_inv_scale, C_inv_scale, return_b_fp, return_b_rowmax):
// fused_split_rotate_quant_xBC without D_QK
PyObject* split_rotate(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) Py_RETURN_NONE;
  c10::Device dev(c10::DeviceType::CPU);
  Tensor xBC, signs, binv, cinv;
  int64_t H, G, N, P;
  if (!device_of(arg[0], dev) || !plain(arg[0], dev, xBC) || !optional(arg[1], dev, signs) || !plain(arg[6], dev, binv) || !plain(arg[7], dev, cinv)) Py_RETURN_NONE;
  if (!integer(arg[2], H) || !integer(arg[3], G) || !integer(arg[4], N) || !integer(arg[5], P)) Py_RETURN_NONE;
  const int want_fp = PyObject_IsTrue(arg[8]), want_max = PyObject_IsTrue(arg[9]);
  if (want_fp < 0 || want_max < 0) return nullptr;
  if (xBC.dim() != 3 || xBC.scalar_type() != ScalarType::Half || !fits(xBC.sizes()) || xBC.stride(2) != 1) Py_RETURN_NONE;
  const int64_t B = xBC.size(0), T = xBC.size(1), d_ssm = H * P;
  if ((N != 64 && N != 128) || G <= 0 || d_ssm <= 0 || xBC.size(2) != d_ssm + 2 * G * N || (want_max && !want_fp)) Py_RETURN_NONE;
  if (!table(binv, G) || !table(cinv, G)) Py_RETURN_NONE;
  int signs_dtype = 0;
  if (signs.defined()) {
    const ScalarType st = signs.scalar_type();
    if ((st != ScalarType::Half && st != ScalarType::Float && st != ScalarType::Char) || !signs.is_contiguous() || signs.numel() != G * N) Py_RETURN_NONE;
    signs_dtype = st == ScalarType::Half ? LQ_DT_F16 : (st == ScalarType::Float ? LQ_DT_F32 : LQ_DT_I8);
  }
  Tensor x, qB, qC, b_fp, b_max;
  lq_split_rotate_quant_xBC_args a = {};
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    x = xBC.slice(2, 0, d_ssm).view({B, T, H, P});
    qB = empty({B, T, G, N}, ScalarType::Char, dev), qC = empty({B, T, G, N}, ScalarType::Char, dev);
    if (want_fp) b_fp = empty({B, T, G, N}, ScalarType::Half, dev);
    if (want_max) b_max = empty({B, T, G}, ScalarType::Float, dev);
    a.xBC = xBC.const_data_ptr(), a.xBC_stride_b = xBC.stride(0), a.xBC_stride_t = xBC.stride(1);
    a.qB = (int8_t*)qB.data_ptr(), a.qC = (int8_t*)qC.data_ptr(), a.b_fp = want_fp ? b_fp.data_ptr() : nullptr;
    a.signs = signs.defined() ? signs.const_data_ptr() : nullptr, a.signs_dtype = signs_dtype;
    a.B_inv_scale = f32(binv), a.C_inv_scale = f32(cinv);
    a.batch = (int)B, a.seqlen = (int)T, a.d_ssm = (int)d_ssm, a.ngroups = (int)G, a.dstate = (int)N;
    a.b_rowmax = want_max ? (float*)b_max.data_ptr() : nullptr;
    rc = split_rotate_entry(&a, stream_of(dev));
  }
  if (rc != 0) return failed("lq_split_rotate_quant_xBC", rc);
  PyObject *px = THPVariable_Wrap(x), *pb = THPVariable_Wrap(qB), *pc = THPVariable_Wrap(qC);
  if (want_max) return Py_BuildValue("(NNNNN)", px, pb, pc, THPVariable_Wrap(b_fp), THPVariable_Wrap(b_max));
  if (want_fp) return Py_BuildValue("(NNNN)", px, pb, pc, THPVariable_Wrap(b_fp));
  return Py_BuildValue("(NNN)", px, pb, pc);
  END_HANDLE_TH_ERRORS
}

bool scalar(const Tensor& t) { return t.scalar_type() == ScalarType::Float && t.numel() == 1; }
bool rows(const Tensor& t, int64_t B, int64_t L, ScalarType st) {  // (B, L, *, *) with dense rows
  return t.dim() == 4 && t.size(0) == B && t.size(1) == L && t.scalar_type() == st && t.stride(3) == 1 && fits(t.sizes());
}

// ---- ssd(x, dt, dt_scale, A_log, A_log_scale, q_B, B_scale, q_C, C_scale, chunk_size, D, D_scale, dt_bias, dt_softplus, dt_limit,
// state_scale, cb_scale, alpha_hp, bscale_g, keyside, x_scale_hp, b_fp, b_gate_scale, b_rowmax, gate_shift): the SSD forward
PyObject* ssd(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 25) Py_RETURN_NONE;
  c10::Device dev(c10::DeviceType::CPU);
  Tensor x, dt, dts, A, als, qB, Bs, qC, Cs, D, dsc, bias, ss, cbs, alpha, bsg, xs, bfp, bgs, bmax;
  if (!device_of(arg[0], dev)) Py_RETURN_NONE;
  const int keyside = PyObject_IsTrue(arg[19]), softplus = PyObject_IsTrue(arg[13]);
  if (keyside < 0 || softplus < 0) return nullptr;
  if (!plain(arg[0], dev, x) || !plain(arg[1], dev, dt) || !plain(arg[2], dev, dts) || !plain(arg[3], dev, A) || !plain(arg[4], dev, als) ||
      !plain(arg[5], dev, qB) || !plain(arg[6], dev, Bs) || !plain(arg[7], dev, qC) || !plain(arg[8], dev, Cs) || !optional(arg[10], dev, D) ||
      !optional(arg[12], dev, bias) || !plain(arg[15], dev, ss) || !plain(arg[16], dev, cbs))
    Py_RETURN_NONE;
  if (D.defined() && !plain(arg[11], dev, dsc)) Py_RETURN_NONE;
  if (x.dim() != 4 || qC.dim() != 4) Py_RETURN_NONE;
  const int64_t B = x.size(0), L = x.size(1), H = x.size(2), P = x.size(3), G = qC.size(2), N = qC.size(3);
  if (!rows(x, B, L, ScalarType::Half) || !rows(qC, B, L, ScalarType::Char) || qB.sizes() != qC.sizes()) Py_RETURN_NONE;
  if (dt.dim() != 3 || dt.size(0) != B || dt.size(1) != L || dt.size(2) != H) Py_RETURN_NONE;
  const ScalarType dtt = dt.scalar_type();
  if (dtt != ScalarType::Half && dtt != ScalarType::Float && dtt != ScalarType::Char) Py_RETURN_NONE;
  if (A.dim() != 1 || A.size(0) != H || A.scalar_type() != ScalarType::Char || !scalar(dts) || !scalar(als)) Py_RETURN_NONE;
  if (!table(Bs, G) || !table(Cs, G) || !table(cbs, G) || cbs.dim() != 1) Py_RETURN_NONE;
  if (ss.dim() != 2 || ss.size(0) != H || ss.size(1) != P || ss.scalar_type() != ScalarType::Float) Py_RETURN_NONE;
  if (bias.defined() && (bias.dim() != 1 || bias.size(0) != H || bias.scalar_type() != ScalarType::Float)) Py_RETURN_NONE;
  if (D.defined() && (D.scalar_type() != ScalarType::Char || D.dim() < 1 || D.dim() > 2 || D.size(0) != H || (D.dim() == 2 && D.size(1) != P) ||
                      D.stride(-1) != 1 || !scalar(dsc)))
    Py_RETURN_NONE;
  int64_t Q, shift;
  double lo, hi;
  if (!integer(arg[9], Q) || !integer(arg[24], shift)) Py_RETURN_NONE;
  if (!PyTuple_CheckExact(arg[14]) || PyTuple_GET_SIZE(arg[14]) != 2 || !number(PyTuple_GET_ITEM(arg[14], 0), lo) || !number(PyTuple_GET_ITEM(arg[14], 1), hi)) Py_RETURN_NONE;
  lq_ssd_combined_args a = {};
  if (keyside) {
    if (!plain(arg[20], dev, xs) || !plain(arg[21], dev, bfp) || !plain(arg[22], dev, bgs) || !optional(arg[23], dev, bmax)) Py_RETURN_NONE;
    if (xs.dim() != 2 || xs.size(0) != H || xs.size(1) != P || xs.scalar_type() != ScalarType::Float) Py_RETURN_NONE;
    if (!rows(bfp, B, L, ScalarType::Half) || bfp.sizes() != qC.sizes()) Py_RETURN_NONE;
    if (bgs.dim() != 4 || bgs.scalar_type() != ScalarType::Float) Py_RETURN_NONE;
    const int64_t full[4] = {B, (L + Q - 1) / std::max<int64_t>(Q, 1), H, N};
    int64_t st[4];
    for (int i = 0; i < 4; ++i) {
      if (bgs.size(i) != 1 && bgs.size(i) != full[i]) Py_RETURN_NONE;
      st[i] = bgs.size(i) > 1 ? bgs.stride(i) : 0;
    }
    if (bmax.defined() && (!table(bmax, B * L * G) || bmax.dim() != 3 || bmax.size(0) != B || bmax.size(1) != L)) Py_RETURN_NONE;
    a.b_fp = bfp.const_data_ptr(), a.bfp_stride_b = bfp.stride(0), a.bfp_stride_l = bfp.stride(1), a.bfp_stride_g = bfp.stride(2);
    a.x_scale_hp = f32(xs), a.xs_stride_h = xs.stride(0), a.xs_stride_p = xs.stride(1);
    a.b_gate_scale = f32(bgs), a.bgs_stride_b = st[0], a.bgs_stride_c = st[1], a.bgs_stride_h = st[2], a.bgs_stride_n = st[3];
    a.b_rowmax = f32(bmax);
  } else {
    if (!plain(arg[17], dev, alpha) || !plain(arg[18], dev, bsg)) Py_RETURN_NONE;
    if (!rows(qB, B, L, ScalarType::Char)) Py_RETURN_NONE;
    if (alpha.dim() != 2 || alpha.size(0) != H || alpha.size(1) != P || alpha.scalar_type() != ScalarType::Float) Py_RETURN_NONE;
    if (bsg.dim() != 1 || bsg.size(0) != G || bsg.scalar_type() != ScalarType::Float) Py_RETURN_NONE;
    a.qB = (const int8_t*)qB.const_data_ptr(), a.qB_stride_b = qB.stride(0), a.qB_stride_l = qB.stride(1), a.qB_stride_g = qB.stride(2);
    a.alpha_hp = f32(alpha), a.alpha_stride_h = alpha.stride(0), a.alpha_stride_p = alpha.stride(1);
    a.bscale_g = f32(bsg), a.bscale_stride_g = bsg.stride(0);
  }
  a.x = x.const_data_ptr(), a.x_stride_b = x.stride(0), a.x_stride_l = x.stride(1), a.x_stride_h = x.stride(2);
  a.dt = dt.const_data_ptr(), a.dt_dtype = dtt == ScalarType::Half ? LQ_DT_F16 : (dtt == ScalarType::Float ? LQ_DT_F32 : LQ_DT_I8);
  a.dt_stride_b = dt.stride(0), a.dt_stride_l = dt.stride(1), a.dt_stride_h = dt.stride(2), a.dt_scale = f32(dts);
  a.A_log = (const int8_t*)A.const_data_ptr(), a.A_log_stride_h = A.stride(0), a.A_log_scale = f32(als);
  a.dt_bias = f32(bias), a.dt_bias_stride_h = bias.defined() ? bias.stride(0) : 0;
  a.dt_softplus = softplus, a.dt_min = (float)lo, a.dt_max = (float)hi;
  a.qC = (const int8_t*)qC.const_data_ptr(), a.qC_stride_b = qC.stride(0), a.qC_stride_l = qC.stride(1), a.qC_stride_g = qC.stride(2);
  a.B_scale = f32(Bs), a.C_scale = f32(Cs), a.cb_scale = f32(cbs);
  if (D.defined()) a.D = (const int8_t*)D.const_data_ptr(), a.D_stride_h = D.stride(0), a.D_has_hdim = D.dim() == 2, a.D_scale = f32(dsc);
  a.state_scale = f32(ss), a.ss_stride_h = ss.stride(0), a.ss_stride_p = ss.stride(1);
  a.keyside = keyside, a.gate_shift = (int)shift;
  a.batch = (int)B, a.seqlen = (int)L, a.nheads = (int)H, a.headdim = (int)P, a.ngroups = (int)G, a.dstate = (int)N, a.chunk_size = (int)Q;
  int64_t bytes = 0;
  if (ssd_bytes(&a, &bytes) != 0) Py_RETURN_NONE;
  Tensor o;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    o = empty({B, L, H, P}, ScalarType::Half, dev);
    Tensor ws = empty({bytes}, ScalarType::Byte, dev);
    a.out = o.data_ptr(), a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
    rc = ssd_entry(&a, stream_of(dev));
  }
  if (rc != 0) return failed("lq_ssd_combined", rc);
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// whether the library was built from the header that this file was: its ABI version and the structs that are filled here
bool same_abi(decltype(&lq_abi_version) version, decltype(&lq_args_size) size) {
  const int v = version();
  if (v != LQ_ABI_VERSION) return PyErr_Format(PyExc_RuntimeError, "ABI version %d, the library has %d", LQ_ABI_VERSION, v), false;
#define LQ_SAME_SIZE(T)                                                                                                          \
  if (const int n = size(#T); n != (int)sizeof(T))                                                                               \
    return PyErr_Format(PyExc_RuntimeError, #T ": sizeof %d, the library has %d", (int)sizeof(T), n), false
  LQ_SAME_SIZE(lq_zoo_simple_gla_args);
  LQ_SAME_SIZE(lq_zoo_chunk_forward_args);
  LQ_SAME_SIZE(lq_zoo_rotate_qkv_args);
  LQ_SAME_SIZE(lq_split_rotate_quant_xBC_args);
  LQ_SAME_SIZE(lq_ssd_combined_args);
#undef LQ_SAME_SIZE
  return true;
}

// init(raise_failed, {entry point: address})
PyObject* init(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 2 || !PyCallable_Check(arg[0]) || !PyDict_Check(arg[1])) {
    PyErr_SetString(PyExc_TypeError, "init(raise_failed, addresses)");
    return nullptr;
  }
  auto entry = [&](const char* name) { PyObject* o = PyDict_GetItemString(arg[1], name); return o ? PyLong_AsVoidPtr(o) : nullptr; };
  const auto version = (decltype(&lq_abi_version))entry("lq_abi_version");
  const auto size = (decltype(&lq_args_size))entry("lq_args_size");
  if (!version || !size) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "lq_abi_version or lq_args_size is missing");
    return nullptr;
  }
  if (!same_abi(version, size)) return nullptr;
  simple_gla_entry = (decltype(simple_gla_entry))entry("lq_zoo_simple_gla");
  simple_gla_bytes = (decltype(simple_gla_bytes))entry("lq_zoo_simple_gla_workspace_bytes");
  split_rotate_entry = (decltype(split_rotate_entry))entry("lq_split_rotate_quant_xBC");
  ssd_entry = (decltype(ssd_entry))entry("lq_ssd_combined");
  ssd_bytes = (decltype(ssd_bytes))entry("lq_ssd_combined_workspace_bytes");
  chunk_forward_entry = (decltype(chunk_forward_entry))entry("lq_zoo_chunk_forward");
  chunk_forward_bytes = (decltype(chunk_forward_bytes))entry("lq_zoo_chunk_forward_workspace_bytes");
  rotate_entry = (decltype(rotate_entry))entry("lq_zoo_rotate_qkv");
  if (!simple_gla_entry || !simple_gla_bytes || !chunk_forward_entry || !chunk_forward_bytes || !rotate_entry || !split_rotate_entry || !ssd_entry || !ssd_bytes) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "an entry point is missing");
    return nullptr;
  }
  Py_INCREF(arg[0]);
  Py_XSETREF(raise_failed, arg[0]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"init", (PyCFunction)(void*)init, METH_FASTCALL, nullptr},
                         {"simple_gla", (PyCFunction)(void*)simple_gla, METH_FASTCALL, nullptr},
                         {"chunk_forward", (PyCFunction)(void*)chunk_forward, METH_FASTCALL, nullptr},
                         {"rotate_qkv", (PyCFunction)(void*)rotate_qkv, METH_FASTCALL, nullptr},
                         {"split_rotate", (PyCFunction)(void*)split_rotate, METH_FASTCALL, nullptr},
                         {"ssd", (PyCFunction)(void*)ssd, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__binding() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", LQ_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
