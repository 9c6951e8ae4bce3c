// Native call path of the Python module's append and decode entry points
// (sglang_mlx_amd._native): argument checks, output allocation and the C-ABI
// call in one C++ function, where the Python form of the same steps (_ext.py,
// through ctypes) costs 13 us an append and 19 us a decode, more than most of
// these kernels run.
//
// Every function takes the ordinary calls only and returns None for any other:
// tensor subclasses and wrapped tensors, other devices and index types,
// sources that need a copy, scratch that has to be allocated, values out of
// range.  The caller then runs the Python path, which has the general forms and
// every error message.  A status other than success comes back as an int; for
// a refused call (nothing was launched) the Python path runs as well.
//
// Other Python threads run while the output is allocated and the kernel is
// launched, as under ctypes: a launch can wait for room in a full queue, and a
// host callback ahead of it in the stream may need the interpreter.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <limits>

#include "../../include/pagedkv.h"

namespace {

using at::Tensor;

// A plain strided tensor on a HIP device: nothing but the dense backend and
// autograd keys, so that its data pointer and strides are what they seem.
bool plain(PyObject* o) { return THPVariable_CheckExact(o); }
bool usable(const Tensor& t, const c10::Device& dev) {
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
      c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
  return t.defined() && t.device() == dev && (t.key_set().raw_repr() & ~allowed.raw_repr()) == 0;
}

// Function modes, tracing, vmap and functional transforms see Python calls
// that this path would hide from them.
bool transformed() {
  using c10::DispatchKey;
  auto on = [](DispatchKey k) { return c10::impl::tls_is_dispatch_key_included(k); };
  return at::impl::torch_function_mode_enabled() || on(DispatchKey::Tracer) || on(DispatchKey::Python) ||
         on(DispatchKey::PythonTLSSnapshot) || on(DispatchKey::Functionalize) ||
         on(DispatchKey::FuncTorchDynamicLayerFrontMode) || on(DispatchKey::FuncTorchBatched);
}

bool as_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  v = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0 && v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max();
}
bool as_double(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o)) return false;
  v = PyFloat_AS_DOUBLE(o);
  return true;
}

// The C ABI's code of a dtype, -1 if it has none; fp8: uint8 holds codes.
int code_of(const Tensor& t, bool fp8) {
  switch (t.scalar_type()) {
    case at::kFloat: return PKV_F32;
    case at::kHalf: return PKV_F16;
    case at::kBFloat16: return PKV_BF16;
    case at::kByte: return fp8 ? PKV_FP8_E4M3 : -1;
    default: return -1;
  }
}
int64_t bytes_of(int code) { return code == PKV_F32 ? 4 : code == PKV_FP8_E4M3 ? 1 : 2; }
bool i32_contiguous(const Tensor& t, int64_t dims) {
  return t.scalar_type() == at::kInt && t.dim() == dims && t.is_contiguous();
}
// float32 holds the scale as a finite, nonzero value (the C ABI refuses
// others, with the Python path's messages).
bool good_scale(double s) { return std::isfinite((float)s) && (float)s != 0.f; }

// The device becomes current for the launch, as under torch.cuda.device.
struct OnDevice {
  c10::OptionalDeviceGuard guard;
  explicit OnDevice(const c10::Device& dev) {
    if (c10::hip::current_device() != dev.index()) guard.reset_device(dev);
  }
};

// (key, value, key_cache, value_cache, slot_mapping, k_scale, v_scale)
PyObject* reshape_and_cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  for (int i = 0; i < 5; ++i)
    if (!plain(a[i])) Py_RETURN_NONE;
  double k_scale, v_scale;
  if (!as_double(a[5], k_scale) || !as_double(a[6], v_scale) || transformed()) Py_RETURN_NONE;
  // (Copies: the tensors stay alive while other threads run.)
  const Tensor key = THPVariable_Unpack(a[0]), value = THPVariable_Unpack(a[1]), kc = THPVariable_Unpack(a[2]),
               vc = THPVariable_Unpack(a[3]), slots = THPVariable_Unpack(a[4]);
  const c10::Device dev = key.device();
  if (!dev.is_cuda() || !usable(key, dev) || !usable(value, dev) || !usable(kc, dev) || !usable(vc, dev) ||
      !usable(slots, dev))
    Py_RETURN_NONE;
  if (key.dim() != 3 || value.sizes() != key.sizes() || !i32_contiguous(slots, 1)) Py_RETURN_NONE;
  const int64_t N = key.size(0), H = key.size(1), D = key.size(2);
  if (N == 0 || H <= 0 || D <= 0 || slots.size(0) != N) Py_RETURN_NONE;
  const int kv = code_of(key, false), cc = code_of(kc, true);
  if (kv < 0 || cc < 0 || value.scalar_type() != key.scalar_type() || vc.scalar_type() != kc.scalar_type())
    Py_RETURN_NONE;
  const bool fp8 = cc == PKV_FP8_E4M3;
  if (!(kv == cc || kv == PKV_F32 || fp8) || (fp8 && !(good_scale(k_scale) && good_scale(v_scale)))) Py_RETURN_NONE;
  const int64_t x = 16 / bytes_of(cc);
  int32_t layout;
  int64_t bs, num_slots;
  if (kc.dim() == 5 && vc.dim() == 4) {
    layout = PKV_LAYOUT_PAGED5D;
    const int64_t nb = kc.size(0);
    bs = kc.size(3);
    if (D % x != 0 || kc.size(1) != H || kc.size(2) != D / x || kc.size(4) != x || vc.size(0) != nb ||
        vc.size(1) != H || vc.size(2) != D || vc.size(3) != bs)
      Py_RETURN_NONE;
    num_slots = nb * bs;
  } else if (kc.dim() == 3 && vc.sizes() == kc.sizes()) {
    layout = PKV_LAYOUT_TOKEN_MAJOR;
    bs = 1;
    if (kc.size(1) != H || kc.size(2) != D || (fp8 && (H * D) % 8 != 0)) Py_RETURN_NONE;
    num_slots = kc.size(0);
  } else {
    Py_RETURN_NONE;
  }
  if (!kc.is_contiguous() || !vc.is_contiguous()) Py_RETURN_NONE;
  auto row_stride = [&](const Tensor& t, int64_t& stride) {
    if (t.stride(1) != D || t.stride(2) != 1 || (N > 1 && t.stride(0) < H * D)) return false;
    stride = N > 1 ? t.stride(0) : H * D;
    return true;
  };
  int64_t ks, vs;
  if (!row_stride(key, ks) || !row_stride(value, vs)) Py_RETURN_NONE;
  const OnDevice on(dev);
  int st;
  {
    pybind11::gil_scoped_release release;
    st = pkv_reshape_and_cache(
        key.data_ptr(), value.data_ptr(), kc.data_ptr(), vc.data_ptr(), static_cast<const int32_t*>(slots.data_ptr()),
        N, (int32_t)H, (int32_t)D, ks, vs, layout, (int32_t)bs, (int32_t)x, num_slots, kv, cc, (float)k_scale,
        (float)v_scale, c10::hip::getCurrentHIPStream(dev.index()).stream());
  }
  if (st != PKV_OK) return PyLong_FromLong(st);
  PyObject* out = PyList_New(2);
  if (out == nullptr) return nullptr;
  Py_INCREF(a[2]);
  Py_INCREF(a[3]);
  PyList_SET_ITEM(out, 0, a[2]);
  PyList_SET_ITEM(out, 1, a[3]);
  return out;
  END_HANDLE_TH_ERRORS
}

// (scratch buffers by (device index, stream), query, key_cache, value_cache,
// block_tables, context_lens, num_kv_heads, scale, block_size, max_seq_len,
// alibi_slopes, partition_size, k_scale, v_scale)
PyObject* paged_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 14 || !PyDict_CheckExact(a[0])) Py_RETURN_NONE;
  for (int i = 1; i < 6; ++i)
    if (!plain(a[i])) Py_RETURN_NONE;
  int64_t Hkv, bs, max_seq, partition;
  double scale, k_scale, v_scale;
  if (!as_int(a[6], Hkv) || !as_double(a[7], scale) || !as_int(a[8], bs) || !as_int(a[9], max_seq) ||
      !as_int(a[11], partition) || !as_double(a[12], k_scale) || !as_double(a[13], v_scale) || transformed())
    Py_RETURN_NONE;
  const Tensor q = THPVariable_Unpack(a[1]), kc = THPVariable_Unpack(a[2]), vc = THPVariable_Unpack(a[3]),
               bt = THPVariable_Unpack(a[4]), lens = THPVariable_Unpack(a[5]);
  const c10::Device dev = q.device();
  if (!dev.is_cuda() || !usable(q, dev) || !usable(kc, dev) || !usable(vc, dev) || !usable(bt, dev) ||
      !usable(lens, dev))
    Py_RETURN_NONE;
  Tensor slopes;
  const float* alibi = nullptr;
  if (a[10] != Py_None) {
    if (!plain(a[10])) Py_RETURN_NONE;
    slopes = THPVariable_Unpack(a[10]);
    if (!usable(slopes, dev) || slopes.scalar_type() != at::kFloat || slopes.dim() != 1 || !slopes.is_contiguous() ||
        q.dim() != 3 || slopes.size(0) != q.size(1))
      Py_RETURN_NONE;
    alibi = static_cast<const float*>(slopes.data_ptr());
  }
  if (q.dim() != 3 || !i32_contiguous(bt, 2) || !i32_contiguous(lens, 1)) Py_RETURN_NONE;
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2);
  if (B == 0 || bt.size(0) != B || lens.size(0) != B || Hkv <= 0 || Hq % Hkv != 0 || bs <= 0 || max_seq <= 0 ||
      partition < 0 || max_seq > bt.size(1) * bs)
    Py_RETURN_NONE;
  const int qc = code_of(q, false), cc = code_of(kc, true);
  if (qc < 0 || cc < 0 || vc.scalar_type() != kc.scalar_type()) Py_RETURN_NONE;
  const bool fp8 = cc == PKV_FP8_E4M3;
  if (!(qc == cc || qc == PKV_F32 || fp8) || (fp8 && !(good_scale(k_scale) && good_scale(v_scale)))) Py_RETURN_NONE;
  int32_t layout;
  int64_t khs, vhs;
  if (kc.dim() == 5 && vc.dim() == 4) {
    layout = PKV_LAYOUT_PAGED5D;
    const int64_t x = 16 / bytes_of(cc);
    if (kc.size(1) != Hkv || vc.size(1) != Hkv || kc.size(2) * x != D || kc.size(4) != x || vc.size(2) != D ||
        kc.size(0) != vc.size(0) || kc.size(3) != bs || vc.size(3) != bs || kc.stride(2) != bs * x ||
        kc.stride(3) != x || kc.stride(4) != 1 || vc.stride(2) != bs || vc.stride(3) != 1)
      Py_RETURN_NONE;
    khs = kc.stride(1);
    vhs = vc.stride(1);
  } else if (kc.dim() == 3 && vc.dim() == 3 && bs == 1 && !fp8 && cc != PKV_F32) {
    layout = PKV_LAYOUT_TOKEN_MAJOR;
    if (kc.sizes() != vc.sizes() || kc.size(1) != Hkv || kc.size(2) != D || kc.stride(1) != D || kc.stride(2) != 1 ||
        vc.stride(1) != D || vc.stride(2) != 1)
      Py_RETURN_NONE;
    khs = vhs = D;
  } else {
    Py_RETURN_NONE;
  }
  if (q.stride(2) != 1 || q.stride(1) != D || (q.stride(0) * bytes_of(qc)) % 16 != 0) Py_RETURN_NONE;
  const size_t need = pkv_paged_attention_full_workspace_size((int32_t)B, (int32_t)Hq, (int32_t)Hkv, (int32_t)D,
                                                              (int32_t)max_seq, (int32_t)partition);
  if (need == 0) Py_RETURN_NONE;
  const auto stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  // The scratch of this device and stream, kept alive by the table; a first
  // or larger need goes to the Python path, which allocates it.
  PyObject* id = Py_BuildValue("(iK)", (int)dev.index(), (unsigned long long)reinterpret_cast<uintptr_t>(stream));
  if (id == nullptr) return nullptr;
  PyObject* held = PyDict_GetItemWithError(a[0], id);  // (borrowed)
  Py_DECREF(id);
  if (held == nullptr) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  if (!plain(held)) Py_RETURN_NONE;
  const Tensor ws = THPVariable_Unpack(held);
  if (ws.scalar_type() != at::kByte || (size_t)ws.numel() < need) Py_RETURN_NONE;
  const OnDevice on(dev);
  Tensor out;
  int st;
  {
    pybind11::gil_scoped_release release;
    out = at::empty({B, Hq, D}, q.options());
    st = pkv_paged_attention(
        out.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), static_cast<const int32_t*>(bt.data_ptr()),
        static_cast<const int32_t*>(lens.data_ptr()), alibi, (int32_t)B, (int32_t)Hq, (int32_t)Hkv, (int32_t)D,
        (int32_t)bs, (int32_t)bt.size(1), (int32_t)max_seq, kc.size(0), (float)scale, q.stride(0), kc.stride(0), khs,
        vc.stride(0), vhs, layout, (int32_t)partition, ws.data_ptr(), (size_t)ws.numel(), qc, cc, (float)k_scale,
        (float)v_scale, stream);
  }
  if (st != PKV_OK) return PyLong_FromLong(st);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (stream handle) -> a number that names the HIP graph capture under way on
// the stream, 0 if there is none.
PyObject* capture_id(PyObject*, PyObject* handle) {
  HANDLE_TH_ERRORS
  const unsigned long long h = PyLong_AsUnsignedLongLong(handle);
  if (PyErr_Occurred()) return nullptr;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(reinterpret_cast<hipStream_t>((uintptr_t)h), &status, &id) != hipSuccess) {
    (void)hipGetLastError();  // the legacy stream beside another stream's capture: it captures nothing itself
    return PyLong_FromLong(0);
  }
  return PyLong_FromUnsignedLongLong(status == hipStreamCaptureStatusNone ? 0 : id + 1);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"reshape_and_cache", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(reshape_and_cache)),
     METH_FASTCALL, nullptr},
    {"paged_attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(paged_attention)), METH_FASTCALL,
     nullptr},
    {"capture_id", capture_id, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", "Append and decode calls without the Python checks.", -1,
                          methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module_def); }
