// The common Int8Linear call without Python between the module and the kernels: pyraquant_amd._direct.
//
//   linear(instance_dict, buffers, x) -> y, None, or a negative status of the library
//
// One call takes the place of the checks, the two allocations and the twenty-argument foreign call of
// Int8Linear._forward_direct: an eager layer of few rows (one launch) costs the host 5.0 us, 14.2 before (two launches,
// 5.5 us, and the rest Python and the foreign call). It looks its tensors up and checks them on every call, and holds them
// until the launch (the module may be given others meanwhile: by another thread while the GIL is released, or by a dispatch
// mode's Python during an allocation); nothing is kept between calls. It takes layers without a low-rank branch, whose tensors and x are plain torch tensors in the state
// the kernels read; for everything else it returns None and the Python paths decide, as they do without it. Results,
// allocations (torch's caching allocator, on the current stream) and refusals are those of the Python path.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/pyraquant_amd.h"

namespace pq {   // (pq_common.h declares them too, among device code)
bool linear_small_size(int64_t M, int64_t K, int64_t N, hipStream_t stream);
int linear_small(const void* x, int32_t x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t* w_packed,
                 const float* s_w, const float* bias, void* y, int64_t ldy, int64_t N, bool& taken, hipStream_t stream);
}

namespace {

enum Name { kWeight, kScale, kScaleGroups, kBias, kLrA, kGroup, kIn, kOut, kNames };
const char* const kNameText[kNames] = {"weight_packed", "w_scale",     "w_scale_gn",   "bias",
                                       "lr_A",          "group_size",  "in_features", "out_features"};
PyObject* g_name[kNames];

// An attribute as nn.Module resolves it: the instance's own dict first, then the registered buffers (borrowed). A name in
// neither is not None: it may be a parameter or a property, and Python decides.
PyObject* attribute(PyObject* inst, PyObject* buffers, Name n) {
  PyObject* v = PyDict_GetItemWithError(inst, g_name[n]);
  if (!v && !PyErr_Occurred()) v = PyDict_GetItemWithError(buffers, g_name[n]);
  return v;
}

bool integer(PyObject* o, int64_t& v) {
  if (!o || !PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  return !(v == -1 && PyErr_Occurred());
}

// A plain tensor on `dev` with the type, element count and contiguous storage the kernels read.
bool plain(PyObject* o, c10::ScalarType dt, int64_t numel, c10::Device dev) {
  if (!o || !THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.has_storage() && t.scalar_type() == dt && t.device() == dev && t.numel() == numel &&
         t.is_contiguous();
}

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3 || !PyDict_Check(args[0]) || !PyDict_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "linear(instance dict, buffers, x)");
    return nullptr;
  }
  PyObject *inst = args[0], *buffers = args[1];
  if (!THPVariable_CheckExact(args[2])) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(args[2]);
  PyObject* const lr = attribute(inst, buffers, kLrA);
  int64_t K, N, group;
  if (lr != Py_None || !integer(attribute(inst, buffers, kIn), K) || !integer(attribute(inst, buffers, kOut), N) ||
      !integer(attribute(inst, buffers, kGroup), group)) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  const auto dt = x.scalar_type();
  const bool bf16 = dt == at::kBFloat16;
  if ((!bf16 && dt != at::kHalf) || !x.has_storage() || !x.is_cuda() || x.dim() < 1 || x.size(-1) != K || K < 64 || N < 64 ||
      (group != 0 && group != 32))
    Py_RETURN_NONE;
  const c10::Device dev = x.device();
  PyObject* const wo = attribute(inst, buffers, kWeight);
  PyObject* const so = attribute(inst, buffers, group ? kScaleGroups : kScale);
  PyObject* const bo = attribute(inst, buffers, kBias);
  if (!plain(wo, at::kChar, (N + 15) / 16 * 16 * K, dev) || !plain(so, at::kFloat, group ? N * K / 32 : N, dev) ||
      (bo != Py_None && !plain(bo, at::kFloat, N, dev))) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  const at::Tensor weight = THPVariable_Unpack(wo), scale = THPVariable_Unpack(so);
  const at::Tensor bias = bo != Py_None ? THPVariable_Unpack(bo) : at::Tensor();
  const at::Tensor x2 = x.dim() == 2 ? x : x.reshape({-1, K});
  const int64_t M = x2.size(0), ldx = x2.stride(0);
  const void* const xp = x2.const_data_ptr();
  if (x2.stride(1) != 1 || ldx % 8 || (uintptr_t)xp % 16) Py_RETURN_NONE;

  const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  const bool small = M > 0 && group == 0 && pq::linear_small_size(M, K, N, stream);   // few rows: one kernel, no workspace
  at::Tensor ws;
  auto workspace = [&] {
    ws = at::empty({pq_int8_linear_workspace_size(M, K, 0)}, x2.options().dtype(at::kByte).requires_grad(false));
  };
  // The workspace before the output, as the Python path: call after call then takes the same workspace and gives each
  // output another block, where the other order let the codes move into the block of the last output (a layer of 3235 x
  // 640 x 1600 19.2 us that way, 17.2 this way).
  if (M > 0 && !small) workspace();
  at::Tensor y = at::empty({M, N}, x2.options().requires_grad(false));
  int st = PQ_OK;
  if (M > 0) {
    const int32_t code = bf16 ? PQ_BF16 : PQ_F16;
    const int8_t* const w = static_cast<const int8_t*>(weight.const_data_ptr());
    const float* const s = static_cast<const float*>(scale.const_data_ptr());
    const float* const b = bias.defined() ? static_cast<const float*>(bias.const_data_ptr()) : nullptr;
    void* const yp = y.data_ptr();
    bool taken = false;
    if (small) {
      Py_BEGIN_ALLOW_THREADS
      st = pq::linear_small(xp, code, M, K, ldx, w, s, b, yp, N, N, taken, stream);
      Py_END_ALLOW_THREADS
    }
    if (!taken) {
      if (!ws.defined()) workspace();   // (the one kernel's size, not its alignment)
      void* const wsp = ws.data_ptr();
      const int64_t bytes = ws.numel();
      Py_BEGIN_ALLOW_THREADS
      st = pq_int8_linear(xp, code, M, K, ldx, w, s, group, b, nullptr, nullptr, 0, nullptr, 0, yp, N, N, wsp, bytes, stream);
      Py_END_ALLOW_THREADS
    }
  }
  if (st != PQ_OK) return PyLong_FromLong(st);
  if (x.dim() != 2) {
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    y = y.reshape(shape);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(linear)), METH_FASTCALL,
     "linear(instance_dict, buffers, x): the Int8Linear call, or None where the Python paths have to decide"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_direct", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__direct() {
  for (int i = 0; i < kNames; ++i)
    if (!g_name[i] && !(g_name[i] = PyUnicode_InternFromString(kNameText[i]))) return nullptr;
  return PyModule_Create(&kModule);
}
