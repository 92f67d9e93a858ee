#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include "ops/framework/torch_bridge.h"

namespace ms_custom_ops {
namespace {
struct TypePair {
  int type_id;
  at::ScalarType scalar;
};
// the numeric values of MindSpore's TypeId (tensor.h)
constexpr TypePair kTypes[] = {{30, at::kBool}, {32, at::kChar},   {33, at::kShort},  {34, at::kInt},    {35, at::kLong},  {37, at::kByte},
                               {40, at::kUInt64}, {42, at::kHalf}, {43, at::kFloat}, {44, at::kDouble}, {45, at::kBFloat16}};
}  // namespace

int ViewTorchTensor(PyObject *object, TorchTensorView *view) {
  if (!THPVariable_Check(object)) return 0;
  HANDLE_TH_ERRORS
  const at::Tensor &t = THPVariable_Unpack(object);
  view->on_gpu = t.is_cuda();
  view->type_id = 0;
  for (const TypePair &p : kTypes)
    if (p.scalar == t.scalar_type()) view->type_id = p.type_id;
  const auto sizes = t.sizes(), strides = t.strides();
  view->dims = sizes.size();
  view->sizes = sizes.data();
  view->strides = strides.data();
  view->data = view->on_gpu ? t.data_ptr() : nullptr;
  return 1;
  END_HANDLE_TH_ERRORS_RET(-1)
}

PyObject *NewTorchTensor(int type_id, const int64_t *sizes, size_t dims, void **data) {
  HANDLE_TH_ERRORS
  at::ScalarType scalar = at::kByte;
  bool known = false;
  for (const TypePair &p : kTypes)
    if (p.type_id == type_id) {
      scalar = p.scalar;
      known = true;
    }
  TORCH_CHECK(known, "no torch dtype for TypeId ", type_id);
  at::Tensor t = at::empty(at::IntArrayRef(sizes, dims), at::TensorOptions().dtype(scalar).device(at::kCUDA));
  *data = t.data_ptr();
  return THPVariable_Wrap(std::move(t));
  END_HANDLE_TH_ERRORS
}

int CurrentTorchDevice() {
  HANDLE_TH_ERRORS
  return static_cast<int>(c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index());
  END_HANDLE_TH_ERRORS_RET(-1)
}
}  // namespace ms_custom_ops
