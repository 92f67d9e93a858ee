// Minimal tensor view and type ids for the operator layer.
//
// The reference's operator glue is written against MindSpore's ms::Tensor / TypeId
// (ops/framework/utils.h:24, ops/framework/module.h:24).  This backend has no MindSpore: a tensor is
// a device pointer plus dtype, shape and strides, handed over by the host framework (PyTorch-ROCm
// tensors are converted as an operator's arguments are read, torch_bridge.h), and `owner` keeps the framework object alive.
#ifndef MS_CUSTOM_OPS_FRAMEWORK_TENSOR_H_
#define MS_CUSTOM_OPS_FRAMEWORK_TENSOR_H_

#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <cstdint>
#include <memory>
#include <numeric>
#include <optional>
#include <string>
#include <vector>

namespace mindspore {
// Numeric values follow MindSpore's TypeId so that integer dtype arguments keep their meaning
// (quant_batch_matmul's default output_dtype is 42 == float16, quant_batch_matmul.cc:161).
enum TypeId : int {
  kTypeUnknown = 0,
  kMetaTypeNone = 9,
  kNumberTypeBool = 30,
  kNumberTypeInt8 = 32,
  kNumberTypeInt16 = 33,
  kNumberTypeInt32 = 34,
  kNumberTypeInt64 = 35,
  kNumberTypeUInt8 = 37,
  kNumberTypeUInt16 = 38,
  kNumberTypeUInt32 = 39,
  kNumberTypeUInt64 = 40,
  kNumberTypeFloat16 = 42,
  kNumberTypeFloat32 = 43,
  kNumberTypeFloat64 = 44,
  kNumberTypeBFloat16 = 45,
  kNumberTypeInt4 = 50,
};
using ShapeVector = std::vector<int64_t>;
using ShapeArray = std::vector<ShapeVector>;
using TypeIdList = std::vector<TypeId>;

inline std::string TypeIdToString(TypeId t) {
  switch (t) {
    case kMetaTypeNone: return "None";
    case kNumberTypeBool: return "Bool";
    case kNumberTypeInt8: return "Int8";
    case kNumberTypeInt16: return "Int16";
    case kNumberTypeInt32: return "Int32";
    case kNumberTypeInt64: return "Int64";
    case kNumberTypeUInt8: return "UInt8";
    case kNumberTypeUInt64: return "UInt64";
    case kNumberTypeFloat16: return "Float16";
    case kNumberTypeFloat32: return "Float32";
    case kNumberTypeFloat64: return "Float64";
    case kNumberTypeBFloat16: return "BFloat16";
    case kNumberTypeInt4: return "Int4";
    default: return "TypeId(" + std::to_string(static_cast<int>(t)) + ")";
  }
}

inline size_t TypeIdSize(TypeId t) {
  switch (t) {
    case kNumberTypeBool: case kNumberTypeInt8: case kNumberTypeUInt8: return 1;
    case kNumberTypeInt4: return 1;   // qint4x2 storage: one byte per element of the stored shape (two 4-bit values)
    case kNumberTypeInt16: case kNumberTypeUInt16: case kNumberTypeFloat16: case kNumberTypeBFloat16: return 2;
    case kNumberTypeInt32: case kNumberTypeUInt32: case kNumberTypeFloat32: return 4;
    case kNumberTypeInt64: case kNumberTypeUInt64: case kNumberTypeFloat64: return 8;
    default: return 0;
  }
}
}  // namespace mindspore

namespace ms {
using mindspore::ShapeVector;
using mindspore::TypeId;

// Copies share one description (an operator hands its tensors on several times per call).
class Tensor {
 public:
  Tensor() = default;
  Tensor(uintptr_t data, int type_id, ShapeVector shape, ShapeVector strides, pybind11::object owner)
      : d_(std::make_shared<Description>(Description{reinterpret_cast<void *>(data), static_cast<TypeId>(type_id), std::move(shape),
                                                     std::move(strides), std::move(owner)})) {}

  bool is_defined() const { return d_ != nullptr; }
  void *GetDataPtr() const { return d_ ? d_->data : nullptr; }
  TypeId data_type() const { return d_ ? d_->dtype : mindspore::kMetaTypeNone; }
  const ShapeVector &shape() const { return d_ ? d_->shape : Nothing(); }
  const ShapeVector &strides() const { return d_ ? d_->strides : Nothing(); }   // may be empty where contiguous
  pybind11::object owner() const { return d_ ? d_->owner : pybind11::object(); }
  int64_t numel() const {
    return std::accumulate(shape().begin(), shape().end(), static_cast<int64_t>(1), std::multiplies<int64_t>());
  }
  size_t nbytes() const { return static_cast<size_t>(numel()) * mindspore::TypeIdSize(data_type()); }
  bool is_contiguous() const { return strides().empty() || ContiguousStrides(shape().data(), strides().data(), shape().size()); }
  static bool ContiguousStrides(const int64_t *shape, const int64_t *strides, size_t dims) {
    int64_t expect = 1;
    for (size_t i = dims; i-- > 0;) {
      if (shape[i] != 1 && strides[i] != expect) return false;
      expect *= shape[i];
    }
    return true;
  }
  // A view on a sub-range of the same buffer (used to walk batches).
  Tensor Slice(int64_t elem_offset, ShapeVector shape) const {
    char *at = static_cast<char *>(GetDataPtr()) + elem_offset * static_cast<int64_t>(mindspore::TypeIdSize(data_type()));
    return Tensor(reinterpret_cast<uintptr_t>(at), data_type(), std::move(shape), ShapeVector(), owner());
  }

 private:
  struct Description {
    void *data;
    TypeId dtype;
    ShapeVector shape;
    ShapeVector strides;
    pybind11::object owner;
  };
  static const ShapeVector &Nothing() {
    static const ShapeVector nothing;
    return nothing;
  }
  std::shared_ptr<const Description> d_;
};
}  // namespace ms

namespace ms_custom_ops {
// A torch.Tensor or a QInt4x2 as an operator sees it.  False for None and for objects of the compiled Tensor class; a tensor that is not
// on the GPU or has a dtype without a TypeId raises, and so does anything else.
bool TensorFromObject(pybind11::handle object, ms::Tensor *tensor);
// an operator's list argument: None, or any iterable of tensors but a tensor itself
struct TensorListArg {
  bool given{false};
  std::vector<ms::Tensor> list;
};
TensorListArg TensorListFromObject(pybind11::handle object);
}  // namespace ms_custom_ops

// Operators take the host framework's tensors and return them: no Python object stands between.
namespace pybind11 {
namespace detail {
template <>
class type_caster<ms::Tensor> : public type_caster_base<ms::Tensor> {
  using Base = type_caster_base<ms::Tensor>;

 public:
  bool load(handle src, bool convert) {
    if (!ms_custom_ops::TensorFromObject(src, &local_)) return Base::load(src, convert);
    this->value = &local_;
    return true;
  }
  static handle cast(const ms::Tensor &src, return_value_policy policy, handle parent) {
    const object owner = src.owner();
    return owner && !owner.is_none() ? owner.inc_ref() : Base::cast(src, policy, parent);
  }
  static handle cast(ms::Tensor &&src, return_value_policy policy, handle parent) { return cast(static_cast<const ms::Tensor &>(src), policy == return_value_policy::move ? return_value_policy::copy : policy, parent); }
  static handle cast(const ms::Tensor *src, return_value_policy policy, handle parent) { return src ? cast(*src, policy, parent) : none().release(); }

 private:
  ms::Tensor local_;
};
template <>
class type_caster<ms_custom_ops::TensorListArg> {
 public:
  PYBIND11_TYPE_CASTER(ms_custom_ops::TensorListArg, const_name("list"));
  bool load(handle src, bool) {
    value = ms_custom_ops::TensorListFromObject(src);
    return true;
  }
  static handle cast(const ms_custom_ops::TensorListArg &src, return_value_policy policy, handle parent) {
    return src.given ? make_caster<std::vector<ms::Tensor>>::cast(src.list, policy, parent) : none().release();
  }
};
}  // namespace detail
}  // namespace pybind11
#endif  // MS_CUSTOM_OPS_FRAMEWORK_TENSOR_H_
