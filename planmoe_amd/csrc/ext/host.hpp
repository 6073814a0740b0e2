// What the extension's parts share: raw pointers of tensors, workspaces, errors of the C ABI.
#pragma once
#include "planmoe_hip.h"

#include <ATen/hip/HIPEvent.h>
#include <hip/hip_runtime_api.h>
#include <torch/extension.h>

#include <algorithm>
#include <stdexcept>

namespace planmoe_host {

using torch::Tensor;

// an error an entry point of libplanmoe_hip reports: PlanMoEError in Python
struct Failure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
#define PM_CALL(expr) do { if ((expr) != 0) throw ::planmoe_host::Failure(planmoe_last_error()); } while (0)

inline void *current_stream() { return (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }
inline bool pm_dtype_ok(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16 || t == at::kHalf; }
inline int pm_dtype(at::ScalarType t)
{
    TORCH_CHECK(pm_dtype_ok(t), "planmoe: unsupported dtype (float32, bfloat16 or float16)");
    return t == at::kFloat ? PLANMOE_F32 : t == at::kBFloat16 ? PLANMOE_BF16 : PLANMOE_F16;
}
inline const int32_t *ints(const Tensor &t) { return t.data_ptr<int32_t>(); }
inline const float *floats(const Tensor &t) { return t.data_ptr<float>(); }
inline void *raw(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
inline Tensor bytes(int64_t n, const Tensor &like) { return at::empty({std::max<int64_t>(n, 16)}, like.options().dtype(at::kByte)); }

} // namespace planmoe_host

void def_routing(pybind11::module_ &m);
