// What the translation units of the PyTorch C++ binding share: operand checks with the reference's messages, status codes
// as exceptions, torch's current stream.  Host C++ only.
#pragma once
#include <torch/extension.h>
// torch's ROCm build presents its devices under the device type "cuda": the guard and stream types that know this
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <string>
#include <vector>

#include "managan_hip.h"

namespace mgt {

inline void check_input(const at::Tensor& t, const char* name, at::ScalarType dtype = at::kFloat) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == dtype, "expected scalar type ", c10::toString(dtype), " but found ",
                c10::toString(t.scalar_type()), " for ", name);
}

// a non-zero status as the exception the reference would raise (the same texts as the ctypes route)
inline void check(int status) {
    if (status == MG_OK) return;
    TORCH_CHECK(status != MG_ERR_BOX_TOO_SMALL, "box dimension must be greater than 3*cutoff");
    const char* text = mg_last_error();
    TORCH_CHECK(false, mg_status_string(status), text[0] ? ": " : "", text);
}

inline mg_stream_t stream_of(const at::Tensor& t) {
    return reinterpret_cast<mg_stream_t>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream());
}

inline const float* fp(const at::Tensor& t) { return t.data_ptr<float>(); }
inline float* fp(at::Tensor& t) { return t.data_ptr<float>(); }
using OptTensor = c10::optional<at::Tensor>;
inline const float* fp(const OptTensor& t) { return t.has_value() ? t->data_ptr<float>() : nullptr; }
inline bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

}  // namespace mgt

// the functions of torch_ops.cpp
void register_ops(pybind11::module_& m);
