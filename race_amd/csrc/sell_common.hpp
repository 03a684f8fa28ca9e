// sell_common.hpp -- value storage of the row-parallel products.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "exec_common.hpp"

namespace race {

namespace {

// matrix value storage (double, float, or bfloat16 bits); the arithmetic
// runs in the vector type XT: FP64, or FP32 accumulation for FP32 / BF16
template <typename VT>
VT toStorage(double v) {
    if constexpr (sizeof(VT) == 2)
        return toBf16(v);
    else
        return (VT)v;
}
template <typename XT>
__device__ __forceinline__ XT fromStorage(double v) {
    return (XT)v;
}
template <typename XT>
__device__ __forceinline__ XT fromStorage(float v) {
    return (XT)v;
}
template <typename XT>
__device__ __forceinline__ XT fromStorage(uint16_t v) {
    return (XT)__uint_as_float((unsigned)v << 16);
}

}  // namespace

}  // namespace race
