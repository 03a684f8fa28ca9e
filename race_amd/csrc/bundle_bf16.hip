// bundle_bf16.hip -- the bundle kernels for BF16 values, FP32 vectors.
#include "bundle_exec.hpp"

namespace race {

template int makeBundleOf<uint16_t, float>(const race_kernel_desc&, const ExecContext&, std::unique_ptr<DeviceFn>*);
template int makeBundleBatchOf<uint16_t, float>(const std::vector<BatchItem>&, const ExecContext&, std::unique_ptr<DeviceFn>*);

}  // namespace race
