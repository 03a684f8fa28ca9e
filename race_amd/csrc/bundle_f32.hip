// bundle_f32.hip -- the bundle kernels for FP32 values and vectors.
#include "bundle_exec.hpp"

namespace race {

template int makeBundleOf<float, float>(const race_kernel_desc&, const ExecContext&, std::unique_ptr<DeviceFn>*);
template int makeBundleBatchOf<float, float>(const std::vector<BatchItem>&, const ExecContext&, std::unique_ptr<DeviceFn>*);

}  // namespace race
