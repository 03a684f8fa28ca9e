// bundle_f64.hip -- the bundle kernels for FP64 values and vectors.
#include "bundle_exec.hpp"

namespace race {

template int makeBundleOf<double, double>(const race_kernel_desc&, const ExecContext&, std::unique_ptr<DeviceFn>*);
template int makeBundleBatchOf<double, double>(const std::vector<BatchItem>&, const ExecContext&, std::unique_ptr<DeviceFn>*);

}  // namespace race
