// bundle_make.hpp -- factories of the bundle functions per value and vector type.
#pragma once
#include <memory>
#include <vector>

#include "exec.hpp"

namespace race {

template <typename VT, typename XT>
int makeBundleOf(const race_kernel_desc& d, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out);
template <typename VT, typename XT>
int makeBundleBatchOf(const std::vector<BatchItem>& items, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out);

}  // namespace race
