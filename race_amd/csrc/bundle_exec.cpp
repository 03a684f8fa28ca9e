// bundle_exec.cpp -- the bundle functions by precision.
#include "bundle_make.hpp"

namespace race {

int makeBundleBatchFn(const std::vector<BatchItem>& items, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    if (items.empty()) return ERR_INVALID_ARG;
    if (ctx.bundleThreads != 64 && ctx.bundleThreads != 128 && ctx.bundleThreads != 256 && ctx.bundleThreads != 512 &&
        ctx.bundleThreads != 1024)
        return ERR_INVALID_ARG;
    const race_kernel_desc& d0 = items[0].d;
    for (const BatchItem& it : items)
        if (it.d.kind != d0.kind || it.d.val_precision != d0.val_precision ||
            it.d.vec_precision != d0.vec_precision || it.d.nrhs != d0.nrhs || !it.fwd || !it.rev)
            return ERR_INVALID_ARG;
    if (d0.kind != RACE_K_GS && d0.kind != RACE_K_KACZ) return ERR_INVALID_ARG;
    if (d0.vec_precision == RACE_FP64) {
        if (d0.val_precision != RACE_FP64) return ERR_NOT_IMPLEMENTED;
        return makeBundleBatchOf<double, double>(items, ctx, out);
    }
    if (d0.val_precision == RACE_BF16) return makeBundleBatchOf<uint16_t, float>(items, ctx, out);
    return makeBundleBatchOf<float, float>(items, ctx, out);
}

int makeBundleFn(const race_kernel_desc& d, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    if (ctx.bundleThreads != 64 && ctx.bundleThreads != 128 && ctx.bundleThreads != 256 && ctx.bundleThreads != 512 &&
        ctx.bundleThreads != 1024)
        return ERR_INVALID_ARG;
    if (d.vec_precision == RACE_FP64) {
        if (d.val_precision != RACE_FP64) return ERR_NOT_IMPLEMENTED;
        return makeBundleOf<double, double>(d, ctx, out);
    }
    if (d.val_precision == RACE_BF16) return makeBundleOf<uint16_t, float>(d, ctx, out);
    return makeBundleOf<float, float>(d, ctx, out);
}

}  // namespace race
