// exec_common.hpp -- helpers shared by the kernel files.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <vector>

#include "engine.hpp"
#include "hip_util.hpp"

namespace race {

constexpr int kBlock = 256;
constexpr size_t kMaxLds = 64 * 1024;  // LDS bytes of a workgroup that shares its CU

template <int W>
__device__ __forceinline__ double groupSum(double v) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, W);
    return v;
}

// bfloat16 bits of v (through float, round to nearest even)
inline uint16_t toBf16(double v) {
    float f = (float)v;
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// Which of a function's `sets` of scratch memory a launch on a stream may use:
// launches of one function on different streams may overlap, so each of the
// first streams gets a set of its own, for good: to learn when a stream's last
// launch has ended, so that another may take its set, an event would have to be
// recorded after each (Gauss-Seidel 27-point 14^3: 81.5 us a step, 87.5 so).  -1
// (run without scratch) for further streams, for the streams whose handle stands
// for several, and while the stream is captured (a graph may be replayed
// anywhere).  A caller destroys a stream after its launches have ended: the handle
// of the next one may be the same.
class StreamSets {
  public:
    int find(hipStream_t st, int sets) {
        if (st == nullptr || st == hipStreamLegacy || st == hipStreamPerThread) return -1;
        hipStreamCaptureStatus cap;
        if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return -1;
        std::lock_guard<std::mutex> g(lock);
        const auto at = std::find(owner.begin(), owner.end(), st);
        if (at != owner.end()) return (int)(at - owner.begin());
        if ((int)owner.size() >= sets) return -1;
        owner.push_back(st);
        return (int)owner.size() - 1;
    }

  private:
    std::mutex lock;
    std::vector<hipStream_t> owner;
};

inline unsigned gridFor(long n, int block = kBlock) {
    long g = (n + block - 1) / block;
    return (unsigned)(g < 1 ? 1 : g);
}

template <typename T>
int upload(DevBuf<T>& d, const T* h, size_t n) {
    RACE_HIP(d.reserve(n));
    if (n) RACE_HIP(hipMemcpy(d.p, h, n * sizeof(T), hipMemcpyHostToDevice));
    return OK;
}

// lanes per row from the mean row length (row-parallel CRS kernels)
inline int pickTpr(long nnz, int n) {
    double m = n ? (double)nnz / n : 1;
    if (m <= 6) return 4;
    if (m <= 12) return 8;
    if (m <= 24) return 16;
    return 32;
}

}  // namespace race
