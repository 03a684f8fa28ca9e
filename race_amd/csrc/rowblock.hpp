// rowblock.hpp -- products over blocks of whole rows with up to 1024 entries.
//
// A workgroup loads its block's entries in CRS order, four per thread,
// gathers x, leaves values and x in LDS and sums each row with as many lanes as
// the block's row count leaves (a power of two).  Values and x, not their
// products: a row summed by one lane is then the same chain of fused multiply-
// adds as in a SELL chunk, with one rounding per entry.  With products rounded
// before the sum, rows of 5 to 7 entries had up to 18 % more error.  Rows of more than
// kLaneEntries entries a lane are summed by a whole wavefront afterwards, so
// that no lane walks a hub row alone (a graph of 200000 rows and 1.2M entries,
// hubs of 400 entries: 19.6 us without this, 11.3 us with it).  No entry is
// padding: two dependent memory levels whatever the row lengths.  In a SELL
// chunk 64 rows take as many steps as the longest of them.  A row of more than
// 1024 entries is a block of its own, summed by the whole workgroup.
//
// What bounds it: memory (nothing but the entries is read twice) and, for
// scattered columns, the address unit, which looks up one cache line per lane
// and cycle, and the 128-byte line each lane moves into L1.  SpMV on a
// Chung-Lu graph of 150000 rows and 3.0M entries in FP64: 103 us in SELL chunks,
// 19.2 us here.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "exec.hpp"
#include "exec_common.hpp"
#include "sell_common.hpp"

namespace race {

namespace {

constexpr int kRbEntries = 4 * kBlock;  // entries of a block of several rows
constexpr int kRbRows = kBlock;         // rows of a block
constexpr int kLaneEntries = 16;        // entries a lane sums alone

// 32 bytes, one scalar load
struct alignas(32) RowBlk {
    int row0;  // rows of its matrix
    uint16_t nrows, longest;  // its longest row, at most 65535
    int e0;           // first entry, in units of 4
    int ne;           // entries
    int base;         // smallest column (16-bit ids)
    int mat;          // its matrix (batches)
    int rp0;          // row pointers of its rows, at rp + rp0
    int p0;           // rp[rp0]
};

// per matrix of a batch
struct RowBlkVecs {
    const void* x;
    void* y;
    long n;
};

template <typename CT, typename VT>
struct RowBlkView {
    const RowBlk* blks;
    const int* rp;
    const CT* col;
    const VT* val;
    const RowBlkVecs* vecs;
};

template <typename VT>
struct RowBlocks {
    bool narrowIds = true;
    std::vector<RowBlk> hb;
    std::vector<int> hrp, hcol;
    std::vector<VT> hval;
    DevBuf<RowBlk> blks;
    DevBuf<int> rp, col32;
    DevBuf<uint16_t> col16;
    DevBuf<VT> val;
    int nBlk = 0;
    int cap = kRbEntries;  // entries of a block of several rows, set before add

    // rows [0, n) of one more matrix
    void add(int n, const int* R, const int* C, const double* V, int mat) {
        const int rp0 = (int)hrp.size();
        hrp.insert(hrp.end(), R, R + n + 1);
        // exactly for the first matrix, at least doubled for further ones: a
        // batch that reserves just what it needs copies all entries so far
        // with every matrix (256 matrices of 0.5M entries 102 s)
        const size_t need = hcol.size() + R[n] + R[n] / 64 + 8;
        if (need > hcol.capacity()) {
            hcol.reserve(std::max(need, 2 * hcol.capacity()));
            hval.reserve(hcol.capacity());
        }
        for (int r = 0; r < n;) {
            RowBlk k{r, 0, 0, (int)(hcol.size() / 4), 0, INT32_MAX, mat, rp0 + r, R[r]};
            while (r < n && k.nrows < kRbRows && (k.nrows == 0 || R[r + 1] - k.p0 <= cap)) {
                k.longest = (uint16_t)std::max<int>(k.longest, std::min(R[r + 1] - R[r], 65535));
                ++r;
                ++k.nrows;
                if (R[r] - k.p0 > cap) break;  // a long row, alone
            }
            k.ne = R[r] - k.p0;
            int hi = 0;
            for (int j = k.p0; j < R[r]; ++j) {
                k.base = std::min(k.base, C[j]);
                hi = std::max(hi, C[j]);
            }
            if (k.ne == 0) k.base = 0;
            narrowIds &= hi - k.base <= 65535;
            hcol.insert(hcol.end(), C + k.p0, C + R[r]);
            for (int j = k.p0; j < R[r]; ++j) hval.push_back(toStorage<VT>(V[j]));
            // the last thread's four entries: the block's smallest column,
            // value 0.  A block of empty rows has four of its own too (column
            // 0): its threads load them, and gather x of its own matrix, which
            // the entries of the next block need not (batches).
            for (int q = 0; (k.ne == 0 && q < 4) || hcol.size() % 4; ++q) {
                hcol.push_back(k.base);
                hval.push_back(VT(0));
            }
            hb.push_back(k);
        }
    }
    bool fits() const { return hcol.size() / 4 <= (size_t)INT32_MAX && hrp.size() <= (size_t)INT32_MAX; }
    int finish() {
        nBlk = (int)hb.size();
        int e;
        if (!fits()) return ERR_INVALID_ARG;
        if (narrowIds) {
            std::vector<uint16_t> h(hcol.size(), 0);
            for (const RowBlk& k : hb)
                for (int j = 0; j < (k.ne + 3) / 4 * 4; ++j)
                    h[(size_t)k.e0 * 4 + j] = (uint16_t)(hcol[(size_t)k.e0 * 4 + j] - k.base);
            if ((e = upload(col16, h.data(), h.size()))) return e;
        } else {
            for (RowBlk& k : hb) k.base = 0;
            if ((e = upload(col32, hcol.data(), hcol.size()))) return e;
        }
        if ((e = upload(blks, hb.data(), hb.size()))) return e;
        if ((e = upload(rp, hrp.data(), hrp.size()))) return e;
        if ((e = upload(val, hval.data(), hval.size()))) return e;
        hb = {};
        hrp = hcol = {};
        hval = {};
        return OK;
    }
    template <typename CT>
    RowBlkView<CT, VT> view(const RowBlkVecs* vecs) const {
        const CT* c;
        if constexpr (sizeof(CT) == 2)
            c = col16.p;
        else
            c = col32.p;
        return RowBlkView<CT, VT>{blks.p, rp.p, c, val.p, vecs};
    }
};

// Where thread t of a block of ne entries reads its four in k_rowblk, and its
// entry j in k_rowblk_packed: past the block's last the first again, which are
// not summed.
__host__ __device__ inline int firstOf4(int t, int ne) { return 4 * t < ne ? 4 * t : 0; }
__host__ __device__ inline int entryAt(int j, int ne) { return j < ne ? j : 0; }

// four consecutive entries, aligned to their size
template <typename T>
__device__ __forceinline__ void load4(const T* __restrict__ p, T (&out)[4]) {
    struct alignas(4 * sizeof(T) < 16 ? 4 * sizeof(T) : 16) P {
        T v[4];
    };
    const P a = *reinterpret_cast<const P*>(p);
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = a.v[k];
}

template <int NR, bool BATCH, typename CT, typename VT, typename XT>
__global__ void __launch_bounds__(kBlock) k_rowblk(RowBlkView<CT, VT> A, const XT* __restrict__ x0,
                                                   XT* __restrict__ y0, long n0, int nrhs, int acc) {
    __shared__ __align__(16) XT gx[NR][kRbEntries];
    __shared__ __align__(16) VT gv[kRbEntries];
    __shared__ int nHub, hub[kRbEntries / kLaneEntries];
    const int t = threadIdx.x;
    const RowBlk k = A.blks[blockIdx.x];
    const XT* __restrict__ x = x0;
    XT* __restrict__ y = y0;
    long n = n0;
    if (BATCH) {
        const RowBlkVecs v = A.vecs[k.mat];
        x = (const XT*)v.x;
        y = (XT*)v.y;
        n = v.n;
    }
    const CT* __restrict__ col = A.col + (long)k.e0 * 4;
    const VT* __restrict__ val = A.val + (long)k.e0 * 4;
    const int ne = k.ne;
    CT c[4];
    VT v[4];
    load4(col + firstOf4(t, ne), c);
    load4(val + firstOf4(t, ne), v);
    if (ne <= kRbEntries) {
        // lanes per row: the largest power of two the rows leave room for, at
        // most a wavefront
        const int lg = min(31 - __clz(kBlock / k.nrows), 6);
        const int r = t >> lg, l = t & ((1 << lg) - 1);
        const bool live = r < k.nrows;
        const int lo = live ? A.rp[k.rp0 + r] - k.p0 : 0, hi = live ? A.rp[k.rp0 + r + 1] - k.p0 : 0;
        const bool isHub = hi - lo > kLaneEntries << lg;
        const bool hubs = k.longest > kLaneEntries << lg;
        if (hubs && t == 0) nHub = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) gv[4 * t + u] = v[u];
        for (int q0 = 0; q0 < nrhs; q0 += NR) {
            XT old[NR];
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                const long vo = (long)min(q0 + q, nrhs - 1) * n;
                const XT* __restrict__ xq = x + vo;
                XT g[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) g[u] = xq[(unsigned)k.base + (unsigned)c[u]];
                old[q] = acc && live && l == 0 ? y[vo + k.row0 + r] : XT(0);
#pragma unroll
                for (int u = 0; u < 4; ++u) gx[q][4 * t + u] = g[u];
            }
            __syncthreads();
            // the hubs' rows, once; each takes more than kLaneEntries of the
            // block's entries, so the list holds them all
            if (q0 == 0 && isHub && l == 0) hub[atomicAdd(&nHub, 1)] = r;
            XT s[NR] = {};
            if (!isHub)
                for (int i = lo + l; i < hi; i += 1 << lg) {
                    const XT a = fromStorage<XT>(gv[i]);
#pragma unroll
                    for (int q = 0; q < NR; ++q) s[q] += a * gx[q][i];
                }
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                for (int o = (1 << lg) / 2; o > 0; o >>= 1) s[q] += __shfl_xor(s[q], o);
                if (live && !isHub && l == 0 && q0 + q < nrhs) y[(long)(q0 + q) * n + k.row0 + r] = old[q] + s[q];
            }
            if (hubs || q0 + NR < nrhs) __syncthreads();
            if (hubs) {
                for (int h = t >> 6; h < nHub; h += kBlock / 64) {
                    const int hr = hub[h], h0 = A.rp[k.rp0 + hr] - k.p0, h1 = A.rp[k.rp0 + hr + 1] - k.p0;
#pragma unroll
                    for (int q = 0; q < NR; ++q) {
                        XT s = XT(0);
                        for (int i = h0 + (t & 63); i < h1; i += 64) s += fromStorage<XT>(gv[i]) * gx[q][i];
                        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
                        if ((t & 63) == 0 && q0 + q < nrhs) {
                            const long at = (long)(q0 + q) * n + k.row0 + hr;
                            y[at] = acc ? y[at] + s : s;
                        }
                    }
                }
                if (q0 + NR < nrhs) __syncthreads();
            }
        }
    } else {
        for (int q = 0; q < nrhs; ++q) {
            const XT* __restrict__ xq = x + (long)q * n;
            XT s = XT(0);
            for (int j = 4 * t; j < ne; j += kRbEntries) {
                CT cc[4];
                VT vv[4];
                load4(col + j, cc);
                load4(val + j, vv);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (j + u < ne) s += fromStorage<XT>(vv[u]) * xq[(unsigned)k.base + (unsigned)cc[u]];
            }
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
            if ((t & 63) == 0) gx[0][t >> 6] = s;
            __syncthreads();
            if (t == 0) {
                for (int w = 1; w < kBlock / 64; ++w) s += gx[0][w];
                const long at = (long)q * n + k.row0;
                y[at] = acc ? y[at] + s : s;
            }
            __syncthreads();
        }
    }
}

__device__ __forceinline__ float fmaOf(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaOf(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The R values of one row of packed right-hand sides (k_pack_rhs).
template <int R, typename XT>
__device__ __forceinline__ void loadRow(const XT* __restrict__ p, XT (&out)[R]) {
    constexpr int B = R * (int)sizeof(XT), V = B < 16 ? R : 16 / (int)sizeof(XT);
    struct alignas(V * sizeof(XT)) P {
        XT v[V];
    };
#pragma unroll
    for (int s = 0; s < R / V; ++s) {
        const P a = reinterpret_cast<const P*>(p)[s];
#pragma unroll
        for (int k = 0; k < V; ++k) out[s * V + k] = a.v[k];
    }
}

// Right-hand sides q0 .. q0 + R - 1 (zeros past the last), row by row.  An
// entry's R values of x are then R * sizeof(XT) consecutive bytes instead of R
// separate cache lines.
template <int R, typename XT>
__global__ void __launch_bounds__(kBlock) k_pack_rhs(const XT* __restrict__ x, XT* __restrict__ packed, long n,
                                                     int nrhs) {
    const long r = (long)blockIdx.x * kBlock + threadIdx.x;
    const int q0 = (int)blockIdx.y * R;
    if (r >= n) return;
    XT v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = q0 + q < nrhs ? x[(long)(q0 + q) * n + r] : XT(0);
    constexpr int V = R * sizeof(XT) < 16 ? R : 16 / (int)sizeof(XT);
    struct alignas(V * sizeof(XT)) P {
        XT v[V];
    };
    P* o = reinterpret_cast<P*>(packed + ((long)blockIdx.y * n + r) * R);
#pragma unroll
    for (int s = 0; s < R / V; ++s) {
        P a;
#pragma unroll
        for (int k = 0; k < V; ++k) a.v[k] = v[s * V + k];
        o[s] = a;
    }
}

// k_rowblk over packed right-hand sides, R per blockIdx.y.  Entries go to the
// threads one by one (t, t + 256, ...), so that the rows of x of neighbouring
// lanes are neighbours in LDS.  Blocks of kPackedEntries take 20 KB of LDS at most.
constexpr int kPackedEntries = 2 * kBlock;
constexpr int kPackedLaneEntries = 64;  // with fewer lanes per row than k_rowblk, and up to eight entries in flight
template <int R, typename CT, typename VT, typename XT>
__global__ void __launch_bounds__(kBlock) k_rowblk_packed(RowBlkView<CT, VT> A, const XT* __restrict__ packed,
                                                          XT* __restrict__ y, long n, int nrhs, int acc) {
    __shared__ __align__(16) XT gx[kPackedEntries * R];
    __shared__ __align__(16) VT gv[kPackedEntries];
    __shared__ int nHub, hub[kPackedEntries / kPackedLaneEntries];
    const int t = threadIdx.x;
    const RowBlk k = A.blks[blockIdx.x];
    const int q0 = (int)blockIdx.y * R, q = t % R, slot = t / R;
    const XT* __restrict__ x = packed + ((long)blockIdx.y * n + k.base) * R;
    const CT* __restrict__ col = A.col + (long)k.e0 * 4;
    const VT* __restrict__ val = A.val + (long)k.e0 * 4;
    const int ne = k.ne;
    auto put = [&](int at, const XT (&v)[R]) {
#pragma unroll
        for (int u = 0; u < R; ++u) gx[at * R + u] = v[u];
    };
    if (ne <= kPackedEntries) {
        constexpr int N = kPackedEntries / kBlock;
        CT c[N];
        VT v[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int j = entryAt(t + u * kBlock, ne);
            c[u] = col[j];
            v[u] = val[j];
        }
        XT g[N][R];
#pragma unroll
        for (int u = 0; u < N; ++u) loadRow<R>(x + (long)(unsigned)c[u] * R, g[u]);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            gv[t + u * kBlock] = v[u];
            put(t + u * kBlock, g[u]);
        }
        if (t == 0) nHub = 0;
        __syncthreads();
        // slots of R lanes; as many slots per row as the rows leave, inside
        // one wavefront
        constexpr int S = kBlock / R, W = 64 / R;
        const int lg = min(31 - __clz(max(1, S / k.nrows)), 31 - __clz(W));
        const int l = slot & ((1 << lg) - 1);
        for (int r0 = 0; r0 < k.nrows; r0 += S >> lg) {
            const int r = r0 + (slot >> lg);
            const bool live = r < k.nrows;
            const int lo = live ? A.rp[k.rp0 + r] - k.p0 : 0, hi = live ? A.rp[k.rp0 + r + 1] - k.p0 : 0;
            const bool isHub = hi - lo > kPackedLaneEntries << lg;
            if (isHub && l == 0 && q == 0) hub[atomicAdd(&nHub, 1)] = r;
            const long at = (long)(q0 + q) * n + k.row0 + r;
            const bool store = live && !isHub && l == 0 && q0 + q < nrhs;
            const XT old = acc && store ? y[at] : XT(0);
            // Rows of less than 8 entries a lane are one chain of fused
            // multiply-adds, longer ones sums of pairs, which err less (rows of
            // 17 entries on average in FP32: 1.2e-7 as one chain, 7.8e-8 so).
            XT s = XT(0);
            const int step = 1 << lg, end = isHub ? 0 : hi;
            int i = lo + l;
            auto pairs = [&](const XT* a, const XT* c4) {
                return fmaOf(a[1], c4[1], a[0] * c4[0]) + fmaOf(a[3], c4[3], a[2] * c4[2]);
            };
            auto load = [&](auto& a, auto& c4) {
                constexpr int N = sizeof(a) / sizeof(XT);
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    a[u] = fromStorage<XT>(gv[i + u * step]);
                    c4[u] = gx[(i + u * step) * R + q];
                }
                i += N * step;
            };
            const bool deep = i + 7 * step < end;
            while (i + 7 * step < end) {
                XT a[8], c4[8];
                load(a, c4);
                s += pairs(a, c4) + pairs(a + 4, c4 + 4);
            }
            if (i + 3 * step < end) {
                XT a[4], c4[4];
                load(a, c4);
                if (deep)
                    s += pairs(a, c4);
                else
#pragma unroll
                    for (int u = 0; u < 4; ++u) s = fmaOf(a[u], c4[u], s);
            }
            for (; i < end; i += step) s = fmaOf(fromStorage<XT>(gv[i]), gx[i * R + q], s);
            for (int o = (1 << lg) / 2; o > 0; o >>= 1) s += __shfl_xor(s, o * R);
            if (store) y[at] = old + s;
        }
        if (k.longest <= kPackedLaneEntries) return;
        __syncthreads();
        for (int h = t >> 6; h < nHub; h += kBlock / 64) {
            const int hr = hub[h], h0 = A.rp[k.rp0 + hr] - k.p0, h1 = A.rp[k.rp0 + hr + 1] - k.p0;
            XT s = XT(0);
            for (int i = h0 + (t & 63) / R; i < h1; i += W) s += fromStorage<XT>(gv[i]) * gx[i * R + q];
            for (int o = W / 2; o > 0; o >>= 1) s += __shfl_xor(s, o * R);
            if ((t & 63) < R && q0 + q < nrhs) {
                const long at = (long)(q0 + q) * n + k.row0 + hr;
                y[at] = acc ? y[at] + s : s;
            }
        }
    } else {
        XT s[R] = {};
        for (int j = t; j < ne; j += kBlock) {
            XT g[R];
            loadRow<R>(x + (long)(unsigned)col[j] * R, g);
            const XT v = fromStorage<XT>(val[j]);
#pragma unroll
            for (int u = 0; u < R; ++u) s[u] += v * g[u];
        }
        put(t, s);
        __syncthreads();
        for (int o = kBlock / 2; o > 0; o >>= 1) {
            for (int i = t; i < o * R; i += kBlock) gx[i] += gx[i + o * R];
            __syncthreads();
        }
        if (t < R && q0 + t < nrhs) {
            const long at = (long)(q0 + t) * n + k.row0;
            y[at] = acc ? y[at] + gx[t] : gx[t];
        }
    }
}

template <int R, typename VT, typename XT>
void launchRowBlkPacked(const RowBlocks<VT>& A, const XT* packed, XT* y, long n, int nrhs, bool acc, hipStream_t st) {
    const dim3 grid(A.nBlk, (nrhs + R - 1) / R);
    if (A.narrowIds)
        hipLaunchKernelGGL((k_rowblk_packed<R, uint16_t, VT, XT>), grid, dim3(kBlock), 0, st,
                           A.template view<uint16_t>(nullptr), packed, y, n, nrhs, (int)acc);
    else
        hipLaunchKernelGGL((k_rowblk_packed<R, int, VT, XT>), grid, dim3(kBlock), 0, st, A.template view<int>(nullptr),
                           packed, y, n, nrhs, (int)acc);
}

// one launch over all blocks.  Right-hand sides share a pass over the entries
// in blocks of 1, 2, 4 or 8, as many as 40 KB of LDS hold beside the values
// (three workgroups per CU in FP64, four in FP32).
template <int NR, bool BATCH, typename VT, typename XT>
void launchRowBlkNr(const RowBlocks<VT>& A, const RowBlkVecs* vecs, const void* x, void* y, long n, int nrhs, bool acc,
                    hipStream_t st) {
    if (A.narrowIds)
        hipLaunchKernelGGL((k_rowblk<NR, BATCH, uint16_t, VT, XT>), dim3(A.nBlk), dim3(kBlock), 0, st,
                           A.template view<uint16_t>(vecs), (const XT*)x, (XT*)y, n, nrhs, (int)acc);
    else
        hipLaunchKernelGGL((k_rowblk<NR, BATCH, int, VT, XT>), dim3(A.nBlk), dim3(kBlock), 0, st,
                           A.template view<int>(vecs), (const XT*)x, (XT*)y, n, nrhs, (int)acc);
}
template <bool BATCH, typename VT, typename XT>
void launchRowBlk(const RowBlocks<VT>& A, const RowBlkVecs* vecs, const void* x, void* y, long n, int nrhs, bool acc,
                  hipStream_t st) {
    if (nrhs == 1)
        launchRowBlkNr<1, BATCH, VT, XT>(A, vecs, x, y, n, nrhs, acc, st);
    else if (nrhs == 2)
        launchRowBlkNr<2, BATCH, VT, XT>(A, vecs, x, y, n, nrhs, acc, st);
    else if (sizeof(XT) == 8 || nrhs <= 4 || (nrhs > 8 && nrhs % 8 >= 1 && nrhs % 8 <= 4))
        launchRowBlkNr<4, BATCH, VT, XT>(A, vecs, x, y, n, nrhs, acc, st);
    else
        launchRowBlkNr<sizeof(XT) == 8 ? 4 : 8, BATCH, VT, XT>(A, vecs, x, y, n, nrhs, acc, st);
}

}  // namespace

}  // namespace race
