// sell.hip -- SELL-C matrices for the row-parallel kernels: SpMV, SymmSpMV,
// SpMTV, the refinement's residual and the matrix powers (MPK).
//
// A chunk is 64 consecutive rows, one wavefront, one row per lane.  Rows keep
// their order (sigma = 1): RACE's level order keeps the x entries of a chunk
// close.  The entries of a chunk are cut into blocks of 8 entries per row and
// one last block each of 4, 2 and 1 (the binary digits of width % 8); inside a
// block a lane's entries are packed so that it reads them 16 bytes at a time
// (packPos).  Column ids are 16-bit offsets from the smallest column of their
// slot (entry position j of the chunk), whose 32-bit base comes through the
// scalar unit; matrices with a slot wider than 65535 columns keep 32-bit ids.
//
// What bounds these kernels is memory: per entry a value and a column id, per
// row its x and y.  One 64-lane load instruction costs the address unit 16
// cycles whatever its width, so with 2-byte and 4-byte loads per entry the
// 27-point BF16 product (81 loads per row) was bound by that unit and not by
// its bytes.  Measured against one 4-byte column id and one value load per
// entry (both on the same matrices): SpMTV 27-point 96^3 BF16 30.6 -> 21.6 us,
// SpMV 27-point 96^3 FP64 51.0 -> 38.4 us, 8 right-hand sides 524 -> 135 us
// (the entries were read once per right-hand side), 7-point 192^3 FP64 130.2 ->
// 116.9 us (106 without the loop over full blocks), SymmSpMV 7-point 64^3 FP64 6.9 -> 6.5 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <functional>
#include <type_traits>

#include "exec.hpp"
#include "exec_common.hpp"
#include "parallel.hpp"
#include "rowblock.hpp"
#include "sell_common.hpp"

namespace race {

namespace {

constexpr int kC = 64;               // rows per chunk (one wavefront)
constexpr int kWavesPerBlock = kBlock / kC;

// A block of E entries per lane of elements T: a lane reads V of them at once
template <typename T>
constexpr int packWidth(int E) {
    return E * (int)sizeof(T) <= 16 ? E : 16 / (int)sizeof(T);
}
template <typename T>
__host__ __device__ inline int packPos(int E, int e, int lane) {
    const int V = packWidth<T>(E);
    return (e / V) * kC * V + lane * V + e % V;
}
// entry j of a chunk of width W: the block's first entry and its size
__host__ __device__ inline void blockOf(int W, int j, int& j0, int& E) {
    const int full = W & ~7;
    if (j < full) {
        j0 = j & ~7;
        E = 8;
        return;
    }
    j0 = full;
    E = W & 4;
    if (E == 0 || j >= j0 + 4) {
        j0 += E;
        E = W & 2;
        if (E == 0 || j >= j0 + 2) {
            j0 += E;
            E = 1;
        }
    }
}

struct SellChunk {
    int width, off64;  // entry offset in units of 64
};

// what a kernel needs of a SELL matrix
template <typename CT, typename VT>
struct SellView {
    const SellChunk* chunks;
    const int* base;      // smallest column of every slot (CT uint16_t), at off64 + j
    const CT* col;
    const VT* val;
    const uint8_t* pad;   // per row: chunk width - row length, or null:
    const int* rowPtr;    // then the row length from the row pointers
    int n, nChunk, W;     // W >= 0: every chunk has this width
};

template <typename VT>
struct SellMatrix {
    int n = 0, nChunk = 0;
    int uniformW = -1;          // >= 0: every chunk has this width, chunk c at c * 64 * width
    bool narrowIds = false;     // 16-bit column ids
    int perPass = 8;            // right-hand sides per pass, at most
    long bytes = 0;             // stored entries
    DevBuf<SellChunk> chunks;
    DevBuf<int> base, rowPtr;
    DevBuf<uint16_t> col16;
    DevBuf<int> col32;
    DevBuf<VT> val;
    DevBuf<uint8_t> pad;

    template <typename CT>
    SellView<CT, VT> view() const {
        const CT* c;
        if constexpr (sizeof(CT) == 2)
            c = col16.p;
        else
            c = col32.p;
        return SellView<CT, VT>{chunks.p, base.p, c, val.p, pad.n ? pad.p : nullptr, rowPtr.p, n, nChunk, uniformW};
    }

    // With chunk widths close to each other (padding every chunk to the
    // widest adds at most 1/8), all chunks get the widest width: the kernels
    // then compute a chunk's place instead of loading it.
    int build(const race_kernel_desc& d) {
        n = d.nrow;
        const int* rp = d.rowPtr;
        nChunk = (n + kC - 1) / kC;
        std::vector<SellChunk> ch(nChunk);
        long total = 0;
        int wmax = 0;
        for (int c = 0; c < nChunk; ++c) {
            int w = 0;
            for (int r = c * kC; r < std::min(n, (c + 1) * kC); ++r) w = std::max(w, rp[r + 1] - rp[r]);
            ch[c] = SellChunk{w, (int)total};
            total += w;
            wmax = std::max(wmax, w);
        }
        uniformW = -1;
        if ((long)wmax * nChunk * 8 <= total * 9) {
            uniformW = wmax;
            for (int c = 0; c < nChunk; ++c) ch[c] = SellChunk{wmax, (int)std::min<long>((long)c * wmax, INT32_MAX)};
            total = (long)wmax * nChunk;
        }
        if (total > (long)INT32_MAX) return ERR_INVALID_ARG;  // offsets in units of 64 must fit an int
        // per slot its smallest column; 16-bit ids if no slot spans more
        std::vector<int> lo((size_t)total, 0);
        std::vector<uint8_t> pd((size_t)nChunk * kC, 0);
        std::vector<char> wide(nChunk, 0), deep(nChunk, 0);
        parallelRanges(nChunk, 256, [&](int c0, int c1) {
            std::vector<int> hi;
            for (int c = c0; c < c1; ++c) {
                const int w = ch[c].width;
                int* l = lo.data() + ch[c].off64;
                std::fill(l, l + w, INT32_MAX);
                hi.assign(w, -1);
                for (int i = 0; i < kC && c * kC + i < n; ++i) {
                    const int r = c * kC + i, len = rp[r + 1] - rp[r];
                    for (int j = 0; j < len; ++j) {
                        l[j] = std::min(l[j], d.col[rp[r] + j]);
                        hi[j] = std::max(hi[j], d.col[rp[r] + j]);
                    }
                    if (w - len > 255) deep[c] = 1;
                    pd[(size_t)c * kC + i] = (uint8_t)std::min(w - len, 255);
                }
                for (int j = 0; j < w; ++j) {
                    if (hi[j] < 0) l[j] = 0;  // no row reaches this slot (uniform widths)
                    if (hi[j] - l[j] > 65535) wide[c] = 1;
                }
            }
        });
        narrowIds = std::find(wide.begin(), wide.end(), 1) == wide.end();
        bytes = total * kC * (long)((narrowIds ? sizeof(uint16_t) : sizeof(int)) + sizeof(VT));
        const bool shallow = std::find(deep.begin(), deep.end(), 1) == deep.end();
        std::vector<uint16_t> h16(narrowIds ? (size_t)total * kC : 0);
        std::vector<int> h32(narrowIds ? 0 : (size_t)total * kC);
        std::vector<VT> hv((size_t)total * kC);
        parallelRanges(nChunk, 256, [&](int c0, int c1) {
            for (int c = c0; c < c1; ++c) {
                const int w = ch[c].width;
                for (int j = 0; j < w; ++j) {
                    int j0, E;
                    blockOf(w, j, j0, E);
                    const size_t at = (size_t)(ch[c].off64 + j0) * kC;
                    const int l = lo[ch[c].off64 + j];
                    for (int i = 0; i < kC; ++i) {
                        const int r = c * kC + i;
                        const bool live = r < n && j < rp[r + 1] - rp[r];
                        const int col = live ? d.col[rp[r] + j] : l;
                        if (narrowIds)
                            h16[at + packPos<uint16_t>(E, j - j0, i)] = (uint16_t)(col - l);
                        else
                            h32[at + packPos<int>(E, j - j0, i)] = col;
                        hv[at + packPos<VT>(E, j - j0, i)] = live ? toStorage<VT>(d.val[rp[r] + j]) : VT(0);
                    }
                }
            }
        });
        int e;
        if ((e = upload(chunks, ch.data(), ch.size()))) return e;
        if (narrowIds && (e = upload(base, lo.data(), lo.size()))) return e;
        if (narrowIds && (e = upload(col16, h16.data(), h16.size()))) return e;
        if (!narrowIds && (e = upload(col32, h32.data(), h32.size()))) return e;
        if (shallow && (e = upload(pad, pd.data(), pd.size()))) return e;
        if (!shallow && (e = upload(rowPtr, rp, (size_t)n + 1))) return e;
        return upload(val, hv.data(), hv.size());
    }
};

// E consecutive entries of every lane of a block (NT: with non-temporal loads)
template <int E, bool NT, typename T>
__device__ __forceinline__ void loadPack(const T* __restrict__ p, int lane, T (&out)[E]) {
    constexpr int V = packWidth<T>(E), B = V * (int)sizeof(T);
    typedef unsigned W4 __attribute__((ext_vector_type(4)));
    using P = std::conditional_t<B == 16, W4,
                                 std::conditional_t<B == 8, uint64_t, std::conditional_t<B == 4, uint32_t, uint16_t>>>;
    const P* __restrict__ q = reinterpret_cast<const P*>(p) + lane;
#pragma unroll
    for (int s = 0; s < E / V; ++s) {
        const P a = NT ? __builtin_nontemporal_load(q + s * kC) : q[s * kC];
        __builtin_memcpy(out + s * V, &a, B);
    }
}

// t[q] += the products of one block with NR right-hand sides (x[q] their
// vectors).  Entries past the row's length multiply 0 by 0: a padding entry
// never brings an x that the row does not have into its sum.
template <int E, int NR, typename CT, typename VT, typename XT>
__device__ __forceinline__ void sellBlock(const CT (&c)[E], const VT (&v)[E], const int* __restrict__ base, int left,
                                          const XT* const (&x)[NR], XT (&t)[NR]) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        XT g[E];
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = x[q][sizeof(CT) == 2 ? (unsigned)base[e] + (unsigned)c[e] : (unsigned)c[e]];
#pragma unroll
        for (int e = 0; e < E; ++e) t[q] += fromStorage<XT>(v[e]) * (e < left ? g[e] : XT(0));
    }
}

// the row sums of one chunk for NR right-hand sides; sequential in the
// row's entries, as the CRS row order.  The entries of the last blocks are
// requested first, those of each full block while the x entries of the one
// before it arrive.
template <int NR, bool NT, bool SHORT, typename CT, typename VT, typename XT>
__device__ __forceinline__ void sellRow(const SellView<CT, VT>& A, int c, int lane, const XT* const (&x)[NR],
                                        XT (&t)[NR]) {
    int W = A.W;
    long s0 = (long)c * W;  // first slot
    if (W < 0) {
        const SellChunk k = A.chunks[c];
        W = __builtin_amdgcn_readfirstlane(k.width);
        s0 = __builtin_amdgcn_readfirstlane(k.off64);
    }
    const int r = c * kC + lane;
    const int len = A.pad ? W - (int)A.pad[r] : r < A.n ? A.rowPtr[r + 1] - A.rowPtr[r] : 0;
    const CT* __restrict__ col = A.col + s0 * kC;
    const VT* __restrict__ val = A.val + s0 * kC;
    const int* __restrict__ base = A.base + (sizeof(CT) == 2 ? s0 : 0);
    const int full = SHORT ? 0 : W & ~7, at2 = full + (W & 4), at1 = at2 + (W & 2);
    CT c4[4], c2[2], c1[1];
    VT v4[4], v2[2], v1[1];
    if (W & 4) {
        loadPack<4, NT>(col + (long)full * kC, lane, c4);
        loadPack<4, NT>(val + (long)full * kC, lane, v4);
    }
    if (W & 2) {
        loadPack<2, NT>(col + (long)at2 * kC, lane, c2);
        loadPack<2, NT>(val + (long)at2 * kC, lane, v2);
    }
    if (W & 1) {
        loadPack<1, NT>(col + (long)at1 * kC, lane, c1);
        loadPack<1, NT>(val + (long)at1 * kC, lane, v1);
    }
    if (full) {
        CT c8[8];
        VT v8[8];
        loadPack<8, NT>(col, lane, c8);
        loadPack<8, NT>(val, lane, v8);
        for (int j = 0; j < full; j += 8) {
            CT cn[8] = {};
            VT vn[8] = {};
            if (j + 8 < full) {
                loadPack<8, NT>(col + (long)(j + 8) * kC, lane, cn);
                loadPack<8, NT>(val + (long)(j + 8) * kC, lane, vn);
            }
            sellBlock<8, NR>(c8, v8, base + j, len - j, x, t);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                c8[e] = cn[e];
                v8[e] = vn[e];
            }
        }
    }
    if (W & 4) sellBlock<4, NR>(c4, v4, base + full, len - full, x, t);
    if (W & 2) sellBlock<2, NR>(c2, v2, base + at2, len - at2, x, t);
    if (W & 1) sellBlock<1, NR>(c1, v1, base + at1, len - at1, x, t);
}

// y = A x (acc: y += A x) for nrhs right-hand sides (vectors column-major,
// v[r + k n]), NR at a time: the entries are read once for NR of them.
template <int NR, bool NT, bool SHORT, typename CT, typename VT, typename XT>
__global__ void __launch_bounds__(kBlock) k_sell(SellView<CT, VT> A, const XT* __restrict__ x, XT* __restrict__ y,
                                                 int nrhs, int acc, int perXcd) {
    // the chunk is uniform over its wavefront: its tables load through the scalar unit
    const int blk = perXcd ? ((int)blockIdx.x & 7) * perXcd + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    const int c = blk * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x / kC);
    const int lane = threadIdx.x % kC;
    if (c >= A.nChunk) return;
    const int r = c * kC + lane;
    for (int q0 = 0; q0 < nrhs; q0 += NR) {
        const XT* xq[NR];
        XT t[NR], old[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            const long vo = (long)min(q0 + q, nrhs - 1) * A.n;
            xq[q] = x + vo;
            t[q] = XT(0);
            old[q] = acc && r < A.n ? y[vo + r] : XT(0);
        }
        sellRow<NR, NT, SHORT>(A, c, lane, xq, t);
        if (r < A.n)
#pragma unroll
            for (int q = 0; q < NR; ++q)
                if (q0 + q < nrhs) y[(long)(q0 + q) * A.n + r] = old[q] + t[q];
    }
}

// SymmSpMV over the upper triangle (diagonal included) in one pass:
// b[r] += a_rr x_r + sum_{c>r} a_rc x_c and b[c] += a_rc x_r, the update of
// SYMM_SPMV_KERNEL (examples/src/helpers/kernels.cpp:403-427).  Rows of
// different leaves of a distance-2 colour never write the same b entry, but
// rows inside a leaf do, and all rows run at once here: every write to b is
// a device-scope FP64 atomic add.
template <typename CT>
__global__ void __launch_bounds__(kBlock) k_sell_symm_atomic(SellView<CT, double> A, const double* __restrict__ x,
                                                             double* b, int nrhs) {
    const int c = blockIdx.x * kWavesPerBlock + threadIdx.x / kC;
    const int lane = threadIdx.x % kC;
    const int r = c * kC + lane;
    if (c >= A.nChunk || r >= A.n) return;
    const int W = A.W >= 0 ? A.W : A.chunks[c].width;
    const long s0 = A.W >= 0 ? (long)c * W : A.chunks[c].off64;
    const int len = A.pad ? W - (int)A.pad[r] : A.rowPtr[r + 1] - A.rowPtr[r];
    for (int q = 0; q < nrhs; ++q) {
        const double* __restrict__ xq = x + (long)q * A.n;
        double* bq = b + (long)q * A.n;
        const double xr = xq[r];
        double t = 0.0;
        for (int j = 0; j < len; ++j) {
            int j0, E;
            blockOf(W, j, j0, E);
            const int cj = (sizeof(CT) == 2 ? A.base[s0 + j] : 0) +
                           (int)A.col[(s0 + j0) * kC + packPos<CT>(E, j - j0, lane)];
            const double v = A.val[(s0 + j0) * kC + packPos<double>(E, j - j0, lane)];
            if (cj == r) {
                t += v * xr;
            } else {
                t += v * xq[cj];
                atomicAdd(&bq[cj], v * xr);
            }
        }
        atomicAdd(&bq[r], t);
    }
}

// Where the matrix stays between calls decides how it is read.  Larger than
// the 256 MB Infinity Cache it comes from HBM every time: non-temporal loads
// keep x and y in the caches instead (7-point 192^3 FP64 125.5 -> 116.9 us,
// 160^3 75.9 -> 70.6; below 256 MB they cost: 140^3 47.9 -> 50.9).  Between the
// 32 MB of the eight L2 caches and 256 MB every XCD gets one contiguous part
// of the rows (workgroups are dealt round-robin over the XCDs), so that an
// x line is fetched by one L2 and not by all whose rows touch it (140^3 47.9 ->
// 41.0 us, 100^3 20.1 -> 18.4; 27-point 96^3 40.5 -> 38.4).  Above 256 MB eight
// such streams are slower than one (192^3 125.5 -> 134.8), below 32 MB the
// mapping only unbalances a short launch (7-point 64^3 5.2 -> 6.1).
constexpr long kL2Bytes = 32l << 20, kInfinityCacheBytes = 256l << 20;

// Matrices whose chunks all have the same width below 8 (SHORT) run without the
// loop over full blocks, whose double buffer costs 94 registers instead of 42
// in FP64 and so 5 waves per SIMD instead of 8: 7-point 256^3 FP64 321 -> 288
// us, 224^3 214 -> 190, 192^3 119 -> 106, 96^3 16.4 -> 13.6, 64^3 the same.
//
// one launch of y = A x or y += A x.  Right-hand sides are taken 1, 2, 4 or 8
// at a time, the smallest block that covers them (8 for 5 to 8, blocks of 4
// otherwise): a pass over the entries costs more than idle columns of a block,
// but for scattered columns (Product::Plan).
template <int NR, typename CT, typename VT, typename XT>
void launchSellNr(const SellMatrix<VT>& A, const void* x, void* y, int nrhs, bool acc, hipStream_t st) {
    const int g = std::max(1, (A.nChunk + kWavesPerBlock - 1) / kWavesPerBlock);
    const long all = A.bytes + 2l * nrhs * A.n * (long)sizeof(XT);
    const int perXcd = A.bytes <= kInfinityCacheBytes && all > kL2Bytes ? (g + 7) / 8 : 0;
    const dim3 grid(perXcd ? 8 * perXcd : g);
    const bool nt = A.bytes > kInfinityCacheBytes;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, A.template view<CT>(), (const XT*)x, (XT*)y, nrhs,
                           (int)acc, perXcd);
    };
    if (A.uniformW >= 0 && A.uniformW < 8)
        nt ? launch(k_sell<NR, true, true, CT, VT, XT>) : launch(k_sell<NR, false, true, CT, VT, XT>);
    else
        nt ? launch(k_sell<NR, true, false, CT, VT, XT>) : launch(k_sell<NR, false, false, CT, VT, XT>);
}
template <typename CT, typename VT, typename XT>
void launchSellIds(const SellMatrix<VT>& A, const void* x, void* y, int nrhs, bool acc, hipStream_t st) {
    if (nrhs == 1 || A.perPass == 1)
        launchSellNr<1, CT, VT, XT>(A, x, y, nrhs, acc, st);
    else if (nrhs == 2)
        launchSellNr<2, CT, VT, XT>(A, x, y, nrhs, acc, st);
    else if (nrhs <= 4 || (nrhs > 8 && nrhs % 8 >= 1 && nrhs % 8 <= 4))
        launchSellNr<4, CT, VT, XT>(A, x, y, nrhs, acc, st);
    else
        launchSellNr<8, CT, VT, XT>(A, x, y, nrhs, acc, st);
}
template <typename VT, typename XT>
void launchSell(const SellMatrix<VT>& A, const void* x, void* y, int nrhs, bool acc, hipStream_t st) {
    if (A.narrowIds)
        launchSellIds<uint16_t, VT, XT>(A, x, y, nrhs, acc, st);
    else
        launchSellIds<int, VT, XT>(A, x, y, nrhs, acc, st);
}

// Whether rows whose chunks store `slots` slots for nnz entries go to row blocks:
// more than 11 slots for 8 entries with one right-hand side, more than 5 for 4
// with several, which the row blocks read in fewer passes.  Both sides measured
// (us, SELL chunks / row blocks, FP64, FP32): rows of 12 +- 4 entries (1.33 slots an
// entry) 9.0 10.5, 6.3 7.1, +- 6 (1.50) 11.7 10.6, 7.2 7.1; random bands of 200000
// rows, 40 entries a row (1.27) 25.3 25.5, 17.7 19.4, of 90001 rows, 21 entries
// (1.39) 6.9 6.3, 5.4 5.2; three sides: the band of 1.27 64.9 51.8, 46.8 37.9, rows of
// 1.33 30.6 25.7, 20.1 19.0; 27-point grids (1.0 to 1.1) one side 64^3 13.1 18.8,
// three 23.2 37.1; Chung-Lu graphs (2 to 5) of 150000 rows 103 19, 20000 rows 35.5 5.5.
inline bool raggedSlots(long slots, long nnz, int nrhs) { return nrhs > 1 ? slots * 4 > nnz * 5 : slots * 8 > nnz * 11; }

// A matrix that is multiplied with vectors, in the layout its rows ask for: SELL
// chunks or row blocks (raggedSlots).  Regular rows whose right-hand sides are
// packed have both: launches without scratch run over the chunks.
template <typename VT, typename XT>
struct Product {
    SellMatrix<VT> sell;
    RowBlocks<VT> blocks;
    int n = 0;
    bool useBlocks = false;
    // Several right-hand sides over row blocks may be packed row by row first
    // (k_pack_rhs, one more launch and pass over x), into scratch of the
    // launch's stream (StreamSets).  Then an entry takes one cache line of x
    // for all of them instead of one each, and one or two trips through the
    // address unit instead of nrhs.  It pays where columns are scattered over
    // x, so that every gather is a line of its own; where lines are shared
    // only with many entries, and for regular rows, whose chunks gather
    // coalesced lines of one side at a time, only with enough entries and sides
    // (Plan).  us, separate columns / packed, ragged rows: Chung-Lu graph of
    // 150000 rows, 3.0M entries FP32 2 / 3 / 8 sides 37 / 23, 71 / 26, 162 / 39, FP64 8 sides
    // 224 / 63; 20000 rows, 0.4M, FP32 2 / 8 sides 13.0 / 7.3, 50 / 10.7.  Regular rows of
    // random columns, chunks / packed: FP32 40000 rows of 20 entries 2 sides 8.7 /
    // 8.3, 10000 rows 2 / 3 sides 5.1 / 5.7, 7.4 / 6.0; 50000 rows of 6 3 / 8 sides 5.9 /
    // 7.9, 11.9 / 10.6; 100000 rows of 24 within 4000 columns (0.42 lines an entry) 2 / 3
    // / 4 sides 10.4 / 13.8, 15.0 / 16.8, 19.9 / 17.0, 200000 rows of 12 within 8000 (0.61)
    // 15.5 / 16.4, 22.9 / 20.4, 30.6 / 20.7; 27-point 96^3 FP64 8 sides 135 / 158.  Two sides
    // of ragged rows: Poisson(12) 20000 rows FP32 4.3 / 6.5, 50000 rows 7.4 / 7.8;
    // with hub rows, Chung-Lu 60000 rows of 6 FP32 9.6 / 8.7.
    static constexpr int kSets = 2;
    DevBuf<XT> packed[kSets];
    StreamSets streamSets;
    int rhs = 1, R = 0;  // R: right-hand sides of a packed row, 0: not packed
    int sets = 0;        // scratch there was memory for
    // how the rows of a matrix and their columns are laid out
    struct Plan {
        bool ragged = false, packed = false;
        long slots = 0;
        int longest = 0;
        int perPass = 8;  // right-hand sides per pass over the chunks, at most
        int width = 1;    // right-hand sides of a packed row
        Plan(const race_kernel_desc& d, int rhs) {
            ragged = Product::ragged(d, rhs, &slots, &longest);
            if (rhs == 1) return;
            width = rhs == 2 ? 2 : rhs <= 4 || sizeof(XT) == 8 ? 4 : 8;
            const long nnz = d.rowPtr[d.nrow], planes = (rhs + width - 1) / width;
            const double lines = linesPerEntry(d);
            if (ragged)
                packed = (nnz * (rhs - 1) >= (rhs > 2 ? 200000 : longest > 64 ? 350000 : 700000) && lines > 0.4) ||
                         nnz * (rhs - planes) >= 10000000;
            else
                packed = nnz * (rhs - 1) > 300000 + 3l * d.nrow * rhs && lines > (rhs == 2 ? 0.65 : rhs == 3 ? 0.45 : 0.4);
            // Columns that share few lines: two or three sides one after the
            // other, where each side's part of x stays in the caches.  us,
            // sides together / one after the other: the rows of 0.42 lines an
            // entry FP32 2 / 3 sides 12.8 / 10.4, 18.6 / 15.0; of 0.24 FP64 3 sides
            // 19.8 / 17.3, 8 sides 35.5 / 42.6.
            if (rhs <= 3 && lines > (rhs == 2 ? 0.4 : 0.1)) perPass = 1;
        }
    };
    int build(const race_kernel_desc& d) {
        n = d.nrow;
        rhs = d.kind == RACE_K_MPK || d.kind == RACE_K_MPK_HIGHEST ? 1 : std::max(1, d.nrhs);
        const Plan plan(d, rhs);
        useBlocks = plan.ragged;
        if (plan.packed) reserveSets((size_t)n * ((rhs + plan.width - 1) / plan.width) * plan.width);
        if (sets > 0) R = plan.width;
        if (!useBlocks) {
            sell.perPass = plan.perPass;
            if (int e = sell.build(d)) return e;
        }
        if (!useBlocks && R == 0) return OK;
        if (R) blocks.cap = kPackedEntries;
        blocks.add(n, d.rowPtr, d.col, d.val, 0);
        return blocks.finish();
    }
    // as many sets as there is memory for: none is no error, the product then
    // runs without packing
    void reserveSets(size_t count) {
        while (sets < kSets && packed[sets].reserve(count) == hipSuccess) ++sets;
        if (sets < kSets) (void)hipGetLastError();
    }
    // distinct 128-byte lines of x per entry, in runs of kPackedEntries entries
    // (up to 2000 runs, spread over the matrix)
    static double linesPerEntry(const race_kernel_desc& d) {
        const long nnz = d.rowPtr[d.nrow], run = kPackedEntries;
        if (nnz < run) return 0.0;
        const long runs = nnz / run, step = std::max(1l, runs / 2000);
        constexpr int perLine = 128 / (int)sizeof(XT);
        std::vector<int> seen((size_t)d.nrow / perLine + 1, -1);
        long lines = 0, entries = 0;
        for (long k = 0; k < runs; k += step, entries += run)
            for (long j = k * run; j < (k + 1) * run; ++j) {
                int& s = seen[d.col[j] / perLine];
                lines += s != (int)k;
                s = (int)k;
            }
        return (double)lines / (double)entries;
    }
    template <int RR>
    void runPacked(const XT* x, XT* y, XT* buf, bool acc, hipStream_t st) const {
        hipLaunchKernelGGL((k_pack_rhs<RR, XT>), dim3(gridFor(n), (rhs + RR - 1) / RR), dim3(kBlock), 0, st, x, buf,
                           (long)n, rhs);
        launchRowBlkPacked<RR, VT, XT>(blocks, buf, y, n, rhs, acc, st);
    }
    static bool ragged(const race_kernel_desc& d, int rhs, long* stored, int* longest) {
        long slots = 0;
        *longest = 0;
        for (int r0 = 0; r0 < d.nrow; r0 += kC) {
            int w = 0;
            for (int r = r0; r < std::min(d.nrow, r0 + kC); ++r) w = std::max(w, d.rowPtr[r + 1] - d.rowPtr[r]);
            slots += w;
            *longest = std::max(*longest, w);
        }
        // the steps of few short rows take less time than a block's way through
        // LDS: rows of Poisson(6) entries, us, chunks / row blocks, one side FP64, FP32:
        // 20000 rows 3.3 3.8, 3.1 3.7, 100000 rows 5.3 6.0, 5.0 5.6, 200000 rows 11.5 8.6, 8.7
        // 7.9; three sides FP32 50000 rows 7.4 9.3, 5000 rows 5.4 4.2
        *stored = slots * kC;
        const bool few = *longest <= 22 && d.nrow <= 100000 && (rhs == 1 || (rhs <= 3 && d.nrow > 10000));
        return !few && raggedSlots(*stored, d.rowPtr[d.nrow], rhs);
    }
    // y = A x (acc: y += A x)
    void run(const void* x, void* y, int nrhs, bool acc, hipStream_t st) {
        const int set = R && nrhs == rhs ? streamSets.find(st, sets) : -1;
        if (set >= 0) {
            XT* buf = packed[set].p;
            if (R == 2) return runPacked<2>((const XT*)x, (XT*)y, buf, acc, st);
            if (R == 4) return runPacked<4>((const XT*)x, (XT*)y, buf, acc, st);
            if constexpr (sizeof(XT) == 4) return runPacked<8>((const XT*)x, (XT*)y, buf, acc, st);
        }
        if (useBlocks)
            launchRowBlk<false, VT, XT>(blocks, nullptr, x, y, n, nrhs, acc, st);
        else
            launchSell<VT, XT>(sell, x, y, nrhs, acc, st);
    }
};

// b = A x
template <typename VT, typename XT>
class SellSpmvFn : public DeviceFn {
  public:
    Product<VT, XT> A;
    int launches(bool) const override { return A.R ? 2 : 1; }
    int nrhs = 1;
    int init(const race_kernel_desc& d) {
        kind = d.kind;
        x = d.x;
        b = d.b;
        nrhs = d.nrhs > 0 ? d.nrhs : 1;
        return A.build(d);
    }
    int run(bool, hipStream_t st) override {
        A.run(x, b, nrhs, false, st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// full CRS of a symmetric matrix from its upper triangle (diagonal first):
// row r holds its upper entries, then (c, r) of the rows c < r
static void expandUpper(const race_kernel_desc& d, std::vector<int>& rp, std::vector<int>& fc,
                        std::vector<double>& fv) {
    const int n = d.nrow;
    std::vector<int> cnt(n + 1, 0);
    for (int r = 0; r < n; ++r)
        for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
            ++cnt[r + 1];
            if (d.col[j] != r) ++cnt[d.col[j] + 1];
        }
    for (int r = 0; r < n; ++r) cnt[r + 1] += cnt[r];
    rp = cnt;
    fc.assign(cnt[n], 0);
    fv.assign(cnt[n], 0.0);
    std::vector<int> pos(cnt.begin(), cnt.end() - 1);
    for (int r = 0; r < n; ++r)
        for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
            fc[pos[r]] = d.col[j];
            fv[pos[r]++] = d.val[j];
        }
    for (int r = 0; r < n; ++r)
        for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
            const int c = d.col[j];
            if (c == r) continue;
            fc[pos[c]] = r;
            fv[pos[c]++] = d.val[j];
        }
}

// SymmSpMV b += A x from the upper triangle, in one launch:
//  mode 2: SELL-C upper triangle, FP64 atomics for every write to b (FP64 only);
//  mode 3: the full matrix (upper triangle and its transpose) built once at
//          registration, SELL-C SpMV accumulating into b (no atomics, reads
//          the strict upper part twice).
template <typename VT, typename XT>
class SymmSellFn : public DeviceFn {
  public:
    Product<VT, XT> A;
    int launches(bool) const override { return A.R ? 2 : 1; }
    int mode = 2, nrhs = 1;
    int init(const race_kernel_desc& d, int mode_) {
        kind = d.kind;
        x = d.x;
        b = d.b;
        mode = mode_;
        nrhs = d.nrhs > 0 ? d.nrhs : 1;
        if (mode == 2) {
            if (!std::is_same<VT, double>::value || !std::is_same<XT, double>::value) return ERR_NOT_IMPLEMENTED;
            return A.sell.build(d);
        }
        std::vector<int> rp, fc;
        std::vector<double> fv;
        expandUpper(d, rp, fc, fv);
        race_kernel_desc f = d;
        f.rowPtr = rp.data();
        f.col = fc.data();
        f.val = fv.data();
        return A.build(f);
    }
    int run(bool, hipStream_t st) override {
        if constexpr (std::is_same<VT, double>::value && std::is_same<XT, double>::value) {
            if (mode == 2) {
                const unsigned g = (unsigned)std::max(1, (A.sell.nChunk + kWavesPerBlock - 1) / kWavesPerBlock);
                if (A.sell.narrowIds)
                    hipLaunchKernelGGL(k_sell_symm_atomic<uint16_t>, dim3(g), dim3(kBlock), 0, st,
                                       A.sell.template view<uint16_t>(), (const double*)x, (double*)b, nrhs);
                else
                    hipLaunchKernelGGL(k_sell_symm_atomic<int>, dim3(g), dim3(kBlock), 0, st,
                                       A.sell.template view<int>(), (const double*)x, (double*)b, nrhs);
                RACE_HIP(hipGetLastError());
                return OK;
            }
        }
        A.run(x, b, nrhs, true, st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// Matrix powers x_q = A x_{q-1}, q = 1..k, x_q at x + q n: one SpMV launch
// per power.  RACE blocks the powers by level groups so that A stays in a
// CPU cache between them (src/matrixPower.cpp:88-140, 685-940); the host
// executor follows that schedule, the device does not.  Per row and power
// the products and their order are the same, only the launches differ.  A
// slope-2 wavefront over the groups (power q on group L - 2 (q - 1) in launch
// L) was measured on 7-point 192^3, k = 8, 256 MB blocking, FP64: 100 launches,
// 1.23 ms, against 1.02 ms for 8 launches over the same SELL layout (0.84 ms
// with packed entries and the SHORT kernels); 27-point 33^3, k = 5, 4 MB, FP32: 31 launches,
// 139.7 us, against 19.3 us.  The 256 MB Infinity Cache serves a
// gathering SpMV little faster than HBM, so the reuse does not pay for the
// extra launches (3-5 us each) at any size.
//
// Only-highest variant (MAT_SPMV_KERNEL_only_highest
// examples/src/helpers/kernels.cpp:706-734): two vector slots, power q in
// slot q % 2.
//
// setPower(p <= k) runs the first p powers.  With FP32 / BF16 values the
// powers are FP32 vectors accumulated in FP32.
template <typename VT, typename XT>
class MpkFn : public DeviceFn {
  public:
    Product<VT, XT> A;
    int nslot = 2;
    int init(const race_kernel_desc& d, const ExecContext& ctx) {
        kind = d.kind;
        x = d.x;
        b = d.b;
        if (!ctx.mpk) return ERR_INVALID_ARG;
        // powers x sub-powers: every (pow, subPow) pair of the reference's
        // power executor is one product with A, in order
        // (FuncManager::powerCallGeneral src/functionManager.cpp:618-822)
        power = d.power > 0 ? d.power : 1;
        subPower = d.sub_power > 0 ? d.sub_power : 1;
        powerMax = power * subPower;
        nslot = d.kind == RACE_K_MPK_HIGHEST ? 2 : powerMax + 1;
        const std::vector<int>& gp = ctx.mpk->groupPtr;
        if (gp.size() < 2 || gp.front() != 0 || gp.back() != d.nrow) return ERR_INVALID_ARG;
        const int G = (int)gp.size() - 1;
        // RACE's schedule computes power q of a group from power q - 1 of
        // the neighbouring groups.  BFS levels guarantee that this is enough;
        // with mtxType "L" / "U" (row order as levels) it holds only for
        // matrices whose entries stay within neighbouring groups, so
        // anything else is refused, as the schedule cannot run it.
        {
            std::vector<int> grp(d.nrow);
            for (int g = 0; g < G; ++g)
                for (int r = gp[g]; r < gp[g + 1]; ++r) grp[r] = g;
            for (int r = 0; r < d.nrow; ++r)
                for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
                    const int dg = grp[d.col[j]] - grp[r];
                    if (dg < -1 || dg > 1) return ERR_INCOMPATIBILITY;
                }
        }
        return A.build(d);
    }
    bool graphable() const override { return true; }
    int launches(bool) const override {
        const int steps = power * subPower;
        return steps < 1 || steps > powerMax ? 0 : steps;
    }
    int run(bool, hipStream_t st) override {
        const int steps = power * subPower;
        if (steps < 1 || steps > powerMax) return ERR_INVALID_ARG;
        for (int q = 1; q <= steps; ++q)
            A.run((const XT*)x + (size_t)((q - 1) % nslot) * A.n, (XT*)x + (size_t)(q % nslot) * A.n, 1, false, st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// SpMTV b += A^T x for nrhs right-hand sides (SPMTV_KERNEL
// examples/src/helpers/kernels.cpp:106-124, which scatters
// b[c_j] += a_j x[r] row by row under a distance-2 colouring).  The
// transpose is formed once at registration, so a call is one gather SpMV
// over the SELL-C rows of A^T accumulating into b: no atomics, no colour
// phases, every b entry written once.  Row c of A^T holds its entries in
// increasing r, the order a sequential sweep adds them in.
template <typename VT, typename XT>
class SpmtvFn : public DeviceFn {
  public:
    Product<VT, XT> A;
    int launches(bool) const override { return A.R ? 2 : 1; }
    int nrhs = 1;
    int init(const race_kernel_desc& d) {
        kind = d.kind;
        x = d.x;
        b = d.b;
        nrhs = d.nrhs > 0 ? d.nrhs : 1;
        const int n = d.nrow;
        std::vector<int> rp(n + 1, 0);
        for (int j = 0; j < d.rowPtr[n]; ++j) ++rp[d.col[j] + 1];
        for (int r = 0; r < n; ++r) rp[r + 1] += rp[r];
        std::vector<int> tc(rp[n]), pos(rp.begin(), rp.end() - 1);
        std::vector<double> tv(rp[n]);
        for (int r = 0; r < n; ++r)
            for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
                const int c = d.col[j];
                tc[pos[c]] = r;
                tv[pos[c]++] = d.val[j];
            }
        race_kernel_desc t = d;
        t.rowPtr = rp.data();
        t.col = tc.data();
        t.val = tv.data();
        return A.build(t);
    }
    int run(bool, hipStream_t st) override {
        A.run(x, b, nrhs, true, st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// r = b - A x (FP64 product, r stored as RT) and the sums of r^2 and b^2
// for the refinement; grid-stride over chunks so few workgroups add to the
// two norm accumulators
template <typename RT, bool NT, typename CT>
__global__ void __launch_bounds__(kBlock) k_sell_residual(SellView<CT, double> A, const double* __restrict__ x,
                                                          const double* __restrict__ b, RT* __restrict__ r, int nrhs,
                                                          double* __restrict__ norms) {
    __shared__ double sr[kWavesPerBlock], sb[kWavesPerBlock];
    const int lane = threadIdx.x % kC, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kC);
    double rr = 0.0, bb = 0.0;
    for (int c = blockIdx.x * kWavesPerBlock + wv; c < A.nChunk; c += gridDim.x * kWavesPerBlock) {
        const int row = c * kC + lane;
        const bool live = row < A.n;  // lanes past the last row compute, store nothing
        for (int q = 0; q < nrhs; ++q) {
            const long vo = (long)q * A.n;
            const double* const xq[1] = {x + vo};
            double t[1] = {0.0};
            const double bv = b[vo + (live ? row : 0)];
            sellRow<1, NT, false>(A, c, lane, xq, t);
            if (!live) continue;
            const double rv = bv - t[0];
            r[vo + row] = (RT)rv;
            rr += rv * rv;
            bb += bv * bv;
        }
    }
    rr = groupSum<kC>(rr);
    bb = groupSum<kC>(bb);
    if (lane == 0) {
        sr[wv] = rr;
        sb[wv] = bb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, e = 0.0;
        for (int w = 0; w < kWavesPerBlock; ++w) {
            a += sr[w];
            e += sb[w];
        }
        atomicAdd(&norms[0], a);
        atomicAdd(&norms[1], e);
    }
}

class SellResidual : public ResidualOp {
  public:
    SellMatrix<double> A;
    int init(const race_kernel_desc& d) { return A.build(d); }
    template <typename RT, typename CT>
    void launch(const double* x, const double* b, void* r, int nrhs, double* norms, hipStream_t st) {
        const int blocks = std::max(1, std::min(4096, (A.nChunk + kWavesPerBlock - 1) / kWavesPerBlock));
        if (A.bytes > kInfinityCacheBytes)
            hipLaunchKernelGGL((k_sell_residual<RT, true, CT>), dim3(blocks), dim3(kBlock), 0, st,
                               A.template view<CT>(), x, b, (RT*)r, nrhs, norms);
        else
            hipLaunchKernelGGL((k_sell_residual<RT, false, CT>), dim3(blocks), dim3(kBlock), 0, st,
                               A.template view<CT>(), x, b, (RT*)r, nrhs, norms);
    }
    int run(const double* x, const double* b, void* r, bool rFp32, int nrhs, double* norms,
            hipStream_t st) override {
        if (rFp32 && A.narrowIds)
            launch<float, uint16_t>(x, b, r, nrhs, norms, st);
        else if (rFp32)
            launch<float, int>(x, b, r, nrhs, norms, st);
        else if (A.narrowIds)
            launch<double, uint16_t>(x, b, r, nrhs, norms, st);
        else
            launch<double, int>(x, b, r, nrhs, norms, st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// ---------------------------------------------------------------------------
// Generalised SELL-C-sigma for batches and the layout tuner: chunk height
// C in {8, 16, 32, 64} (a wavefront holds 64 / C chunks), rows sorted by
// length (longest first) inside windows of sigma rows so that a chunk holds
// rows of similar length, and every chunk tagged with its matrix, whose
// vectors it uses.  Entry j of slot i of a chunk at off + j C + i.
struct SellGChunk {
    int rows, width, slot0, mat;
    long off;
};

template <int C, bool PERM, typename XT, bool ACC>
__global__ void __launch_bounds__(kBlock) k_sellg_spmv(const SellGChunk* __restrict__ chunks, int nChunk,
                                                       const int* __restrict__ rowOf, const int* __restrict__ col,
                                                       const XT* __restrict__ val, const XT* const* __restrict__ mx,
                                                       XT* const* __restrict__ my, const int* __restrict__ mn,
                                                       int nrhs) {
    const int lane = threadIdx.x % 64;
    const int c = (int)((blockIdx.x * (long)blockDim.x + threadIdx.x) / 64) * (64 / C) + lane / C;
    const int i = lane % C;
    if (c >= nChunk) return;
    const SellGChunk k = chunks[c];
    if (i >= k.rows) return;
    const int row = PERM ? rowOf[k.slot0 + i] : k.slot0 + i;
    const XT* __restrict__ x = mx[k.mat];
    XT* __restrict__ y = my[k.mat];
    const long n = mn[k.mat];
    const int* __restrict__ cc = col + k.off + i;
    const XT* __restrict__ vv = val + k.off + i;
    for (int q = 0; q < nrhs; ++q) {
        const XT* __restrict__ xq = x + q * n;
        XT t = XT(0);
        int j = 0;
        for (; j + 2 <= k.width; j += 2) {
            const int c0 = cc[j * C], c1 = cc[(j + 1) * C];
            const XT v0 = vv[j * C], v1 = vv[(j + 1) * C];
            t += v0 * xq[c0];
            t += v1 * xq[c1];
        }
        if (j < k.width) t += vv[j * C] * xq[cc[j * C]];
        if (ACC)
            y[q * n + row] += t;
        else
            y[q * n + row] = t;
    }
}

// SpMV (b = A x) or SymmSpMV (b += A x, expanded from the upper triangle)
// on a batch of matrices: one launch over the SELL chunks of all matrices
// that fit the layout, one over the row blocks of the others (chooseBlocks): with 8
// right-hand sides a chunk holding a hub row runs its up to 400 steps once per
// right-hand side.  16 matrices of 2000 to 40000 rows, FP32, 8 right-hand sides: 864 us
// in chunks of 64 rows alone, 80 us.
template <typename XT>
class SellBatchFn : public DeviceFn {
  public:
    int C = 64, sigma = 1, nrhs = 1, nChunk = 0;
    bool perm = false;
    DevBuf<SellGChunk> chunks;
    DevBuf<int> rowOf, col, mn;
    DevBuf<XT> val;
    DevBuf<const XT*> mx;
    DevBuf<XT*> my;
    RowBlocks<XT> blocks;
    DevBuf<RowBlkVecs> vecs;

    // The matrices that go to row blocks: those over 5 slots for 4 entries in
    // chunks, or with a chunk wider than 64 entries.  Where none is over 11 for 8
    // and they hold less than a 16th of the batch's entries, all stay in chunks: a
    // second launch for a few small matrices costs more (stencils, 27-point 10^3 of
    // 1.26 slots an entry among them, one side FP64, us: 13.6 in chunks, 17.2 in two
    // launches).
    std::vector<char> chooseBlocks(const std::vector<BatchItem>& items) const {
        std::vector<char> in(items.size(), 0);
        std::vector<int> len;
        long entries = 0, over = 0;
        bool far = false;
        for (size_t m = 0; m < items.size(); ++m) {
            const race_kernel_desc& d = items[m].d;
            const int n = d.nrow;
            len.assign(n, 0);
            for (int r = 0; r < n; ++r)
                for (int j = d.rowPtr[r]; j < d.rowPtr[r + 1]; ++j) {
                    ++len[r];
                    if (kind == RACE_K_SYMMSPMV && d.col[j] != r) ++len[d.col[j]];
                }
            if (perm)
                for (int w0 = 0; w0 < n; w0 += sigma)
                    std::sort(len.begin() + w0, len.begin() + std::min(n, w0 + sigma), std::greater<int>());
            long slots = 0, nnz = 0;
            int widest = 0;
            for (int r0 = 0; r0 < n; r0 += C) {
                int w = 0;
                for (int r = r0; r < std::min(n, r0 + C); ++r) {
                    w = std::max(w, len[r]);
                    nnz += len[r];
                }
                slots += (long)w * C;
                widest = std::max(widest, w);
            }
            entries += nnz;
            in[m] = widest > 64 || slots * 4 > nnz * 5;
            if (in[m]) over += nnz;
            far = far || widest > 64 || slots * 8 > nnz * 11;
        }
        if (!far && over * 16 < entries) in.assign(items.size(), 0);
        return in;
    }

    int init(const std::vector<BatchItem>& items, const ExecContext& ctx) {
        kind = items[0].d.kind;
        nrhs = items[0].d.nrhs > 0 ? items[0].d.nrhs : 1;
        C = ctx.sellC;
        sigma = std::max(1, ctx.sellSigma);
        perm = sigma > 1;
        if (C != 8 && C != 16 && C != 32 && C != 64) return ERR_INVALID_ARG;
        std::vector<SellGChunk> hc;
        std::vector<int> hrow, hcol, hn;
        std::vector<XT> hval;
        std::vector<const XT*> hx;
        std::vector<XT*> hy;
        std::vector<RowBlkVecs> hv;
        std::vector<int> rp, fc, order;
        std::vector<double> fv;
        const std::vector<char> inBlocks = chooseBlocks(items);
        for (size_t m = 0; m < items.size(); ++m) {
            const race_kernel_desc& d = items[m].d;
            const int n = d.nrow;
            const int* R = d.rowPtr;
            const int* Cc = d.col;
            const double* V = d.val;
            if (kind == RACE_K_SYMMSPMV) {
                expandUpper(d, rp, fc, fv);
                R = rp.data();
                Cc = fc.data();
                V = fv.data();
            }
            order.resize(n);
            for (int r = 0; r < n; ++r) order[r] = r;
            if (perm)
                for (int w0 = 0; w0 < n; w0 += sigma) {
                    const int w1 = std::min(n, w0 + sigma);
                    std::stable_sort(order.begin() + w0, order.begin() + w1, [&](int a, int b) {
                        return R[a + 1] - R[a] > R[b + 1] - R[b];
                    });
                }
            hx.push_back((const XT*)d.x);
            hy.push_back((XT*)d.b);
            hn.push_back(n);
            hv.push_back(RowBlkVecs{d.x, d.b, n});
            if (inBlocks[m]) {
                blocks.add(n, R, Cc, V, (int)m);
                continue;
            }
            for (int r0 = 0; r0 < n; r0 += C) {
                const int rows = std::min(C, n - r0);
                int w = 0;
                for (int i = 0; i < rows; ++i) w = std::max(w, R[order[r0 + i] + 1] - R[order[r0 + i]]);
                const long off = (long)hcol.size();
                const int slot0 = perm ? (int)hrow.size() : r0;
                hc.push_back(SellGChunk{rows, w, slot0, (int)m, off});
                hcol.resize(off + (long)w * C);
                hval.resize(off + (long)w * C);
                for (int i = 0; i < C; ++i) {
                    const int r = order[r0 + std::min(i, rows - 1)];
                    const int len = i < rows ? R[r + 1] - R[r] : 0;
                    for (int j = 0; j < w; ++j) {
                        const long pos = off + (long)j * C + i;
                        hcol[pos] = j < len ? Cc[R[r] + j] : r;
                        hval[pos] = j < len ? (XT)V[R[r] + j] : XT(0);
                    }
                    if (perm && i < rows) hrow.push_back(r);
                }
            }
        }
        nChunk = (int)hc.size();
        int e;
        if ((e = blocks.finish())) return e;
        if ((e = upload(vecs, hv.data(), hv.size()))) return e;
        if ((e = upload(chunks, hc.data(), hc.size()))) return e;
        if ((e = upload(rowOf, hrow.data(), hrow.size()))) return e;
        if ((e = upload(col, hcol.data(), hcol.size()))) return e;
        if ((e = upload(val, hval.data(), hval.size()))) return e;
        if ((e = upload(mx, hx.data(), hx.size()))) return e;
        if ((e = upload(my, hy.data(), hy.size()))) return e;
        if ((e = upload(mn, hn.data(), hn.size()))) return e;
        return OK;
    }
    template <int CC, bool P>
    void launch(hipStream_t st) {
        const long waves = ((long)nChunk + (64 / CC) - 1) / (64 / CC);
        const unsigned g = (unsigned)std::max(1l, (waves + kWavesPerBlock - 1) / kWavesPerBlock);
        if (kind == RACE_K_SYMMSPMV)
            hipLaunchKernelGGL((k_sellg_spmv<CC, P, XT, true>), dim3(g), dim3(kBlock), 0, st, chunks.p, nChunk,
                               rowOf.p, col.p, val.p, mx.p, my.p, mn.p, nrhs);
        else
            hipLaunchKernelGGL((k_sellg_spmv<CC, P, XT, false>), dim3(g), dim3(kBlock), 0, st, chunks.p, nChunk,
                               rowOf.p, col.p, val.p, mx.p, my.p, mn.p, nrhs);
    }
    int launches(bool) const override { return (nChunk > 0) + (blocks.nBlk > 0); }
    int run(bool, hipStream_t st) override {
        if (blocks.nBlk > 0)
            launchRowBlk<true, XT, XT>(blocks, vecs.p, nullptr, nullptr, 0, nrhs, kind == RACE_K_SYMMSPMV, st);
        if (nChunk > 0) runChunks(st);
        RACE_HIP(hipGetLastError());
        return OK;
    }
    void runChunks(hipStream_t st) {
        switch (C * 2 + (perm ? 1 : 0)) {
            case 16: launch<8, false>(st); break;
            case 17: launch<8, true>(st); break;
            case 32: launch<16, false>(st); break;
            case 33: launch<16, true>(st); break;
            case 64: launch<32, false>(st); break;
            case 65: launch<32, true>(st); break;
            case 128: launch<64, false>(st); break;
            default: launch<64, true>(st); break;
        }
    }
};

}  // namespace

int makeSellBatchFn(const std::vector<BatchItem>& items, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    if (items.empty()) return ERR_INVALID_ARG;
    const race_kernel_desc& d0 = items[0].d;
    for (const BatchItem& it : items)
        if (it.d.kind != d0.kind || it.d.val_precision != d0.val_precision ||
            it.d.vec_precision != d0.vec_precision || it.d.nrhs != d0.nrhs)
            return ERR_INVALID_ARG;
    if (d0.kind != RACE_K_SYMMSPMV && d0.kind != RACE_K_SPMV) return ERR_INVALID_ARG;
    if (d0.val_precision != d0.vec_precision) return ERR_NOT_IMPLEMENTED;
    int e;
    if (d0.vec_precision == RACE_FP64) {
        auto f = std::make_unique<SellBatchFn<double>>();
        e = f->init(items, ctx);
        *out = std::move(f);
    } else if (d0.vec_precision == RACE_FP32) {
        auto f = std::make_unique<SellBatchFn<float>>();
        e = f->init(items, ctx);
        *out = std::move(f);
    } else {
        return ERR_NOT_IMPLEMENTED;
    }
    return e;
}

// the storage / arithmetic pairs of the single-matrix SELL functions:
// FP64 / FP64, FP32 / FP32, BF16 / FP32
template <template <typename, typename> class F, typename Init>
int makeTyped(const race_kernel_desc& d, std::unique_ptr<DeviceFn>* out, Init&& init) {
    int e;
    if (d.val_precision == RACE_FP64 && d.vec_precision == RACE_FP64) {
        auto f = std::make_unique<F<double, double>>();
        e = init(*f);
        *out = std::move(f);
    } else if (d.val_precision == RACE_FP32 && d.vec_precision == RACE_FP32) {
        auto f = std::make_unique<F<float, float>>();
        e = init(*f);
        *out = std::move(f);
    } else if (d.val_precision == RACE_BF16 && d.vec_precision == RACE_FP32) {
        auto f = std::make_unique<F<uint16_t, float>>();
        e = init(*f);
        *out = std::move(f);
    } else {
        return ERR_NOT_IMPLEMENTED;
    }
    return e;
}

int makeSellResidual(const race_kernel_desc& d, std::unique_ptr<ResidualOp>* out) {
    auto f = std::make_unique<SellResidual>();
    int e = f->init(d);
    *out = std::move(f);
    return e;
}

bool spmvByLanes(const race_kernel_desc& d) {
    const long n = d.nrow, nnz = d.rowPtr[d.nrow];
    if (d.val_precision != RACE_FP64 || d.vec_precision != RACE_FP64 || d.nrhs <= 1) return false;
    if (nnz > 450000 || nnz <= 4 * n || nnz * d.nrhs > 2500000) return false;
    for (int r = 0; r < d.nrow; ++r)
        if (d.rowPtr[r + 1] - d.rowPtr[r] > 64) return false;
    const Product<double, double>::Plan plan(d, d.nrhs);
    if (nnz <= 8 * n && (d.nrhs > 3 || !raggedSlots(plan.slots, nnz, 1))) return false;
    return nnz * d.nrhs <= 1200000 || (!plan.ragged && !plan.packed);
}

int makeSellSpmvFn(const race_kernel_desc& d, std::unique_ptr<DeviceFn>* out) {
    return makeTyped<SellSpmvFn>(d, out, [&](auto& f) { return f.init(d); });
}

int makeSymmSellFn(const race_kernel_desc& d, int mode, std::unique_ptr<DeviceFn>* out) {
    return makeTyped<SymmSellFn>(d, out, [&](auto& f) { return f.init(d, mode); });
}

int makeSpmtvFn(const race_kernel_desc& d, std::unique_ptr<DeviceFn>* out) {
    return makeTyped<SpmtvFn>(d, out, [&](auto& f) { return f.init(d); });
}

int makeMpkFn(const race_kernel_desc& d, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    return makeTyped<MpkFn>(d, out, [&](auto& f) { return f.init(d, ctx); });
}

}  // namespace race
