// bundle_exec.hpp -- Gauss-Seidel and Kaczmarz over leaf bundles.
//
// Included once per pair of value and vector type (bundle_f64.hip,
// bundle_f32.hip, bundle_bf16.hip), so that the instantiations compile in
// parallel.
//
// One workgroup runs one bundle (a run of whole, mutually independent
// leaves of one colour phase).  TPR lanes share a row; each lane keeps E
// (local column, value) pairs of its row in registers for the whole launch.
// The bundle's local column space lives in LDS; the dependency waves of the
// leaves (rows of equal depth in RACE's sequential leaf order) run one after
// the other with a workgroup barrier in between.  Only the prologue touches
// HBM: the entry block, the outside columns of x, and the write-back.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <type_traits>

#include "bundle.hpp"
#include "bundle_make.hpp"
#include "exec.hpp"
#include "exec_common.hpp"

namespace race {

namespace {

// matrix value storage: double, float, or bfloat16 bits (uint16_t).  The
// prologue keeps a value as loaded (ValBits) and converts it where it is
// used, after every load of the prologue has been issued.  A bfloat16 shift
// next to its load makes the wave wait for that load before it issues the
// next entry's loads (13 round trips in a row); the empty asm statement,
// which emits no instruction, keeps the compiler from moving the shift back
// next to the load.
template <typename VT>
struct ValBits {
    using T = VT;
};
template <>
struct ValBits<uint16_t> {
    using T = unsigned;
};
template <typename XT>
__device__ __forceinline__ XT valOf(double v) {
    return (XT)v;
}
template <typename XT>
__device__ __forceinline__ XT valOf(float v) {
    return (XT)v;
}
template <typename XT>
__device__ __forceinline__ XT valOf(unsigned v) {
    asm volatile("" : "+v"(v));
    return (XT)__uint_as_float(v << 16);
}

// Sum over the TPR lanes of a row.  The lanes of a row lie in one quad
// (TPR <= 4), so the partner's value comes through a DPP quad permutation,
// a VALU move with no LDS round trip: lane ^ 2 is quad_perm [2,3,0,1]
// (0x4E), lane ^ 1 is quad_perm [1,0,3,2] (0xB1).  The partner lanes of a
// row are always active together.  Same additions, in the same order, as a
// butterfly over shuffles.
template <int CTRL>
__device__ __forceinline__ float quadSwap(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double quadSwap(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xF, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int TPR, typename T>
__device__ __forceinline__ T laneSum(T v) {
    static_assert(TPR == 1 || TPR == 2 || TPR == 4, "the lanes of a row must lie in one quad");
    if (TPR == 4) v += quadSwap<0x4E>(v);
    if (TPR >= 2) v += quadSwap<0xB1>(v);
    return v;
}

// bundle handled by this workgroup: with xcd != 0, consecutive bundles of the
// phase go to the same XCD (workgroups are dealt round-robin over 8 XCDs), so
// the outside columns they share stay in one L2.  Returns -1 for the padding
// workgroups of that mapping.
__device__ __forceinline__ int bundleOfBlock(int nbnd, int xcd) {
    if (!xcd) return blockIdx.x;
    const int chunk = (nbnd + 7) >> 3;
    const int q = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
    return q < nbnd ? q : -1;
}

// the lane of a row that reads and writes its x (the first of its lanes)
__device__ __forceinline__ bool own(bool active, int lane) { return active && lane == 0; }

// ---------------------------------------------------------------------------
// The dependency waves of a bundle.  Slots are sorted by wave, so the lanes of
// a wave are contiguous and each wavefront holds a contiguous range of waves.
// A wavefront's LDS accesses execute in order, so waves that lie inside one
// wavefront need no workgroup barrier between them: only that wavefront runs
// them while the others wait at the next barrier.  A wave spread over several
// wavefronts is run by all of them between two barriers.  That is at most two
// barriers per wavefront of the workgroup instead of two per wave.  A wave is
// bound by its chain of LDS reads, products, the sum over the lanes of a row
// and LDS writes.  Used with variable lanes per row, whose waves needed two
// barriers and a serial sum: a forward Kaczmarz sweep over a Chung-Lu graph of
// 36425 rows (one chain of 7009 waves), FP32, 6.76 ms before, 4.34 ms with this,
// rowSum and the batched column gathers.  Not used with uniform lanes, where one
// barrier per wave is cheaper than finding the spans for some ten waves a
// launch (Gauss-Seidel, 27-point 14^3: 124.3 us a step, 143.3 us with spans).
//
// WaveSpans: first and last wave of every wavefront, in LDS; set before a
// barrier and read by runWaves after it.
template <int NW>
struct WaveSpans {
    int first[NW], last[NW];
};
template <int NW>
__device__ __forceinline__ void setSpans(WaveSpans<NW>& sp, bool active, int myWave) {
    const unsigned long long m = __ballot(active);
    const int v = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // active lanes are the first of their wavefront
    const int end = 64 - (m ? __clzll((long long)m) : 64);
    if (lane == 0) sp.first[v] = m ? myWave : INT32_MAX;
    if (lane == (m ? end - 1 : 0)) sp.last[v] = m ? myWave : -1;
}
// row(w, spread) runs wave w on the lanes that belong to it; spread: several
// wavefronts run it at once and every thread of the workgroup calls it (it
// may hold barriers then).  Ends with a barrier if the bundle has any wave.
template <int NW, class Row>
__device__ __forceinline__ void runWaves(const WaveSpans<NW>& sp, int nw, Row&& row) {
    const int me = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lf = lane < NW ? sp.first[lane] : INT32_MAX, ll = lane < NW ? sp.last[lane] : -1;
    int next = 0;
    for (int v = 0; v < NW && next < nw;) {
        const int vl = __builtin_amdgcn_readlane(ll, v);
        if (vl < next) {
            ++v;
            continue;
        }
        // waves of v alone, then the one it shares with its successors
        const bool shares = v + 1 < NW && __builtin_amdgcn_readlane(lf, v + 1) == vl;
        const bool spread = shares && next == vl;
        const int end = spread ? vl : shares ? vl - 1 : vl;
        if (spread || me == v)
            for (int w = next; w <= end; ++w) {
                row(w, spread);
                // the next wave's reads stay behind this one's writes
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        next = end + 1;
        __syncthreads();
    }
}

// Vectors of a bundle: the launch's x, b and n, or, for a batch of matrices
// (BATCH), the bundle's own (each matrix keeps its vectors).
template <bool BATCH, typename XT>
struct BundleVec {
    XT* x;
    const XT* b;
    int n;
    __device__ __forceinline__ BundleVec(XT* x0, const XT* b0, int n0, XT* const* bx, const XT* const* bb,
                                         const int* bn, int bnd) {
        if (BATCH) {
            x = bx[bnd];
            b = bb[bnd];
            n = bn[bnd];
        } else {
            x = x0;
            b = b0;
            n = n0;
        }
    }
};

// The prologue has three dependent memory levels: the bundle's offsets;
// then, all issued together, its entry block, row ids, inverse diagonals,
// wave numbers and outside-column ids; then the gathers of x and b.  Row
// and column ids are unsigned: widening them for the 64-bit address is then
// a zero high half, not a sign extension that has to wait for the loaded
// value.  A phase whose chains are single bundles (bundle0 >= 0) skips the
// chain table.
template <int BS, int TPR, int E, typename VT, typename XT, bool ONE_RHS, bool BATCH, int NX = 2>
__global__ void __launch_bounds__(BS) k_gs_bundle(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const XT* __restrict__ rdiag, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* __restrict__ x0,
    const XT* __restrict__ b0, int n0, int nrhs, const int* __restrict__ chainPtr, int chain0, int nchain,
    int bundle0, int xcd, XT* const* __restrict__ bX, const XT* const* __restrict__ bB,
    const int* __restrict__ bN) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);

    const int q = bundleOfBlock(nchain, xcd);
    if (q < 0) return;
    // a chain: one bundle, or the segments of a leaf too large for one bundle,
    // run in order (each segment reads what the previous one wrote)
    const int cLo = bundle0 >= 0 ? bundle0 + q : chainPtr[chain0 + q];
    const int cHi = bundle0 >= 0 ? cLo + 1 : chainPtr[chain0 + q + 1];
    auto runBundle = [&](const int bnd) {
        const BundleVec<BATCH, XT> vec(x0, b0, n0, bX, bB, bN, bnd);
        XT* __restrict__ x = vec.x;
        const XT* __restrict__ b = vec.b;
        const int n = vec.n;
        const int s0 = bSlot[bnd], nb = bSlot[bnd + 1] - s0;
        const long off = bOff[bnd];
        const int wb = bLen[bnd];
        const int nw = bWave[bnd + 1] - bWave[bnd];
        const int e0 = bExt[bnd], ne = bExt[bnd + 1] - e0;
        const int t = threadIdx.x, i = t / TPR, l = t % TPR;
        const bool active = i < nb;
        const long lanes = (long)nb * TPR;

        // Branch-free prologue.  An entry load past the bundle's width or of
        // a padding row reads the zero entry (local column 0, value 0) that
        // ends the entry arrays, at index `zero`.  Any other load whose lane
        // is idle reads element 0 of its array (every device array holds at
        // least one element); the lane ignores it, and an id read that way
        // is replaced by 0 before it indexes x.  Without branches the wait
        // before the gathers counts exactly the entry loads still in flight,
        // so the gathers overlap the entry block.  The ids the gathers need
        // go out first.
        const int sr = active ? s0 + i : 0;
        const unsigned row = (unsigned)rowId[sr];
        // ids of the first NX*BS outside columns, in one batch (columns
        // beyond are gathered round by round)
        unsigned ex[NX];
#pragma unroll
        for (int k = 0; k < NX; ++k) ex[k] = (unsigned)ext[t + k * BS < ne ? e0 + t + k * BS : 0];
        int li[E];
        typename ValBits<VT>::T lv[E];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const long e = (active && u < wb) ? off + (long)u * lanes + t : zero;
            li[u] = (int)sidx[e];
            lv[u] = sval[e];
        }
        const XT rd = rdiag[sr];
        const int myWave = (int)slotWave[sr];

        // right-hand sides are independent: grid.y splits them over workgroups
        const int k0 = ONE_RHS ? 0 : (int)blockIdx.y;
        const int k1 = ONE_RHS ? 1 : (gridDim.y > 1 ? k0 + 1 : nrhs);
        const bool own = active && l == 0;
        for (int k = k0; k < k1; ++k) {
            const size_t vo = (size_t)k * n;
            // every gather in flight before the first LDS write
            XT g[NX];
#pragma unroll
            for (int q = 0; q < NX; ++q) g[q] = x[vo + (t + q * BS < ne ? ex[q] : 0u)];
            const XT gr = x[vo + (own ? row : 0u)];
            const XT br = b[vo + (own ? row : 0u)];
#pragma unroll
            for (int q = 0; q < NX; ++q)
                if (t + q * BS < ne) xl[nb + t + q * BS] = g[q];
            if (own) xl[i] = gr;
            for (int c = t + NX * BS; c < ne; c += BS) xl[nb + c] = x[vo + ext[e0 + c]];
            __syncthreads();
            for (int w = 0; w < nw; ++w) {
                if (active && myWave == w) {
                    // two partial sums: half the dependent FMA chain
                    XT sa = XT(0), sb = XT(0);
#pragma unroll
                    for (int u = 0; u + 1 < E; u += 2) {
                        sa += valOf<XT>(lv[u]) * xl[li[u]];
                        sb += valOf<XT>(lv[u + 1]) * xl[li[u + 1]];
                    }
                    if (E % 2) sa += valOf<XT>(lv[E - 1]) * xl[li[E - 1]];
                    const XT sm = laneSum<TPR>(sa + sb);
                    if (l == 0) xl[i] = (br - sm) * rd;
                }
                __syncthreads();
            }
            if (own) x[vo + row] = xl[i];
            __syncthreads();
        }
    };
    // the common case, one bundle per workgroup, as its own straight-line copy
    if (cHi == cLo + 1) {
        runBundle(cLo);
    } else {
        for (int bnd = cLo; bnd < cHi; ++bnd) {
            runBundle(bnd);
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// One launch per sweep ("flow"): the chains of every phase are handed out in
// chain order (phase order) from a ticket counter, and a chain waits only for
// the earlier chains it conflicts with (chainDeps), through a completion flag
// per chain, instead of for the whole previous phase at a launch boundary.
// Tickets go out in an order in which every dependency comes first, and a
// workgroup takes a ticket only when it can run it, so the chain with the
// smallest unfinished number always has its dependencies done: the launch
// cannot deadlock, whatever the number of resident workgroups.
//
// Values of x that another workgroup may have written during the launch are
// read and written with agent-scope relaxed atomics (each XCD has its own
// L2; these accesses are coherent across them).  A chain publishes its flag
// after every wave of the workgroup has waited for its stores of x; a waiter
// reads the flag, then issues its loads of x.
struct FlowState {
    int ticket;  // next chain to hand out
    int done;    // workgroups finished in this launch
    int epoch;   // launch number: a chain's flag holds the epoch it finished in
    int abort;   // a wait exceeded its poll budget in this launch
    int aborts;  // launches that aborted (kept for the host)
    int tail;    // readiness-driven sweeps: next free slot of the ready queue
    int pad[2];
};

__device__ __forceinline__ int ldAgent(const int* p) {
    return __hip_atomic_load(const_cast<int*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stAgent(int* p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T ldCoh(const T* p) {
    return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void stCoh(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wait until chain a has finished in this launch.  After pollLimit polls
// (a broken dependency table), or once another wait has given up, the
// launch is marked aborted and the wait returns, so every workgroup ends.
__device__ __forceinline__ void waitChain(const int* flag, int a, int epoch, FlowState* fs, int pollLimit) {
    int polls = 0;
    while (ldAgent(&flag[a]) != epoch) {
        if ((++polls & 255) == 0 && (polls >= pollLimit || ldAgent(&fs->abort))) {
            stAgent(&fs->abort, 1);
            return;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Gauss-Seidel, one right-hand side, all phases of a sweep in one launch.
// The bundle body is k_gs_bundle's, with the dependency wait between the
// prologue's matrix loads and its gathers of x.
// NX register slots per lane for outside-column ids and values: NX*BS
// columns are gathered in one batch (bundles of a 27-point stencil at small
// leaves have about 900-2500 outside columns).
template <int BS, int TPR, int E, typename VT, typename XT, int NX = 6>
__global__ void __launch_bounds__(BS) k_gs_flow(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const XT* __restrict__ rdiag, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* x, const XT* __restrict__ b,
    const int* __restrict__ tLo, const int* __restrict__ tHi, int nchain, const int* __restrict__ depPtr,
    const int* __restrict__ dep, int* flag, FlowState* fs, int pollLimit) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);
    __shared__ int sTicket;
    const int t = threadIdx.x, i = t / TPR, l = t % TPR;
    const int epoch = ldAgent(&fs->epoch);
    if (t == 0) sTicket = atomicAdd(&fs->ticket, 1);
    __syncthreads();
    // the chain index is uniform: its table entries load through the scalar unit
    int cur = __builtin_amdgcn_readfirstlane(sTicket);
    // The previous chain's flag goes out at the next chain's first wait for
    // memory, which covers the previous chain's stores of x: their
    // completion overlaps the next prologue.  It is published before that
    // chain waits for anything, so no wait can depend on it.
    int pending = -1;
    auto publish = [&]() {
        if (pending >= 0) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (t == 0) stAgent(&flag[pending], epoch);
            pending = -1;
        }
    };
    while (cur < nchain) {
        int next = 0;
        const int cLo = tLo[cur], cHi = tHi[cur];
        for (int bnd = cLo; bnd < cHi; ++bnd) {
            const bool first = bnd == cLo;
            const int d0 = first ? depPtr[cur] : 0, nd = first ? depPtr[cur + 1] - d0 : 0;
            // branch-free: the dependency ids load with the prologue (every
            // device array holds at least one element)
            const int dj = dep[t < nd ? d0 + t : 0];
            const int s0 = bSlot[bnd], nb = bSlot[bnd + 1] - s0;
            const long off = bOff[bnd];
            const int wb = bLen[bnd];
            const int nw = bWave[bnd + 1] - bWave[bnd];
            const int e0 = bExt[bnd], ne = bExt[bnd + 1] - e0;
            const bool active = i < nb;
            const long lanes = (long)nb * TPR;
            // branch-free prologue (as in k_gs_bundle)
            const int sr = active ? s0 + i : 0;
            const unsigned row = (unsigned)rowId[sr];
            // ids of the first NX*BS outside columns, in one batch
            unsigned ex[NX];
#pragma unroll
            for (int k = 0; k < NX; ++k) ex[k] = (unsigned)ext[t + k * BS < ne ? e0 + t + k * BS : 0];
            int li[E];
            typename ValBits<VT>::T lv[E];
#pragma unroll
            for (int u = 0; u < E; ++u) {
                const long e = (active && u < wb) ? off + (long)u * lanes + t : zero;
                li[u] = (int)sidx[e];
                lv[u] = sval[e];
            }
            const XT rd = rdiag[sr];
            const int myWave = (int)slotWave[sr];
            const XT br = b[own(active, l) ? row : 0u];
            // Columns no earlier chain of the launch writes (bit 31 clear)
            // still hold the launch's starting value: they are gathered now,
            // with the matrix, through the caches.  So is the row's own x
            // (only this chain writes it).
            XT g[NX];
#pragma unroll
            for (int k = 0; k < NX; ++k) g[k] = x[t + k * BS < ne && !(ex[k] >> 31) ? ex[k] : 0u];
            const XT gr = x[own(active, l) ? row : 0u];
            // the next ticket is requested here, behind the prologue's loads
            // (the wave waits for it where it waits for them), and read after
            // this chain
            if (first && t == 0) next = atomicAdd(&fs->ticket, 1);
            publish();
            // the chains this one conflicts with, then the columns they wrote
            if (t < nd) waitChain(flag, dj, epoch, fs, pollLimit);
            for (int j = t + BS; j < nd; j += BS) waitChain(flag, dep[d0 + j], epoch, fs, pollLimit);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NX; ++k)
                if (t + k * BS < ne && (ex[k] >> 31)) g[k] = ldCoh(&x[ex[k] & 0x7fffffffu]);
#pragma unroll
            for (int k = 0; k < NX; ++k)
                if (t + k * BS < ne) xl[nb + t + k * BS] = g[k];
            if (own(active, l)) xl[i] = gr;
            for (int c = t + NX * BS; c < ne; c += BS) {
                const unsigned ec = (unsigned)ext[e0 + c];
                xl[nb + c] = (ec >> 31) ? ldCoh(&x[ec & 0x7fffffffu]) : x[ec];
            }
            __syncthreads();
            for (int w = 0; w < nw; ++w) {
                if (active && myWave == w) {
                    XT sa = XT(0), sb = XT(0);
#pragma unroll
                    for (int u = 0; u + 1 < E; u += 2) {
                        sa += valOf<XT>(lv[u]) * xl[li[u]];
                        sb += valOf<XT>(lv[u + 1]) * xl[li[u + 1]];
                    }
                    if (E % 2) sa += valOf<XT>(lv[E - 1]) * xl[li[E - 1]];
                    const XT sm = laneSum<TPR>(sa + sb);
                    if (l == 0) xl[i] = (br - sm) * rd;
                }
                __syncthreads();
            }
            if (own(active, l)) stCoh(&x[row], xl[i]);
            __syncthreads();
        }
        // the flag goes out once every wave's stores of x are complete
        pending = cur;
        if (t == 0) sTicket = next;
        __syncthreads();
        cur = __builtin_amdgcn_readfirstlane(sTicket);
    }
    publish();
    // the last workgroup to finish prepares the next launch
    if (t == 0 && atomicAdd(&fs->done, 1) == (int)gridDim.x - 1) {
        if (ldAgent(&fs->abort)) {
            atomicAdd(&fs->aborts, 1);
            stAgent(&fs->abort, 0);
        }
        stAgent(&fs->ticket, 0);
        stAgent(&fs->done, 0);
        stAgent(&fs->epoch, epoch + 1);
    }
}

// Loads and stores of x in a Kaczmarz chain.  FLOW: the column id may carry
// bit 31 (written earlier in the one-launch sweep: read coherently), and
// every store is coherent; otherwise plain accesses.
template <bool FLOW, typename XT>
__device__ __forceinline__ XT ldX(const XT* x, unsigned id) {
    if constexpr (FLOW) {
        const XT* p = x + (id & 0x7fffffffu);
        return (id >> 31) ? ldCoh(p) : *p;
    } else {
        return x[id];
    }
}
template <bool FLOW, typename XT>
__device__ __forceinline__ void stX(XT* x, unsigned id, XT v) {
    if constexpr (FLOW)
        stCoh(x + (id & 0x7fffffffu), v);
    else
        x[id] = v;
}

// The local columns of a Kaczmarz bundle.  Each thread holds the ids of up to
// kColSlots columns (a bundle has at most 6144 by default, 4096 of them in one
// batch of 512 threads), so that all gathers of x are in flight together: one
// column per thread and round cost two dependent memory round trips per round,
// and the bundles of a long leaf have 4000 to 6000 columns
// (the graph of WaveSpans: 6.02 -> 5.60 ms).
//
// The ids that a thread holds over the waves of a bundle cost registers, so the
// kernels come with K of them; columns past K per thread are taken in further
// rounds.
//   kColSlots   where the time of a chain counts
//   kFewSlots   no bundle has more columns than that: the same loads with 16 to
//               24 registers less (256 threads, 8 entries a lane, FP64: 4 workgroups
//               per CU with kColSlots, 5 with kFewSlots), for sweeps with more
//               chains than find a place at once.  us per symmetric step, phase
//               launches, kColSlots / kFewSlots: 7-point 96^3 FP64 8 right-hand
//               sides 1292 / 1099, 128^3 3185 / 2625, FP32 2242 / 1504, one side 484
//               / 385; 27-point 112^3 8 sides FP64 5707 / 5581, FP32 3972 / 3390.
//               Larger bundles lose by it (band of 154560 rows, 1500 columns a
//               bundle of 256 threads 2246 / 2398).
//   kLeanSlots  batches that keep every place of the chip busy for several times
//               the longest chain path: also without the second index array of
//               an update, so that three workgroups of 512 threads share a CU
//               instead of two (BundleBatchFn::leanBatch)
constexpr int kColSlots = 8, kFewSlots = 4, kLeanSlots = 2;
template <int BS, int K>
__device__ __forceinline__ void loadCols(const int* __restrict__ ext, int e0, int ne, unsigned (&ex)[K]) {
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 2; ++k) ex[k] = (unsigned)ext[t + k * BS < ne ? e0 + t + k * BS : 0];
    if (K > 2 && ne > 2 * BS)
#pragma unroll
        for (int k = 2; k < K; ++k) ex[k] = (unsigned)ext[t + k * BS < ne ? e0 + t + k * BS : 0];
}
// x of the columns: to g first (issued together), then to LDS
template <int BS, bool FLOW, int K, typename XT>
__device__ __forceinline__ void gatherCols(const XT* x, int ne, const unsigned (&ex)[K], XT (&g)[K]) {
    const int t = threadIdx.x;
    auto slots = [&](auto k0, auto k1) {
#pragma unroll
        for (int k = k0; k < k1; ++k) g[k] = x[t + k * BS < ne && !(FLOW && ex[k] >> 31) ? ex[k] : 0u];
        if constexpr (FLOW)
#pragma unroll
            for (int k = k0; k < k1; ++k)
                if (t + k * BS < ne && ex[k] >> 31) g[k] = ldCoh(&x[ex[k] & 0x7fffffffu]);
    };
    slots(std::integral_constant<int, 0>{}, std::integral_constant<int, 2>{});
    if constexpr (K > 2)
        if (ne > 2 * BS) slots(std::integral_constant<int, 2>{}, std::integral_constant<int, K>{});
}
// columns of a round after the first
template <int K>
constexpr int kRound = K < 4 ? 4 : K;
template <int BS, bool FLOW, int K, typename XT>
__device__ __forceinline__ void placeCols(const XT* x, const int* __restrict__ ext, int e0, int ne, const XT (&g)[K],
                                          XT* xl) {
    constexpr int N = kRound<K>;
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (t + k * BS < ne) xl[t + k * BS] = g[k];
    for (int c0 = t + K * BS; c0 < ne; c0 += N * BS) {
        unsigned id[N];
        XT v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) id[k] = (unsigned)ext[e0 + (c0 + k * BS < ne ? c0 + k * BS : c0)];
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = ldX<FLOW>(x, id[k]);
#pragma unroll
        for (int k = 0; k < N; ++k)
            if (c0 + k * BS < ne) xl[c0 + k * BS] = v[k];
    }
}
template <int BS, bool FLOW, int K, typename XT>
__device__ __forceinline__ void storeCols(XT* x, const int* __restrict__ ext, int e0, int ne, const unsigned (&ex)[K],
                                          const XT* xl) {
    constexpr int N = kRound<K>;
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (t + k * BS < ne) stX<FLOW>(x, ex[k], xl[t + k * BS]);
    for (int c0 = t + K * BS; c0 < ne; c0 += N * BS) {
        unsigned id[N];
#pragma unroll
        for (int k = 0; k < N; ++k) id[k] = (unsigned)ext[e0 + (c0 + k * BS < ne ? c0 + k * BS : c0)];
#pragma unroll
        for (int k = 0; k < N; ++k)
            if (c0 + k * BS < ne) stX<FLOW>(x, id[k], xl[c0 + k * BS]);
    }
}

// The quotient d / rn by the row norm of which inv is the reciprocal: a
// division costs a wave's chain some twenty dependent FP64 operations, this
// three.  One Newton step makes it as exact as the division; a norm whose
// reciprocal is not finite is divided by.  For FP32 vectors the product alone
// is exact beyond the rounding to FP32.
template <typename XT>
__device__ __forceinline__ XT rowScale(double d, double rn, double inv) {
    const double q = d * inv;
    if constexpr (sizeof(XT) == 4) return (XT)q;
    if (!(inv <= 1.7976931348623157e308)) return (XT)(d / rn);
    const double c = __builtin_fma(__builtin_fma(-q, rn, d), inv, q);
    return (XT)(c == c ? c : q);  // an infinite quotient has no remainder
}

// Kaczmarz, the bundles [cLo, cHi) of a chain for right-hand side k: every
// column a bundle touches lives in LDS; rows of one wave share no column.  The
// row norms stay FP64.  The next bundle's offsets, column ids and row ids are
// requested before the current one's waves run, so that a bundle starts with
// the gathers of x and the entries.
template <int BS, int TPR, int E, typename VT, typename XT, bool BATCH, bool FLOW, int K>
__device__ __forceinline__ void kaczChain(
    const int cLo, const int cHi, const int k, XT* xl, const int spare, const int* __restrict__ bSlot,
    const int* __restrict__ bWave, const long* __restrict__ bOff, const int* __restrict__ bLen,
    const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave, const int* __restrict__ rowId,
    const double* __restrict__ rowNorm, const int* __restrict__ ext, const uint16_t* __restrict__ sidx,
    const VT* __restrict__ sval, long zero, XT* x0, const XT* __restrict__ b0, int n0, XT* const* __restrict__ bX,
    const XT* const* __restrict__ bB, const int* __restrict__ bN) {
    constexpr bool LEAN = K == kLeanSlots;
    if (cLo >= cHi) return;
    const BundleVec<BATCH, XT> vec(x0, b0, n0, bX, bB, bN, cLo);
    const size_t vo = (size_t)k * vec.n;
    XT* __restrict__ x = vec.x + vo;
    const XT* __restrict__ b = vec.b + vo;
    const int t = threadIdx.x, i = t / TPR;

    int s0 = bSlot[cLo], nb = bSlot[cLo + 1] - s0;
    int e0 = bExt[cLo], ne = bExt[cLo + 1] - e0;
    unsigned ex[K], row = (unsigned)rowId[i < nb ? s0 + i : 0];
    loadCols<BS>(ext, e0, ne, ex);
    for (int bnd = cLo;;) {
        const long off = bOff[bnd];
        const int wb = bLen[bnd];
        const int nw = bWave[bnd + 1] - bWave[bnd];
        const bool active = i < nb;
        const long lanes = (long)nb * TPR;
        // branch-free entry loads (as in k_gs_bundle)
        const int sr = active ? s0 + i : 0;
        int li[E];
        typename ValBits<VT>::T lv[E];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const long e = (active && u < wb) ? off + (long)u * lanes + t : zero;
            li[u] = (int)sidx[e];
            lv[u] = sval[e];
        }
        const double rn = rowNorm[sr];
        const int myWave = (int)slotWave[sr];
        XT g[K];
        gatherCols<BS, FLOW>(x, ne, ex, g);
        const XT br = b[active ? row : 0u];
        placeCols<BS, FLOW>(x, ext, e0, ne, g, xl);
        // behind the gathers, as these wait for the entries
        const double rnInv = 1.0 / rn;
        // where an entry's update goes: an entry of value 0 (a padding entry
        // may name a column another row updates) to a spare place behind the
        // columns, or, LEAN, nowhere
        int lw[LEAN ? 1 : E];
        if constexpr (!LEAN)
#pragma unroll
            for (int u = 0; u < E; ++u) lw[u] = valOf<XT>(lv[u]) != XT(0) ? li[u] : ne + (t & (spare - 1));
        __syncthreads();
        const bool more = bnd + 1 < cHi;
        int s0n = 0, nbn = 0, e0n = 0, nen = 0;
        unsigned exn[K] = {}, rown = 0;
        if (more) {
            s0n = bSlot[bnd + 1], nbn = bSlot[bnd + 2] - s0n;
            e0n = bExt[bnd + 1], nen = bExt[bnd + 2] - e0n;
            rown = (unsigned)rowId[i < nbn ? s0n + i : 0];
            loadCols<BS>(ext, e0n, nen, exn);
        }
        for (int w = 0; w < nw; ++w) {
            if (active && myWave == w) {
                // the row's x entries, read once in one batch (no other
                // row of this wave writes them)
                XT cur[E];
#pragma unroll
                for (int u = 0; u < E; ++u) cur[u] = xl[li[u]];
                // two partial sums: half the dependent FMA chain
                XT sa = XT(0), sb = XT(0);
#pragma unroll
                for (int u = 0; u + 1 < E; u += 2) {
                    sa += valOf<XT>(lv[u]) * cur[u];
                    sb += valOf<XT>(lv[u + 1]) * cur[u + 1];
                }
                if (E % 2) sa += valOf<XT>(lv[E - 1]) * cur[E - 1];
                const XT dot = laneSum<TPR>(sa + sb);
                const XT scale = rowScale<XT>((double)dot - (double)br, rn, rnInv);
#pragma unroll
                for (int u = 0; u < E; ++u) {
                    const XT a = valOf<XT>(lv[u]);
                    if constexpr (!LEAN)
                        xl[lw[u]] = cur[u] - scale * a;
                    else if (a != XT(0))
                        xl[li[u]] = cur[u] - scale * a;
                }
            }
            __syncthreads();
        }
        storeCols<BS, FLOW>(x, ext, e0, ne, ex, xl);
        __syncthreads();
        if (!more) break;
        ++bnd;
        s0 = s0n, nb = nbn, e0 = e0n, ne = nen, row = rown;
#pragma unroll
        for (int q = 0; q < K; ++q) ex[q] = exn[q];
    }
}

template <int BS, int TPR, int E, typename VT, typename XT, bool BATCH, int K>
__global__ void __launch_bounds__(BS) k_kacz_bundle(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const double* __restrict__ rowNorm, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* __restrict__ x0,
    const XT* __restrict__ b0, int n0, int nrhs, const int* __restrict__ chainPtr, int chain0, int nchain, int xcd,
    int spare, XT* const* __restrict__ bX, const XT* const* __restrict__ bB, const int* __restrict__ bN) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);

    const int q = bundleOfBlock(nchain, xcd);
    if (q < 0) return;
    // a chain: one bundle, or the segments of a leaf too large for one bundle,
    // run in order (each segment reads what the previous one wrote)
    const int cLo = chainPtr[chain0 + q], cHi = chainPtr[chain0 + q + 1];
    // right-hand sides are independent: one per grid.y
    kaczChain<BS, TPR, E, VT, XT, BATCH, false, K>(cLo, cHi, (int)blockIdx.y, xl, spare, bSlot, bWave, bOff, bLen, bExt,
                                                slotWave, rowId, rowNorm, ext, sidx, sval, zero, x0, b0, n0, bX, bB, bN);
}

// Readiness-driven one-launch sweep.  A workgroup takes a queue position
// (ticket) and runs the chain stored there: the chains without dependencies
// occupy the first positions (roots), every other chain is appended by the
// workgroup that completes its last dependency.  So a workgroup never holds
// a chain whose dependencies are still running (with tickets in chain order,
// a matrix of a batch with a few long chains holds the slots of every other
// matrix's later phases).  No deadlock: a workgroup takes a position only
// after releasing the successors of its previous chain, and while positions
// wait for chains, some chain with finished dependencies has been queued.
// Per right-hand side (blockIdx.y) its own queue, arrival counters and state.
struct ReadyTables {
    const int* lo;             // chain -> first bundle
    const int* hi;             // chain -> end of its bundles
    const int* depPtr;         // chain -> its dependencies (their count)
    const int* succPtr;        // chain -> chains depending on it
    const int* succ;
    const int* roots;          // chains without dependencies
    unsigned* arrivals;        // per side: completed dependencies, summed over launches
    unsigned long long* queue; // per side: (epoch << 32) | chain, from position nroots on
    FlowState* fs;             // per side
    int nchain, nroots, pollLimit;
};

// the chain at queue position h (>= nroots) once it has been written, or
// -1 when the launch gives up (see waitChain)
__device__ __forceinline__ int waitQueue(const unsigned long long* q, int h, int epoch, FlowState* fs, int pollLimit) {
    int polls = 0;
    for (;;) {
        const unsigned long long v =
            __hip_atomic_load(const_cast<unsigned long long*>(&q[h]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((int)(v >> 32) == epoch) return (int)(unsigned)v;
        if ((++polls & 255) == 0 && (polls >= pollLimit || ldAgent(&fs->abort))) {
            stAgent(&fs->abort, 1);
            return -1;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

template <int BS, class Body>
__device__ __forceinline__ void readyLoop(const ReadyTables& r, Body&& body) {
    __shared__ int sChain;
    const int t = threadIdx.x;
    FlowState* fs = r.fs + blockIdx.y;
    unsigned* arr = r.arrivals + (size_t)blockIdx.y * r.nchain;
    unsigned long long* q = r.queue + (size_t)blockIdx.y * r.nchain;
    const int epoch = ldAgent(&fs->epoch);
    for (;;) {
        if (t == 0) {
            const int h = atomicAdd(&fs->ticket, 1);
            sChain = h < r.nroots ? r.roots[h] : h < r.nchain ? waitQueue(q, h, epoch, fs, r.pollLimit) : -1;
        }
        __syncthreads();
        const int c = __builtin_amdgcn_readfirstlane(sChain);
        if (c < 0) break;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        body(r.lo[c], r.hi[c]);
        // every wave's stores of x are complete before any successor is released
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        const int s0 = r.succPtr[c], ns = r.succPtr[c + 1] - s0;
        for (int j = t; j < ns; j += BS) {
            const int sc = r.succ[s0 + j];
            const unsigned need = (unsigned)epoch * (unsigned)(r.depPtr[sc + 1] - r.depPtr[sc]);
            if (atomicAdd(&arr[sc], 1u) + 1u == need) {
                const int slot = atomicAdd(&fs->tail, 1);
                __hip_atomic_store(&q[slot], ((unsigned long long)(unsigned)epoch << 32) | (unsigned)sc,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    // the last workgroup to finish prepares the next launch
    if (t == 0 && atomicAdd(&fs->done, 1) == (int)gridDim.x - 1) {
        if (ldAgent(&fs->abort)) {
            atomicAdd(&fs->aborts, 1);
            stAgent(&fs->abort, 0);
        }
        stAgent(&fs->ticket, 0);
        stAgent(&fs->tail, r.nroots);
        stAgent(&fs->done, 0);
        stAgent(&fs->epoch, epoch + 1);
    }
}

// Kaczmarz, all phases of a sweep in one readiness-driven launch; grid.y =
// right-hand sides.
template <int BS, int TPR, int E, typename VT, typename XT, bool BATCH, int K>
__global__ void __launch_bounds__(BS) k_kacz_flow(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const double* __restrict__ rowNorm, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* x0, const XT* __restrict__ b0,
    int n0, int spare, XT* const* __restrict__ bX, const XT* const* __restrict__ bB, const int* __restrict__ bN,
    ReadyTables rt) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);
    const int k = (int)blockIdx.y;
    readyLoop<BS>(rt, [&](int cLo, int cHi) {
        kaczChain<BS, TPR, E, VT, XT, BATCH, true, K>(cLo, cHi, k, xl, spare, bSlot, bWave, bOff, bLen, bExt, slotWave,
                                                   rowId, rowNorm, ext, sidx, sval, zero, x0, b0, n0, bX, bB, bN);
    });
}

// v of the lane that the DPP control names; 0 where there is none (MASK: the
// 16-lane rows that take part)
template <int CTRL, int MASK>
__device__ __forceinline__ float dppMove(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, MASK, 0xF, false));
}
template <int CTRL, int MASK>
__device__ __forceinline__ double dppMove(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, MASK, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, MASK, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The sum over the lanes [lo, hi) of a row, for all of them, in a fixed order
// without atomics; lanes of rows that are not summed now pass mine = false.
// A row inside one wavefront: a segmented scan with DPP moves (VALU, no LDS
// round trips), whose last lane's total goes to the others (the graph of
// WaveSpans: 5.60 ms with a tree of LDS shuffles, 4.36 with this).  Rows of a
// wave spread over wavefronts: through LDS, with a barrier for every thread.
template <typename XT>
__device__ __forceinline__ XT rowSum(bool mine, bool spread, XT v, XT* part, int lo, int hi) {
    const int t = threadIdx.x;
    if (!spread) {
        const int lane = t & 63, l0 = mine ? lo & 63 : 64;
        XT u;
        u = dppMove<0x111, 0xF>(v);  // row_shr:1, 2, 4, 8: inside 16 lanes
        v += lane - 1 >= l0 ? u : XT(0);
        u = dppMove<0x112, 0xF>(v);
        v += lane - 2 >= l0 ? u : XT(0);
        u = dppMove<0x114, 0xF>(v);
        v += lane - 4 >= l0 ? u : XT(0);
        u = dppMove<0x118, 0xF>(v);
        v += lane - 8 >= l0 ? u : XT(0);
        u = dppMove<0x142, 0xA>(v);  // row_bcast:15: lane 15 to 16-31, 47 to 48-63
        v += (lane & 48) > l0 ? u : XT(0);
        u = dppMove<0x143, 0xC>(v);  // row_bcast:31: lane 31 to 32-63
        v += (lane & 32) > l0 ? u : XT(0);
        return __shfl(v, mine ? (hi - 1) & 63 : 0);
    }
    if (mine) part[t] = v;
    __syncthreads();
    XT s = XT(0);
    if (mine)
        for (int l = lo; l < hi; ++l) s += part[l];
    return s;
}

// ---------------------------------------------------------------------------
// Variable lanes per row (matrices with a few very long rows): the row of
// slot i owns lanes [lane0(i), lane0(i+1)) of the bundle, each holding up to
// kVarE entries in registers, and the lanes of a row add up their partial sums
// (rowSum).
template <int BS, typename VT, typename XT, bool BATCH>
__global__ void __launch_bounds__(BS) k_gs_bundle_vl(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const XT* __restrict__ diag, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* __restrict__ x0,
    const XT* __restrict__ b0, int n0, int nrhs, const int* __restrict__ chainPtr, int chain0, int nchain, int xcd,
    int ldsLocal, const int* __restrict__ lanePtr, const uint16_t* __restrict__ laneSlot,
    XT* const* __restrict__ bX, const XT* const* __restrict__ bB, const int* __restrict__ bN) {
    constexpr int E = kVarE;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ WaveSpans<BS / 64> spans;
    XT* xl = reinterpret_cast<XT*>(smem);
    XT* part = xl + ldsLocal;                               // BS partial sums
    int* rl0 = reinterpret_cast<int*>(part + BS);           // row -> first lane

    const int q = bundleOfBlock(nchain, xcd);
    if (q < 0) return;
    const int cLo = chainPtr[chain0 + q], cHi = chainPtr[chain0 + q + 1];
    auto runBundle = [&](const int bnd) {
        const BundleVec<BATCH, XT> vec(x0, b0, n0, bX, bB, bN, bnd);
        XT* __restrict__ x = vec.x;
        const XT* __restrict__ b = vec.b;
        const int n = vec.n;
        const int s0 = bSlot[bnd], nb = bSlot[bnd + 1] - s0;
        const long off = bOff[bnd];
        const int wb = bLen[bnd];
        const int nw = bWave[bnd + 1] - bWave[bnd];
        const int e0 = bExt[bnd], ne = bExt[bnd + 1] - e0;
        const int lp = lanePtr[bnd], nl = lanePtr[bnd + 1] - lp;
        const int t = threadIdx.x;
        const bool active = t < nl;
        // branch-free prologue, ids first (as in k_gs_bundle); the first
        // lane of every row goes to LDS and is read after the barrier that
        // follows the gathers
        const unsigned ex0 = (unsigned)ext[t < ne ? e0 + t : 0];
        const unsigned ex1 = (unsigned)ext[t + BS < ne ? e0 + t + BS : 0];
        const int i = (int)laneSlot[active ? lp + t : 0];  // used by active lanes only
        const int iPrev = (int)laneSlot[active && t > 0 ? lp + t - 1 : 0];
        int li[E];
        typename ValBits<VT>::T lv[E];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const long e = (active && u < wb) ? off + (long)u * nl + t : zero;
            li[u] = (int)sidx[e];
            lv[u] = sval[e];
        }
        const bool first = active && (t == 0 || iPrev != i);
        const int sr = active ? s0 + i : 0;
        const unsigned row = (unsigned)rowId[sr];
        const XT dg = diag[sr];  // 1 / a_rr
        const int myWave = (int)slotWave[sr];
        if (first) rl0[i] = t;
        if (t == 0) rl0[nb] = nl;
        int rowL0 = 0, rowL1 = 0;

        const int k0 = (int)blockIdx.y;
        const int k1 = gridDim.y > 1 ? k0 + 1 : nrhs;
        for (int k = k0; k < k1; ++k) {
            const size_t vo = (size_t)k * n;
            const XT g0 = x[vo + (t < ne ? ex0 : 0u)];
            const XT g1 = x[vo + (t + BS < ne ? ex1 : 0u)];
            const XT gr = x[vo + (first ? row : 0u)];
            const XT br = b[vo + (first ? row : 0u)];
            if (k == k0) setSpans(spans, active, myWave);
            if (t < ne) xl[nb + t] = g0;
            if (t + BS < ne) xl[nb + t + BS] = g1;
            if (first) xl[i] = gr;
            for (int c = t + 2 * BS; c < ne; c += BS) xl[nb + c] = x[vo + ext[e0 + c]];
            __syncthreads();
            if (k == k0 && active) {
                rowL0 = rl0[i];
                rowL1 = rl0[i + 1];
            }
            runWaves(spans, nw, [&](int w, bool spread) {
                const bool mine = active && myWave == w;
                XT sum = XT(0);
                if (mine) {
                    XT sb = XT(0);
#pragma unroll
                    for (int u = 0; u < E; u += 2) {
                        sum += valOf<XT>(lv[u]) * xl[li[u]];
                        sb += valOf<XT>(lv[u + 1]) * xl[li[u + 1]];
                    }
                    sum += sb;
                }
                sum = rowSum(mine, spread, sum, part, rowL0, rowL1);
                if (mine && first) xl[i] = (br - sum) * dg;
            });
            if (first) x[vo + row] = xl[i];
            __syncthreads();
        }
    };
    if (cHi == cLo + 1) {
        runBundle(cLo);
    } else {
        for (int bnd = cLo; bnd < cHi; ++bnd) {
            runBundle(bnd);
            __syncthreads();
        }
    }
}

// Variable lanes per row, Kaczmarz (see kaczChain).  part: BS partial
// sums, rl0: the first lane of every row of the bundle.  A bundle without
// columns of its own works in those of the bundle before it (residentChains);
// they are stored before the next bundle that has columns and after the last.
template <int BS, typename VT, typename XT, bool BATCH, bool FLOW, int K>
__device__ __forceinline__ void kaczChainVL(
    const int cLo, const int cHi, const int k, XT* xl, const int spare, XT* part, int* rl0,
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const double* __restrict__ rowNorm, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* x0, const XT* __restrict__ b0,
    int n0, const int* __restrict__ lanePtr, const uint16_t* __restrict__ laneSlot, XT* const* __restrict__ bX,
    const XT* const* __restrict__ bB, const int* __restrict__ bN) {
    constexpr int E = kVarE;
    __shared__ WaveSpans<BS / 64> spans;
    constexpr bool LEAN = K == kLeanSlots;
    if (cLo >= cHi) return;
    const BundleVec<BATCH, XT> vec(x0, b0, n0, bX, bB, bN, cLo);
    const size_t vo = (size_t)k * vec.n;
    XT* __restrict__ x = vec.x + vo;
    const XT* __restrict__ b = vec.b + vo;
    const int t = threadIdx.x;

    int s0 = bSlot[cLo], e0 = bExt[cLo], ne = bExt[cLo + 1] - e0;
    int lp = lanePtr[cLo], nl = lanePtr[cLo + 1] - lp;
    unsigned ex[K];
    loadCols<BS>(ext, e0, ne, ex);
    int i = (int)laneSlot[t < nl ? lp + t : 0];  // used by active lanes only
    bool load = true;
    for (int bnd = cLo;;) {
        const int nb = bSlot[bnd + 1] - s0;
        const long off = bOff[bnd];
        const int wb = bLen[bnd];
        const int nw = bWave[bnd + 1] - bWave[bnd];
        const bool active = t < nl;
        const int sr = active ? s0 + i : 0;
        const unsigned row = (unsigned)rowId[sr];
        const double rn = rowNorm[sr];
        const int myWave = (int)slotWave[sr];
        const int iPrev = (int)laneSlot[active && t > 0 ? lp + t - 1 : 0];
        int li[E];
        typename ValBits<VT>::T lv[E];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const long e = (active && u < wb) ? off + (long)u * nl + t : zero;
            li[u] = (int)sidx[e];
            lv[u] = sval[e];
        }
        XT g[K];
        if (load) gatherCols<BS, FLOW>(x, ne, ex, g);
        const XT br = b[active ? row : 0u];
        if (load) placeCols<BS, FLOW>(x, ext, e0, ne, g, xl);
        // behind the gathers, as in kaczChain
        setSpans(spans, active, myWave);
        if (active && (t == 0 || iPrev != i)) rl0[i] = t;
        if (t == 0) rl0[nb] = nl;
        const double rnInv = 1.0 / rn;
        int lw[LEAN ? 1 : E];
        if constexpr (!LEAN)
#pragma unroll
            for (int u = 0; u < E; ++u) lw[u] = valOf<XT>(lv[u]) != XT(0) ? li[u] : ne + (t & (spare - 1));
        __syncthreads();
        const int rowL0 = active ? rl0[i] : 0, rowL1 = active ? rl0[i + 1] : 0;
        const bool more = bnd + 1 < cHi;
        int s0n = 0, e0n = 0, nen = 0, lpn = 0, nln = 0, in = 0;
        unsigned exn[K] = {};
        if (more) {
            s0n = bSlot[bnd + 1];
            e0n = bExt[bnd + 1], nen = bExt[bnd + 2] - e0n;
            lpn = lanePtr[bnd + 1], nln = lanePtr[bnd + 2] - lpn;
            if (LEAN || nen > 0) loadCols<BS>(ext, e0n, nen, exn);
            in = (int)laneSlot[t < nln ? lpn + t : 0];
        }
        runWaves(spans, nw, [&](int w, bool spread) {
            const bool mine = active && myWave == w;
            // the lane's x entries, read once in one batch and kept
            // (no other row of this wave writes them)
            XT cur[E], dot = XT(0);
            if (mine) {
#pragma unroll
                for (int u = 0; u < E; ++u) cur[u] = xl[li[u]];
                XT sb = XT(0);
#pragma unroll
                for (int u = 0; u < E; u += 2) {
                    dot += valOf<XT>(lv[u]) * cur[u];
                    sb += valOf<XT>(lv[u + 1]) * cur[u + 1];
                }
                dot += sb;
            }
            const XT rowDot = rowSum(mine, spread, dot, part, rowL0, rowL1);
            if (mine) {
                const XT scale = rowScale<XT>((double)rowDot - (double)br, rn, rnInv);
#pragma unroll
                for (int u = 0; u < E; ++u) {
                    const XT a = valOf<XT>(lv[u]);
                    if constexpr (!LEAN)
                        xl[lw[u]] = cur[u] - scale * a;
                    else if (a != XT(0))
                        xl[li[u]] = cur[u] - scale * a;
                }
            }
        });
        load = LEAN || nen > 0;
        if (load || !more) storeCols<BS, FLOW>(x, ext, e0, ne, ex, xl);
        __syncthreads();
        if (!more) break;
        ++bnd;
        s0 = s0n, lp = lpn, nl = nln, i = in;
        if (load) {
            e0 = e0n, ne = nen;
#pragma unroll
            for (int q = 0; q < K; ++q) ex[q] = exn[q];
        }
    }
}

template <int BS, typename VT, typename XT, bool BATCH, int K>
__global__ void __launch_bounds__(BS) k_kacz_bundle_vl(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const double* __restrict__ rowNorm, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* __restrict__ x0,
    const XT* __restrict__ b0, int n0, int nrhs, const int* __restrict__ chainPtr, int chain0, int nchain, int xcd,
    int ldsLocal, int spare, const int* __restrict__ lanePtr, const uint16_t* __restrict__ laneSlot,
    XT* const* __restrict__ bX, const XT* const* __restrict__ bB, const int* __restrict__ bN) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);
    XT* part = xl + ldsLocal + spare;                       // BS partial sums
    int* rl0 = reinterpret_cast<int*>(part + BS);           // row -> first lane

    const int q = bundleOfBlock(nchain, xcd);
    if (q < 0) return;
    const int cLo = chainPtr[chain0 + q], cHi = chainPtr[chain0 + q + 1];
    kaczChainVL<BS, VT, XT, BATCH, false, K>(cLo, cHi, (int)blockIdx.y, xl, spare, part, rl0, bSlot, bWave, bOff, bLen,
                                          bExt, slotWave, rowId, rowNorm, ext, sidx, sval, zero, x0, b0, n0, lanePtr,
                                          laneSlot, bX, bB, bN);
}

// Kaczmarz with variable lanes per row, all phases of a sweep in one launch.
template <int BS, typename VT, typename XT, bool BATCH, int K>
__global__ void __launch_bounds__(BS, K == kLeanSlots ? 4 : 1) k_kacz_flow_vl(
    const int* __restrict__ bSlot, const int* __restrict__ bWave, const long* __restrict__ bOff,
    const int* __restrict__ bLen, const int* __restrict__ bExt, const uint16_t* __restrict__ slotWave,
    const int* __restrict__ rowId, const double* __restrict__ rowNorm, const int* __restrict__ ext,
    const uint16_t* __restrict__ sidx, const VT* __restrict__ sval, long zero, XT* x0, const XT* __restrict__ b0,
    int n0, int ldsLocal, int spare, const int* __restrict__ lanePtr, const uint16_t* __restrict__ laneSlot,
    XT* const* __restrict__ bX, const XT* const* __restrict__ bB, const int* __restrict__ bN,
    ReadyTables rt) {
    extern __shared__ __align__(16) unsigned char smem[];
    XT* xl = reinterpret_cast<XT*>(smem);
    XT* part = xl + ldsLocal + spare;
    int* rl0 = reinterpret_cast<int*>(part + BS);
    const int k = (int)blockIdx.y;
    readyLoop<BS>(rt, [&](int cLo, int cHi) {
        kaczChainVL<BS, VT, XT, BATCH, true, K>(cLo, cHi, k, xl, spare, part, rl0, bSlot, bWave, bOff, bLen, bExt, slotWave,
                                             rowId, rowNorm, ext, sidx, sval, zero, x0, b0, n0, lanePtr, laneSlot, bX,
                                             bB, bN);
    });
}

// (lanes per row, register width) pairs with a uniform kernel
// instantiation; longer rows use variable lanes per row
int pickE(int tpr, int need) {
    static const int e1[] = {4, 8, 16}, e2[] = {8, 13, 16}, e4[] = {8, 16};
    if (tpr != 1 && tpr != 2 && tpr != 4) return -1;
    const int* c = tpr == 1 ? e1 : tpr == 2 ? e2 : e4;
    const int nc = tpr == 4 ? 2 : 3;
    for (int q = 0; q < nc; ++q)
        if (c[q] >= need) return c[q];
    return -1;
}

// LDS of a workgroup: bytes, and the spare places behind the local columns
// (one per lane of a wavefront, or what 32 bytes hold where LDS is short)
struct LdsPlan {
    size_t bytes;
    int spare;
};
// beside the local columns: with variable lanes a partial sum per lane and the
// first lane of every row
template <typename XT>
size_t ldsBeside(int rows, int tpr, int bs) {
    return tpr == 0 ? (size_t)bs * sizeof(XT) + (size_t)(rows + 1) * sizeof(int) : 0;
}
template <typename XT>
LdsPlan ldsPlan(int local, int rows, int tpr, int bs, size_t limit) {
    const size_t need = (size_t)local * sizeof(XT) + ldsBeside<XT>(rows, tpr, bs);
    const int spare = need + 64 * sizeof(XT) <= limit ? 64 : 32 / (int)sizeof(XT);
    return {need + spare * sizeof(XT), spare};
}

// a bundle's prologue, gathers and stores, in dependency waves (weight of a
// bundle in the longest-path estimate of a readiness-driven sweep)
constexpr int kBundleFixedWaves = 4;

// A sweep in dependency waves plus kBundleFixedWaves per bundle: all its
// chains, the longest of them, and the longest of every phase added up
struct SweepCost {
    long all = 0, longest = 0, phases = 0;
    explicit SweepCost(const BundleTable& t) {
        for (int p = 0; p < t.numPhases(); ++p) {
            long most = 0;
            for (int c = t.phaseChain[p]; c < t.phaseChain[p + 1]; ++c) {
                const int b0 = t.chainPtr[c], b1 = t.chainPtr[c + 1];
                const long cost = t.wave[b1] - t.wave[b0] + (long)kBundleFixedWaves * (b1 - b0);
                all += cost;
                most = std::max(most, cost);
            }
            longest = std::max(longest, most);
            phases += most;
        }
    }
};

// Long Kaczmarz chains whose columns fit the LDS of a whole CU keep them there
// from the first bundle to the last instead of gathering and storing some 5000
// scattered columns per bundle (the graph of WaveSpans: 4.34 -> 3.65 ms a sweep;
// a batch with eight such graphs and eight right-hand sides, both sweeps and a
// symmetric product: 10.2 -> 7.6 ms).  Loading the next bundle's entries and row
// data behind the current waves as well gave nothing (3.71 ms).
// A workgroup then has its CU to itself, so only where one workgroup per CU
// gets through all other chains in the time of the longest one.  Short chains
// gain nothing.
constexpr int kResidentBundles = 8;
constexpr size_t kStaticLds = 1024;  // spans, tickets: less than this
// most columns of a chain to keep, 0 for none; limit: LDS of a workgroup then
template <typename XT>
int residentCols(const BundleTable& t, int nrhs, int bs, size_t* limit, int* cols) {
    *cols = 0;
    const SweepCost sweep(t);
    int dev = 0, cus = 0, lds = 0, rows = 0;
    RACE_HIP(hipGetDevice(&dev));
    RACE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    RACE_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    for (int r : t.phRows) rows = std::max(rows, r);
    *limit = (size_t)std::max(0, lds) > kStaticLds ? (size_t)lds - kStaticLds : 0;
    const size_t beside = ldsBeside<XT>(rows, t.tpr, bs) + 64 * sizeof(XT);
    if (sweep.all * nrhs <= sweep.longest * cus && *limit > std::max(beside, kMaxLds))
        *cols = (int)((*limit - beside) / sizeof(XT));
    return OK;
}

template <typename VT, typename XT>
struct BundleDev {
    BundleTable h;
    DevBuf<int> slot, wave, len, ext, extPtr, rowId, chainPtr, lanePtr;
    DevBuf<uint16_t> laneSlot, slotWave;
    DevBuf<long> off;
    DevBuf<uint16_t> sidx;
    DevBuf<VT> sval;
    long zero = 0;  // index of the zero entry in sidx / sval
    DevBuf<XT> diag;
    DevBuf<double> rowNorm;
    size_t maxLds = kMaxLds;
    bool fewCols = false;  // Kaczmarz, uniform lanes: kernels with kFewSlots hold the columns of every bundle
    // LDS a workgroup of bs threads needs, at most maxLds: false if a phase
    // needs more
    bool fits(int bs) const {
        for (int p = 0; p < h.numPhases(); ++p)
            if (lds(p, bs).bytes > maxLds) return false;
        return true;
    }
    int load(BundleTable&& t, int bs, int nrhs) {
        h = std::move(t);
        int e;
        if (h.kind == RACE_K_KACZ && h.tpr == 0 && fits(bs)) {
            size_t limit = 0;
            int cols = 0;
            if ((e = residentCols<XT>(h, nrhs, bs, &limit, &cols))) return e;
            if (cols > 0 && residentChains(h, kResidentBundles, cols)) maxLds = limit;
        }
        if (h.kind == RACE_K_KACZ && h.tpr > 0) {
            int widest = 0;
            for (size_t b = 0; b + 1 < h.extPtr.size(); ++b) widest = std::max(widest, h.extPtr[b + 1] - h.extPtr[b]);
            fewCols = widest <= kFewSlots * bs;
        }
        if ((e = upload(slot, h.slot.data(), h.slot.size()))) return e;
        if ((e = upload(wave, h.wave.data(), h.wave.size()))) return e;
        if ((e = upload(len, h.len.data(), h.len.size()))) return e;
        if ((e = upload(off, h.off.data(), h.off.size()))) return e;
        if ((e = upload(ext, h.ext.data(), h.ext.size()))) return e;
        if ((e = upload(extPtr, h.extPtr.data(), h.extPtr.size()))) return e;
        if ((e = upload(chainPtr, h.chainPtr.data(), h.chainPtr.size()))) return e;
        if (h.tpr == 0) {
            if ((e = upload(lanePtr, h.lanePtr.data(), h.lanePtr.size()))) return e;
            if ((e = upload(laneSlot, h.laneSlot.data(), h.laneSlot.size()))) return e;
        }
        if ((e = upload(rowId, h.rowId.data(), h.rowId.size()))) return e;
        // the zero entry: what a lane loads for an entry it does not have
        zero = (long)h.sidx.size();
        h.sidx.push_back(0);
        h.sval.push_back(0.0);
        if ((e = upload(sidx, h.sidx.data(), h.sidx.size()))) return e;
        std::vector<VT> v(h.sval.size());
        for (size_t q = 0; q < v.size(); ++q) v[q] = conv(h.sval[q]);
        if ((e = upload(sval, v.data(), v.size()))) return e;
        if (h.kind == RACE_K_KACZ) {
            if ((e = upload(rowNorm, h.rowNorm.data(), h.rowNorm.size()))) return e;
        } else {
            // Gauss-Seidel multiplies by the inverse diagonal
            std::vector<XT> dg(h.diag.size());
            for (size_t q = 0; q < dg.size(); ++q) dg[q] = (XT)(1.0 / h.diag[q]);
            if ((e = upload(diag, dg.data(), dg.size()))) return e;
        }
        // slot -> its wave inside the bundle (a bundle holds at most 8192 rows)
        std::vector<uint16_t> sw(h.rowId.size(), 0);
        for (size_t bd = 0; bd + 1 < h.wave.size(); ++bd)
            for (int w = h.wave[bd]; w < h.wave[bd + 1]; ++w)
                for (int sl = h.waveSlot[w]; sl < h.waveSlot[w + 1]; ++sl)
                    sw[sl] = (uint16_t)(w - h.wave[bd]);
        if ((e = upload(slotWave, sw.data(), sw.size()))) return e;
        // the host copies of the big arrays are no longer needed
        std::vector<uint16_t>().swap(h.sidx);
        std::vector<double>().swap(h.sval);
        return OK;
    }
    static VT conv(double v) {
        if constexpr (sizeof(VT) == 2)
            return toBf16(v);
        else
            return (VT)v;
    }
    // LDS bytes of phase p for workgroups of bs threads: the local column
    // space, the spare places behind it and, with variable lanes, a partial
    // sum per lane and the first lane of every row
    LdsPlan lds(int p, int bs) const { return ldsPlan<XT>(h.phLocal[p], h.phRows[p], h.tpr, bs, maxLds); }
};

// one fused or plain launch of the chains [c0, c0 + nchain) of phase p
template <int BS, int TPR, int EE, typename VT, typename XT, bool BATCH>
void launchBundles(int kind, int nrhs, const BundleDev<VT, XT>& d, int c0, int nchain, int p, int xcd, XT* x,
                   const XT* b, int n, XT* const* bX, const XT* const* bB, const int* bN, hipStream_t st) {
    const dim3 grid(xcd ? 8u * (unsigned)((nchain + 7) / 8) : (unsigned)nchain, (unsigned)std::max(1, nrhs));
    // chains of one bundle each: the kernel indexes bundles directly
    const std::vector<int>& cp = d.h.chainPtr;
    const int bundle0 = cp[c0 + nchain] - cp[c0] == nchain ? cp[c0] : -1;
    if (kind == RACE_K_KACZ) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(BS), d.lds(p, BS).bytes, st, d.slot.p, d.wave.p, d.off.p, d.len.p,
                               d.extPtr.p, d.slotWave.p, d.rowId.p, d.rowNorm.p, d.ext.p, d.sidx.p, d.sval.p, d.zero, x,
                               b, n, nrhs, d.chainPtr.p, c0, nchain, xcd, d.lds(p, BS).spare, bX, bB, bN);
        };
        if (d.fewCols)
            launch(k_kacz_bundle<BS, TPR, EE, VT, XT, BATCH, kFewSlots>);
        else
            launch(k_kacz_bundle<BS, TPR, EE, VT, XT, BATCH, kColSlots>);
    } else if (nrhs == 1 && (BS == 256 || BS == 512) && !BATCH && d.h.phExt[p] > 2 * BS)
        // many outside columns: gather up to 1536 (256 threads) or 2048
        // (512 threads) of them in one batch
        hipLaunchKernelGGL((k_gs_bundle<BS, TPR, EE, VT, XT, true, BATCH, (BS == 256 ? 6 : 4)>), dim3(grid.x), dim3(BS),
                           d.lds(p, BS).bytes, st, d.slot.p, d.wave.p, d.off.p, d.len.p, d.extPtr.p, d.slotWave.p, d.rowId.p, d.diag.p,
                           d.ext.p, d.sidx.p, d.sval.p, d.zero, x, b, n, nrhs, d.chainPtr.p, c0, nchain, bundle0, xcd, bX,
                           bB, bN);
    else if (nrhs == 1)
        hipLaunchKernelGGL((k_gs_bundle<BS, TPR, EE, VT, XT, true, BATCH>), dim3(grid.x), dim3(BS), d.lds(p, BS).bytes, st,
                           d.slot.p, d.wave.p, d.off.p, d.len.p, d.extPtr.p, d.slotWave.p, d.rowId.p, d.diag.p,
                           d.ext.p, d.sidx.p, d.sval.p, d.zero, x, b, n, nrhs, d.chainPtr.p, c0, nchain, bundle0, xcd, bX,
                           bB, bN);
    else
        hipLaunchKernelGGL((k_gs_bundle<BS, TPR, EE, VT, XT, false, BATCH>), grid, dim3(BS), d.lds(p, BS).bytes,
                           st, d.slot.p, d.wave.p, d.off.p, d.len.p, d.extPtr.p, d.slotWave.p, d.rowId.p,
                           d.diag.p, d.ext.p, d.sidx.p, d.sval.p, d.zero, x, b, n, nrhs, d.chainPtr.p, c0, nchain, bundle0,
                           xcd, bX, bB, bN);
}

// the variable-lanes kernels (tpr == 0)
template <int BS, typename VT, typename XT, bool BATCH>
void launchBundlesVL(int kind, int nrhs, const BundleDev<VT, XT>& d, int c0, int nchain, int p, int xcd, XT* x,
                     const XT* b, int n, XT* const* bX, const XT* const* bB, const int* bN, hipStream_t st) {
    const dim3 grid(xcd ? 8u * (unsigned)((nchain + 7) / 8) : (unsigned)nchain, (unsigned)std::max(1, nrhs));
    if (kind == RACE_K_KACZ)
        hipLaunchKernelGGL((k_kacz_bundle_vl<BS, VT, XT, BATCH, kColSlots>), grid, dim3(BS), d.lds(p, BS).bytes, st, d.slot.p, d.wave.p,
                           d.off.p, d.len.p, d.extPtr.p, d.slotWave.p, d.rowId.p, d.rowNorm.p, d.ext.p, d.sidx.p,
                           d.sval.p, d.zero, x, b, n, nrhs, d.chainPtr.p, c0, nchain, xcd, d.h.phLocal[p], d.lds(p, BS).spare,
                           d.lanePtr.p, d.laneSlot.p, bX, bB, bN);
    else
        hipLaunchKernelGGL((k_gs_bundle_vl<BS, VT, XT, BATCH>), grid, dim3(BS), d.lds(p, BS).bytes, st, d.slot.p, d.wave.p,
                           d.off.p, d.len.p, d.extPtr.p, d.slotWave.p, d.rowId.p, d.diag.p, d.ext.p, d.sidx.p,
                           d.sval.p, d.zero, x, b, n, nrhs, d.chainPtr.p, c0, nchain, xcd, d.h.phLocal[p],
                           d.lanePtr.p, d.laneSlot.p, bX, bB, bN);
}

template <typename VT, typename XT, bool BATCH>
void launchPhase(int bs, int tpr, int E, int kind, int nrhs, const BundleDev<VT, XT>& d, int c0, int nchain, int p,
                 int xcd, XT* x, const XT* b, int n, XT* const* bX, const XT* const* bB, const int* bN,
                 hipStream_t st) {
#define RACE_BUNDLE_CASE(BS_)                                                                              \
    switch (tpr * 100 + E) {                                                                               \
        case 104: launchBundles<BS_, 1, 4, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;   \
        case 108: launchBundles<BS_, 1, 8, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;   \
        case 116: launchBundles<BS_, 1, 16, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;  \
        case 208: launchBundles<BS_, 2, 8, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;   \
        case 213: launchBundles<BS_, 2, 13, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;  \
        case 216: launchBundles<BS_, 2, 16, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;  \
        case 416: launchBundles<BS_, 4, 16, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;  \
        case 16: launchBundlesVL<BS_, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;        \
        default: launchBundles<BS_, 4, 8, VT, XT, BATCH>(kind, nrhs, d, c0, nchain, p, xcd, x, b, n, bX, bB, bN, st); break;   \
    }
    switch (bs) {
        case 64: RACE_BUNDLE_CASE(64) break;
        case 128: RACE_BUNDLE_CASE(128) break;
        case 512: RACE_BUNDLE_CASE(512) break;
        case 1024: RACE_BUNDLE_CASE(1024) break;
        default: RACE_BUNDLE_CASE(256) break;
    }
#undef RACE_BUNDLE_CASE
}

// polls of one dependency flag or queue position before a launch gives up
// (about seconds; a correct dependency table never gets near it)
constexpr int kFlowPollLimit = 1 << 22;
// and of a launch that the caller did not ask for by the option (and whose
// aborts it will not look for): 16 times as long, about a minute, longer than any
// pause of the device.  A table that would need it is refused at registration
// (FlowDev::init, BundleFn::init: every dependency on an earlier chain of an
// earlier phase); should one be wrong all the same, the launch ends.
constexpr int kAutoPollLimit = 1 << 26;

// Device state of the one-launch sweep of one direction: the bundle range
// and the dependencies of every chain, column ids with the coherent-read
// bit, and per right-hand side a flag per chain (tickets in chain order) or
// an arrival counter per chain and a ready queue (readiness-driven), and a
// ticket/epoch state.
struct FlowDev {
    DevBuf<int> depPtr, dep, ext, lo, hi;
    // readiness-driven sweeps (Kaczmarz): successors and roots
    DevBuf<int> succPtr, succ, roots;
    // what a running sweep changes; sweeps on different streams may overlap
    // if each uses a set of its own
    struct Live {
        DevBuf<int> flag;
        DevBuf<FlowState> fs;
        // readiness-driven: arrival counters and ready queues
        DevBuf<unsigned> arrivals;
        DevBuf<unsigned long long> queue;
    };
    std::vector<std::unique_ptr<Live>> live;
    bool readyMode = false;
    int nroots = 0, pollLimit = kFlowPollLimit;
    // readiness-driven: the longest dependency path of the sweep, in
    // dependency waves plus kBundleFixedWaves per bundle
    long longestPath = 0;
    int nchain = 0, grid = 0, nrhs = 1, maxLocal = 0, maxRows = 0, spare = 64;
    size_t lds = 0;
    bool fits = false;
    // chains whose conflicts lie inside one phase (0 for a valid colouring)
    long samePhase = 0;
    int held = kColSlots;  // Kaczmarz: column ids a thread holds, which kernel
    // nkeys / colBase: the key space of the rows and columns (chainDeps)
    // ready: readiness-driven (queue) instead of tickets in chain order
    // sets: sweeps that may overlap
    template <typename VT, typename XT>
    int init(const BundleDev<VT, XT>& d, long nkeys, const std::vector<long>* colBase, int bs, int nrhs_,
             bool ready, int sets = 1) {
        readyMode = ready;
        std::vector<int> dp, dd;
        samePhase = chainDeps(d.h, nkeys, colBase, &dp, &dd);
        nchain = (int)d.h.chainPtr.size() - 1;
        nrhs = std::max(1, nrhs_);
        for (int p = 0; p < d.h.numPhases(); ++p) {
            maxLocal = std::max(maxLocal, d.h.phLocal[p]);
            maxRows = std::max(maxRows, d.h.phRows[p]);
        }
        // one layout for every phase: the largest local column space, then
        // (variable lanes) the partial sums and the first lane of every row
        const LdsPlan plan = ldsPlan<XT>(maxLocal, maxRows, d.h.tpr, bs, d.maxLds);
        lds = plan.bytes;
        spare = plan.spare;
        if (!(fits = lds <= d.maxLds)) return OK;  // not used
        // tickets in chain order (phase order)
        for (int c = 0; c < nchain; ++c)
            for (int j = dp[c]; j < dp[c + 1]; ++j)
                if (dd[j] >= c) return ERR_INTERNAL;  // a dependency after its chain
        const std::vector<int>& cp = d.h.chainPtr;
        int e;
        if ((e = upload(depPtr, dp.data(), dp.size()))) return e;
        if ((e = upload(dep, dd.data(), dd.size()))) return e;
        if ((e = upload(lo, cp.data(), (size_t)nchain))) return e;
        if ((e = upload(hi, cp.data() + 1, (size_t)nchain))) return e;
        const std::vector<int> fx = flowExt(d.h, nkeys, colBase);
        if ((e = upload(ext, fx.data(), fx.size()))) return e;
        if (ready) {
            std::vector<int> sp(nchain + 1, 0), sv(dd.size()), rv;
            for (int c = 0; c < nchain; ++c)
                for (int j = dp[c]; j < dp[c + 1]; ++j) ++sp[dd[j] + 1];
            for (int c = 0; c < nchain; ++c) sp[c + 1] += sp[c];
            std::vector<int> fill(sp.begin(), sp.end() - 1);
            for (int c = 0; c < nchain; ++c)
                for (int j = dp[c]; j < dp[c + 1]; ++j) sv[fill[dd[j]]++] = c;
            for (int c = 0; c < nchain; ++c)
                if (dp[c + 1] == dp[c]) rv.push_back(c);
            nroots = (int)rv.size();
            // queue positions are chain numbers (order is the identity)
            for (long p : chainLongestPaths(d.h, dp, dd, kBundleFixedWaves)) longestPath = std::max(longestPath, p);
            if ((e = upload(succPtr, sp.data(), sp.size()))) return e;
            if ((e = upload(succ, sv.data(), sv.size()))) return e;
            if ((e = upload(roots, rv.data(), rv.size()))) return e;
        }
        // flags start below the first epoch, queue entries of epoch 0 never
        // match a launch
        const size_t cells = (size_t)std::max(nchain, 1) * nrhs;
        FlowState f0{};
        f0.epoch = 1;
        f0.tail = nroots;
        const std::vector<FlowState> fv(nrhs, f0);
        for (int k = 0; k < sets; ++k) {
            live.push_back(std::make_unique<Live>());
            Live& v = *live.back();
            if ((e = upload(v.fs, fv.data(), fv.size()))) return e;
            if (!ready) {
                if ((e = upload(v.flag, std::vector<int>(cells, 0).data(), cells))) return e;
                continue;
            }
            if ((e = upload(v.arrivals, std::vector<unsigned>(cells, 0u).data(), cells))) return e;
            if ((e = upload(v.queue, std::vector<unsigned long long>(cells, 0ull).data(), cells))) return e;
        }
        return OK;
    }
    // as many workgroups per right-hand side of the kernel that will run it as
    // are resident at once, at most `most` per CU, all sides together (more would
    // only find the tickets gone)
    int occupy(const void* kern, int bs, int most = INT32_MAX) {
        if (!kern) return ERR_INTERNAL;
        if (!fits) return OK;  // not used
        int per = 0, dev = 0, cus = 0;
        RACE_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, bs, lds));
        RACE_HIP(hipGetDevice(&dev));
        RACE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const int slots = std::max(1, std::max(std::min(per, most), 1) * cus / nrhs);
        grid = std::max(1, std::min(nchain, slots));
        return OK;
    }
    ReadyTables tables(int set) const {
        ReadyTables r;
        r.lo = lo.p;
        r.hi = hi.p;
        r.depPtr = depPtr.p;
        r.succPtr = succPtr.p;
        r.succ = succ.p;
        r.roots = roots.p;
        r.arrivals = live[set]->arrivals.p;
        r.queue = live[set]->queue.p;
        r.fs = live[set]->fs.p;
        r.nchain = nchain;
        r.nroots = nroots;
        r.pollLimit = pollLimit;
        return r;
    }
    int aborts(int* out) const {
        *out = 0;
        for (const auto& v : live) {
            std::vector<FlowState> f(nrhs);
            RACE_HIP(hipMemcpy(f.data(), v->fs.p, sizeof(FlowState) * nrhs, hipMemcpyDeviceToHost));
            for (const FlowState& q : f) *out += q.aborts;
        }
        return OK;
    }
};

template <int BS, int TPR, int EE, typename VT, typename XT>
int launchFlow(const BundleDev<VT, XT>& d, FlowDev& f, int set, XT* x, const XT* b, hipStream_t st) {
    auto kern = k_gs_flow<BS, TPR, EE, VT, XT, BS == 512 ? 4 : 6>;
    hipLaunchKernelGGL(kern, dim3(f.grid), dim3(BS), f.lds, st, d.slot.p, d.wave.p, d.off.p, d.len.p, d.extPtr.p,
                       d.slotWave.p, d.rowId.p, d.diag.p, f.ext.p, d.sidx.p, d.sval.p, d.zero, x, b, f.lo.p, f.hi.p,
                       f.nchain, f.depPtr.p, f.dep.p, f.live[set]->flag.p, f.live[set]->fs.p, f.pollLimit);
    RACE_HIP(hipGetLastError());
    return OK;
}

template <typename VT, typename XT>
int launchFlowShape(int bs, int tpr, int E, const BundleDev<VT, XT>& d, FlowDev& f, int set, XT* x, const XT* b,
                    hipStream_t st) {
    // 512 threads: four lanes per row only (BundleFn::fourLanes)
    if (bs == 512 && tpr == 4) return launchFlow<512, 4, 8>(d, f, set, x, b, st);
    switch (tpr * 100 + E) {
        case 104: return launchFlow<256, 1, 4>(d, f, set, x, b, st);
        case 108: return launchFlow<256, 1, 8>(d, f, set, x, b, st);
        case 116: return launchFlow<256, 1, 16>(d, f, set, x, b, st);
        case 208: return launchFlow<256, 2, 8>(d, f, set, x, b, st);
        case 213: return launchFlow<256, 2, 13>(d, f, set, x, b, st);
        case 216: return launchFlow<256, 2, 16>(d, f, set, x, b, st);
        case 408: return launchFlow<256, 4, 8>(d, f, set, x, b, st);
        case 416: return launchFlow<256, 4, 16>(d, f, set, x, b, st);
        default: return ERR_INTERNAL;
    }
}

// Kaczmarz one-launch sweep: grid (resident workgroups per side, nrhs)
template <int BS, int TPR, int EE, typename VT, typename XT, bool BATCH>
int launchKaczFlow(const BundleDev<VT, XT>& d, FlowDev& f, int set, XT* x, const XT* b, int n, XT* const* bX,
                   const XT* const* bB, const int* bN, hipStream_t st) {
    if constexpr (TPR == 0) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(f.grid, f.nrhs), dim3(BS), f.lds, st, d.slot.p, d.wave.p, d.off.p, d.len.p,
                               d.extPtr.p, d.slotWave.p, d.rowId.p, d.rowNorm.p, f.ext.p, d.sidx.p, d.sval.p, d.zero, x,
                               b, n, f.maxLocal, f.spare, d.lanePtr.p, d.laneSlot.p, bX, bB, bN, f.tables(set));
        };
        if constexpr (BATCH)
            if (f.held == kLeanSlots) {
                launch(k_kacz_flow_vl<BS, VT, XT, BATCH, kLeanSlots>);
                RACE_HIP(hipGetLastError());
                return OK;
            }
        launch(k_kacz_flow_vl<BS, VT, XT, BATCH, kColSlots>);
    } else {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(f.grid, f.nrhs), dim3(BS), f.lds, st, d.slot.p, d.wave.p, d.off.p, d.len.p,
                               d.extPtr.p, d.slotWave.p, d.rowId.p, d.rowNorm.p, f.ext.p, d.sidx.p, d.sval.p, d.zero, x,
                               b, n, f.spare, bX, bB, bN, f.tables(set));
        };
        constexpr int fewer = BATCH ? kLeanSlots : kFewSlots;
        if (f.held == fewer)
            launch(k_kacz_flow<BS, TPR, EE, VT, XT, BATCH, fewer>);
        else
            launch(k_kacz_flow<BS, TPR, EE, VT, XT, BATCH, kColSlots>);
    }
    RACE_HIP(hipGetLastError());
    return OK;
}

template <typename VT, typename XT, bool BATCH>
int launchKaczFlowShape(int bs, int tpr, int E, const BundleDev<VT, XT>& d, FlowDev& f, int set, XT* x, const XT* b,
                        int n, XT* const* bX, const XT* const* bB, const int* bN, hipStream_t st) {
#define RACE_KFLOW_CASE(BS_)                                                                                       \
    switch (tpr * 100 + E) {                                                                                       \
        case 104: return launchKaczFlow<BS_, 1, 4, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                  \
        case 108: return launchKaczFlow<BS_, 1, 8, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                  \
        case 116: return launchKaczFlow<BS_, 1, 16, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                 \
        case 208: return launchKaczFlow<BS_, 2, 8, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                  \
        case 213: return launchKaczFlow<BS_, 2, 13, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                 \
        case 216: return launchKaczFlow<BS_, 2, 16, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                 \
        case 408: return launchKaczFlow<BS_, 4, 8, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                  \
        case 416: return launchKaczFlow<BS_, 4, 16, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);                 \
        case 16: return launchKaczFlow<BS_, 0, kVarE, VT, XT, BATCH>(d, f, set, x, b, n, bX, bB, bN, st);               \
        default: return ERR_INTERNAL;                                                                              \
    }
    switch (bs) {
        case 256: RACE_KFLOW_CASE(256)
        case 512: RACE_KFLOW_CASE(512)
        case 1024: RACE_KFLOW_CASE(1024)
        default: return ERR_INTERNAL;
    }
#undef RACE_KFLOW_CASE
}
// workgroup sizes the one-launch Kaczmarz sweep is built for
inline bool kaczFlowBs(int bs) { return bs == 256 || bs == 512 || bs == 1024; }

// the kernel a one-launch sweep of this shape runs (for its occupancy)
template <typename VT, typename XT>
const void* gsFlowKernel(int bs, int tpr, int E) {
    if (bs == 512 && tpr == 4) return reinterpret_cast<const void*>(k_gs_flow<512, 4, 8, VT, XT, 4>);
    switch (tpr * 100 + E) {
        case 104: return reinterpret_cast<const void*>(k_gs_flow<256, 1, 4, VT, XT>);
        case 108: return reinterpret_cast<const void*>(k_gs_flow<256, 1, 8, VT, XT>);
        case 116: return reinterpret_cast<const void*>(k_gs_flow<256, 1, 16, VT, XT>);
        case 208: return reinterpret_cast<const void*>(k_gs_flow<256, 2, 8, VT, XT>);
        case 213: return reinterpret_cast<const void*>(k_gs_flow<256, 2, 13, VT, XT>);
        case 216: return reinterpret_cast<const void*>(k_gs_flow<256, 2, 16, VT, XT>);
        case 408: return reinterpret_cast<const void*>(k_gs_flow<256, 4, 8, VT, XT>);
        case 416: return reinterpret_cast<const void*>(k_gs_flow<256, 4, 16, VT, XT>);
        default: return nullptr;
    }
}
template <int BS, int K, typename VT, typename XT, bool BATCH>
const void* kaczFlowKernelOf(int tpr, int E) {
    switch (tpr * 100 + E) {
        case 104: return reinterpret_cast<const void*>(k_kacz_flow<BS, 1, 4, VT, XT, BATCH, K>);
        case 108: return reinterpret_cast<const void*>(k_kacz_flow<BS, 1, 8, VT, XT, BATCH, K>);
        case 116: return reinterpret_cast<const void*>(k_kacz_flow<BS, 1, 16, VT, XT, BATCH, K>);
        case 208: return reinterpret_cast<const void*>(k_kacz_flow<BS, 2, 8, VT, XT, BATCH, K>);
        case 213: return reinterpret_cast<const void*>(k_kacz_flow<BS, 2, 13, VT, XT, BATCH, K>);
        case 216: return reinterpret_cast<const void*>(k_kacz_flow<BS, 2, 16, VT, XT, BATCH, K>);
        case 408: return reinterpret_cast<const void*>(k_kacz_flow<BS, 4, 8, VT, XT, BATCH, K>);
        case 416: return reinterpret_cast<const void*>(k_kacz_flow<BS, 4, 16, VT, XT, BATCH, K>);
    }
    if constexpr (K != kFewSlots)
        if (tpr == 0) return reinterpret_cast<const void*>(k_kacz_flow_vl<BS, VT, XT, BATCH, K>);
    return nullptr;
}
template <int BS, typename VT, typename XT, bool BATCH>
const void* kaczFlowKernelBs(int held, int tpr, int E) {
    constexpr int fewer = BATCH ? kLeanSlots : kFewSlots;
    return held == fewer ? kaczFlowKernelOf<BS, fewer, VT, XT, BATCH>(tpr, E)
                         : kaczFlowKernelOf<BS, kColSlots, VT, XT, BATCH>(tpr, E);
}
// held: column ids a thread holds (kLeanSlots: batches only, kFewSlots: others)
template <typename VT, typename XT, bool BATCH>
const void* kaczFlowKernel(int held, int bs, int tpr, int E) {
    switch (bs) {
        case 256: return kaczFlowKernelBs<256, VT, XT, BATCH>(held, tpr, E);
        case 512: return kaczFlowKernelBs<512, VT, XT, BATCH>(held, tpr, E);
        case 1024: return kaczFlowKernelBs<1024, VT, XT, BATCH>(held, tpr, E);
        default: return nullptr;
    }
}

// lanes per row and register width for the longest row (diagonal excluded
// for Gauss-Seidel); E < 0 if no kernel instantiation fits.  Rows longer
// than 64 entries select variable lanes per row (tpr 0, kVarE registers
// per lane), so a few long rows do not widen every row of the matrix.
void pickShape(int kind, int maxRowLen, int forcedTpr, int* tpr, int* E) {
    int m = maxRowLen - (kind != RACE_K_KACZ ? 1 : 0);
    m = std::max(m, 1);
    if (forcedTpr <= 0 && m > 64) {
        *tpr = 0;
        *E = kVarE;
        return;
    }
    *tpr = forcedTpr > 0 ? forcedTpr : (m <= 16 ? 1 : m <= 32 ? 2 : 4);
    *E = pickE(*tpr, (m + *tpr - 1) / *tpr);
}

// rows per bundle: the workgroup's lanes divided by the lanes per row, or
// (variable lanes) the row limit alone, lanes checked by the builder
int rowsCapFor(int bundleRows, int bs, int tpr) { return tpr > 0 ? std::min(bundleRows, bs / tpr) : bundleRows; }

template <typename VT, typename XT>
class BundleFn : public DeviceFn {
  public:
    using Dev = BundleDev<VT, XT>;
    Dev df, dr;
    int nrhs = 1, n = 0, bs = 256, tpr = 2, E = 16, xcd = 1;
    std::unique_ptr<DeviceFn> fallback;
    // one launch per sweep (the "flow" option): Gauss-Seidel with one
    // right-hand side, 256-thread workgroups and uniform lanes per row;
    // Kaczmarz with 256-1024-thread workgroups
    bool flow = false;
    FlowDev ff, fr;
    // Small matrices sweep in one launch without the option.  A phase launch
    // costs about 4.7 us however few its bundles, a level of the one-launch
    // sweep about 3.3 us (a store, a flag, a poll and a gather through memory)
    // while every chain finds a workgroup at once.  us per symmetric step, phase
    // launches / one launch: Gauss-Seidel 27-point FP64 14^3 127 / 87, 40^3 141 /
    // 108, 48^3 145 / 130 (864 chains), 52^3 147 / 155 (1100), FP32 48^3 132 / 127,
    // 52^3 133 / 151: 896 chains, 3.5 per CU.  Kaczmarz 7-point FP64 20^3 102 / 67,
    // 45^3 208 / 192, 64^3 266 / 219; FP32 20^3 90 / 62, 48^3 192 / 192, 50^3 194 /
    // 205: with FP32 up to 1280 chains (48^3), with FP64 as far as measured.
    // Long chains are left out: their coherent stores cost more than the
    // launches (Chung-Lu graph of 20000 rows, 4 launches: 1916 / 2064).
    // Sweeps that overlap need sets of their own, so each of the first kSets
    // streams gets one (a flag or two numbers per chain); other streams and
    // captured launches run the phases.
    static constexpr int kSets = 8, kAutoBundles = 4;
    static int autoChains(int kind) { return kind == RACE_K_GS ? 896 : sizeof(XT) == 8 ? 16384 : 1280; }
    bool autoFlow = false;
    StreamSets streamSets;
    // the set for a launch on st, -1 for the phase launches
    int setFor(hipStream_t st) { return flow ? 0 : autoFlow ? streamSets.find(st, kSets) : -1; }
    // Gauss-Seidel rows of 17 to 32 entries off the diagonal: four lanes per
    // row (8 entries a lane instead of 16) and 64 rows per bundle where the
    // chain of waves counts more than the bytes.  us per symmetric step of a
    // 27-point grid, 128 rows x 2 lanes / 64 x 4.  One launch per sweep, FP64
    // 14^3 87 / 82, FP32 84 / 72; 40^3 FP64 107 / 136, as twice the chains no longer
    // find a workgroup at once: up to 256 bundles of 64 rows.  One launch per
    // phase, past the sizes of the one-launch sweep: FP32 56^3 167 / 156, 100^3 229 /
    // 213, 128^3 324 / 318, BF16 56^3 207 / 178; FP64 gains 2 % at 56^3 and loses 4 %
    // at 128^3 to the outside columns that smaller bundles share less, and keeps
    // two lanes.  By size alone, not by the flow option: the lanes of a row set
    // the order of its sum, and both kinds of launches give the same bits.  With
    // the option on, larger matrices take 512 threads for the same 128 rows
    // (FP32 64^3 204 us with two lanes, 177 with 512 threads, 268 with 64 rows).
    bool fourLanes() const {
        if (kind != RACE_K_GS || nrhs != 1) return false;
        return n <= 256 * 64 || (sizeof(XT) == 4 && n > 128 * autoChains(kind));
    }
    // Kaczmarz in one launch: kFewSlots where more chains could run at once than
    // 1536 threads per CU hold, on a grid of as many.  Below, more workgroups than
    // kColSlots leaves room for only wait for chains (7-point 64^3 FP64, one side:
    // 166 chains at once 217 us, with kFewSlots 242).  Eight sides, kColSlots /
    // kFewSlots: 7-point 64^3 FP32 (1325 at once) 377 / 389, 27-point 80^3 FP32
    // (2001) 1150 / 970, FP64 1643 / 1619, 7-point 96^3 FP64 (3197) 1309 / 1138.
    int occupyKacz(FlowDev& f, const Dev& d) const {
        constexpr int kThreads = 1536;
        int dev = 0, cus = 0;
        RACE_HIP(hipGetDevice(&dev));
        RACE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        const SweepCost sweep(d.h);
        const bool few = d.fewCols && sweep.all * nrhs * bs > sweep.phases * cus * kThreads;
        f.held = few ? kFewSlots : kColSlots;
        return f.occupy(kaczFlowKernel<VT, XT, false>(f.held, bs, tpr, E), bs, few ? kThreads / bs : INT32_MAX);
    }
    static bool autoFits(const BundleTable& t) {
        int longest = 0;
        for (size_t c = 0; c + 1 < t.chainPtr.size(); ++c) longest = std::max(longest, t.chainPtr[c + 1] - t.chainPtr[c]);
        return t.numPhases() >= 3 && longest <= kAutoBundles;
    }

    int init(const race_kernel_desc& d, const ExecContext& ctx) {
        kind = d.kind;
        nrhs = d.nrhs > 0 ? d.nrhs : 1;
        n = d.nrow;
        x = d.x;
        b = d.b;
        bs = ctx.bundleThreads;
        xcd = ctx.xcdOrder;
        int maxLen = 0;
        for (int r = 0; r < n; ++r) maxLen = std::max(maxLen, d.rowPtr[r + 1] - d.rowPtr[r]);
        pickShape(kind, maxLen, ctx.bundleTpr, &tpr, &E);
        int rowsCap = rowsCapFor(ctx.bundleRows, bs, tpr);
        bool flowWide = false;
        if (tpr == 2 && ctx.bundleTpr == 0 && ctx.bundleRows == 128 && bs == 256 && fourLanes()) {
            tpr = 4;
            E = pickE(4, (maxLen - 1 + 3) / 4);
            flowWide = ctx.flow > 0 && n > 256 * 64;
            if (flowWide) bs = 512;
            rowsCap = rowsCapFor(ctx.bundleRows, bs, tpr);
        }
        const bool fp64 = std::is_same<VT, double>::value && std::is_same<XT, double>::value;
        auto fallBack = [&]() -> int {
            if (ctx.layout == 2 || !fp64) return ERR_INCOMPATIBILITY;  // bundles required
            return makeWaveFn(d, ctx, &fallback);
        };
        if (E < 0 || rowsCap < 1) return fallBack();
        BundleTable tf = buildBundles(*ctx.fwd, kind, n, d.rowPtr, d.col, d.val, rowsCap,
                                      ctx.bundleLocal, tpr, bs);
        if (!tf.ok) return fallBack();
        BundleTable tr = buildBundles(*ctx.rev, kind, n, d.rowPtr, d.col, d.val, rowsCap,
                                      ctx.bundleLocal, tpr, bs);
        if (!tr.ok) return fallBack();
        int e;
        if ((e = df.load(std::move(tf), bs, nrhs))) return e;
        if ((e = dr.load(std::move(tr), bs, nrhs))) return e;
        if (!df.fits(bs) || !dr.fits(bs)) return fallBack();
        const bool gsFlow = kind == RACE_K_GS && nrhs == 1 && (bs == 256 || flowWide) && tpr > 0;
        const bool kaczFlow = kind == RACE_K_KACZ && kaczFlowBs(bs);
        const int chains = std::max((int)df.h.chainPtr.size(), (int)dr.h.chainPtr.size()) - 1;
        const bool small =
            ctx.flow < 0 && (long)chains * nrhs <= autoChains(kind) && autoFits(df.h) && autoFits(dr.h);
        if ((ctx.flow > 0 || small) && (gsFlow || kaczFlow)) {
            const int sets = small ? kSets : 1;
            const int sides = kind == RACE_K_KACZ ? nrhs : 1;
            const bool ready = kind == RACE_K_KACZ;
            if ((e = ff.init(df, n, nullptr, bs, sides, ready, sets)) ||
                (e = fr.init(dr, n, nullptr, bs, sides, ready, sets)))
                return e;
            if ((e = ready ? occupyKacz(ff, df) : ff.occupy(gsFlowKernel<VT, XT>(bs, tpr, E), bs)) ||
                (e = ready ? occupyKacz(fr, dr) : fr.occupy(gsFlowKernel<VT, XT>(bs, tpr, E), bs)))
                return e;
            // conflicts inside a phase would serialise its chains, and one
            // LDS layout serves every phase: keep the phase launches if
            // either does not hold
            const bool ok = ff.samePhase == 0 && fr.samePhase == 0 && ff.fits && fr.fits;
            flow = ok && !small;
            autoFlow = ok && small;
            if (small) ff.pollLimit = fr.pollLimit = kAutoPollLimit;
        }
        return OK;
    }
    int flowAborts(int* out) const override {
        *out = 0;
        if (!flow && !autoFlow) return OK;
        int a = 0, c = 0, e;
        if ((e = ff.aborts(&a)) || (e = fr.aborts(&c))) return e;
        *out = a + c;
        return OK;
    }

    int waves(bool rev) const override {
        if (fallback) return fallback->waves(rev);
        return (int)(rev ? dr.h.critical : df.h.critical);
    }
    bool graphable() const override { return fallback ? fallback->graphable() : true; }
    int launches(bool rev) const override {
        if (fallback) return fallback->launches(rev);
        if (flow || autoFlow) return 1;
        const std::vector<int>& pc = (rev ? dr : df).h.phaseChain;
        int k = 0;
        for (size_t p = 0; p + 1 < pc.size(); ++p) k += pc[p + 1] > pc[p];
        return k;
    }
    int run(bool rev, hipStream_t st) override {
        if (fallback) {
            fallback->x = x;
            fallback->b = b;
            return fallback->run(rev, st);
        }
        const Dev& d = rev ? dr : df;
        const int set = setFor(st);
        if (set >= 0 && kind == RACE_K_KACZ)
            return launchKaczFlowShape<VT, XT, false>(bs, tpr, E, d, rev ? fr : ff, set, (XT*)x, (const XT*)b, n,
                                                      nullptr, nullptr, nullptr, st);
        if (set >= 0) return launchFlowShape<VT, XT>(bs, tpr, E, d, rev ? fr : ff, set, (XT*)x, (const XT*)b, st);
        const std::vector<int>& pc = d.h.phaseChain;
        for (int p = 0; p + 1 < (int)pc.size(); ++p) {
            const int c0 = pc[p], nchain = pc[p + 1] - pc[p];
            if (nchain <= 0) continue;
            launchPhase<VT, XT, false>(bs, tpr, E, kind, nrhs, d, c0, nchain, p, xcd, (XT*)x, (const XT*)b, n,
                                       nullptr, nullptr, nullptr, st);
        }
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

// Gauss-Seidel or Kaczmarz on a batch of matrices, each with its own
// colouring and vectors: one fused launch per phase index runs the bundles
// of that phase of every matrix (concatBundles), so a batch of small
// matrices fills the device instead of issuing a few tiny launches per
// matrix and phase.  All matrices share the kernel shape (lanes per row,
// register width, workgroup size), chosen from the longest row.
template <typename VT, typename XT>
class BundleBatchFn : public DeviceFn {
  public:
    using Dev = BundleDev<VT, XT>;
    // matrices with the same kernel shape share fused tables
    struct Group {
        int tpr = 1, E = 4;
        Dev dev[2];
        DevBuf<XT*> bx[2];
        DevBuf<const XT*> bb[2];
        DevBuf<int> bn[2];
        FlowDev flow[2];
    };
    std::vector<std::unique_ptr<Group>> groups;
    int nrhs = 1, bs = 256, xcd = 0, maxPhases[2] = {0, 0};
    long critical[2] = {0, 0};
    // one launch per group and sweep (the "flow" option, Kaczmarz): every
    // matrix advances through its own phases, waiting only for its own
    // earlier chains, instead of every fused phase waiting for the slowest
    // matrix
    bool flow = false, flowOk = true;
    // flow: the groups hold different matrices, so their launches run
    // concurrently, the group with the longest dependency path first (on
    // the caller's stream), so that its long chains start at once and the
    // other groups (each on a stream of its own, forked from and joined back
    // into the caller's stream by events) fill the remaining workgroup slots
    std::vector<hipStream_t> side;
    std::vector<hipEvent_t> joinEv;
    hipEvent_t forkEv = nullptr;
    std::vector<int> launchOrder[2];

    ~BundleBatchFn() override {
        for (hipStream_t s : side) (void)hipStreamDestroy(s);
        for (hipEvent_t e : joinEv) (void)hipEventDestroy(e);
        if (forkEv) (void)hipEventDestroy(forkEv);
    }

    int init(const std::vector<BatchItem>& items, const ExecContext& ctx) {
        if (items.empty()) return ERR_INVALID_ARG;
        kind = items[0].d.kind;
        nrhs = items[0].d.nrhs > 0 ? items[0].d.nrhs : 1;
        bs = ctx.bundleThreads;
        xcd = ctx.xcdOrder;
        std::vector<int> shape(items.size());
        std::vector<std::pair<int, int>> shapes;
        for (size_t m = 0; m < items.size(); ++m) {
            const BatchItem& it = items[m];
            int maxLen = 0;
            for (int r = 0; r < it.d.nrow; ++r) maxLen = std::max(maxLen, it.d.rowPtr[r + 1] - it.d.rowPtr[r]);
            int tpr, E;
            pickShape(kind, maxLen, ctx.bundleTpr, &tpr, &E);
            if (E < 0 && ctx.bundleTpr > 0) pickShape(kind, maxLen, 0, &tpr, &E);  // row too long for the forced width
            if (E < 0 || rowsCapFor(ctx.bundleRows, bs, tpr) < 1) return ERR_INCOMPATIBILITY;
            const std::pair<int, int> key(tpr, E);
            auto f = std::find(shapes.begin(), shapes.end(), key);
            shape[m] = (int)(f - shapes.begin());
            if (f == shapes.end()) shapes.push_back(key);
        }
        for (size_t g = 0; g < shapes.size(); ++g) {
            auto grp = std::make_unique<Group>();
            grp->tpr = shapes[g].first;
            grp->E = shapes[g].second;
            const int rowsCap = rowsCapFor(ctx.bundleRows, bs, grp->tpr);
            for (int dir = 0; dir < 2; ++dir) {
                std::vector<int> members;
                for (size_t m = 0; m < items.size(); ++m)
                    if (shape[m] == (int)g) members.push_back((int)m);
                // the matrices' tables are independent: build them on host threads
                std::vector<BundleTable> tabs(members.size());
                std::atomic<size_t> next{0};
                std::atomic<bool> bad{false};
                auto work = [&]() {
                    for (size_t q; (q = next++) < members.size();) {
                        const BatchItem& it = items[members[q]];
                        tabs[q] = buildBundles(dir ? *it.rev : *it.fwd, kind, it.d.nrow, it.d.rowPtr, it.d.col,
                                               it.d.val, rowsCap, ctx.bundleLocal, grp->tpr, bs);
                        if (!tabs[q].ok) bad = true;
                    }
                };
                const size_t nth = std::min<size_t>(members.size(),
                                                    std::max(1u, std::min(16u, std::thread::hardware_concurrency())));
                std::vector<std::thread> pool;
                for (size_t t = 1; t < nth; ++t) pool.emplace_back(work);
                work();
                for (std::thread& th : pool) th.join();
                if (bad) return ERR_INCOMPATIBILITY;
                std::vector<const BundleTable*> ptrs;
                for (size_t q = 0; q < members.size(); ++q) ptrs.push_back(&tabs[q]);
                std::vector<int> owner;
                BundleTable fused = concatBundles(ptrs, &owner);
                std::vector<BundleTable>().swap(tabs);
                std::vector<XT*> hx(owner.size());
                std::vector<const XT*> hb(owner.size());
                std::vector<int> hn(owner.size());
                for (size_t k = 0; k < owner.size(); ++k) {
                    const race_kernel_desc& d = items[members[owner[k]]].d;
                    hx[k] = (XT*)d.x;
                    hb[k] = (const XT*)d.b;
                    hn[k] = d.nrow;
                }
                int e;
                if ((e = upload(grp->bx[dir], hx.data(), hx.size()))) return e;
                if ((e = upload(grp->bb[dir], hb.data(), hb.size()))) return e;
                if ((e = upload(grp->bn[dir], hn.data(), hn.size()))) return e;
                if ((e = grp->dev[dir].load(std::move(fused), bs, nrhs))) return e;
                if (!grp->dev[dir].fits(bs)) return ERR_INCOMPATIBILITY;
                maxPhases[dir] = std::max(maxPhases[dir], grp->dev[dir].h.numPhases());
                if (ctx.flow && kind == RACE_K_KACZ && kaczFlowBs(bs)) {
                    // every matrix its own range of row / column keys
                    std::vector<long> base(members.size() + 1, 0);
                    for (size_t q = 0; q < members.size(); ++q) base[q + 1] = base[q] + items[members[q]].d.nrow;
                    std::vector<long> colBase(owner.size());
                    for (size_t k = 0; k < owner.size(); ++k) colBase[k] = base[owner[k]];
                    if ((e = grp->flow[dir].init(grp->dev[dir], base.back(), &colBase, bs, nrhs, true))) return e;
                    // conflicts inside a phase, or one LDS layout for all
                    // phases too large: the fused phase launches then
                    if (grp->flow[dir].samePhase != 0 || !grp->flow[dir].fits) flowOk = false;
                }
            }
            groups.push_back(std::move(grp));
        }
        flow = flowOk && ctx.flow && kind == RACE_K_KACZ && kaczFlowBs(bs);
        for (int dir = 0; dir < 2 && flow; ++dir) {
            int e;
            bool lean = false;
            if ((e = leanBatch(dir, &lean))) return e;
            for (const auto& g : groups) {
                FlowDev& f = g->flow[dir];
                f.held = lean ? kLeanSlots : kColSlots;
                const int most = lean && g->tpr == 0 && groups.size() > 1 ? 1 : INT32_MAX;
                if ((e = f.occupy(kaczFlowKernel<VT, XT, true>(f.held, bs, g->tpr, g->E), bs, most))) return e;
            }
        }
        for (int dir = 0; dir < 2; ++dir) {
            launchOrder[dir].resize(groups.size());
            for (size_t g = 0; g < groups.size(); ++g) launchOrder[dir][g] = (int)g;
            std::stable_sort(launchOrder[dir].begin(), launchOrder[dir].end(), [&](int a, int b) {
                return groups[a]->flow[dir].longestPath > groups[b]->flow[dir].longestPath;
            });
        }
        if (flow && groups.size() > 1) {
            RACE_HIP(hipEventCreateWithFlags(&forkEv, hipEventDisableTiming));
            for (size_t g = 1; g < groups.size(); ++g) {
                hipStream_t s = nullptr;
                hipEvent_t e = nullptr;
                RACE_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
                side.push_back(s);
                RACE_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
                joinEv.push_back(e);
            }
        }
        for (int dir = 0; dir < 2; ++dir)
            for (int p = 0; p < maxPhases[dir]; ++p) {
                int w = 0;
                for (const auto& g : groups)
                    if (p < g->dev[dir].h.numPhases()) w = std::max(w, g->dev[dir].h.phWaves[p]);
                critical[dir] += w;
            }
        return OK;
    }
    // One-launch sweeps: kLeanSlots where the work of all matrices keeps the
    // places of the chip (the workgroups per CU that the group with the most work
    // has with kColSlots) busy for more than three times the longest dependency
    // path.  Chains are slower then, but three workgroups of 512 threads share a
    // CU.  ms per forward / backward sweep of eight right-hand sides, half banded
    // matrices and half Chung-Lu graphs of 2000 to 200000 rows, 512 threads x 256
    // rows x 4 lanes, kColSlots / kLeanSlots: FP32 384 matrices (ratio 2.7) 49.1 49.2
    // / 54.3 50.4, 512 (3.5) 68.7 66.1 / 66.6 62.8, the banded ones of them (18.8)
    // 48.5 48.4 / 42.2 42.1; FP64 128 (2.0) 37.5 38.4 / 38.8 39.3, 256 (3.9) 62.9 65.5
    // / 52.3 52.4.  Groups run at once, and the longest path's, mostly that of the
    // graphs (variable lanes), starts first: it gets one workgroup per CU, as more
    // leave the other groups no place until it ends (the 512 and 256 matrices 78.3
    // 80.3 and 60.1 67.0).
    static constexpr int kLeanRatio = 3;
    int leanBatch(int dir, bool* lean) const {
        int dev = 0, cus = 0, per = 0;
        RACE_HIP(hipGetDevice(&dev));
        RACE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        long all = 0, most = -1, path = 1;
        for (const auto& g : groups) {
            if (g->dev[dir].maxLds != kMaxLds) return OK;  // lean kernels know no chains kept in LDS
            const long cost = SweepCost(g->dev[dir].h).all;
            all += cost;
            path = std::max(path, g->flow[dir].longestPath);
            if (cost <= most) continue;
            most = cost;
            RACE_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per, kaczFlowKernel<VT, XT, true>(kColSlots, bs, g->tpr, g->E), bs, g->flow[dir].lds));
        }
        *lean = (double)all * nrhs > (double)kLeanRatio * path * cus * std::max(per, 1);
        return OK;
    }
    int waves(bool rev) const override { return (int)critical[rev ? 1 : 0]; }
    int launches(bool rev) const override {
        if (flow) return (int)groups.size();
        int k = 0;
        const int dir = rev ? 1 : 0;
        for (int p = 0; p < maxPhases[dir]; ++p)
            for (const auto& g : groups)
                if (p < g->dev[dir].h.numPhases() && g->dev[dir].h.phaseChain[p + 1] > g->dev[dir].h.phaseChain[p]) ++k;
        return k;
    }
    int flowAborts(int* out) const override {
        *out = 0;
        if (!flow) return OK;
        for (const auto& g : groups)
            for (int dir = 0; dir < 2; ++dir) {
                int a = 0, e;
                if ((e = g->flow[dir].aborts(&a))) return e;
                *out += a;
            }
        return OK;
    }
    int run(bool rev, hipStream_t st) override {
        const int dir = rev ? 1 : 0;
        if (flow) {
            if (!side.empty()) RACE_HIP(hipEventRecord(forkEv, st));
            for (size_t q = 0; q < groups.size(); ++q) {
                Group& g = *groups[launchOrder[dir][q]];
                hipStream_t s = q == 0 ? st : side[q - 1];
                if (q > 0) RACE_HIP(hipStreamWaitEvent(s, forkEv, 0));
                int e = launchKaczFlowShape<VT, XT, true>(bs, g.tpr, g.E, g.dev[dir], g.flow[dir], 0, nullptr, nullptr,
                                                          0, g.bx[dir].p, g.bb[dir].p, g.bn[dir].p, s);
                if (e) return e;
                if (q > 0) RACE_HIP(hipEventRecord(joinEv[q - 1], s));
            }
            for (hipEvent_t e : joinEv) RACE_HIP(hipStreamWaitEvent(st, e, 0));
            return OK;
        }
        // phase p of every group before phase p + 1 of any (stream order)
        for (int p = 0; p < maxPhases[dir]; ++p)
            for (const auto& g : groups) {
                const Dev& d = g->dev[dir];
                if (p >= d.h.numPhases()) continue;
                const int c0 = d.h.phaseChain[p], nchain = d.h.phaseChain[p + 1] - c0;
                if (nchain <= 0) continue;
                launchPhase<VT, XT, true>(bs, g->tpr, g->E, kind, nrhs, d, c0, nchain, p, xcd, nullptr, nullptr, 0,
                                          g->bx[dir].p, g->bb[dir].p, g->bn[dir].p, st);
            }
        RACE_HIP(hipGetLastError());
        return OK;
    }
};

}  // namespace

template <typename VT, typename XT>
int makeBundleOf(const race_kernel_desc& d, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    auto f = std::make_unique<BundleFn<VT, XT>>();
    const int e = f->init(d, ctx);
    *out = std::move(f);
    return e;
}

template <typename VT, typename XT>
int makeBundleBatchOf(const std::vector<BatchItem>& items, const ExecContext& ctx, std::unique_ptr<DeviceFn>* out) {
    auto f = std::make_unique<BundleBatchFn<VT, XT>>();
    const int e = f->init(items, ctx);
    *out = std::move(f);
    return e;
}

}  // namespace race
