// Host-only check of residentChains (race_amd/csrc/bundle.cpp), built with g++
// by tests/test_resident_chains.py, on 5-point grids whose lines are chains of
// several bundles, colouring and bundles made so that every chain has more than
// the minimum of bundles:
//  * no column allowed, or fewer than a bundle has: nothing is changed and no
//    memory taken that grows with the table;
//  * fewer than a chain touches: nothing is changed;
//  * otherwise every entry names the column it named before, in the list of
//    its chain's first bundle.
// Prints "ok" and exits 0 on success.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "bundle.hpp"
#include "race_amd.h"

using namespace race;

static size_t taken = 0;
void* operator new(size_t n) {
    taken += n;
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

int failures = 0;
void expect(bool ok, const char* what, int w) {
    if (ok) return;
    ++failures;
    std::printf("%s (width %d)\n", what, w);
}

void check(int h, int w, int cap) {
    const int n = h * w;
    std::vector<int> rp{0}, col;
    for (int r = 0; r < n; ++r) {
        const int i = r / w, j = r % w;
        col.push_back(r);
        if (i > 0) col.push_back(r - w);
        if (i + 1 < h) col.push_back(r + w);
        if (j > 0) col.push_back(r - 1);
        if (j + 1 < w) col.push_back(r + 1);
        rp.push_back((int)col.size());
    }
    const std::vector<double> val(col.size(), 1.5);
    Schedule s;  // leaves: the lines; phases: the line number modulo 3
    s.phasePtr.push_back(0);
    for (int q = 0; q < 3; ++q) {
        for (int i = q; i < h; i += 3) {
            s.leafLo.push_back(i * w);
            s.leafHi.push_back((i + 1) * w);
        }
        s.phasePtr.push_back((int)s.leafLo.size());
    }
    const BundleTable t0 = buildBundles(s, RACE_K_KACZ, n, rp.data(), col.data(), val.data(), cap, 6144, 1, 256);
    expect(t0.ok, "table", w);
    int bundles = 1 << 30;
    for (size_t c = 0; c + 1 < t0.chainPtr.size(); ++c) bundles = std::min(bundles, t0.chainPtr[c + 1] - t0.chainPtr[c]);
    expect(bundles >= 8, "chains are long", w);
    for (int cols : {0, 1}) {
        BundleTable t = t0;
        const size_t before = taken;
        expect(residentChains(t, 8, cols) == 0, "kept without room", w);
        expect(taken - before <= 4096, "memory taken without room", w);
        expect(t.ext == t0.ext && t.extPtr == t0.extPtr && t.sidx == t0.sidx && t.phLocal == t0.phLocal, "changed", w);
    }
    {
        BundleTable t = t0;
        expect(residentChains(t, 8, 2 * w - 1) == 0, "kept a chain that does not fit", w);
        expect(t.ext == t0.ext && t.extPtr == t0.extPtr && t.sidx == t0.sidx && t.phLocal == t0.phLocal, "changed", w);
    }
    BundleTable t = t0;
    expect(residentChains(t, 8, 3 * w) == (int)t0.chainPtr.size() - 1, "not all kept", w);
    for (int p = 0; p < t.numPhases(); ++p)
        for (int c = t.phaseChain[p]; c < t.phaseChain[p + 1]; ++c)
            expect(t.phLocal[p] >= t.extPtr[t.chainPtr[c] + 1] - t.extPtr[t.chainPtr[c]], "phase's columns", w);
    for (size_t c = 0; c + 1 < t.chainPtr.size(); ++c)
        for (int b = t.chainPtr[c]; b < t.chainPtr[c + 1]; ++b) {
            const int first = t.extPtr[t.chainPtr[c]];
            if (b > t.chainPtr[c]) expect(t.extPtr[b] == t.extPtr[b + 1], "a later bundle lists columns", w);
            const long end = b + 2 < (int)t.slot.size() ? t.off[b + 1] : (long)t.sidx.size();
            bool same = true;
            for (long e = t.off[b]; e < end; ++e)
                same = same && t.ext[first + t.sidx[e]] == t0.ext[t0.extPtr[b] + t0.sidx[e]];
            expect(same, "another column", w);
        }
}

}  // namespace

int main() {
    check(9, 512, 16);
    check(3, 2000, 64);
    check(7, 100, 8);
    if (failures == 0) std::puts("ok");
    return failures != 0;
}
