// Host-only check of the row blocks' table (race_amd/csrc/rowblock.hpp:
// RowBlocks::add), built with hipcc by tests/test_rowblock_table.py; it makes
// no HIP call.
//
//   rowblock_table columns
//     a batch of matrices with runs of empty rows at the start, in the middle
//     and at the end, smaller ones before larger ones: every entry that a
//     thread may load lies in the table, names a column of the block's own
//     matrix, and is one of the block's entries or has the value 0; every row
//     of every matrix is in one block with its own entries.
//   rowblock_table growth
//     matrices added one by one: entries are moved to new memory a number of
//     times that grows with the logarithm of their count, and one matrix alone
//     not at all.
// Prints "ok" and exits 0 on success.
#include <cstdio>
#include <cstring>
#include <vector>

#include "rowblock.hpp"

using namespace race;

namespace {

struct Crs {
    int n;
    std::vector<int> rp, col;
    std::vector<double> val;
};

// rows without entries where empty(r); others of 1 to 9 entries, one of `hub`
template <class F>
Crs matrix(int n, int hubRow, int hub, F&& empty) {
    Crs m{n, {0}, {}, {}};
    unsigned s = 12345u + (unsigned)n;
    for (int r = 0; r < n; ++r) {
        const int len = empty(r) ? 0 : r == hubRow ? hub : 1 + (int)((s >> 16) % 9);
        for (int j = 0; j < len; ++j) {
            s = s * 1664525u + 1013904223u;
            m.col.push_back((int)((s >> 8) % (unsigned)n));
            m.val.push_back(1.0 + j);
        }
        m.rp.push_back((int)m.col.size());
    }
    return m;
}

template <typename VT>
int check(int cap) {
    std::vector<Crs> ms;
    ms.push_back(matrix(1000, 3, 40, [](int r) { return r >= 448; }));       // end
    ms.push_back(matrix(100000, 5, 3000, [](int) { return false; }));        // larger
    ms.push_back(matrix(900, 700, 40, [](int r) { return r < 600; }));       // start
    ms.push_back(matrix(70000, 69999, 2000, [](int r) { return r % 1500 < 700; }));
    ms.push_back(matrix(2000, 1, 1500, [](int r) { return r > 1; }));        // behind a long row
    ms.push_back(matrix(300, -1, 0, [](int) { return true; }));              // nothing at all
    ms.push_back(matrix(50000, 9, 100, [](int) { return false; }));
    ms.push_back(matrix(1, -1, 0, [](int) { return true; }));                // the last block is empty
    RowBlocks<VT> rb;
    rb.cap = cap;
    for (size_t m = 0; m < ms.size(); ++m) rb.add(ms[m].n, ms[m].rp.data(), ms[m].col.data(), ms[m].val.data(), (int)m);
    int bad = 0, next = 0, mat = 0;
    auto fail = [&](const char* what, const RowBlk& k) {
        if (++bad <= 5) std::printf("%s: matrix %d row %d rows %d entries %d\n", what, k.mat, k.row0, (int)k.nrows, k.ne);
    };
    for (const RowBlk& k : rb.hb) {
        while (mat < k.mat && next == ms[mat].n) ++mat, next = 0;
        const Crs& m = ms[k.mat];
        if (k.mat != mat || k.row0 != next || k.nrows < 1) fail("rows out of order", k);
        next = k.row0 + k.nrows;
        if (k.ne != m.rp[next] - m.rp[k.row0] || k.p0 != m.rp[k.row0]) fail("entries", k);
        const size_t e0 = (size_t)k.e0 * 4;
        auto entry = [&](int j) {  // of the block, as a kernel loads it
            if (e0 + j >= rb.hcol.size() || e0 + j >= rb.hval.size()) return fail("outside the table", k);
            const int c = rb.hcol[e0 + j];
            if (c < 0 || c >= m.n) return fail("column of another matrix", k);
            if (c < k.base || c - k.base > 65535) {
                if (rb.narrowIds) fail("column past 16 bits", k);
            }
            if (j < k.ne ? c != m.col[k.p0 + j] : rb.hval[e0 + j] != VT(0)) fail("not the block's entry", k);
        };
        for (int t = 0; t < kBlock; ++t) {
            for (int u = 0; u < 4; ++u) entry(firstOf4(t, k.ne) + u);
            for (int u = 0; u < kPackedEntries / kBlock; ++u) entry(entryAt(t + u * kBlock, k.ne));
            for (int j = 4 * t; j < k.ne; j += 4 * kBlock)
                for (int u = 0; u < 4; ++u) entry(j + u);
        }
    }
    while (mat < (int)ms.size() && next == ms[mat].n) ++mat, next = 0;
    if (mat != (int)ms.size()) std::printf("rows missing from matrix %d\n", mat), ++bad;
    return bad;
}

int growth() {
    const Crs m = matrix(20000, 7, 300, [](int) { return false; });
    int bad = 0;
    for (int count : {1, 16, 64, 256}) {
        RowBlocks<float> rb;
        int moves = 0, log2 = 0;
        const int* at = nullptr;
        for (int k = 0; k < count; ++k) {
            rb.add(m.n, m.rp.data(), m.col.data(), m.val.data(), k);
            moves += at != nullptr && at != rb.hcol.data();
            at = rb.hcol.data();
        }
        while (1 << log2 < count) ++log2;
        if (moves > log2 + 1) std::printf("%d matrices: %d moves\n", count, moves), ++bad;
    }
    return bad;
}

}  // namespace

int main(int argc, char** argv) {
    int bad = 1;
    if (argc == 2 && !std::strcmp(argv[1], "columns"))
        bad = check<double>(kRbEntries) + check<float>(kPackedEntries) + check<uint16_t>(kRbEntries);
    else if (argc == 2 && !std::strcmp(argv[1], "growth"))
        bad = growth();
    if (bad == 0) std::puts("ok");
    return bad != 0;
}
