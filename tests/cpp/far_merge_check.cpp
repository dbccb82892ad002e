// Host check of the far field's merged fragments
// (grasph2_amd/csrc/sym_geometry.hpp), no GPU: replays which fragments
// far_kernel's workgroups write (one where far_merged_row says so, else one
// per wavefront and row it works on) and checks that row_fragments gives the
// combine exactly these, each once and in order, for many particle counts,
// wavefront counts and splits.  Prints "ok <cases>" and exits 0, or prints the
// first failure and exits 1.
#include <cstdio>
#include <map>
#include <vector>

#include "../../grasph2_amd/csrc/sym_geometry.hpp"

using namespace grasph;

static bool check(int64_t n, int64_t wanted, int Q, bool merge)
{
    const int64_t nsb = (n + kSB - 1) / kSB, rows = rows_with_units(nsb), U = row_prefix(rows, nsb, Q);
    if (U == 0) return true;
    const int64_t W = far_workgroups(wanted, U);
    std::map<int64_t, std::vector<int64_t>> written;  // per row, in workgroup order
    for (int64_t k0 = 0; k0 < W; k0 += kFarMerge) {
        const int64_t g = merge ? far_merged_row(k0, U, W, nsb, Q) : -1;
        if (g >= 0) {
            written[g].push_back(k0);
            continue;
        }
        for (int64_t k = k0; k < k0 + kFarMerge && k < W; ++k)
            for (int64_t r = row_of_unit(k * U / W, nsb, Q); r < rows && row_prefix(r, nsb, Q) < (k + 1) * U / W; ++r)
                written[r].push_back(k);
    }
    for (int64_t g = 0; g < rows; ++g) {
        const RowFragments R = row_fragments(row_prefix(g, nsb, Q), row_prefix(g + 1, nsb, Q), U, W, merge);
        std::vector<int64_t> read;
        for (int64_t e = 0; e < R.count; ++e) read.push_back(R.wavefront(e));
        if (read != written[g]) {
            std::printf("FAIL n=%lld W=%lld Q=%d merge=%d row %lld: %zu read, %zu written\n", (long long)n, (long long)W,
                        Q, (int)merge, (long long)g, read.size(), written[g].size());
            return false;
        }
    }
    return true;
}

int main()
{
    int cases = 0;
    for (int64_t n : {1025, 2048, 2049, 4097, 13312, 16384, 17001, 20011, 50021, 65537, 131072, 150000})
        for (int64_t W : {1, 2, 3, 4, 5, 7, 8, 40, 63, 255, 2048, 2051, 100000})
            for (int Q : {2, 4, 8, 64})
                for (int merge = 0; merge < 2; ++merge, ++cases)
                    if (!check(n, W, Q, merge)) return 1;
    std::printf("ok %d\n", cases);
    return 0;
}
