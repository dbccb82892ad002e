// sym_geometry.hpp -- how the symmetric sweep (sym_sweep.hip) cuts its work:
// slots in groups of 1024 (one far-field wavefront, 16 slots per lane; a
// super-block is the slots of one far wavefront, here the whole group).  The
// far field's rows are group g against the later groups; one unit is one
// partner super-block, or a piece of one.  Host and device code use these functions, and
// tests/cpp/sym_geometry_check.cpp checks them on the host (every far pair
// exactly once, indices in bounds, every partial that is read was written).
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <vector>

namespace grasph {

// own slots per lane in the far field: the partner-side reduction and the
// partners' DPP moves of a chunk are shared by the lane's slots (16: one
// wavefront owns a group of 1024, 209-235 VGPRs, 2 wavefronts per SIMD; 4 was
// measured 7% slower than 8)
constexpr int kNI = 16;
constexpr int kSB = 64 * kNI;           // slots per super-block (a far wavefront's slots)
constexpr int kGroup = 1024;            // slots per group
constexpr int kGroupSB = kGroup / kSB;  // super-blocks per group (wavefronts per far workgroup)

static_assert(kGroupSB == 1, "the row geometry below takes one far wavefront per group");

// Column batches: the far field may run in batches of partner groups
// [c0, c1) (1 <= c0 < c1 <= nsb), so the partner-side partials, which grow
// with n^2, need only the batch's share.  Row g of a batch holds its
// partner groups [max(g + 1, c0), c1), each cut into Q pieces: rows
// 0 .. c1 - 2 have units.  The unbatched far field is the batch [1, nsb).
__device__ __host__ inline int64_t col_row_units(int64_t g, int64_t c0, int64_t c1, int Q)
{
    const int64_t first = g + 1 > c0 ? g + 1 : c0;
    return first < c1 ? (c1 - first) * Q : 0;
}
// units before row g (g <= c1 - 1): rows below c0 hold c1 - c0 groups
// each, row g' >= c0 holds c1 - 1 - g'
__device__ __host__ inline int64_t col_row_prefix(int64_t g, int64_t c0, int64_t c1, int Q)
{
    const int64_t a = g < c0 ? g : c0, m = g > c0 ? g - c0 : 0;
    return Q * (a * (c1 - c0) + m * (c1 - 1 - c0) - m * (m - 1) / 2);
}
__device__ __host__ inline int64_t col_rows(int64_t c1) { return c1 >= 2 ? c1 - 1 : 0; }
// the row holding unit u of the batch: the largest g with col_row_prefix(g) <= u
__device__ __host__ inline int64_t col_row_of_unit(int64_t u, int64_t c0, int64_t c1, int Q)
{
    int64_t lo = 0, hi = col_rows(c1) - 1;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (col_row_prefix(mid, c0, c1, Q) <= u) lo = mid; else hi = mid - 1;
    }
    return lo;
}
// first partner group of row g in the batch
__device__ __host__ inline int64_t col_first_group(int64_t g, int64_t c0) { return g + 1 > c0 ? g + 1 : c0; }
// first element (of 3 per partner and row) of the batch's partner-side
// partials of group J: the groups c0 .. J - 1 before it take J' rows each
__device__ __host__ inline int64_t col_bpart_base(int64_t J, int64_t c0)
{
    return (int64_t)kGroup * (J * (J - 1) / 2 - c0 * (c0 - 1) / 2);
}

// Column batches of the far field: boundaries c[0] = 1 < c[1] < ... <
// c[last] = nsb, each batch [c[b], c[b + 1]) as wide as keeps its
// partner-side partials within max_elems floats (one group at least).
__host__ inline std::vector<int> sym_columns(int64_t nsb, int64_t max_elems)
{
    std::vector<int> c{1};
    if (nsb <= 1) {
        c.push_back(1);
        return c;
    }
    int64_t c0 = 1;
    while (c0 < nsb) {
        int64_t c1 = c0 + 1;
        while (c1 < nsb && 3 * col_bpart_base(c1 + 1, c0) <= max_elems) ++c1;
        c.push_back((int)c1);
        c0 = c1;
    }
    return c;
}

// far units of row g: each partner super-block of [kGroupSB (g + 1), nsb)
// cut into Q pieces of kSB / Q partners (Q = 1 to 64; more pieces spread the
// work more evenly)
__device__ __host__ inline int64_t row_units(int64_t g, int64_t nsb, int Q = 1)
{
    const int64_t u = nsb - (int64_t)kGroupSB * (g + 1);
    return u > 0 ? u * Q : 0;
}
// units before row g (g <= rows_with_units): sum over g' < g of row_units(g')
__device__ __host__ inline int64_t row_prefix(int64_t g, int64_t nsb, int Q = 1)
{
    return Q * (g * nsb - (int64_t)kGroupSB * (g * (g + 1) / 2));
}
// rows with far work: nsb - kGroupSB (g + 1) >= 1
__device__ __host__ inline int64_t rows_with_units(int64_t nsb) { return nsb >= 1 ? (nsb - 1) / kGroupSB : 0; }
// the row holding unit u (0 <= u < row_prefix(rows_with_units(nsb), nsb, Q)): the largest g with row_prefix(g) <= u
__device__ __host__ inline int64_t row_of_unit(int64_t u, int64_t nsb, int Q = 1)
{
    int64_t lo = 0, hi = rows_with_units(nsb) - 1;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (row_prefix(mid, nsb, Q) <= u) lo = mid; else hi = mid - 1;
    }
    return lo;
}
// pieces per partner super-block for n particles and `wanted` far
// workgroups (as many as run at once): the kernel lasts as long as its
// fullest share, ceil(U / W) units of kSB / Q partners with W = min(wanted,
// U); the Q of 2 to 64 (a piece is at least one chunk of 16 partners) that
// makes that shortest, the fewest pieces on a tie.  A share is one run of
// partners per row whatever Q is, so pieces cost nothing by themselves
// (N = 50021: 8 pieces leave the fullest of 2048 shares 9% above the mean,
// 64 pieces 0.7%; Plummer step 419 -> 391 us, N = 17000 111 -> 83).
constexpr int kMinSplit = 2, kMaxSplit = 64;
__device__ __host__ inline int far_split(int64_t n, int64_t wanted, int most = kMaxSplit)
{
    const int64_t nsb = (n + kSB - 1) / kSB;
    const int64_t u1 = row_prefix(rows_with_units(nsb), nsb, 1);
    if (u1 <= 0 || wanted <= 0) return kMinSplit;
    int best = kMinSplit;
    int64_t best_num = 0, best_den = 1;  // makespan as the fraction num / den super-blocks
    for (int Q = kMinSplit; Q <= most; Q *= 2) {
        const int64_t U = u1 * Q, W = wanted < U ? wanted : U;
        const int64_t num = (U + W - 1) / W;
        if (Q == kMinSplit || num * best_den < best_num * Q) {
            best = Q;
            best_num = num;
            best_den = Q;
        }
    }
    return best;
}
// The most partners whose terms a slot adds in plain FP32 before they join its
// LDS sum: a piece of a partner group by the rule above with 16 pieces at most
// (512 down to 64 by the count: 131072 particles 512, 165000 128, 262144 64),
// and 128 below 131072.  Of the plain sums only this one grows with the count,
// and it shows: with a fixed 512 from 131072 on the error against FP64 (equal /
// unequal masses) is 4.13e-8 / 5.32e-8 of the norm at 165000 and 3.88e-8 /
// 4.68e-8 at 262144, with the rule 3.64e-8 / 4.15e-8 and 3.53e-8 / 3.78e-8, for
// 2.2% and 3.3% of the step.  At 65536 128 instead of the piece's 512 gives
// 3.86e-8 / 5.48e-8 instead of 4.67e-8 / 6.96e-8 for 1.8%; at 131072 it would
// cost 1.6%.
constexpr int kMaxFoldSplit = 16, kShortFold = 128;
constexpr int64_t kShortFoldBelow = 131072;
__device__ __host__ inline int far_fold(int64_t n, int64_t wanted)
{
    const int piece = kSB / far_split(n, wanted, kMaxFoldSplit);
    return n < kShortFoldBelow && piece > kShortFold ? kShortFold : piece;
}
// the workgroup whose share [k U / W, (k + 1) U / W) holds unit u
__device__ __host__ inline int64_t wg_of_unit(int64_t u, int64_t U, int64_t W) { return ((u + 1) * W - 1) / U; }
// Wavefronts of the whole far field's workgroups: workgroup K's are k =
// kFarMerge K and the next.  Where all of them are there and work on one row,
// their own-side sums leave as one fragment, wavefront kFarMerge K's
// (far_merged_row: that row, else -1).  Only plain fragments are merged; a
// merged one has corrections.
constexpr int kFarMerge = 8;
__device__ __host__ inline int64_t far_merged_row(int64_t k0, int64_t U, int64_t W, int64_t nsb, int Q)
{
    if (k0 + kFarMerge > W) return -1;
    const int64_t g = row_of_unit(k0 * U / W, nsb, Q);
    return (k0 + kFarMerge) * U / W <= row_prefix(g + 1, nsb, Q) ? g : -1;
}
// The fragments of a row whose units are [u0, u1): those of wavefronts k0 ..
// k0 + lead - 1, `merged` of whole workgroups, and the wavefronts' after them.
struct RowFragments {
    int64_t k0, lead, merged, count;
    __device__ __host__ int64_t wavefront(int64_t e) const  // whose the e-th is
    {
        return k0 + e + (e < lead ? 0 : e < lead + merged ? (kFarMerge - 1) * (e - lead) : (kFarMerge - 1) * merged);
    }
};
__device__ __host__ inline RowFragments row_fragments(int64_t u0, int64_t u1, int64_t U, int64_t W, bool merge)
{
    RowFragments R;
    R.k0 = wg_of_unit(u0, U, W);
    const int64_t k1 = wg_of_unit(u1 - 1, U, W) + 1;  // wavefronts [k0, k1)
    R.lead = R.count = k1 - R.k0;
    R.merged = 0;
    if (!merge) return R;
    const int64_t first = (R.k0 + (R.k0 * U / W < u0) + kFarMerge - 1) / kFarMerge;  // workgroups [first, last)
    const int64_t last = (k1 - (k1 * U / W > u1)) / kFarMerge;
    if (first < last) {
        R.lead = kFarMerge * first - R.k0;
        R.merged = last - first;
        R.count -= (kFarMerge - 1) * R.merged;
    }
    return R;
}
// workgroups of the far kernel: at most the units, so every one has a share and a row's
// fragments come from consecutive workgroups
__host__ inline int far_workgroups(int64_t wanted, int64_t units)
{
    const int64_t w = wanted < units ? wanted : units;
    return (int)(w > 1 ? w : 1);
}
// A batch's far rows go to its wavefronts whole or in pieces: row g of an
// instance (row_units(g, nsb) partner groups) is cut into
// batch_row_pieces(units, most) pieces of consecutive partner groups, piece h
// starting at batch_piece_begin(units, h, most); each piece leaves its own-side
// sums as its own fragment (`most` fragments per row), so the longest
// rows do not set the kernel's length.
// Batches with fewer pieces than wavefronts cut their rows finer, kBatchPiecesMost
// at most (one instance of 60000 among 300 of 100 7544 -> 2235 us a derivative
// call, 8 of 32768 4535 -> 1540: a piece held up to 15 groups, one wavefront
// alone on its SIMD).
constexpr int kBatchPieces = 4, kBatchPiecesMost = 16;
__device__ __host__ inline int batch_row_pieces(int64_t units, int most = kBatchPieces)
{
    return units < most ? (int)units : most;
}
__device__ __host__ inline int64_t batch_piece_begin(int64_t units, int h, int most = kBatchPieces)
{
    return h * units / batch_row_pieces(units, most);
}
// first element of the partner-side partials of group h (the h groups before it contribute)
__device__ __host__ inline int64_t bpart_group_base(int64_t h) { return (int64_t)kGroup * (h * (h - 1) / 2); }

// Own-side fragments: one per (row, wavefront that worked on the row), in
// float4 elements, 2 kGroup of them: for each 64 slots of the group, their
// 64 sums (x y z, w unused), then those sums' 64 corrections (slot s: sums
// at frag_elem(s), corrections 64 further).  A wavefront folds its own-side
// sums into LDS sums every so many partners and those into the fragment every
// kFoldsPerFlush folds and at the end of its stay on the row.  The first flush
// writes the sums (their corrections are exactly zero).  When no stay has more
// than kFoldsPerFlush folds, every fragment is flushed once: it is
// plain, and neither the far field nor the combine touch its corrections
// (except a merged one's, which its wavefronts' sums leave);
// otherwise the first flush writes zero corrections too.
constexpr int kFoldsPerFlush = 16;
constexpr int kFragElems = 2 * kGroup;
__device__ __host__ inline int frag_elem(int slot) { return 128 * (slot >> 6) + (slot & 63); }
__device__ __host__ inline bool fragments_plain(int64_t max_folds_per_visit)
{
    return max_folds_per_visit <= kFoldsPerFlush;
}

}  // namespace grasph
