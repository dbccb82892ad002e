// sym_sweep.hip -- the all-pairs gravity sweep evaluated once per unordered
// pair (gfx950).
//
// Same results as the sweep of sweep.hip (softened gravity of
// calcAcceleration, src/computeDerivatives.h:229-235), organised by groups
// of 1024 consecutive slots:
//  - in-group gravity, one-sided (own_block.hpp);
//  - far field: every pair of slots in different groups is computed once,
//    for both sides (Newton's third law).  One wavefront owns a group (16
//    slots per lane).  The later groups' particles come 16 at a time, one
//    per lane of each 16-lane DPP row, and go once round the row
//    (far_rotation.hpp); a lane sums its own slots' gravity in registers,
//    and each partner's sum travels with it.  Two swaps then add the four
//    rows, and the values are stored as the (group, partner) partial
//    straight away;
//  - a combine kernel adds, per slot and in a fixed order, the in-group sum,
//    the far own-side fragments and the far partner-side partials
//    (compensated), then finishes the acceleration as the one-range sweep.
// Per far pair: 3 sub, 3 FMA for r^2 + H^2, one v_rsq_f32, 2 mul, 3 FMA for
// the own side and 3 FMA for the partner side (2 more mul with unequal
// masses), plus 6 DPP instructions per rotation of 16 pairs: for two
// interactions per lane and slot, against 11 and a v_rsq_f32 for one in the
// one-sided sweep.
// Every sum is in a fixed order, so results do not vary from run to run.
#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

#include "far_rotation.hpp"
#include "own_block.hpp"
#include "sym_geometry.hpp"

namespace grasph {
namespace {

constexpr int kBlock = 256;
constexpr int kFarThreads = 64;  // one wavefront owns a group
static_assert(kGroupSB == 1 && kSB == kGroup, "the far field assumes one wavefront per group");

// ------------------------------------------------------------------ cross-lane reduction

__device__ __forceinline__ float swap32_sum(float p, float q)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(p), __float_as_uint(q), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_sum(float p, float q)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(p), __float_as_uint(q), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// ------------------------------------------------------------------ kernels

// In-group gravity: a workgroup takes 64 NI slots of a group, its wavefronts
// a share of len (times their number at least the group's slots) of the
// group's slots as partners each.  store(t, x, y, z) gets every slot's
// compensated sums.
template <int NI, bool SOFT, typename F>
__device__ __forceinline__ void ingroup_block(const float4* __restrict__ xs, const int o0, const int g0, const int g1,
                                              const int len, const float h2, const float* __restrict__ um, float* lds,
                                              F&& store)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = blockDim.x >> 6;
    if (um && um[0] != 0.0f)
        own_block<NI, true, SOFT>(xs, o0, g1, g0, g1, len, h2, um[1], wave, waves, lds, store);
    else
        own_block<NI, false, SOFT>(xs, o0, g1, g0, g1, len, h2, 1.0f, wave, waves, lds, store);
}

// a slot's compensated sums as two float4
__device__ __forceinline__ void store_near(float4* __restrict__ near_part, const int t, const CSum& x, const CSum& y,
                                           const CSum& z)
{
    near_part[2 * (size_t)t] = make_float4(x.s, y.s, z.s, 0.0f);
    near_part[2 * (size_t)t + 1] = make_float4(x.c, y.c, z.c, 0.0f);
}

template <bool SOFT>
__global__ __launch_bounds__(64 * kOwnMaxWaves) void ingroup_kernel(const float4* __restrict__ xs, const int n,
                                                                    float4* __restrict__ near_part, const float h2,
                                                                    const float* __restrict__ umass)
{
    extern __shared__ float lds[];
    const int o0 = 64 * blockIdx.x, g0 = o0 / kGroup * kGroup;
    ingroup_block<1, SOFT>(xs, o0, g0, min(n, g0 + kGroup), kGroup / (int)(blockDim.x >> 6), h2, umass, lds,
                           [&](int t, const CSum& x, const CSum& y, const CSum& z) { store_near(near_part, t, x, y, z); });
}

// One chunk of 16 partners (pj: row lane l holds partner l) against the
// lane's kNI slots.  Own side into o.a*; returns the partner side: lanes
// 0-15 hold partner l's x, lanes 16-31 partner l - 16's z, lanes 32-47
// partner l - 32's y (UM: without the common mass; else with the slots' masses).
template <bool UM, bool SOFT, bool WIDE>
__device__ __forceinline__ float far_chunk_rot(const float4 pj, FarOwn& o, const float H2)
{
    FarPartner p{pj.x, pj.y, pj.z, pj.w, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int k = 0; k < kRow; ++k) {
        if constexpr (SOFT)
            far_rotation_soft<UM, WIDE>(p, o, H2);
        else
            far_rotation_hard<UM, WIDE>(p, o);
    }
    // the last rotation's contribution, then home
    const float tx = ror<1>(ror<1>(p.tx) + p.px), ty = ror<1>(ror<1>(p.ty) + p.py), tz = ror<1>(ror<1>(p.tz) + p.pz);
    // rows 0 + 2 and 1 + 3: x to lanes 0-31, y to lanes 32-63; z everywhere
    const float xy = swap32_sum(tx, ty);
    const float zz = swap32_sum(tz, tz);
    // row 0: x, row 1: z, row 2: y (row 3: z again)
    return swap16_sum(xy, zz);
}

// partner b + (lane & 15) of an instance of n particles (clamped to n - 1:
// a look-ahead past the end loads values nobody uses).  UM loads x y z
// alone: a loaded register left unused would be reused at once, and that
// write would wait for the load, a chunk too early.
template <bool UM>
__device__ __forceinline__ float4 load_partner_row(const float4* __restrict__ xs, const int b, const int n,
                                                   const int lane)
{
    const int jc = min(b + (lane & (kRow - 1)), n - 1);
    if (UM) {
        const float3 p = *reinterpret_cast<const float3*>(xs + jc);
        return make_float4(p.x, p.y, p.z, 0.0f);
    }
    return xs[jc];
}
// partners at or past n: far away and massless (applied where the chunk is
// used, so the load's wait stays there)
__device__ __forceinline__ float4 bound_partner_row(const float4 v, const int b, const int n, const int lane)
{
    return b + (lane & (kRow - 1)) >= n ? make_float4(3.0e18f, 3.0e18f, 3.0e18f, 0.0f) : v;
}

// component of the partner side this lane holds after far_chunk_rot: row 0
// x, row 2 y, rows 1 and 3 z (the same value, bit for bit, stored to the
// same place: every lane stores, so an unbounded chunk's store needs no
// branch, behind which the compiler would sink the chunk's own-side sums)
__device__ __forceinline__ int partner_comp_rot(const int lane)
{
    const int row = lane >> 4;
    return row == 0 ? 0 : row == 2 ? 1 : 2;
}

// The own slots of row g (slots 1024 g + 64 q + lane, q < kNI) of an
// instance of n particles at xs (slots past n sit far away and massless),
// the wavefront's LDS sums lsum, and the row's fragment of workgroup k:
// frag (fresh until the first flush).
__device__ __forceinline__ void far_load_row(const float4* __restrict__ xs, const int n, const int64_t g,
                                             const int lane, float* lsum, float4* frag, const bool plain, FarOwn& o)
{
#pragma unroll
    for (int q = 0; q < kNI; ++q) {
        const int t = kSB * (int)g + 64 * q + lane;
        o.x[q] = o.y[q] = o.z[q] = -3.0e18f;
        o.m[q] = 0.0f;
        if (t < n) {
            const float4 p = xs[t];
            o.x[q] = p.x; o.y[q] = p.y; o.z[q] = p.z; o.m[q] = p.w;
        }
        o.ax[q] = o.ay[q] = o.az[q] = 0.0f;
    }
    o.lsum = lsum;
    o.frag = frag;
    o.folds = 0;
    o.fresh = true;
    o.plain = plain;
}

// The lane's slot of own slot q, through an empty asm statement: indexed
// by it, the LDS sums and the fragment are never kept in registers across
// a row's folds by the compiler (96 more live values, which the pair loop
// cannot spare).
__device__ __forceinline__ int own_lane(const int lane)
{
    int l = lane;
    __asm__ volatile("" : "+v"(l));
    return l;
}

// The LDS sums of the lane's slots added (compensated) into the row's
// fragment; the first flush stores them (and zero corrections unless the
// fragments are plain).
__device__ __forceinline__ void far_flush_own(FarOwn& o, const int lane)
{
    if (o.folds == 0) return;
    const int l = own_lane(lane);
    float4* const fr = o.frag;
#pragma unroll
    for (int q = 0; q < kNI; ++q) {
        const int slot = 64 * q + l, e = 128 * q + l;  // e: frag_elem(slot)
        float4 sv = make_float4(0.f, 0.f, 0.f, 0.f), cv = sv;
        if (!o.fresh) {
            sv = fr[e];
            cv = fr[e + 64];
        }
        CSum x{sv.x, cv.x}, y{sv.y, cv.y}, z{sv.z, cv.z};
        x.add(o.lsum[slot]);
        y.add(o.lsum[kGroup + slot]);
        z.add(o.lsum[2 * kGroup + slot]);
        fr[e] = make_float4(x.s, y.s, z.s, 0.0f);
        if (!o.plain) fr[e + 64] = make_float4(x.c, y.c, z.c, 0.0f);
    }
    o.fresh = false;
    o.folds = 0;
}

// The lane's plain own-side sums added to its LDS sums, then cleared;
// every kFoldsPerFlush folds the LDS sums go to the fragment.
template <bool UM>
__device__ __forceinline__ void far_fold_own(FarOwn& o, const float m, const int lane)
{
    if (o.folds == kFoldsPerFlush) far_flush_own(o, lane);
    float* const sum = o.lsum + own_lane(lane);
    float old[3][kNI];  // all read before the first is used: one by one they waited 32 times a fold
    if (o.folds > 0) {
#pragma unroll
        for (int q = 0; q < kNI; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) old[c][q] = sum[kGroup * c + 64 * q];
    } else {
#pragma unroll
        for (int q = 0; q < kNI; ++q) old[0][q] = old[1][q] = old[2][q] = 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kNI; ++q) {
        const float ax = UM ? o.ax[q] * m : o.ax[q];
        const float ay = UM ? o.ay[q] * m : o.ay[q];
        const float az = UM ? o.az[q] * m : o.az[q];
        sum[64 * q] = old[0][q] + ax;
        sum[kGroup + 64 * q] = old[1][q] + ay;
        sum[2 * kGroup + 64 * q] = old[2][q] + az;
        o.ax[q] = o.ay[q] = o.az[q] = 0.0f;
    }
    ++o.folds;
}

// Partners [b0, b1) (multiples of 16; those past n are left out) against the
// slots of row g, a chunk of 16 at a time; each chunk's partner side (summed
// over the whole group: one wavefront owns it) goes straight to row g's
// partials of its group (element 3 (bpart_group_base(J) - boff) on holds
// group J's; boff: the groups before the column batch).  UM: the row's slots
// have mass mo and the partners mass mp, which the sums take as a factor.  The
// store has no condition: partners of the last chunk past n (their group's
// partials are allocated whole) get values nobody reads, and a store behind a
// branch makes the compiler spill the chunk's registers.
// The own side is folded every `fold` partners and at the end, so a slot
// adds at most that many terms in plain FP32 before they join its LDS sum
// (and at most kFoldsPerFlush such sums before they join the compensated
// fragment): far_fold's number, in batches half a group.
constexpr int kBatchFold = 512;
template <bool UM, bool SOFT, bool WIDE>
__device__ __forceinline__ void far_range(const float4* __restrict__ xs, const int n, const int64_t g, const int b0,
                                          const int b1, const int fold, FarOwn& o, float* __restrict__ bpart,
                                          const int64_t boff, const float H2, const float mo, const float mp,
                                          const int lane)
{
    const int end = min(b1, n);
    if (b0 >= end) {  // a share of the last group past n: zeros in its fragment
        far_fold_own<UM>(o, mp, lane);
        return;
    }
    float* bp = nullptr;  // row g's partials of the chunk's first partner, for this lane
    int terms = 0;
    float4 A = load_partner_row<UM>(xs, b0, n, lane);
    for (int b = b0; b < end; b += kRow) {
        if (b == b0 || b % kGroup == 0)
            bp = bpart + 3 * (bpart_group_base(b / kGroup) - boff + g * kGroup + b % kGroup) +
                 3 * (lane & (kRow - 1)) + partner_comp_rot(lane);
        const float4 B = load_partner_row<UM>(xs, b + kRow, n, lane);  // unused after the last
        if (b + kRow > end) A = bound_partner_row(A, b, n, lane);
        const float v = far_chunk_rot<UM, SOFT, WIDE>(A, o, H2);
        *bp = UM ? v * mo : v;
        bp += 3 * kRow;
        A = B;
        terms += kRow;
        if (terms == fold || b + kRow >= end) {
            far_fold_own<UM>(o, mp, lane);
            terms = 0;
        }
    }
}

// Far field of one instance, or (COL) column batch [c0, c1) of its partner
// groups.  Workgroup k of W takes the units [k U / W, (k + 1) U / W) of the
// rows g (group g against its later groups, or those in the batch, each cut
// into Q pieces) laid end to end: consecutive partners, row by row.  Its
// own-side sums of row g go to fragment g + k (plain: every fragment is
// flushed once).  The whole far field keeps a kernel of its own (far_kernel),
// so the row arithmetic of the batches does not change its code.
// umass null: each run finds out for itself whether its own slots have one
// mass and its partners one (one more read of their masses, the first ones
// with the row's slots; a kernel that looks at all particles first costs 5 us,
// 8% of a Plummer step at 16384).
template <bool SOFT, bool COL, bool WIDE>
__device__ __forceinline__ void far_work(const float4* __restrict__ xs, const int n, const int64_t nsb, const int c0,
                                         const int c1, const int64_t U, const int W, const int Q, const int fold,
                                         float4* __restrict__ apart, const bool plain, const int k, const bool merge,
                                         float* __restrict__ bpart, const float H2,
                                         const float* __restrict__ umass, float* lsum)
{
    if (k >= W) return;
    const int lane = threadIdx.x & 63, len = kSB / Q;
    int64_t u = (int64_t)k * U / W;
    const int64_t u1 = (int64_t)(k + 1) * U / W;
    if (u >= u1) return;
    const int64_t boff = COL ? bpart_group_base(c0) : 0;
    int64_t g = COL ? col_row_of_unit(u, c0, c1, Q) : row_of_unit(u, nsb, Q);
    int64_t s = u - (COL ? col_row_prefix(g, c0, c1, Q) : row_prefix(g, nsb, Q));  // first unit within row g
    FarOwn o;
    for (; u < u1; ++g, s = 0) {
        const int64_t row = COL ? col_row_units(g, c0, c1, Q) : row_units(g, nsb, Q);
        const int64_t cnt = min(row - s, u1 - u);
        const int first = kSB * (int)(COL ? col_first_group(g, c0) : g + 1) + len * (int)s;
        const int end = first + len * (int)cnt;
        float mo, mp = 0.0f, mj = 0.0f;
        if (!umass) {
            mp = xs[min(first, n - 1)].w;
            mj = xs[min(first + lane, min(end, n) - 1)].w;
        }
        far_load_row(xs, n, g, lane, lsum, apart + (size_t)kFragElems * (g + k), plain, o);
        bool one_mass;
        if (umass) {
            one_mass = umass[0] != 0.0f;
            mo = mp = umass[1];
        } else {
            mo = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(o.m[0])));
            int differ = __float_as_int(mj) ^ __float_as_int(mp);
#pragma unroll
            for (int q = 0; q < kNI; ++q) differ |= __float_as_int(o.m[q]) ^ __float_as_int(mo);
#pragma unroll 4
            for (int j = first + 64 + lane; j < min(end, n); j += 64)
                differ |= __float_as_int(xs[j].w) ^ __float_as_int(mp);
            one_mass = !__any(differ != 0);
        }
        if (one_mass)
            far_range<true, SOFT, false>(xs, n, g, first, end, fold, o, bpart, boff, H2, mo, mp, lane);
        else
            far_range<false, SOFT, WIDE>(xs, n, g, first, end, fold, o, bpart, boff, H2, 1.0f, 1.0f, lane);
        if (!merge) far_flush_own(o, lane);
        u += cnt;
    }
}

// Wavefronts share a workgroup so that, when their ranges lie in one row (all
// but two a row), their own-side sums leave as one fragment: a fragment per
// wavefront was 34 MB written and read again, whatever the count (Plummer
// N = 16384: 69.6 -> 66.6 us per step, 50021: 441 -> 434).
// WIDE (below kSymOneSided particles, down to where the one-sided sweep takes over):
// unequal masses in any units, as there (unequal masses, N = 13000: 51.6 -> 53.6 us
// a step; from 16384 on 1 / r^3 has to be in range by itself).
template <bool SOFT, bool WIDE>
__global__ __launch_bounds__(64 * kFarMerge, 2) void far_kernel(const float4* __restrict__ xs, const int n,
                                                               const int64_t nsb, const int64_t U, const int W,
                                                               const int Q, const int fold,
                                                               float4* __restrict__ apart, const int plain,
                                                               float* __restrict__ bpart, const float H2,
                                                               const float* __restrict__ umass)
{
    __shared__ float lsum[kFarMerge][3 * kGroup];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int k0 = kFarMerge * (int)blockIdx.x;
    const int64_t g = plain ? far_merged_row(k0, U, W, nsb, Q) : -1;
    const bool merge = g >= 0;  // the same for the whole workgroup
    far_work<SOFT, false, WIDE>(xs, n, nsb, 1, (int)nsb, U, W, Q, fold, apart, plain, k0 + wave, merge, bpart, H2, umass,
                          lsum[wave]);
    if (!merge) return;
    __syncthreads();
    float4* const fr = apart + (size_t)kFragElems * (g + k0);
    for (int q = wave; q < kNI; q += kFarMerge) {
        const int slot = 64 * q + lane;
        CSum v[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v[c] = CSum{lsum[0][kGroup * c + slot], 0.0f};
#pragma unroll
            for (int w = 1; w < kFarMerge; ++w) v[c].add(lsum[w][kGroup * c + slot]);
        }
        fr[128 * q + lane] = make_float4(v[0].s, v[1].s, v[2].s, 0.0f);  // frag_elem(slot)
        fr[128 * q + lane + 64] = make_float4(v[0].c, v[1].c, v[2].c, 0.0f);
    }
}

// one column batch [c0, c1) of the far field
template <bool SOFT>
__global__ __launch_bounds__(kFarThreads, 2) void far_column_kernel(const float4* __restrict__ xs, const int n,
                                                                   const int c0, const int c1, const int64_t U,
                                                                   const int W, const int Q, const int fold,
                                                                   float4* __restrict__ apart, const int plain,
                                                                   float* __restrict__ bpart, const float H2,
                                                                   const float* __restrict__ umass)
{
    __shared__ float lsum[3 * kGroup];
    far_work<SOFT, true, false>(xs, n, 0, c0, c1, U, W, Q, fold, apart, plain, blockIdx.x, false, bpart, H2, umass, lsum);
}

// The far field's part p of PARTS of slot t's sums: the own-side fragments of
// its row, then the partner-side partials, every PARTS-th from the p-th on.
template <int PARTS, bool PLAIN>
__device__ __forceinline__ void far_sums(const float4* __restrict__ apart, const float* __restrict__ bpart,
                                         const int t, const int p, const int64_t nsb, const int64_t U, const int W,
                                         const int Q, CSum& x, CSum& y, CSum& z)
{
    const int64_t g = t / kGroup, local = t - g * kGroup;
    if (U > 0 && g < rows_with_units(nsb)) {
        // one fragment per wavefront that touched the row (every wavefront
        // has a share: W <= U), or per workgroup of them; eight fragments'
        // loads in flight before their ordered adds
        const RowFragments R = row_fragments(row_prefix(g, nsb, Q), row_prefix(g + 1, nsb, Q), U, W, PLAIN);
        const float4* const row = apart + (size_t)kFragElems * g + frag_elem((int)local);
        // fragments [e0, e1), with their corrections
        const auto add = [&](const int64_t e0, const int64_t e1, auto corrections) {
            int64_t k = e0 + p;
            for (; k + 7 * PARTS < e1; k += 8 * PARTS) {
                float4 f[8], fc[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float4* fr = row + (size_t)kFragElems * R.wavefront(k + u * PARTS);
                    f[u] = fr[0];
                    if constexpr (corrections) fc[u] = fr[64];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    x.add(f[u].x); y.add(f[u].y); z.add(f[u].z);
                    if constexpr (corrections) { x.c += fc[u].x; y.c += fc[u].y; z.c += fc[u].z; }
                }
            }
            for (; k < e1; k += PARTS) {
                const float4* fr = row + (size_t)kFragElems * R.wavefront(k);
                const float4 f = fr[0];
                x.add(f.x); y.add(f.y); z.add(f.z);
                if constexpr (corrections) {
                    const float4 fc = fr[64];
                    x.c += fc.x; y.c += fc.y; z.c += fc.z;
                }
            }
        };
        if constexpr (PLAIN) {
            add(0, R.lead, std::false_type());
            add(R.lead, R.lead + R.merged, std::true_type());
            add(R.lead + R.merged, R.count, std::false_type());
        } else {
            add(0, R.count, std::true_type());
        }
    }
    const int64_t base = bpart_group_base(g) + local;
    const int ng = (int)g;
    // eight groups' loads in flight before their (ordered) adds
    int gp = p;
    for (; gp + 7 * PARTS < ng; gp += 8 * PARTS) {
        float v[8][3];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t e = 3 * (size_t)(base + (int64_t)(gp + u * PARTS) * kGroup);
            v[u][0] = bpart[e]; v[u][1] = bpart[e + 1]; v[u][2] = bpart[e + 2];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            x.add(-v[u][0]); y.add(-v[u][1]); z.add(-v[u][2]);
        }
    }
    for (; gp < ng; gp += PARTS) {
        const size_t e = 3 * (size_t)(base + (int64_t)gp * kGroup);
        x.add(-bpart[e]); y.add(-bpart[e + 1]); z.add(-bpart[e + 2]);
    }
}

// The parts' sums added in part order, in part 0's threads (thread q kSlots +
// l holds part q of the workgroup's l-th slot).
template <int PARTS, int SLOTS>
__device__ __forceinline__ void add_parts(const int p, CSum& x, CSum& y, CSum& z)
{
    __shared__ float red[6][PARTS * SLOTS];  // every thread reaches the barrier
    if (p > 0) {
        red[0][threadIdx.x] = x.s; red[1][threadIdx.x] = x.c;
        red[2][threadIdx.x] = y.s; red[3][threadIdx.x] = y.c;
        red[4][threadIdx.x] = z.s; red[5][threadIdx.x] = z.c;
    }
    __syncthreads();
    if (p > 0) return;
#pragma unroll
    for (int q = 1; q < PARTS; ++q) {
        const int o = (int)threadIdx.x + q * SLOTS;
        x.add(red[0][o]); x.c += red[1][o];
        y.add(red[2][o]); y.c += red[3][o];
        z.add(red[4][o]); z.c += red[5][o];
    }
}

// slot t's gravity into the acceleration of its particle
__device__ __forceinline__ void finish_slot(const int t, CSum x, CSum y, CSum z, const int* __restrict__ perm,
                                            float4* __restrict__ acc, const int finish, const int add_acc,
                                            float4* __restrict__ xvel, float* __restrict__ maxvsig,
                                            const DevParams& P)
{
    const int i = perm ? perm[t] : t;
    if (add_acc) {  // the SPH terms (and environment), summed before the far field was done
        const float4 a = acc[i];
        x.add(a.x); y.add(a.y); z.add(a.z);
    }
    float ax = x.value(), ay = y.value(), az = z.value();
    if (finish) {
        environment_acceleration(P, ax, ay, az);
        if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (maxvsig) maxvsig[i] = 0.0f;
    }
    acc[i] = make_float4(ax, ay, az, 0.0f);
}

// Per slot, in a fixed order: the in-group sums, the far own-side fragments
// (workgroup order), the far partner-side partials (group order, negated:
// they were summed as seen from the other side), compensated; then the
// acceleration is finished as the one-range sweep does.  With PARTS > 1
// (small counts: the slots alone would not fill the GPU, and a slot's row
// has up to hundreds of fragments), PARTS threads share a slot: part p
// takes every PARTS-th term of each list from the p-th on, and part 0 adds
// the parts' compensated sums in part order.  PLAIN: the fragments hold
// sums alone (their corrections are zero and were not stored).
template <int PARTS, bool PLAIN>
__global__ __launch_bounds__(kBlock) void sym_combine_kernel(
    const float4* __restrict__ near_part, const float4* __restrict__ apart, const float* __restrict__ bpart,
    const int n, const int64_t nsb, const int64_t U, const int W, const int Q,
    const int* __restrict__ perm, float4* __restrict__ acc, const int finish, const int add_acc,
    float4* __restrict__ xvel, float* __restrict__ maxvsig, const DevParams P)
{
    constexpr int kSlots = kBlock / PARTS;  // slots per block
    const int p = (int)threadIdx.x / kSlots;
    const int t = blockIdx.x * kSlots + ((int)threadIdx.x - p * kSlots);
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
    if (t < n) {
        if (p == 0) {
            const float4 a = near_part[2 * (size_t)t], c = near_part[2 * (size_t)t + 1];
            x = CSum{a.x, c.x}; y = CSum{a.y, c.y}; z = CSum{a.z, c.z};
        }
        far_sums<PARTS, PLAIN>(apart, bpart, t, p, nsb, U, W, Q, x, y, z);
    }
    if constexpr (PARTS > 1) add_parts<PARTS, kSlots>(p, x, y, z);
    if (p == 0 && t < n) finish_slot(t, x, y, z, perm, acc, finish, add_acc, xvel, maxvsig, P);
}

// In-group gravity and combine in one launch, for counts at which either
// takes as long as its launch: a workgroup of kNearFused wavefronts makes 64
// slots' in-group sums as ingroup_kernel does, then wavefront p is their part
// p of the combine.  The in-group sums are the two kernels'
// bit for bit; the combine has 8 parts whatever the count.  Plummer N =
// 16384: 61.5 -> 59.4 us per step.
constexpr int kNearFused = 8;
template <bool SOFT>
__global__ __launch_bounds__(64 * kNearFused) void near_combine_kernel(
    const float4* __restrict__ xs, const float4* __restrict__ apart, const float* __restrict__ bpart, const int n,
    const int64_t nsb, const int64_t U, const int W, const int Q, const float* __restrict__ umass,
    const int* __restrict__ perm, float4* __restrict__ acc, const int finish, const int add_acc,
    float4* __restrict__ xvel, float* __restrict__ maxvsig, const DevParams P)
{
    __shared__ float lds[own_lds_floats(1, kNearFused)];
    const int p = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int o0 = 64 * blockIdx.x, g0 = o0 / kGroup * kGroup, t = o0 + lane;
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
    ingroup_block<1, SOFT>(xs, o0, g0, min(n, g0 + kGroup), kGroup / kNearFused, P.H2, umass, lds,
                           [&](int, const CSum& a, const CSum& b, const CSum& c) {  // wavefront 0's lanes
                               x = a; y = b; z = c;
                           });
    if (t < n) far_sums<kNearFused, true>(apart, bpart, t, p, nsb, U, W, Q, x, y, z);
    add_parts<kNearFused, 64>(p, x, y, z);
    if (p == 0 && t < n) finish_slot(t, x, y, z, perm, acc, finish, add_acc, xvel, maxvsig, P);
}

// After column batch [c0, c1) of the far field (column-batched far field,
// one thread per slot): the slot's running compensated sums (accsum: 2
// float4 per slot, sums then corrections; none before the first batch)
// take the batch's own-side fragments of the slot's row and, for slots in
// the batch's groups, their partner-side partials, complete now (every row
// before the group was in the batch).  After the last batch the near
// partials join them and the acceleration is finished as in the combine.
__global__ __launch_bounds__(kBlock) void sym_column_combine_kernel(
    const float4* __restrict__ near_part, const float4* __restrict__ apart, const float* __restrict__ bpart,
    float4* __restrict__ accsum, const int n, const int c0, const int c1, const int64_t U,
    const int W, const int Q, const int plain, const int first, const int last, const int* __restrict__ perm,
    float4* __restrict__ acc, const int finish, const int add_acc, float4* __restrict__ xvel,
    float* __restrict__ maxvsig, const DevParams P)
{
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n) return;
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
    if (!first) {
        const float4 a = accsum[2 * (size_t)t], c = accsum[2 * (size_t)t + 1];
        x = CSum{a.x, c.x}; y = CSum{a.y, c.y}; z = CSum{a.z, c.z};
    }
    const int g = t / kGroup, local = t - g * kGroup;
    if (g < col_rows(c1) && U > 0) {
        // the fragments of the workgroups that worked on row g in this batch
        const int64_t k0 = wg_of_unit(col_row_prefix(g, c0, c1, Q), U, W);
        const int64_t k1 = wg_of_unit(col_row_prefix(g + 1, c0, c1, Q) - 1, U, W);
        const int el = frag_elem(local);
        for (int64_t k = k0; k <= k1; ++k) {
            const float4* fr = apart + (size_t)kFragElems * (g + k) + el;
            const float4 f = fr[0];
            x.add(f.x); y.add(f.y); z.add(f.z);
            if (!plain) {
                const float4 fc = fr[64];
                x.c += fc.x; y.c += fc.y; z.c += fc.z;
            }
        }
    }
    if (g >= c0 && g < c1) {
        const int64_t base = col_bpart_base(g, c0) + local;
        int gp = 0;  // eight rows' loads in flight before their (ordered) adds
        for (; gp + 8 <= g; gp += 8) {
            float v[8][3];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t e = 3 * (size_t)(base + (int64_t)(gp + u) * kGroup);
                v[u][0] = bpart[e]; v[u][1] = bpart[e + 1]; v[u][2] = bpart[e + 2];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                x.add(-v[u][0]); y.add(-v[u][1]); z.add(-v[u][2]);
            }
        }
        for (; gp < g; ++gp) {
            const size_t e = 3 * (size_t)(base + (int64_t)gp * kGroup);
            x.add(-bpart[e]); y.add(-bpart[e + 1]); z.add(-bpart[e + 2]);
        }
    }
    if (!last) {
        accsum[2 * (size_t)t] = make_float4(x.s, y.s, z.s, 0.0f);
        accsum[2 * (size_t)t + 1] = make_float4(x.c, y.c, z.c, 0.0f);
        return;
    }
    {
        const float4 a = near_part[2 * (size_t)t], c = near_part[2 * (size_t)t + 1];
        x.add(a.x); y.add(a.y); z.add(a.z);
        x.c += c.x; y.c += c.y; z.c += c.z;
    }
    const int i = perm ? perm[t] : t;
    if (add_acc) {  // the SPH terms (and environment), summed before the far field was done
        const float4 a = acc[i];
        x.add(a.x); y.add(a.y); z.add(a.z);
    }
    float ax = x.value(), ay = y.value(), az = z.value();
    if (finish) {
        environment_acceleration(P, ax, ay, az);
        if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (maxvsig) maxvsig[i] = 0.0f;
    }
    acc[i] = make_float4(ax, ay, az, 0.0f);
}

// ------------------------------------------------------------------ batches
// The same sweep over the larger instances of a batch (slot indices are
// the batch's; the smaller instances stay with the one-sided persistent
// sweep).  Differences: four wavefronts share the in-group gravity of a block
// of slots; the far kernel is persistent and takes rows (instance, group), cut
// into kBatchPieces or a few more pieces, longest first; each piece's own-side sums
// leave as a fragment, numbered by the instance's first row + g and the piece.

// NI 4: blk has blocks of 256 slots, NI 1: of 64.
template <int NI, bool SOFT>
__global__ __launch_bounds__(kBlock) void sym_batch_ingroup_kernel(const float4* __restrict__ xs,
                                                                   const int4* __restrict__ blk,
                                                                   const SymInst* __restrict__ sinst,
                                                                   const BatchInst* __restrict__ insts,
                                                                   float4* __restrict__ near_part,
                                                                   const float* __restrict__ umass)
{
    constexpr int kWaves = kBlock / 64;
    __shared__ float lds[own_lds_floats(NI, kWaves)];
    const int4 bl = blk[xcd_block((int)blockIdx.x, (int)gridDim.x)];  // XCD-contiguous (xcd_block)
    const SymInst S = sinst[bl.x];
    const int g0 = S.off + (bl.y - S.off) / kGroup * kGroup;
    const int g1 = min(S.off + S.n, g0 + kGroup);
    const int len = ((g1 - g0 + kWaves - 1) / kWaves + 7) / 8 * 8;  // even shares: small groups keep all wavefronts busy
    ingroup_block<NI, SOFT>(xs, bl.y, g0, g1, len, insts[bl.x].H2, umass + 2 * bl.x, lds,
                            [&](int t, const CSum& x, const CSum& y, const CSum& z) { store_near(near_part, t, x, y, z); });
}

// one piece of a far row of an instance of the batch: group R.g against
// R.units partner groups from j0 on
template <bool UM, bool SOFT>
__device__ __forceinline__ void batch_far_row(const float4* __restrict__ xk, const int n, const SymRow R, const int j0,
                                              float* lsum, float4* frag, const bool plain, float* __restrict__ bk,
                                              const float H2, const float m, const int lane)
{
    FarOwn o;
    far_load_row(xk, n, R.g, lane, lsum, frag, plain, o);
    far_range<UM, SOFT, false>(xk, n, R.g, kGroup * j0, kGroup * (j0 + R.units), kBatchFold, o, bk, 0, H2, m, m, lane);
    far_flush_own(o, lane);
}

// Persistent far field over the batch's rows: a wavefront's first is its own
// number, the next come from the counter; it leaves past nrows.  (With the
// first from the counter too, where few rows end up was a race: 384 of them
// 545 or 580 us.)  plain: no piece has more than kFoldsPerFlush units.
template <bool SOFT>
__global__ __launch_bounds__(kFarThreads, 2) void sym_batch_far_kernel(
    const float4* __restrict__ xs, const SymInst* __restrict__ sinst, const BatchInst* __restrict__ insts,
    const SymRow* __restrict__ rows, const int nrows, const int most, int* __restrict__ queue,
    float4* __restrict__ apart, const int plain, float* __restrict__ bpart, const float* __restrict__ umass)
{
    __shared__ float lsum[3 * kGroup];
    const int lane = threadIdx.x;
    const int waves = gridDim.x;
    int r = blockIdx.x;
    while (r < nrows) {
        const SymRow R = rows[r];
        const SymInst S = sinst[R.inst];
        const float H2 = insts[R.inst].H2;
        const float4* xk = xs + S.off;
        float* const bk = bpart + S.bpart0;
        const bool um = umass[2 * R.inst] != 0.0f;
        const float m = umass[2 * R.inst + 1];
        const int j0 = R.g + 1 + (int)batch_piece_begin(row_units(R.g, S.nsb), R.piece, most);
        float4* const frag = apart + (size_t)kFragElems * ((size_t)most * (S.row0 + R.g) + R.piece);
        if (um)
            batch_far_row<true, SOFT>(xk, S.n, R, j0, lsum, frag, plain, bk, H2, m, lane);
        else
            batch_far_row<false, SOFT>(xk, S.n, R, j0, lsum, frag, plain, bk, H2, 1.0f, lane);
        if (waves >= nrows) break;
        r = 0;
        if (lane == 0) r = atomicAdd(queue, 1);
        r = __builtin_amdgcn_readfirstlane(r) + waves;
    }
}

// Per slot of the instances in the sweep (256-slot block table), as
// sym_combine_kernel: near partial, the row's pieces' own-side fragments, the
// partner-side partials (group order, negated).
template <bool PLAIN>
__global__ __launch_bounds__(kBlock) void sym_batch_combine_kernel(
    const float4* __restrict__ near_part, const float4* __restrict__ apart, const float* __restrict__ bpart,
    const SymInst* __restrict__ sinst, const int4* __restrict__ blk, const int most, const int* __restrict__ perm,
    float4* __restrict__ acc, const int add_acc)
{
    const int4 bl = blk[blockIdx.x];
    const int t = bl.y + threadIdx.x;
    if (t >= bl.z) return;
    const int k = bl.x;
    const SymInst S = sinst[k];
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
    const float4 a = near_part[2 * (size_t)t], c = near_part[2 * (size_t)t + 1];
    x.add(a.x); y.add(a.y); z.add(a.z);
    x.c += c.x; y.c += c.y; z.c += c.z;
    const int local = t - S.off;
    const int g = local / kGroup, lg = local - g * kGroup;
    if (g < S.nrows) {
        const int pieces = batch_row_pieces(row_units(g, S.nsb), most);
        for (int h = 0; h < pieces; ++h) {
            const float4* fr = apart + (size_t)kFragElems * ((size_t)most * (S.row0 + g) + h) + frag_elem(lg);
            const float4 f = fr[0];
            x.add(f.x); y.add(f.y); z.add(f.z);
            if (!PLAIN) {
                const float4 fc = fr[64];
                x.c += fc.x; y.c += fc.y; z.c += fc.z;
            }
        }
    }
    const float* bk = bpart + S.bpart0;
    const int64_t base = bpart_group_base(g) + lg;
    int gp = 0;  // eight groups' loads in flight before their (ordered) adds
    for (; gp + 8 <= g; gp += 8) {
        float v[8][3];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t e = 3 * (size_t)(base + (int64_t)(gp + u) * kGroup);
            v[u][0] = bk[e]; v[u][1] = bk[e + 1]; v[u][2] = bk[e + 2];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            x.add(-v[u][0]); y.add(-v[u][1]); z.add(-v[u][2]);
        }
    }
    for (; gp < g; ++gp) {
        const size_t e = 3 * (size_t)(base + (int64_t)gp * kGroup);
        x.add(-bk[e]); y.add(-bk[e + 1]); z.add(-bk[e + 2]);
    }
    const int i = perm ? perm[t] : t;
    if (add_acc) {  // the SPH terms (and environment), summed before the far field was done
        const float4 a = acc[i];
        x.add(a.x); y.add(a.y); z.add(a.z);
    }
    acc[i] = make_float4(x.value(), y.value(), z.value(), 0.0f);
}

}  // namespace

int sym_default_workgroups(int cus)
{
    return std::max(1, 8 * cus / kGroupSB);  // 2 wavefronts per SIMD
}

// the most folds a workgroup makes in one row of `units` units cut among wgs
// workgroups (far_range: one for every `fold` partners)
static int64_t far_folds(int64_t units, int wgs, int split, int fold)
{
    return ((units + wgs - 1) / wgs * (kSB / split) + fold - 1) / fold;
}

// one column batch's units, far workgroups (of `wanted`) and fragment kind
SymCol sym_column(int split, int fold, int wanted, int c0, int c1)
{
    SymCol C;
    C.c0 = c0;
    C.c1 = c1;
    C.units = col_row_prefix(col_rows(c1), c0, c1, split);
    C.wgs = far_workgroups(wanted, C.units);
    C.plain = fragments_plain(far_folds(C.units, C.wgs, split, fold));
    return C;
}

SymGeom sym_geometry(int64_t n, int wgs, int64_t col_elems)
{
    SymGeom G;
    G.nsb = (n + kSB - 1) / kSB;
    G.groups = (int)((G.nsb + kGroupSB - 1) / kGroupSB);
    G.split = far_split(n, wgs);
    G.units = row_prefix(rows_with_units(G.nsb), G.nsb, G.split);
    G.wgs = far_workgroups(wgs, G.units);
    G.near_elems = 2 * n;
    G.apart_elems = (int64_t)kFragElems * (G.groups + wgs);
    G.plain = fragments_plain(far_folds(G.units, G.wgs, G.split, far_fold(n, wgs)));
    G.bpart_elems = 3 * bpart_group_base(G.groups);
    G.ncols = 1;
    if (G.bpart_elems > col_elems) {
        const std::vector<int> c = sym_columns(G.nsb, col_elems);
        G.ncols = (int)c.size() - 1;
        G.bpart_elems = 0;
        for (int b = 0; b < G.ncols; ++b) G.bpart_elems = std::max(G.bpart_elems, 3 * col_bpart_base(c[b + 1], c[b]));
    }
    return G;
}

// gravity inside the groups
hipError_t launch_sym_ingroup(const SymLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    const int w = L.near_waves;  // a power of two: the shares cover the group exactly
    if (w < 1 || w > kOwnMaxWaves || (w & (w - 1))) return hipErrorInvalidValue;
    const dim3 grid((L.n + 63) / 64), block(64 * w);
    const size_t lds = sizeof(float) * own_lds_floats(1, w);
    if (P.H2 > 0.0f)
        hipLaunchKernelGGL(ingroup_kernel<true>, grid, block, lds, s, L.xs, L.n, L.near_part, P.H2, L.umass);
    else
        hipLaunchKernelGGL(ingroup_kernel<false>, grid, block, lds, s, L.xs, L.n, L.near_part, P.H2, L.umass);
    return hipGetLastError();
}

bool sym_has_far(const SymLaunch& L) { return L.n > 0 && sym_geometry(L.n, L.wgs).units > 0; }

template <bool SOFT>
void launch_far_column(const SymLaunch& L, const SymCol& C, const int split, const DevParams& P, hipStream_t s)
{
    hipLaunchKernelGGL((far_column_kernel<SOFT>), dim3(C.wgs), dim3(kFarThreads), 0, s, L.xs, L.n, C.c0, C.c1,
                       C.units, C.wgs, split, far_fold(L.n, L.wgs), L.apart, C.plain ? 1 : 0, L.bpart, P.H2, L.umass);
}

void launch_column_combine(const SymLaunch& L, const SymCol& C, const int split, const bool first, const bool last,
                           const DevParams& P, hipStream_t s)
{
    hipLaunchKernelGGL(sym_column_combine_kernel, dim3((L.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, L.near_part,
                       L.apart, L.bpart, L.accsum, L.n, C.c0, C.c1, C.units, C.wgs, split, C.plain ? 1 : 0,
                       first ? 1 : 0, last ? 1 : 0, L.perm, L.acc, L.finish ? 1 : 0, L.add_acc ? 1 : 0, L.xvel,
                       L.maxvsig, P);
}

// far field: gravity between groups, once per pair (needs only xs and
// umass); in column batches when the partials of the whole would not fit,
// each batch but the last followed by its column combine
hipError_t launch_sym_far(const SymLaunch& L, const DevParams& P, hipStream_t s)
{
    if (!sym_has_far(L)) return hipSuccess;
    const SymGeom G = sym_geometry(L.n, L.wgs, L.col_elems);
    if (G.ncols == 1) {
        const int far_groups = (L.wgs + kFarMerge - 1) / kFarMerge;
#define GRASPH_FAR(SOFT, WIDE)                                                                                       \
    hipLaunchKernelGGL((far_kernel<SOFT, WIDE>), dim3(far_groups), dim3(64 * kFarMerge), 0, s, L.xs, L.n, G.nsb,     \
                       G.units, L.wgs, G.split, far_fold(L.n, L.wgs), L.apart, G.plain ? 1 : 0, L.bpart, P.H2, L.umass)
        const bool soft = P.H2 > 0.0f, wide = L.n < kSymOneSided;
        if (soft && wide) GRASPH_FAR(true, true);
        else if (soft) GRASPH_FAR(true, false);
        else if (wide) GRASPH_FAR(false, true);
        else GRASPH_FAR(false, false);
#undef GRASPH_FAR
        return hipGetLastError();
    }
    const std::vector<int> c = sym_columns(G.nsb, L.col_elems);
    for (int b = 0; b < G.ncols; ++b) {
        const SymCol C = sym_column(G.split, far_fold(L.n, L.wgs), L.wgs, c[b], c[b + 1]);
        if (P.H2 > 0.0f) launch_far_column<true>(L, C, G.split, P, s); else launch_far_column<false>(L, C, G.split, P, s);
        if (b + 1 < G.ncols) launch_column_combine(L, C, G.split, b == 0, false, P, s);
    }
    return hipGetLastError();
}

// both of the next two in one launch, where that is the faster way
bool sym_fused(const SymLaunch& L)
{
    if (L.n <= 0 || L.near_waves != kNearFused) return false;
    const SymGeom G = sym_geometry(L.n, L.wgs, L.col_elems);
    return G.ncols == 1 && G.plain;
}
hipError_t launch_sym_near_combine(const SymLaunch& L, const DevParams& P, hipStream_t s)
{
    const SymGeom G = sym_geometry(L.n, L.wgs, L.col_elems);
#define GRASPH_FUSED(SOFT)                                                                                            \
    hipLaunchKernelGGL(near_combine_kernel<SOFT>, dim3((L.n + 63) / 64), dim3(64 * kNearFused), 0, s, L.xs, L.apart, \
                       L.bpart, L.n, G.nsb, G.units, L.wgs, G.split, L.umass, L.perm, L.acc, L.finish ? 1 : 0,       \
                       L.add_acc ? 1 : 0, L.xvel, L.maxvsig, P)
    if (P.H2 > 0.0f) GRASPH_FUSED(true); else GRASPH_FUSED(false);
#undef GRASPH_FUSED
    return hipGetLastError();
}

// combine (after both fields): the acceleration
hipError_t launch_sym_combine(const SymLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    const SymGeom G = sym_geometry(L.n, L.wgs, L.col_elems);
    if (G.ncols > 1 && sym_has_far(L)) {
        // the last column batch's combine, which finishes
        const std::vector<int> c = sym_columns(G.nsb, L.col_elems);
        const SymCol C = sym_column(G.split, far_fold(L.n, L.wgs), L.wgs, c[G.ncols - 1], c[G.ncols]);
        launch_column_combine(L, C, G.split, false, true, P, s);
        return hipGetLastError();
    }
    // threads per slot: about 2^17 threads or more in all (below 65536 particles the fused launch takes the
    // combine, unless option sym_near_shares asks for another in-group shape)
    const int parts = L.n >= 98304 ? 1 : L.n >= 49152 ? 2 : L.n >= 24576 ? 4 : 8;
#define GRASPH_COMBINE(PARTS, PLAIN)                                                                                  \
    hipLaunchKernelGGL((sym_combine_kernel<PARTS, PLAIN>), dim3((L.n + kBlock / PARTS - 1) / (kBlock / PARTS)),        \
                       dim3(kBlock), 0, s, L.near_part, L.apart, L.bpart, L.n, G.nsb, G.units, L.wgs,       \
                       G.split, L.perm, L.acc, L.finish ? 1 : 0, L.add_acc ? 1 : 0,        \
                       L.xvel, L.maxvsig, P)
    if (G.plain) {
        switch (parts) {
        case 1: GRASPH_COMBINE(1, true); break;
        case 2: GRASPH_COMBINE(2, true); break;
        case 4: GRASPH_COMBINE(4, true); break;
        default: GRASPH_COMBINE(8, true); break;
        }
    } else {
        GRASPH_COMBINE(1, false);  // more than kFoldsPerFlush units per workgroup: large counts (or few workgroups)
    }
#undef GRASPH_COMBINE
    return hipGetLastError();
}

SymBatchTables sym_batch_tables(const std::vector<int64_t>& offsets, int64_t min_n, int64_t wgs)
{
    SymBatchTables T;
    const int n_inst = (int)offsets.size() - 1;
    const auto pieces = [&](int most) {
        int64_t count = 0;
        for (int k = 0; k < n_inst; ++k) {
            const int64_t n = offsets[k + 1] - offsets[k], nsb = n >= min_n ? (n + kSB - 1) / kSB : 0;
            for (int64_t g = 0; g < rows_with_units(nsb); ++g) count += batch_row_pieces(row_units(g, nsb), most);
        }
        return count;
    };
    while (T.most < kBatchPiecesMost && pieces(T.most) < std::min(wgs, pieces(2 * T.most))) T.most *= 2;
    int row0 = 0;
    int64_t bpart0 = 0;
    for (int k = 0; k < n_inst; ++k) {
        const int64_t n = offsets[k + 1] - offsets[k];
        const bool sym = n >= min_n && n > 0;
        SymInst S;
        S.off = (int)offsets[k];
        S.n = sym ? (int)n : 0;  // instances left to the one-sided sweep: nothing here
        if (sym) {
            append_blocks(T.blk, k, offsets[k], offsets[k + 1], 256);
            append_blocks(T.blk64, k, offsets[k], offsets[k + 1], 64);
        }
        S.nsb = (int)((S.n + kSB - 1) / kSB);
        S.nrows = (int)rows_with_units(S.nsb);
        S.row0 = row0;
        S.bpart0 = bpart0;
        for (int g = 0; g < S.nrows; ++g) {
            const int64_t u = row_units(g, S.nsb);
            for (int h = 0; h < batch_row_pieces(u, T.most); ++h) {
                const int units = (int)(batch_piece_begin(u, h + 1, T.most) - batch_piece_begin(u, h, T.most));
                T.rows.push_back(SymRow{k, g, h, units});
                T.plain = T.plain && fragments_plain((int64_t)units * kGroup / kBatchFold);
            }
        }
        row0 += S.nrows;
        bpart0 += 3 * bpart_group_base((S.nsb + kGroupSB - 1) / kGroupSB);
        T.insts.push_back(S);
    }
    std::stable_sort(T.rows.begin(), T.rows.end(), [](const SymRow& a, const SymRow& b) { return a.units > b.units; });
    T.apart_elems = (int64_t)kFragElems * T.most * row0;
    T.bpart_elems = bpart0;
    return T;
}

// Blocks of 64 slots, one a lane, where those of 256 leave the GPU idle (so many
// workgroups fill it once: 16 x 4096 particles 48 against 34 us, 32 x
// 4096 56 either way, 512 x 1000 165 against 172) or leave an eighth of the lanes
// without a slot (2000 x 50: 20 us with 256, 8 with 64).
constexpr int kNearBlocksMin = 512;
hipError_t launch_sym_batch_ingroup(const SymBatchLaunch& L, hipStream_t s)
{
    if (L.ntotal <= 0 || L.n_blk <= 0) return hipSuccess;
    const bool small = L.n_blk < kNearBlocksMin || 9 * (int64_t)L.n_blk64 < 32 * (int64_t)L.n_blk;
#define GRASPH_NEAR(NI, SOFT, N, BLK)                                                                                \
    hipLaunchKernelGGL((sym_batch_ingroup_kernel<NI, SOFT>), dim3(N), dim3(kBlock), 0, s, L.xs, BLK, L.sinst, L.insts, \
                       L.near_part, L.umass)
    if (small && L.soft) GRASPH_NEAR(1, true, L.n_blk64, L.blk64);
    else if (small) GRASPH_NEAR(1, false, L.n_blk64, L.blk64);
    else if (L.soft) GRASPH_NEAR(4, true, L.n_blk, L.blk);
    else GRASPH_NEAR(4, false, L.n_blk, L.blk);
#undef GRASPH_NEAR
    return hipGetLastError();
}

hipError_t launch_sym_batch_far(const SymBatchLaunch& L, hipStream_t s)
{
    if (!sym_batch_has_far(L)) return hipSuccess;
    hipError_t e;
    if ((e = launch_reset_queue(L.queue, 1, s)) != hipSuccess) return e;
    if (L.soft)
        hipLaunchKernelGGL((sym_batch_far_kernel<true>), dim3(L.wgs), dim3(kFarThreads), 0, s, L.xs, L.sinst, L.insts,
                           L.rows, L.nrows, L.most, L.queue, L.apart, L.plain ? 1 : 0, L.bpart, L.umass);
    else
        hipLaunchKernelGGL((sym_batch_far_kernel<false>), dim3(L.wgs), dim3(kFarThreads), 0, s, L.xs, L.sinst, L.insts,
                           L.rows, L.nrows, L.most, L.queue, L.apart, L.plain ? 1 : 0, L.bpart, L.umass);
    return hipGetLastError();
}

hipError_t launch_sym_batch_combine(const SymBatchLaunch& L, hipStream_t s)
{
    if (L.ntotal <= 0 || L.n_blk <= 0) return hipSuccess;
    if (L.plain)
        hipLaunchKernelGGL(sym_batch_combine_kernel<true>, dim3(L.n_blk), dim3(kBlock), 0, s, L.near_part, L.apart,
                           L.bpart, L.sinst, L.blk, L.most, L.perm, L.acc, L.add_acc ? 1 : 0);
    else
        hipLaunchKernelGGL(sym_batch_combine_kernel<false>, dim3(L.n_blk), dim3(kBlock), 0, s, L.near_part, L.apart,
                           L.bpart, L.sinst, L.blk, L.most, L.perm, L.acc, L.add_acc ? 1 : 0);
    return hipGetLastError();
}

}  // namespace grasph
