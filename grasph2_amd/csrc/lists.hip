// lists.hip -- the neighbour lists (0 < r^2 <= H^2, src/computeDerivatives.h
// :72,122,238) that the passes of nbr_passes.hip walk (gfx950).
//
// Boxes: every 8, every 64 and every 512 consecutive slots of an instance have
// a bounding box.  In slot (Hilbert) order these are small, and a box
// farther than H from a particle holds none of its neighbours: the box gaps
// and their squared sum round like the exact pair distance (rounding is
// monotonic), so they never exceed it.
//
// One wavefront makes the lists of 8 slots.  Lane l tests box l of 64 boxes
// of 512 against the 8 slots' own box; the 64 lanes then test the boxes of 64
// in 8 near ones at a time (instances of up to 8192 particles begin here),
// then the boxes of 8 in 8 near ones of these, then the particles of the near
// ones, 64 at a time: those within H of the own box are collected in LDS, in slot order.  Lane
// l = 8 i + j takes slot i against every eighth of them from the j-th on; the
// 64 lanes' hits in one ballot give slot i its partners as a byte in slot
// order, so a partner's place in the list is the count so far plus the bits
// below it: the lists come out in increasing slot order, complete and one to a
// slot, whatever the launch shape.
//
// What bounds it: instructions, about 1000 vector ones per wavefront, and the
// chain of dependent loads from level to level.  8 slots meet ~70 boxes within
// H = 2.5 spacings, 560 particles, for ~65 neighbours each, of which ~250 come
// within H of their box: testing the slots against those instead of all 560
// took N = 200003 from 126 to 92 us, 65536 squeezed ones (430 partners each)
// from 190 to 137, 512 instances from 1.63 to 1.15 ms.  The boxes of 64 save
// most of the tests of boxes of 8 (12 to 16 boxes of 512 are near, with 64 of
// 8 each), and with lists short enough for 8 wavefronts per SIMD took SPH
// steps without gravity at 200003 particles from 283 to 275 us, default solids
// at 16384 from 103 to 99, three single passes at 20011 from 221 to 212.  A
// wavefront's stores fill lines of its own (list_entry): where lists are long they
// decide (internal.hpp).
#include "internal.hpp"

namespace grasph {
namespace {

constexpr int kBoxThreads = kBoxCoarse;  // slots of a coarse box: one workgroup
constexpr int kTile = 32;                // slots per workgroup of the list kernel
constexpr int kListThreads = 8 * kTile;
constexpr int kBoxList = 256;            // near fine boxes a wavefront collects before it tests them
constexpr int kMidList = 128;            // near mid boxes it collects before it tests their fine ones
// instances of so many mid boxes test them without the coarse ones (allocation-free steps of 8192 particles 81.4 us
// with the coarse ones, 81.1 without; a two-round test costs what the coarse round and its chain do)
constexpr int kMidDirect = 128;
constexpr int kAhead = 2;                // loads of 8 boxes' partners in flight
constexpr int kPartners = 192;           // close partners a wavefront collects before it tests them

#define GRASPH_INLINE __attribute__((always_inline))
typedef float vec4 __attribute__((ext_vector_type(4)));

// Orders the wavefront's LDS accesses around it (the hardware executes one
// wavefront's in order; the compiler must not move them).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// whether two boxes come within H of each other
__device__ __forceinline__ bool boxes_near(const float4 lo, const float4 hi, const float4 l2, const float4 h2,
                                           const float H2)
{
    const float gx = fmaxf(0.0f, fmaxf(l2.x - hi.x, lo.x - h2.x));
    const float gy = fmaxf(0.0f, fmaxf(l2.y - hi.y, lo.y - h2.y));
    const float gz = fmaxf(0.0f, fmaxf(l2.z - hi.z, lo.z - h2.z));
    return dist2_exact(gx, gy, gz) <= H2;
}

__device__ __forceinline__ float lane_value(const float v, const int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// boxes of a batch: block b of the 256-slot block table makes the coarse box
// its instance-relative slots begin, if they begin one
__global__ __launch_bounds__(kBoxThreads) void batch_box_kernel(const float4* __restrict__ xs,
                                                                const int4* __restrict__ blk,
                                                                const BatchInst* __restrict__ insts,
                                                                float4* __restrict__ fine, float4* __restrict__ mid,
                                                                float4* __restrict__ coarse)
{
    const int4 bl = blk[blockIdx.x];
    const BatchInst I = insts[bl.x];
    const int first = bl.y - I.off;
    if (first % kBoxCoarse) return;  // the whole workgroup leaves
    const int t = first + (int)threadIdx.x;
    const bool act = t < I.n;
    const float4 p = act ? xs[I.off + t] : make_float4(0.f, 0.f, 0.f, 0.f);
    block_boxes(p, act, first, I.n, fine + 2 * (size_t)I.fine0, mid + 2 * (size_t)(kBoxCoarse / kBoxMid) * I.coarse0,
                coarse + 2 * (size_t)I.coarse0);
}

template <bool BATCH>
__global__ __launch_bounds__(kListThreads) void list_kernel(const float4* __restrict__ xs, const int n0,
                                                            const float4* __restrict__ fine0,
                                                            const float4* __restrict__ coarse0,
                                                            const float4* __restrict__ mid0,
                                                            int* __restrict__ nbr, int* __restrict__ nbr_cnt,
                                                            const int kmax, const float h2,
                                                            const int4* __restrict__ blk,
                                                            const BatchInst* __restrict__ insts,
                                                            int* __restrict__ max_dev, int* __restrict__ max_host)
{
    // one wavefront's rows are its own: no barrier
    __shared__ int boxes[kTile / kBoxFine][kBoxList];
    __shared__ int mids[kTile / kBoxFine][kMidList];
    __shared__ int coarses[kTile / kBoxFine][64];
    __shared__ vec4 partners[kTile / kBoxFine][kPartners];
    // XCD-contiguous (xcd_block): neighbouring tiles read the same partners
    const int tile = xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    int off = 0, n = n0, first;  // the instance's slots [off, off + n); this wavefront's 8, instance-relative
    float H2 = h2;
    const float4 *fine = fine0, *coarse = coarse0, *mid = mid0;
    if (BATCH) {
        const int4 bl = blk[tile];
        const BatchInst I = insts[bl.x];
        off = I.off;
        n = I.n;
        H2 = I.H2;
        fine += 2 * (size_t)I.fine0;
        coarse += 2 * (size_t)I.coarse0;
        mid += 2 * (size_t)(kBoxCoarse / kBoxMid) * I.coarse0;
        first = bl.y - off + kBoxFine * wave;
    } else {
        first = kTile * tile + kBoxFine * wave;
    }
    if (first >= n) return;  // whole wavefronts leave
    int* const box = boxes[wave];
    const int i = lane >> 3, j = lane & 7;
    const int t = first + i;
    float xi = __int_as_float(0x7fc00000), yi = xi, zi = xi;  // NaN: a slot past the end hits nothing
    if (t < n) {
        const float4 p = xs[off + t];
        xi = p.x; yi = p.y; zi = p.z;
    }
    const int nf = (n + kBoxFine - 1) / kBoxFine, nm = (n + kBoxMid - 1) / kBoxMid, nc = (n + kBoxCoarse - 1) / kBoxCoarse;
    float4 lo = fine[2 * (first / kBoxFine)], hi = fine[2 * (first / kBoxFine) + 1];
    // Eight slots that span a jump of the slot order (where the curve leaves
    // the particles and comes back) have a box that says little.  Where it is
    // wider than H^2's reach both ways, it is cut in two at the longest step
    // between its slots, and if a part still is, boxes are tested against the
    // slots one by one.  (With the wide box one such wavefront tested every
    // particle: N = 200003, 1736 us instead of 207; with all of them slot by
    // slot those wavefronts were the last by far: liquid of 8192, 20.8 us
    // instead of 14.9.)
    const auto wide = [&](const float4 l, const float4 h) {
        const float w = fmaxf(h.x - l.x, fmaxf(h.y - l.y, h.z - l.z));
        return (bool)__builtin_amdgcn_readfirstlane(w * w > 4.0f * H2);
    };
    const int own = min(kBoxFine, n - first);
    const auto slot = [&](const int q) {
        return make_float4(lane_value(xi, 8 * q), lane_value(yi, 8 * q), lane_value(zi, 8 * q), 0.0f);
    };
    const bool jump = wide(lo, hi);
    bool each = false;
    float4 lo2 = lo, hi2 = hi;  // the second part's box
    if (jump) {
        int cut = 1;
        float longest = -1.0f;
        for (int q = 1; q < own; ++q) {
            const float4 p = slot(q), o = slot(q - 1);
            const float d = dist2_exact(p.x - o.x, p.y - o.y, p.z - o.z);
            if (d > longest) {
                longest = d;
                cut = q;
            }
        }
        lo = hi = slot(0);
        lo2 = hi2 = slot(own - 1);
        for (int q = 0; q < own; ++q) {
            const float4 p = slot(q);
            float4 &l = q < cut ? lo : lo2, &h = q < cut ? hi : hi2;
            l.x = fminf(l.x, p.x); l.y = fminf(l.y, p.y); l.z = fminf(l.z, p.z);
            h.x = fmaxf(h.x, p.x); h.y = fmaxf(h.y, p.y); h.z = fmaxf(h.z, p.z);
        }
        each = wide(lo, hi) || wide(lo2, hi2);
    }
    auto near = [&](const float4 l2, const float4 h2) -> bool {
        if (!each) {
            bool any = boxes_near(lo, hi, l2, h2, H2);
            if (jump) any = any || boxes_near(lo2, hi2, l2, h2, H2);
            return any;
        }
        bool any = false;
        for (int q = 0; q < own; ++q) {
            const float4 p = slot(q);
            any = any || boxes_near(p, p, l2, h2, H2);
        }
        return any;
    };
    // entry k of this lane's slot, in bytes from the wavefront's first tile of
    // the lists (which its 8 slots may leave, in a batch)
    char* const lists = reinterpret_cast<char*>(nbr + list_entry((off + first) & ~63, 0, kmax));
    const uint32_t column = 4u * (uint32_t)(((off + t) >> 6 != (off + first) >> 6 ? kmax * 64 : 0) + ((off + t) & 63) * list_chunk(kmax));
    const uint32_t mask = list_mask(kmax);
    const uint32_t bit = 1u << j, below = bit - 1u;
    const int shift = 8 * (i & 3);
    const float4* const xj = xs + off;
    vec4* const part = partners[wave];
    int cnt = 0, np = 0;  // partners found for this lane's slot; partners collected
    // The pairs of this wavefront's slots with the partners collected.
    auto test_partners = [&]() {
        if (lane < 8) part[np + lane] = __int_as_float(0x7fc00000);  // NaN hits nothing
        wave_lds_order();
        for (int b = 0; b < np; b += 8) {
            const vec4 q = part[b + j];
            const bool hit = is_neighbour(dist2_exact(xi - q.x, yi - q.y, zi - q.z), H2);
            const uint64_t hits = __builtin_amdgcn_ballot_w64(hit);
            const uint32_t half = lane < 32 ? (uint32_t)hits : (uint32_t)(hits >> 32);
            const uint32_t mine = (half >> shift) & 0xffu;
            const int k = cnt + __builtin_popcount(mine & below);
            if (hit && k < kmax) *reinterpret_cast<int*>(lists + (column + 4u * list_offset((uint32_t)k, mask))) = __float_as_int(q.w);
            cnt += __builtin_popcount(mine);
        }
        wave_lds_order();
        np = 0;
    };
    // The particles collected: the `close` lanes' of p, slots a of the instance.
    const auto collect = [&](vec4 p, const int a, const bool close) GRASPH_INLINE {
        const uint64_t all = __builtin_amdgcn_ballot_w64(close);
        p.w = __int_as_float(off + a);
        if (close)
            part[np + __builtin_amdgcn_mbcnt_hi((uint32_t)(all >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)all, 0))] = p;
        np += __builtin_popcountll(all);
        if (np > kPartners - 72) test_partners();
    };
    // The partners in the m boxes of box[] within H of this wavefront's own
    // box, collected: 8 boxes at a time, kAhead times as many on their way.
    auto test_boxes = [&](const int m) {
        if (m == 0) return;  // box[m - 1] is read
        wave_lds_order();
        int at[kAhead];
        vec4 q[kAhead];
        const auto fetch = [&](const int b, int& a, vec4& v) GRASPH_INLINE {
            const int u = b + i;
            a = u < m ? kBoxFine * box[min(u, m - 1)] + j : n;
            v = *reinterpret_cast<const vec4*>(xj + min(a, n - 1));
        };
#pragma unroll
        for (int u = 0; u < kAhead; ++u) fetch(8 * u, at[u], q[u]);
        for (int b0 = 0; b0 < m; b0 += 8 * kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int a = at[u];
                const vec4 p = q[u];
                fetch(b0 + 8 * (u + kAhead), at[u], q[u]);
                const float4 at4 = make_float4(p.x, p.y, p.z, 0.0f);
                bool close = boxes_near(lo, hi, at4, at4, H2);
                if (jump) close = close || boxes_near(lo2, hi2, at4, at4, H2);
                close = close && a < n;
                collect(p, a, close);
            }
        }
    };
    int* const mbox = mids[wave];
    int* const cbox = coarses[wave];
    const uint64_t lower = (1ull << lane) - 1ull;
    int m = 0, mm = 0;  // fine boxes, mid boxes collected
    // The fine boxes of the mid boxes collected, 16 mid boxes at a time, their
    // loads in flight together.
    auto test_mids = [&]() {
        wave_lds_order();
        // The wavefront's slots lie apart and most boxes in a row are near: the
        // slot order keeps nothing together here (option reorder_interval 0, or
        // bodies small beside the distance of a stray particle, on which the
        // curve's cells depend).  Every particle of the boxes is then tested
        // against the 8 slots, 64 particles a load.  60000 particles in random
        // order 2244 -> 1280 us a derivative call, one of them 3000 radii away
        // 1912 -> 1230 (all-pairs lists beside the gravity took 1458 and 1508).
        if (each && mm > kMidList / 4 && mbox[mm - 1] - mbox[0] < 2 * mm) {
            test_boxes(m);
            m = 0;
            // the slots as registers of the loop (the compiler read their lanes anew for
            // every 64 particles: list kernel 1237 us, 673 now), a third of them vector
            // ones: all would leave 6 wavefronts a SIMD instead of 8
            float sx[kBoxFine], sy[kBoxFine], sz[kBoxFine];
#pragma unroll
            for (int q = 0; q < kBoxFine; ++q) {
                const float4 o = slot(q);  // NaN past the end: nothing is close
                sx[q] = o.x; sy[q] = o.y; sz[q] = o.z;
                __asm__ volatile("" : "+v"(sx[q]), "+s"(sy[q]), "+s"(sz[q]));
            }
            const float limit = fmaf(H2, 1.0f + 1.0f / (1 << 20), 1e-37f);  // within H, as the pairs round it
            const auto first_of = [&](const int b) GRASPH_INLINE {
                return kBoxMid * __builtin_amdgcn_readfirstlane(mbox[min(b, mm - 1)]);
            };
            const auto load = [&](const int a) GRASPH_INLINE {
                return *reinterpret_cast<const vec4*>(xj + a + (uint32_t)min(lane, n - 1 - a));
            };
            int ahead = first_of(0);
            vec4 next = load(ahead);
            for (int b = 0; b < mm; ++b) {
                const int a = ahead;
                const vec4 p = next;
                ahead = first_of(b + 1);
                next = load(ahead);
                float d = INFINITY;
#pragma unroll
                for (int q = 0; q < kBoxFine; ++q) {
                    const float dx = p.x - sx[q], dy = p.y - sy[q], dz = p.z - sz[q];
                    d = fminf(d, fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
                }
                const bool close = d <= limit && lane < n - a;
                if (__builtin_amdgcn_ballot_w64(close)) collect(p, a + lane, close);
            }
            wave_lds_order();
            mm = 0;
            return;
        }
        for (int b = 0; b < mm; b += 16) {
            const int ua = b + i, ub = ua + 8;
            const int fa = kBoxMid / kBoxFine * mbox[min(ua, mm - 1)] + j, fb = kBoxMid / kBoxFine * mbox[min(ub, mm - 1)] + j;
            const int ca = min(fa, nf - 1), cb = min(fb, nf - 1);
            const float4 la = fine[2 * ca], ha = fine[2 * ca + 1], lb = fine[2 * cb], hb = fine[2 * cb + 1];
            const uint64_t ma = __builtin_amdgcn_ballot_w64(ua < mm && fa < nf && near(la, ha));
            const uint64_t mb = __builtin_amdgcn_ballot_w64(ub < mm && fb < nf && near(lb, hb));
            if ((ma >> lane) & 1) box[m + __builtin_popcountll(ma & lower)] = fa;
            m += __builtin_popcountll(ma);
            if ((mb >> lane) & 1) box[m + __builtin_popcountll(mb & lower)] = fb;
            m += __builtin_popcountll(mb);
            if (m > kBoxList - 128) {
                test_boxes(m);
                m = 0;
            }
        }
        wave_lds_order();
        mm = 0;
    };
    if (nm <= kMidDirect) {
        for (int b = 0; b < nm; b += 64) {
            const int q = b + lane, cq = min(q, nm - 1);
            const uint64_t ms = __builtin_amdgcn_ballot_w64(q < nm && near(mid[2 * cq], mid[2 * cq + 1]));
            if ((ms >> lane) & 1) mbox[mm + __builtin_popcountll(ms & lower)] = q;
            mm += __builtin_popcountll(ms);
            if (mm > kMidList - 64) test_mids();
        }
    }
    for (int c0 = nm <= kMidDirect ? nc : 0; c0 < nc; c0 += 64) {
        const int c = min(c0 + lane, nc - 1);
        const uint64_t mc = __builtin_amdgcn_ballot_w64(c0 + lane < nc && near(coarse[2 * c], coarse[2 * c + 1]));
        const int cc = __builtin_popcountll(mc);  // near coarse boxes: their mid boxes, 8 coarse ones at a time
        if ((mc >> lane) & 1) cbox[__builtin_popcountll(mc & lower)] = c;
        wave_lds_order();
        for (int b = 0; b < cc; b += 8) {
            const int u = b + i, q = kBoxCoarse / kBoxMid * cbox[min(u, cc - 1)] + j, cq = min(q, nm - 1);
            const float4 l2 = mid[2 * cq], h2 = mid[2 * cq + 1];
            const uint64_t ms = __builtin_amdgcn_ballot_w64(u < cc && q < nm && near(l2, h2));
            if ((ms >> lane) & 1) mbox[mm + __builtin_popcountll(ms & lower)] = q;
            mm += __builtin_popcountll(ms);
            if (mm > kMidList - 64) test_mids();
        }
        wave_lds_order();
    }
    test_mids();
    test_boxes(m);
    test_partners();
    if (j == 0 && t < n) nbr_cnt[off + t] = cnt;
    // a list that overflowed reports the largest count: to the device's
    // maximum of this evaluation, and to the host's when it raises that one
    // (two wavefronts' host stores may land in either order: the host then
    // sees the smaller, and the next evaluation's overflow corrects it)
    if (max_host && __builtin_amdgcn_ballot_w64(t < n && cnt > kmax)) {
        int m = t < n ? cnt : 0;
        for (int o = 32; o >= 8; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
        if (lane == 0 && atomicMax(max_dev, m) < m)
            __hip_atomic_store(max_host, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace

hipError_t launch_lists(const ListLaunch& L, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(list_kernel<false>, dim3((L.n + kTile - 1) / kTile), dim3(kListThreads), 0, s, L.xs, L.n,
                       L.fine, L.coarse, L.mid, L.nbr, L.nbr_cnt, L.kmax, L.H2, nullptr, nullptr, L.max_dev, L.max_host);
    return hipGetLastError();
}

hipError_t launch_batch_lists(const ListLaunch& L, hipStream_t s)
{
    if (L.n <= 0 || L.n_blk <= 0 || L.n_blk32 <= 0) return hipSuccess;
    static_assert(kTile == 32, "the batch's blocks of the list kernel");
    hipLaunchKernelGGL(batch_box_kernel, dim3(L.n_blk), dim3(kBoxThreads), 0, s, L.xs, L.blk, L.insts, L.fine,
                       L.mid, L.coarse);
    hipLaunchKernelGGL(list_kernel<true>, dim3(L.n_blk32), dim3(kListThreads), 0, s, L.xs, 0, L.fine, L.coarse,
                       L.mid, L.nbr, L.nbr_cnt, L.kmax, 0.0f, L.blk32, L.insts, nullptr, nullptr);
    return hipGetLastError();
}

}  // namespace grasph
