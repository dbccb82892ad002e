// own_block.hpp -- one-sided gravity of a workgroup's own slots: up to 16
// wavefronts take the same NI * 64 slots (NI per lane) against a share of the
// partners each, and add their sums in LDS.  Used by the one-sided sweep
// (sweep.hip) and for the pairs inside a group (sym_sweep.hip).
//
// What bounds it is the FP32 vector issue, with the two rates that
// far_rotation.hpp describes: the partners have to be in vector registers
// (with a scalar operand each difference took 4 clocks instead of 2, and the
// pair 46), three reads must not meet in one half of the register file, and
// the v_rsq_f32 have to come in runs.  A wavefront copies 64 partners at a
// time into LDS and reads them back one by one, the same for every lane; 8
// pairs at a time go through one asm block.  Every slot meets the partners in
// their order whatever NI is, so with the same shares NI does not change a bit of
// the result (own_plan chooses other shares for another NI, though).
// Measured: Plummer steps of 1000 particles 59 -> 11 us (28 with one share
// per slot block, 14 with the equal-mass check), of 8192 ~100 -> 31; pairs
// inside the groups of the 512-instance ensemble 1.34 -> 1.10 ms.
#pragma once

#include "far_rotation.hpp"
#include "internal.hpp"

namespace grasph {
namespace {

// partners per plain partial sum before the compensated add (error against FP64
// of the norm with 128 and 64, unequal masses: 8000 particles 1.13e-7, 8.64e-8; pairs
// inside a group at 16384 4.44e-8, 4.37e-8 of all; for 0.5% of the step)
constexpr int kFold = 64;
constexpr int kOwnPairs = 8;      // pairs per asm block
constexpr int kOwnMaxWaves = 16;  // wavefronts sharing their own slots

template <int NI>
struct OwnAcc {
    float x[NI], y[NI], z[NI];     // the lane's own slots
    float ax[NI], ay[NI], az[NI];  // plain sums since the last fold
};

// pair of slot q and partner r, the register of its r^2 + H^2, then 1/r and
// 1/r^3 (even), of dx, dy, dz (odd) and of 1/r^2 (even); v96 holds H^2
#define GRASPH_OWN_PAIRS1(F) \
    F(0, 0, 64, 65, 67, 69, 98) F(0, 1, 66, 71, 73, 75, 100) F(0, 2, 68, 77, 79, 81, 102) F(0, 3, 70, 83, 85, 87, 104) \
    F(0, 4, 72, 89, 91, 93, 106) F(0, 5, 74, 95, 97, 99, 108) F(0, 6, 76, 101, 103, 105, 110) F(0, 7, 78, 107, 109, 111, 112)
#define GRASPH_OWN_PAIRS2(F) \
    F(0, 0, 64, 65, 67, 69, 98) F(1, 0, 66, 71, 73, 75, 100) F(0, 1, 68, 77, 79, 81, 102) F(1, 1, 70, 83, 85, 87, 104) \
    F(0, 2, 72, 89, 91, 93, 106) F(1, 2, 74, 95, 97, 99, 108) F(0, 3, 76, 101, 103, 105, 110) F(1, 3, 78, 107, 109, 111, 112)
#define GRASPH_OWN_PAIRS4(F) \
    F(0, 0, 64, 65, 67, 69, 98) F(1, 0, 66, 71, 73, 75, 100) F(2, 0, 68, 77, 79, 81, 102) F(3, 0, 70, 83, 85, 87, 104) \
    F(0, 1, 72, 89, 91, 93, 106) F(1, 1, 74, 95, 97, 99, 108) F(2, 1, 76, 101, 103, 105, 110) F(3, 1, 78, 107, 109, 111, 112)
#define GRASPH_OWN_CLOBBERS \
    "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", \
    "v79", "v81", "v83", "v85", "v87", "v89", "v91", "v93", "v95", "v96", "v97", "v98", "v99", "v100", "v101", \
    "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112"
#define GRASPH_OWN_SUB(q, r, d, x, y, z, t)                                                                        \
    "v_sub_f32 v" #x ", %[jx" #r "], %[x" #q "]\n v_sub_f32 v" #y ", %[jy" #r "], %[y" #q "]\n"                      \
    "v_sub_f32 v" #z ", %[jz" #r "], %[z" #q "]\n"
#define GRASPH_OWN_R2X(q, r, d, x, y, z, t) GRASPH_FAR_R2X(q, d, x, y, z, t)
#define GRASPH_OWN_R2Y(q, r, d, x, y, z, t) GRASPH_FAR_R2Y(q, d, x, y, z, t)
#define GRASPH_OWN_R2Z(q, r, d, x, y, z, t) GRASPH_FAR_R2Z(q, d, x, y, z, t)
#define GRASPH_OWN_RSQ(q, r, d, x, y, z, t) GRASPH_FAR_RSQ(q, d, x, y, z, t)
#define GRASPH_OWN_INV2(q, r, d, x, y, z, t) GRASPH_FAR_INV2(q, d, x, y, z, t)
#define GRASPH_OWN_INV3(q, r, d, x, y, z, t) GRASPH_FAR_INV3(q, d, x, y, z, t)
// the mass joins 1/r: m / r is in range where 1 / r^3 alone is not (r past 10^13 or
// below 10^-13, with masses to match)
#define GRASPH_OWN_MASS(q, r, d, x, y, z, t) "v_mul_f32 v" #d ", %[jm" #r "], v" #d "\n"
#define GRASPH_OWN_SUMS(q, r, d, x, y, z, t)                                                                       \
    "v_fmac_f32 %[ax" #q "], v" #x ", v" #d "\n v_fmac_f32 %[ay" #q "], v" #y ", v" #d "\n"                         \
    "v_fmac_f32 %[az" #q "], v" #z ", v" #d "\n"
#define GRASPH_OWN_SLOT(q) [x##q] "v"(a.x[q]), [y##q] "v"(a.y[q]), [z##q] "v"(a.z[q])
#define GRASPH_OWN_SUM(q) [ax##q] "+&v"(a.ax[q]), [ay##q] "+&v"(a.ay[q]), [az##q] "+&v"(a.az[q])
#define GRASPH_OWN_PARTNER(r) [jx##r] "v"(p[r].x), [jy##r] "v"(p[r].y), [jz##r] "v"(p[r].z)
#define GRASPH_OWN_PMASS(r) [jm##r] "v"(p[r].w)
#define GRASPH_OWN_BODY(PAIRS, MASS)                                                                               \
    "v_mov_b32 v96, %[h2]\n" PAIRS(GRASPH_OWN_SUB) PAIRS(GRASPH_OWN_R2X) PAIRS(GRASPH_OWN_R2Y)                      \
    PAIRS(GRASPH_OWN_R2Z) "s_setprio 1\n" PAIRS(GRASPH_OWN_RSQ) "s_setprio 0\n s_nop 0\n"                          \
    PAIRS(GRASPH_OWN_INV2) MASS PAIRS(GRASPH_OWN_INV3) PAIRS(GRASPH_OWN_SUMS)
#define GRASPH_OWN_ASM(PAIRS, SUMS, SLOTS, PARTNERS, MASSES)                                                       \
    if constexpr (UM)                                                                                              \
        asm volatile(GRASPH_OWN_BODY(PAIRS, "") : SUMS : [h2] "v"(h2), SLOTS, PARTNERS : GRASPH_OWN_CLOBBERS);     \
    else                                                                                                           \
        asm volatile(GRASPH_OWN_BODY(PAIRS, PAIRS(GRASPH_OWN_MASS))                                                \
                     : SUMS                                                                                        \
                     : [h2] "v"(h2), SLOTS, PARTNERS, MASSES                                                       \
                     : GRASPH_OWN_CLOBBERS)
#define GRASPH_OWN_LIST2(M) M(0), M(1)
#define GRASPH_OWN_LIST4(M) GRASPH_OWN_LIST2(M), M(2), M(3)
#define GRASPH_OWN_LIST8(M) GRASPH_OWN_LIST4(M), M(4), M(5), M(6), M(7)

// kOwnPairs / NI partners against the lane's NI slots
template <int NI, bool UM, bool SOFT>
__device__ __forceinline__ void own_pairs(const float4 (&p)[kOwnPairs / NI], OwnAcc<NI>& a, const float h2)
{
    if constexpr (!SOFT) {  // coincident particles exert nothing (computeDerivatives.h:226)
#pragma unroll
        for (int r = 0; r < kOwnPairs / NI; ++r)
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                const float dx = p[r].x - a.x[q], dy = p[r].y - a.y[q], dz = p[r].z - a.z[q];
                const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                const float inv = __builtin_amdgcn_rsqf(d2);
                const float s = (d2 > 0.0f) ? (UM ? inv : p[r].w * inv) * (inv * inv) : 0.0f;
                a.ax[q] = fmaf(dx, s, a.ax[q]); a.ay[q] = fmaf(dy, s, a.ay[q]); a.az[q] = fmaf(dz, s, a.az[q]);
            }
    } else if constexpr (NI == 1) {
        GRASPH_OWN_ASM(GRASPH_OWN_PAIRS1, GRASPH_OWN_SUM(0), GRASPH_OWN_SLOT(0), GRASPH_OWN_LIST8(GRASPH_OWN_PARTNER),
                       GRASPH_OWN_LIST8(GRASPH_OWN_PMASS));
    } else if constexpr (NI == 2) {
        GRASPH_OWN_ASM(GRASPH_OWN_PAIRS2, GRASPH_OWN_LIST2(GRASPH_OWN_SUM), GRASPH_OWN_LIST2(GRASPH_OWN_SLOT),
                       GRASPH_OWN_LIST4(GRASPH_OWN_PARTNER), GRASPH_OWN_LIST4(GRASPH_OWN_PMASS));
    } else {
        static_assert(NI == 4);
        GRASPH_OWN_ASM(GRASPH_OWN_PAIRS4, GRASPH_OWN_LIST4(GRASPH_OWN_SUM), GRASPH_OWN_LIST4(GRASPH_OWN_SLOT),
                       GRASPH_OWN_LIST2(GRASPH_OWN_PARTNER), GRASPH_OWN_LIST2(GRASPH_OWN_PMASS));
    }
}

// Compensated gravity of the lane's slots from the partners [j0, j1), in
// order; tile: 64 float4 of this wavefront's; m the common mass when UM.
template <int NI, bool UM, bool SOFT>
__device__ __forceinline__ void own_sweep(const float4* __restrict__ xs, const int j0, const int j1, OwnAcc<NI>& a,
                                          CSum (&s)[NI][3], const float h2, const float m, float4* tile,
                                          const int lane)
{
    constexpr int kP = kOwnPairs / NI;
    auto partner = [&](const int j) {  // past the end: far away and massless
        float4 v = xs[min(j, j1 - 1)];
        if (j >= j1) v = make_float4(3.0e18f, 3.0e18f, 3.0e18f, 0.0f);
        return v;
    };
    if (j0 >= j1) return;
    float4 next = partner(j0 + lane);
    for (int j = j0; j < j1; j += 64) {
        tile[lane] = next;
        __builtin_amdgcn_wave_barrier();
        next = partner(j + 64 + lane);
        const int groups = (min(64, j1 - j) + kP - 1) / kP;
        float4 p[kP];
#pragma unroll
        for (int r = 0; r < kP; ++r) p[r] = tile[r];
        for (int g = 0; g < groups; ++g) {
            const int at = min(g + 1, 64 / kP - 1) * kP;
            if constexpr (NI == 1) {  // 8 partners: no registers for 8 more
                own_pairs<NI, UM, SOFT>(p, a, h2);
#pragma unroll
                for (int r = 0; r < kP; ++r) p[r] = tile[at + r];
            } else {  // the next partners on their way while these are summed
                float4 p2[kP];
#pragma unroll
                for (int r = 0; r < kP; ++r) p2[r] = tile[at + r];
                own_pairs<NI, UM, SOFT>(p, a, h2);
#pragma unroll
                for (int r = 0; r < kP; ++r) p[r] = p2[r];
            }
        }
        __builtin_amdgcn_wave_barrier();
        static_assert(kFold == 64);  // a tile
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            s[q][0].add(UM ? a.ax[q] * m : a.ax[q]);
            s[q][1].add(UM ? a.ay[q] * m : a.ay[q]);
            s[q][2].add(UM ? a.az[q] * m : a.az[q]);
            a.ax[q] = a.ay[q] = a.az[q] = 0.0f;
        }
    }
}

// LDS of a workgroup whose `waves` wavefronts share their own slots: a tile
// of partners each, then (when there are several) their sums
__host__ __device__ constexpr int own_lds_floats(int ni, int waves)
{
    return 256 * waves + (waves > 1 ? 6 * 64 * ni * waves : 0);
}

// Gravity of the slots [o0, o0 + 64 NI) below o1 from the partners [j0, j1)
// cut into `waves` shares of len (a multiple of 8): wavefront `wave` takes
// [j0 + wave len, j0 + (wave + 1) len).  store(t, x, y, z) gets every slot's
// sums, the shares' added in share order.  With several wavefronts they are
// the whole workgroup, and every thread calls it.
template <int NI, bool UM, bool SOFT, typename F>
__device__ __forceinline__ void own_block(const float4* __restrict__ xs, const int o0, const int o1, const int j0,
                                          const int j1, const int len, const float h2, const float m,
                                          const int wave, const int waves, float* lds, F&& store)
{
    const int lane = threadIdx.x & 63;
    OwnAcc<NI> a;
    CSum s[NI][3];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const float4 p = xs[min(o0 + 64 * q + lane, o1 - 1)];
        a.x[q] = p.x; a.y[q] = p.y; a.z[q] = p.z;
        a.ax[q] = a.ay[q] = a.az[q] = 0.0f;
        s[q][0] = s[q][1] = s[q][2] = CSum{0.0f, 0.0f};
    }
    const int b = j0 + wave * len, e = min(j1, b + len);
    own_sweep<NI, UM, SOFT>(xs, b, e, a, s, h2, m, reinterpret_cast<float4*>(lds) + 64 * wave, lane);
    if (waves == 1) {
#pragma unroll
        for (int q = 0; q < NI; ++q)
            if (o0 + 64 * q + lane < o1) store(o0 + 64 * q + lane, s[q][0], s[q][1], s[q][2]);
        return;
    }
    constexpr int kN = 64 * NI;
    float* const red = lds + 256 * waves;  // [wave][6][kN]
#pragma unroll
    for (int q = 0; q < NI; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            red[(wave * 6 + c) * kN + 64 * q + lane] = s[q][c].s;
            red[(wave * 6 + 3 + c) * kN + 64 * q + lane] = s[q][c].c;
        }
    __syncthreads();
    for (int i = threadIdx.x; i < kN; i += 64 * waves) {
        if (o0 + i >= o1) continue;
        CSum v[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v[c] = CSum{red[c * kN + i], red[(3 + c) * kN + i]};
            for (int w = 1; w < waves; ++w) {
                v[c].add(red[(w * 6 + c) * kN + i]);
                v[c].c += red[(w * 6 + 3 + c) * kN + i];
            }
        }
        store(o0 + i, v[0], v[1], v[2]);
    }
}

// own_block for few particles: 64 / SPLIT slots, each in SPLIT lanes of a
// wavefront, the q-th of which takes the share wave SPLIT + q of len partners,
// whose masses are taken as they come.  With one slot per lane 1000 particles
// were 16 workgroups of 16 wavefronts, 64 partners long each; four lanes a slot
// make that 63 workgroups of 11 wavefronts and 24 partners (Plummer step 11.0 ->
// 9.6 us, of 4096, in one plane instead of four, 13.7 -> 11.2).
// Every wavefront of the workgroup calls it; lds as for own_block<1>.
template <int SPLIT, bool SOFT, typename F>
__device__ __forceinline__ void own_split_block(const float4* __restrict__ xs, const int o0, const int n,
                                                const int len, const float h2, const int wave, const int waves,
                                                float* lds, F&& store)
{
    constexpr int kSlots = 64 / SPLIT;  // of the workgroup, and partners of a share in a tile
    const int lane = threadIdx.x & 63, slot = lane % kSlots, q = lane / kSlots;
    float4* const tile = reinterpret_cast<float4*>(lds) + 64 * wave;
    const int j0 = (wave * SPLIT + q) * len, j1 = min(n, j0 + len);
    auto partner = [&](const int j) {  // past the end: far away and massless
        float4 v = xs[min(j0 + j + slot, n - 1)];
        if (j0 + j + slot >= j1) v = make_float4(3.0e18f, 3.0e18f, 3.0e18f, 0.0f);
        return v;
    };
    float4 next = partner(0);
    OwnAcc<1> a;
    const float4 own = xs[min(o0 + slot, n - 1)];
    a.x[0] = own.x; a.y[0] = own.y; a.z[0] = own.z;
    a.ax[0] = a.ay[0] = a.az[0] = 0.0f;
    CSum s[3] = {CSum{0.0f, 0.0f}, CSum{0.0f, 0.0f}, CSum{0.0f, 0.0f}};
    for (int j = 0; j < len; j += kSlots) {
        tile[lane] = next;
        __builtin_amdgcn_wave_barrier();
        next = partner(j + kSlots);
#pragma unroll
        for (int g = 0; g < kSlots; g += kOwnPairs) {
            float4 p[kOwnPairs];
#pragma unroll
            for (int r = 0; r < kOwnPairs; ++r) p[r] = tile[lane - slot + g + r];
            own_pairs<1, false, SOFT>(p, a, h2);
        }
        __builtin_amdgcn_wave_barrier();
        if ((j + kSlots) % kFold == 0 || j + kSlots >= len) {
            s[0].add(a.ax[0]);
            s[1].add(a.ay[0]);
            s[2].add(a.az[0]);
            a.ax[0] = a.ay[0] = a.az[0] = 0.0f;
        }
    }
    float* const red = lds + 256 * waves;  // [wave][6][64]
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        red[(wave * 6 + c) * 64 + lane] = s[c].s;
        red[(wave * 6 + 3 + c) * 64 + lane] = s[c].c;
    }
    __syncthreads();
    if (wave != 0) return;
    for (int w = 1; w < waves; ++w)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s[c].add(red[(w * 6 + c) * 64 + lane]);
            s[c].c += red[(w * 6 + 3 + c) * 64 + lane];
        }
#pragma unroll
    for (int o = kSlots; o < 64; o <<= 1)  // lanes q = 0: (0 + 1) + (2 + 3)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float v = __shfl_xor(s[c].s, o, 64), e = __shfl_xor(s[c].c, o, 64);
            s[c].add(v);
            s[c].c += e;
        }
    if (q == 0 && o0 + slot < n) store(o0 + slot, s[0], s[1], s[2]);
}

}  // namespace
}  // namespace grasph
