// far_rotation.hpp -- one rotation of the symmetric sweep's far field: the 16
// slots of every lane against one partner, for both sides (sym_sweep.hip
// includes it; anonymous namespace).
//
// The partners of a chunk sit one per lane of a DPP row (16 partners, the
// same 16 in all four rows).  Sixteen rotations by one lane (row_ror:1) take
// every partner past every lane of its row: in rotation k, lane l's slots
// meet partner (l - k) & 15.  The partner side of a rotation is summed over
// the lane's slots (P) and then joins the partner's running sum T, which
// travels with the partner, one lane per rotation; after the 16th both are
// home, and two swaps add the four rows.
//
// What bounds a rotation is the FP32 vector issue, and gfx950 has two rates.
// A wave64 instruction takes 2 clocks (157 TFLOP/s of plain FMAs) when it
// reads VGPRs only, of which no three lie in the same half (even or odd
// numbers) of the register file; it takes 4 clocks with three reads of one
// half, an SGPR operand, a DPP operand or FP64, and a v_rsq_f32 takes 8.  Two
// wavefronts of a SIMD reach the 2-clock rate only while both issue 2-clock
// instructions; a slow one of either holds both at 4 clocks for some twenty
// instructions more.  Measured with loops of a pair's 14 instructions and its
// v_rsq_f32 at 2 wavefronts per SIMD: 60 clocks with the 16 v_rsq_f32 of a
// rotation in one run, 39.5 with that run at raised wave priority, which
// keeps the other wavefront from mixing its instructions into it (33.7 for
// the 14 alone).  The compiler knows neither the halves nor such runs, so a
// rotation is one asm block: for all 16 slots the differences (odd
// registers) and r^2 + H^2 (even registers), then the 16 v_rsq_f32 and the 6
// DPP instructions in one run at priority 1, then the rest.  With it
// far_kernel alone on the GPU takes 2.28 ms for the 8.52e9 unordered pairs of
// N = 131072 (3.20 before, 150 TFLOP/s at 20 per ordered pair now), and
// 165 ms for N = 1048576 with unequal masses (231 before).
#pragma once

#include "internal.hpp"
#include "sym_geometry.hpp"

namespace grasph {
namespace {

constexpr int kRow = 16;  // partners per rotated chunk (one DPP row)

// Own slots of a lane in the far field: position, mass and the plain
// gravity sums since the last fold.  A fold adds those to the wavefront's
// LDS sums (lsum[1024 c + slot], component c: plain sums of at most
// kFoldsPerFlush folds), and every kFoldsPerFlush folds and at the end of
// the row the LDS sums go into the row's own-side fragment in global
// memory (float4 sums at frag[frag_elem(slot)], their corrections 64
// further), compensated.  Neither level takes registers from the pair loop,
// and the fragment is written about once per row.
struct FarOwn {
    float x[kNI], y[kNI], z[kNI], m[kNI];
    float ax[kNI], ay[kNI], az[kNI];
    float* lsum;
    float4* frag;
    int folds;   // folds in lsum since the last flush (0: lsum holds nothing)
    bool fresh;  // nothing flushed into the fragment yet: the first flush writes it
    bool plain;  // every fragment is flushed once: no correction planes
};

// A chunk's partners on their way round the row: the partner at this lane,
// its partner-side sum T, and the last rotation's contribution P to it.
struct FarPartner {
    float x, y, z, m;
    float tx, ty, tz;
    float px, py, pz;
};

template <int K>
__device__ __forceinline__ float ror(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + K, 0xf, 0xf, true));
}

// One rotation in plain code (no softening: coincident particles exert
// nothing, computeDerivatives.h:226).  WIDE: far_rotation_soft's.
template <bool UM, bool WIDE>
__device__ __forceinline__ void far_rotation_hard(FarPartner& p, FarOwn& o)
{
    float px = 0.0f, py = 0.0f, pz = 0.0f;
#pragma unroll
    for (int q = 0; q < kNI; ++q) {
        const float dx = p.x - o.x[q], dy = p.y - o.y[q], dz = p.z - o.z[q];
        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const float inv = __builtin_amdgcn_rsqf(d2);
        float s = inv * inv;
        s = (d2 > 0.0f) ? s * inv : 0.0f;
        float sa = UM ? s : p.m * s, sb = UM ? s : s * o.m[q];
        if (!UM && WIDE) {
            sa = d2 > 0.0f ? (p.m * inv) * (inv * inv) : 0.0f;
            sb = d2 > 0.0f ? (o.m[q] * inv) * (inv * inv) : 0.0f;
        }
        o.ax[q] = fmaf(dx, sa, o.ax[q]); o.ay[q] = fmaf(dy, sa, o.ay[q]); o.az[q] = fmaf(dz, sa, o.az[q]);
        px = fmaf(dx, sb, px); py = fmaf(dy, sb, py); pz = fmaf(dz, sb, pz);
    }
    p.x = ror<1>(p.x); p.y = ror<1>(p.y); p.z = ror<1>(p.z);
    if (!UM) p.m = ror<1>(p.m);
    p.tx = ror<1>(p.tx) + p.px; p.ty = ror<1>(p.ty) + p.py; p.tz = ror<1>(p.tz) + p.pz;
    p.px = px; p.py = py; p.pz = pz;
}

// The asm block's slots: slot q, the register of its r^2 + H^2, then 1/r and
// 1/r^3 (even), of dx, dy and dz (odd), and of 1/r^2, then the partner
// side's factor (even).  v96 holds H^2.
#define GRASPH_FAR_SLOT0(F) \
    F(0, 64, 65, 67, 69, 98)
#define GRASPH_FAR_SLOTS1(F) \
    F(1, 66, 71, 73, 75, 100) F(2, 68, 77, 79, 81, 102) \
    F(3, 70, 83, 85, 87, 104) F(4, 72, 89, 91, 93, 106) \
    F(5, 74, 95, 97, 99, 108) F(6, 76, 101, 103, 105, 110) \
    F(7, 78, 107, 109, 111, 112) F(8, 80, 113, 115, 117, 114) \
    F(9, 82, 119, 121, 123, 116) F(10, 84, 125, 127, 129, 118) \
    F(11, 86, 131, 133, 135, 120) F(12, 88, 137, 139, 141, 122) \
    F(13, 90, 143, 145, 147, 124) F(14, 92, 149, 151, 153, 126) \
    F(15, 94, 155, 157, 159, 128)
#define GRASPH_FAR_SLOTS(F) GRASPH_FAR_SLOT0(F) GRASPH_FAR_SLOTS1(F)
#define GRASPH_FAR_CLOBBERS \
    "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", \
    "v79", "v80", "v81", "v82", "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", \
    "v94", "v95", "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", \
    "v109", "v110", "v111", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", \
    "v124", "v125", "v126", "v127", "v128", "v129", "v131", "v133", "v135", "v137", "v139", "v141", "v143", "v145", "v147", \
    "v149", "v151", "v153", "v155", "v157", "v159"
#define GRASPH_FAR_SUB(q, d, x, y, z, t)                                                                           \
    "v_sub_f32 v" #x ", %[jx], %[x" #q "]\n v_sub_f32 v" #y ", %[jy], %[y" #q "]\n"                                 \
    "v_sub_f32 v" #z ", %[jz], %[z" #q "]\n"
#define GRASPH_FAR_R2X(q, d, x, y, z, t) "v_fma_f32 v" #d ", v" #x ", v" #x ", v96\n"
#define GRASPH_FAR_R2Y(q, d, x, y, z, t) "v_fmac_f32 v" #d ", v" #y ", v" #y "\n"
#define GRASPH_FAR_R2Z(q, d, x, y, z, t) "v_fmac_f32 v" #d ", v" #z ", v" #z "\n"
#define GRASPH_FAR_RSQ(q, d, x, y, z, t) "v_rsq_f32 v" #d ", v" #d "\n"
#define GRASPH_FAR_INV2(q, d, x, y, z, t) "v_mul_f32 v" #t ", v" #d ", v" #d "\n"
#define GRASPH_FAR_INV3(q, d, x, y, z, t) "v_mul_f32 v" #d ", v" #t ", v" #d "\n"
// unequal masses: the slot's mass for the partner side, the partner's for the slot's
#define GRASPH_FAR_MASS(q, d, x, y, z, t)                                                                          \
    "v_mul_f32 v" #t ", v" #d ", %[m" #q "]\n v_mul_f32 v" #d ", %[jm], v" #d "\n"
// the same from 1/r and 1/r^2, each mass joining 1/r first; v130 in passing
#define GRASPH_FAR_WIDE(q, d, x, y, z, t)                                                                          \
    "v_mul_f32 v130, v" #d ", %[m" #q "]\n v_mul_f32 v" #d ", %[jm], v" #d "\n"                                   \
    "v_mul_f32 v" #d ", v" #t ", v" #d "\n v_mul_f32 v" #t ", v130, v" #t "\n"
// slot q's sums and its partner side with the factor in register f; op starts (v_mul) or continues (v_fmac) P
#define GRASPH_FAR_SUMS(q, d, x, y, z, f, op)                                                                      \
    "v_fmac_f32 %[ax" #q "], v" #x ", v" #d "\n" op " %[px], v" #x ", v" #f "\n"                                    \
    "v_fmac_f32 %[ay" #q "], v" #y ", v" #d "\n" op " %[py], v" #y ", v" #f "\n"                                    \
    "v_fmac_f32 %[az" #q "], v" #z ", v" #d "\n" op " %[pz], v" #z ", v" #f "\n"
#define GRASPH_FAR_START_UM(q, d, x, y, z, t) GRASPH_FAR_SUMS(q, d, x, y, z, d, "v_mul_f32")
#define GRASPH_FAR_SUMS_UM(q, d, x, y, z, t) GRASPH_FAR_SUMS(q, d, x, y, z, d, "v_fmac_f32")
#define GRASPH_FAR_START_M(q, d, x, y, z, t) GRASPH_FAR_SUMS(q, d, x, y, z, t, "v_mul_f32")
#define GRASPH_FAR_SUMS_M(q, d, x, y, z, t) GRASPH_FAR_SUMS(q, d, x, y, z, t, "v_fmac_f32")
#define GRASPH_FAR_IN(q, d, u, v, w, t) , [x##q] "v"(o.x[q]), [y##q] "v"(o.y[q]), [z##q] "v"(o.z[q])
#define GRASPH_FAR_MASS_IN(q, d, u, v, w, t) , [m##q] "v"(o.m[q])
#define GRASPH_FAR_OUT(q, d, u, v, w, t) , [ax##q] "+&v"(o.ax[q]), [ay##q] "+&v"(o.ay[q]), [az##q] "+&v"(o.az[q])
#define GRASPH_FAR_PARTNER                                                                                         \
    [jx] "+&v"(p.x), [jy] "+&v"(p.y), [jz] "+&v"(p.z), [tx] "+&v"(p.tx), [ty] "+&v"(p.ty), [tz] "+&v"(p.tz),              \
        [px] "+&v"(p.px), [py] "+&v"(p.py), [pz] "+&v"(p.pz)
#define GRASPH_FAR_ROR(op, r, a) op " %[" r "], %[" r "]" a " row_ror:1 row_mask:0xf bank_mask:0xf\n"
// differences and r^2 + H^2; then, in one run, the roots, the partners' move
// on to the next lane and the last rotation's P joining T
#define GRASPH_FAR_HEAD                                                                                            \
    "v_mov_b32 v96, %[h2]\n" GRASPH_FAR_SLOTS(GRASPH_FAR_SUB) GRASPH_FAR_SLOTS(GRASPH_FAR_R2X)                      \
    GRASPH_FAR_SLOTS(GRASPH_FAR_R2Y) GRASPH_FAR_SLOTS(GRASPH_FAR_R2Z)                                              \
    "s_setprio 1\n" GRASPH_FAR_SLOTS(GRASPH_FAR_RSQ)                                                               \
    GRASPH_FAR_ROR("v_add_f32_dpp", "tx", ", %[px]") GRASPH_FAR_ROR("v_add_f32_dpp", "ty", ", %[py]")              \
    GRASPH_FAR_ROR("v_add_f32_dpp", "tz", ", %[pz]") GRASPH_FAR_ROR("v_mov_b32_dpp", "jx", "")                     \
    GRASPH_FAR_ROR("v_mov_b32_dpp", "jy", "") GRASPH_FAR_ROR("v_mov_b32_dpp", "jz", "")
#define GRASPH_FAR_SQUARE "s_setprio 0\n" GRASPH_FAR_SLOTS(GRASPH_FAR_INV2)
#define GRASPH_FAR_CUBE GRASPH_FAR_SQUARE GRASPH_FAR_SLOTS(GRASPH_FAR_INV3)

// One rotation with softening; the partner's mass rotates for the next one.
// (Early-clobber outputs: the block writes them before its last input is read.)
// WIDE, unequal masses: the masses join 1/r, not 1/r^3, as in own_block.hpp, one
// multiply per pair more.
template <bool UM, bool WIDE>
__device__ __forceinline__ void far_rotation_soft(FarPartner& p, FarOwn& o, const float h2)
{
    if constexpr (UM) {
        asm volatile(GRASPH_FAR_HEAD GRASPH_FAR_CUBE GRASPH_FAR_SLOT0(GRASPH_FAR_START_UM)
                         GRASPH_FAR_SLOTS1(GRASPH_FAR_SUMS_UM)
                     : GRASPH_FAR_PARTNER GRASPH_FAR_SLOTS(GRASPH_FAR_OUT)
                     : [h2] "v"(h2) GRASPH_FAR_SLOTS(GRASPH_FAR_IN)
                     : GRASPH_FAR_CLOBBERS);
    } else {
        const float jm = p.m;
#define GRASPH_FAR_UNEQUAL(FACTORS, ...)                                                                           \
    asm volatile(GRASPH_FAR_HEAD GRASPH_FAR_ROR("v_mov_b32_dpp", "nm", "") FACTORS                                 \
                     GRASPH_FAR_SLOT0(GRASPH_FAR_START_M) GRASPH_FAR_SLOTS1(GRASPH_FAR_SUMS_M)                     \
                 : GRASPH_FAR_PARTNER, [nm] "+&v"(p.m) GRASPH_FAR_SLOTS(GRASPH_FAR_OUT)                            \
                 : [h2] "v"(h2), [jm] "v"(jm) GRASPH_FAR_SLOTS(GRASPH_FAR_IN) GRASPH_FAR_SLOTS(GRASPH_FAR_MASS_IN) \
                 : GRASPH_FAR_CLOBBERS, ##__VA_ARGS__)
        if constexpr (WIDE)
            GRASPH_FAR_UNEQUAL(GRASPH_FAR_SQUARE GRASPH_FAR_SLOTS(GRASPH_FAR_WIDE), "v130");
        else
            GRASPH_FAR_UNEQUAL(GRASPH_FAR_CUBE GRASPH_FAR_SLOTS(GRASPH_FAR_MASS));
#undef GRASPH_FAR_UNEQUAL
    }
}

}  // namespace
}  // namespace grasph
