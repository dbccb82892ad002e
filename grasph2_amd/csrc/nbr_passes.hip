// nbr_passes.hip -- the O(N k) neighbour-list passes (gfx950).
//
// density: calcDensity (src/computeDerivatives.h:52-91) over the list.
// strain:  calcBalsaraDensityDTDStressDT (:96-162); also writes the
//          per-particle record {sigma/rho^2, balsara, density} that the
//          acceleration pass reads for its j side, hoisting the per-pair
//          Murnaghan pow and nine divides of :246-257.
// prep:    the same record alone, for configurations that skip the strain
//          pass (:322-324).
// accel:   the SPH part of calcAcceleration (:237-295) plus
//          environmentAcceleration (:300-312), added to the gravity the
//          sweep left in acc with compensated (TwoSum) accumulation.
//
// Several lanes share a particle, particles in slot order (slot t ->
// i = perm[t]).  Every input a pass reads for a neighbour sits in one 64-byte
// slot record, rec[j] = {x y z m, vx vy vz rho, sigma/rho^2 (6) balsara rho},
// in slot order: one neighbour costs one contiguous gather, and a particle's
// neighbours' records are close together in memory.  Outputs go to
// particle i of the caller's arrays.  The list is stored in tiles of 64
// slots (list_entry) and holds slot indices in increasing order.  A particle
// whose count exceeds the list capacity falls back to a scan over its
// instance's slots with the exact neighbour test, so a full list never loses
// partners.
//
// What bounds them: a pass mixes FP64 and FP32 work, so every vector
// instruction takes about 4 clocks, and the acceleration pass's gathers look
// up 4 lines of the vector cache per pair, a line per clock and CU: at 200003
// particles 188000 of its 200000 clocks (fetching each record by 4 lanes
// together and exchanging the pieces through LDS halves the look-ups, but the
// exchange's instructions cost what that gives).  Density and strain are
// bound by their instructions.  At small counts a wavefront is alone on its
// SIMD (5.5 clocks per instruction) and the lanes per particle decide.
//
// Every kernel serves one instance (SlotMap from the kernel arguments) or a
// batch (SlotMap and parameters of the block's instance from tables).
#include "internal.hpp"

// No multiply-add contraction in this file: the pair arithmetic is inlined
// into the list walk and into the overflow scan, and contraction decided per
// call site could round the two differently.  Products and sums round as
// written, and fused ones are written as such.
#pragma clang fp contract(off)

namespace grasph {
namespace {

constexpr int kBlock = 256, kWaves = kBlock / 64;
// steps in flight of each pass's walk (for_each_neighbour's D; strain: with 4
// lanes, with 16 one): what hides their latency is wavefronts, and a deeper
// ring costs them registers.  All three passes at 200003 particles: 238 us
// with 4, 2 and 2 steps and the terms added in the order of all neighbours
// (48, 101, 89), now 29, 65 and 83.
constexpr int kDeepDensity = 2, kDeepStrain = 2, kDeepAccel = 1;

// lambdas are inlined by force: called from the list walk and the overflow
// scan, they would otherwise stay calls and pass the records through scratch
#define GRASPH_INLINE __attribute__((always_inline))

struct Tens {  // full 3x3, row-major, as mpu::Mat<float,3,3>
    float m[3][3];
};

__device__ inline Tens sym_to_full(float xx, float yy, float zz, float xy, float xz, float yz)
{
    Tens t;
    t.m[0][0] = xx; t.m[1][1] = yy; t.m[2][2] = zz;
    t.m[0][1] = xy; t.m[1][0] = xy;
    t.m[0][2] = xz; t.m[2][0] = xz;
    t.m[1][2] = yz; t.m[2][1] = yz;
    return t;
}

// src/sph/models.h:250-268, for the unique (d,e) of a symmetric result
__device__ inline float dsdt_entry(const Tens& ed, const Tens& rd, const Tens& S, float shear, int d, int e)
{
    float o = 2.0f * shear * ed.m[d][e];
#pragma unroll
    for (int f = 0; f < 3; ++f) {
        if (d == e) o -= 2.0f * shear * ed.m[f][f] / 3.0f;
        o += S.m[d][f] * rd.m[e][f];
        o += S.m[e][f] * rd.m[d][f];
    }
    return o;
}

struct Lists {
    const int* nbr;
    const int* cnt;
    const float4* coarse;  // boxes of 512 slots
    const float4* mid;     // and of 64
};

// LPP lanes share a particle (4 or 16): lane l of a wavefront serves
// particle l / LPP of the wavefront's 64 / LPP, and in step e of the walk
// neighbour e LPP + l % LPP of its list.  A particle has four sums of each
// quantity, of the neighbours k with k mod 4 = 0, 1, 2, 3 in the list's order,
// added at the end (ClassSums), whatever LPP is: a batch's results equal the
// single instance's bit for bit, and a list's those of its overflow scan.
// Against one lane per particle: 4 to 16 times the wavefronts for small counts
// (8192 particles: density, strain and acceleration 76 -> 26 us), lists of 16
// or 4 particles instead of 64 to wait for, and neighbouring lanes read
// neighbouring records (512 instances: 4.7 -> 3.7 ms).
template <int LPP>
__device__ __forceinline__ int pass_slot(const SlotMap& m)
{
    return m.slot0 + (int)threadIdx.x / LPP;
}

// Orders the wavefront's LDS accesses around it (the hardware executes one
// wavefront's in order; the compiler must not move them).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void acc_add(CSum& a, float v) { a.add(v); }
__device__ __forceinline__ void acc_add(float& a, float v) { a += v; }
__device__ __forceinline__ void acc_add(double& a, double v) { a += v; }

// adds a class's sum to another's: nothing when it is zero, so that an
// infinite gravity without neighbours stays one
__device__ __forceinline__ void acc_merge(CSum& a, const float s, const float c)
{
    if (s != 0.0f) a.add(s);
    a.c += c;
}

// NC sums of a particle (A: the accumulator of terms of type T) by classes of
// neighbours.  With 4 lanes each lane is a class and keeps its own sums (with
// the terms exchanged through LDS and added by all neighbours' order, the
// exchange took density and strain at 200003 particles 38 and 74 us, without
// it 32 and 70).  With
// 16 the four lanes of a class write their terms to LDS, side by side, a row
// per quantity (kRow apart, so the rows start in different banks), and lane
// 4 q + r adds those of class r of the quantities q, q + 4, ....
template <int LPP, int NC, typename T, typename A>
struct ClassSums {
    static constexpr int K = LPP == 4 ? NC : (NC + 3) / 4;
    static constexpr int kRow = 64 + 16 / (int)sizeof(T);
    static constexpr int kLds = LPP == 4 ? 4 : NC * kRow;  // elements of T per wavefront
    A a[K];

    // the quantity of accumulator k in lane sub (lanes without one repeat the last)
    __device__ __forceinline__ static int quantity(int sub, int k)
    {
        return LPP == 4 ? k : min(sub / 4 + 4 * k, NC - 1);
    }
    // what the sum of quantity c starts from
    __device__ __forceinline__ void init(const int c, const T v, const int lane)
    {
        const int sub = lane % LPP;
        if (LPP == 4 ? sub == 0 : sub == 4 * (c % 4)) a[LPP == 4 ? c : c / 4] = start(v);
    }
    // the step's terms (this lane's in v) of the group's first `rem` lanes
    __device__ __forceinline__ void add(const T (&v)[NC], const int rem, T* lds, const int lane)
    {
        const int sub = lane % LPP;
        if constexpr (LPP == 4) {
            if (sub < rem) {
#pragma unroll
                for (int c = 0; c < NC; ++c) acc_add(a[c], v[c]);
            }
        } else {
            T* const group = lds + (lane - sub);
#pragma unroll
            for (int c = 0; c < NC; ++c) group[c * kRow + 4 * (sub % 4) + sub / 4] = v[c];
            wave_lds_order();
            T w[K][4];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const T* row = (const T*)__builtin_assume_aligned(group + quantity(sub, k) * kRow + 4 * (sub % 4), 16);
#pragma unroll
                for (int u = 0; u < 4; ++u) w[k][u] = row[u];
            }
            wave_lds_order();
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (sub % 4 + 4 * u < rem) {
#pragma unroll
                    for (int k = 0; k < K; ++k) acc_add(a[k], w[k][u]);
                }
        }
    }
    // sum c, in every lane of the group (all lanes of the wavefront take part)
    __device__ __forceinline__ T value(const int c, const int lane) const
    {
        const A& m = a[LPP == 4 ? c : c / 4];
        const int first = lane - lane % LPP + (LPP == 4 ? 0 : 4 * (c % 4));  // its class 0
        return total(m, first);
    }

  private:
    __device__ __forceinline__ static CSum start_of(float v, CSum*) { return CSum{v, 0.0f}; }
    __device__ __forceinline__ static T start_of(T v, T*) { return v; }
    __device__ __forceinline__ static A start(T v) { return start_of(v, (A*)nullptr); }
    __device__ __forceinline__ static float total(const CSum& m, const int first)
    {
        float s[4], e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = __shfl(m.s, first + r, 64);
            e[r] = __shfl(m.c, first + r, 64);
        }
        CSum x{s[0], e[0]}, y{s[2], e[2]};
        acc_merge(x, s[1], e[1]);
        acc_merge(y, s[3], e[3]);
        acc_merge(x, y.s, y.c);
        return x.value();
    }
    __device__ __forceinline__ static T total(const T& m, const int first)
    {
        return (__shfl(m, first, 64) + __shfl(m, first + 1, 64)) +
               (__shfl(m, first + 2, 64) + __shfl(m, first + 3, 64));
    }
};

// the scan's collected neighbours: 2 LPP entries to each group of a wavefront's
constexpr int kPending = 2 * 64;
template <int LPP>
__device__ __forceinline__ int* pending_of(int (&pending)[kWaves][kPending])
{
    const int lane = threadIdx.x & 63;
    return pending[threadIdx.x >> 6] + 2 * (lane - lane % LPP);
}

// four floats that the compiler keeps in registers through the walk's rings
// (float4, a class, it copies as 16 bytes of memory, through scratch)
typedef float vec4 __attribute__((ext_vector_type(4)));

// Walk slot t's neighbours: the list, or when it overflowed, a scan of the
// instance's slots, in the boxes of 512 and of 64 within H, with the exact test
// (same partners, same order).
// step(q, rem): q holds the first PIECES float4 of the neighbour's record (of
// STRIDE float4 at src); lane sub has one if sub < rem (the others repeat the
// last).  pend: 2 LPP entries of the group's own, in which the scan collects the
// neighbours until each lane has one (evaluated one by one by the whole group
// they took the list's work LPP times: 32 squeezed instances of 8192 particles,
// 430 neighbours each in lists of 160, 8.3 ms a derivative call, now 4.7).
//
// The walk is software-pipelined D deep: while step e is computed, the
// records of steps e + 1 .. e + D and the indices up to e + 2 D are in
// flight.  A group past its list's end is masked off; within its last steps
// its lanes repeat the last neighbour.
template <int D, int LPP, int PIECES, int STRIDE, typename S>
__device__ __forceinline__ void for_each_neighbour(const vec4* __restrict__ src, const float4* __restrict__ xs,
                                                   const Lists& Ls, const int t, const bool act, const int kmax,
                                                   const float4 pi, const SlotMap& m, const float H2, int* pend,
                                                   S&& step)
{
    const int lane = threadIdx.x & 63, sub = lane % LPP;
    const int cnt = Ls.cnt[t];
    const int c = act && cnt <= kmax ? cnt : 0;
    // what a lane reads past its list's end is some slot of the instance: the
    // list's last entry (a lane without a list walks entry 0 of slot t's
    // overflowed one, or reads slot 0 from a count of 0)
    const int* list = cnt > 0 ? Ls.nbr + list_entry(t, 0, kmax) : Ls.cnt + t;
    const uint32_t mask = list_mask(kmax), lane0 = list_offset((uint32_t)sub, mask);
    const uint32_t last = list_offset((uint32_t)max(c - 1, 0), mask);
    static_assert(LPP % 4 == 0);  // a step's entries begin a chunk
    const auto index = [&](int e) GRASPH_INLINE { return list[min((uint32_t)(64 * LPP * e) + lane0, last)]; };
    const auto fetch = [&](int j, vec4 (&r)[PIECES]) GRASPH_INLINE {
#pragma unroll
        for (int q = 0; q < PIECES; ++q) r[q] = src[STRIDE * (uint64_t)(uint32_t)j + q];
    };
    int jn[D];
    vec4 r[D][PIECES];
    const auto turn = [&](int e, int& j, vec4 (&rr)[PIECES]) GRASPH_INLINE {
        vec4 q[PIECES];
#pragma unroll
        for (int p = 0; p < PIECES; ++p) q[p] = rr[p];
        fetch(j, rr);  // step e + D (its indices came D steps ago)
        j = index(e + 2 * D);
        step(q, c - e * LPP);
    };
#pragma unroll
    for (int u = 0; u < D; ++u) jn[u] = index(u);
#pragma unroll
    for (int u = 0; u < D; ++u) {
        fetch(jn[u], r[u]);
        jn[u] = index(u + D);
    }
    for (int e = 0; e * LPP < c; e += D) {
        turn(e, jn[0], r[0]);
        if constexpr (D > 1) turn(e + 1, jn[1], r[1]);
        if constexpr (D > 2) turn(e + 2, jn[2], r[2]);
        if constexpr (D > 3) turn(e + 3, jn[3], r[3]);
    }
    if (act && cnt > kmax) {
        constexpr int kMids = kBoxCoarse / kBoxMid;
        const float4* const coarse = Ls.coarse + 2 * (size_t)m.coarse0;
        const float4* const mid = Ls.mid + 2 * (size_t)kMids * m.coarse0;
        const int nc = (m.n + kBoxCoarse - 1) / kBoxCoarse, nm = (m.n + kBoxMid - 1) / kBoxMid;
        // the group's lanes look at LPP boxes or slots at once
        const auto bits = [&](bool b) GRASPH_INLINE {
            return (unsigned)(__ballot(b) >> (lane - sub)) & ((1u << LPP) - 1u);
        };
        // a box farther than H holds none of the partners (lists.hip)
        const auto near = [&](const float4* box, int q, int count) GRASPH_INLINE {
            const float4 lo = box[2 * min(q, count - 1)], hi = box[2 * min(q, count - 1) + 1];
            const float bx = fmaxf(0.0f, fmaxf(lo.x - pi.x, pi.x - hi.x));
            const float by = fmaxf(0.0f, fmaxf(lo.y - pi.y, pi.y - hi.y));
            const float bz = fmaxf(0.0f, fmaxf(lo.z - pi.z, pi.z - hi.z));
            return q < count && dist2_exact(bx, by, bz) <= H2;
        };
        const auto collected = [&](int rem) GRASPH_INLINE {
            vec4 q[PIECES];
            fetch(pend[min(sub, rem - 1)], q);
            step(q, rem);
        };
        int fill = 0;
        for (int c0 = 0; c0 < nc; c0 += LPP)
            for (unsigned cb = bits(near(coarse, c0 + sub, nc)); cb != 0u; cb &= cb - 1u) {
                const int m0 = kMids * (c0 + __ffs(cb) - 1);
                for (int h = 0; h < kMids; h += LPP)
                    for (unsigned mb = bits(h + sub < kMids && near(mid, m0 + h + sub, nm)); mb != 0u; mb &= mb - 1u) {
                        const int first = kBoxMid * (m0 + h + __ffs(mb) - 1), end = min(first + kBoxMid, m.n);
                        for (int j0 = first; j0 < end; j0 += LPP) {
                            const int j = m.off + min(j0 + sub, end - 1);
                            const float4 pj = xs[j];
                            const bool is = j0 + sub < end &&
                                            is_neighbour(dist2_exact(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z), H2);
                            const unsigned b = bits(is);
                            if (is) pend[fill + __popc(b & ((1u << sub) - 1u))] = j;
                            fill += __popc(b);
                            if (fill < LPP) continue;
                            wave_lds_order();
                            collected(LPP);
                            fill -= LPP;
                            const int rest = pend[LPP + sub];
                            wave_lds_order();
                            if (sub < fill) pend[sub] = rest;
                        }
                    }
            }
        if (fill > 0) {
            wave_lds_order();
            collected(fill);
        }
    }
}

template <int LPP>
__device__ __forceinline__ void max_subs(float& a)
{
#pragma unroll
    for (int o = 1; o < LPP; o <<= 1) a = fmaxf(a, __shfl_xor(a, o, 64));
}

template <bool BATCH, int LPP>
__global__ __launch_bounds__(kBlock) void density_kernel(const float4* __restrict__ xs, SlotRec* __restrict__ rec,
                                                         const int* __restrict__ perm,
                                                         const Lists Ls,
                                                         const size_t nstride, const int kmax,
                                                         float* __restrict__ density, const BlockTables T,
                                                         const DevParams P0)
{
    using Rho = ClassSums<LPP, 1, float, CSum>;
    __shared__ __attribute__((aligned(16))) float terms[kWaves][Rho::kLds];
    __shared__ int pending[kWaves][kPending];
    const SlotMap m = slot_map<BATCH>(T, (int)nstride, kBlock / LPP, xcd_run((int)nstride, kmax));
    const int t0 = pass_slot<LPP>(m), lane = threadIdx.x & 63;
    const bool act = t0 < m.slot_end;
    const int t = act ? t0 : m.slot_end - 1;  // lanes past the end only take part in the wavefront's exchanges
    float* const lt = terms[threadIdx.x >> 6];
    const DevParams P = BATCH ? T.prm[m.inst] : P0;
    const float4 pi = xs[t];  // positions from the compact slot-ordered array (16 B per partner)
    Rho rho{};
    const auto term = [&](const vec4 (&q)[1], float (&v)[1]) GRASPH_INLINE {
        v[0] = q[0].w * kernel_w_f64(pi.x - q[0].x, pi.y - q[0].y, pi.z - q[0].z, P);
    };
    for_each_neighbour<kDeepDensity, LPP, 1, 1>(
        (const vec4*)xs, xs, Ls, t, act, kmax, pi, m, P.H2, pending_of<LPP>(pending),
        [&](const vec4 (&q)[1], int rem) GRASPH_INLINE {
            float v[1];
            term(q, v);
            rho.add(v, rem, lt, lane);
        });
    float r = rho.value(0, lane);
    if (!act || lane % LPP != 0) return;
    if ((P.flags & GRASPH_DEAL_WITH_NO_PARTNERS) && r < 0.001f) r = P.rho0 * 0.01f;  // :85-88
    density[perm ? perm[t] : t] = r;
    rec[t].vr.w = r;  // the strain / record passes read densities from the slot records
}

template <bool BATCH, int LPP, bool SOLIDS, bool BALS, bool INTD>
__global__ __launch_bounds__(kBlock) void strain_kernel(
    const float4* __restrict__ xs, SlotRec* __restrict__ rec, const float* __restrict__ dstress,
    const int* __restrict__ perm, const Lists Ls, const size_t nstride, const int kmax, float* __restrict__ balsara,
    float* __restrict__ density_dt, float* __restrict__ dstress_dt, const BlockTables T, const DevParams P0)
{
    // Sums and terms in FP64 from the FP32 inputs: the velocity divergence
    // and curl cancel strongly where bodies meet, and the Balsara factor
    // built from them scales the artificial viscosity of the acceleration
    // pass, where FP32 rounding here showed up amplified.  Solids: the nine
    // sums M_ab of vol v_a g_b, which hold the strain rate (-M's symmetric
    // part, models.h:225-248), the rotation rate (-M's antisymmetric part)
    // and div v (-M's trace); liquids: curl v with a Balsara switch, and div v
    // where it is used.
    constexpr int kRot = SOLIDS ? 9 : BALS ? 3 : 0;
    constexpr int NC = kRot + (!SOLIDS && (BALS || INTD) ? 1 : 0);
    constexpr int kTerms = NC > 0 ? NC : 1;
    using Rates = ClassSums<LPP, kTerms, double, double>;
    __shared__ __attribute__((aligned(16))) double terms[kWaves][Rates::kLds];
    __shared__ int pending[kWaves][kPending];
    const SlotMap m = slot_map<BATCH>(T, (int)nstride, kBlock / LPP, xcd_run((int)nstride, kmax));
    const int t0 = pass_slot<LPP>(m), lane = threadIdx.x & 63;
    const bool act = t0 < m.slot_end;
    const int t = act ? t0 : m.slot_end - 1;  // lanes past the end only take part in the wavefront's exchanges
    double* const lt = terms[threadIdx.x >> 6];
    const DevParams P = BATCH ? T.prm[m.inst] : P0;
    const int i = perm ? perm[t] : t;
    const float4 pi = rec[t].pm;
    const float4 vr = rec[t].vr;
    const float rhoi = vr.w;
    const struct { double x, y, z; } vi = {vr.x, vr.y, vr.z};

    float st[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // the stress used after the walk, on its way during it
    if (SOLIDS) {
#pragma unroll
        for (int c = 0; c < 6; ++c) st[c] = dstress[m.plane6(c, i)];
    }
    Rates R{};
    const auto term = [&](const vec4 (&q)[2], double (&v)[kTerms]) GRASPH_INLINE {
        const vec4 pj = q[0], vj = q[1];
        const double rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        const double s = dw_over_r_f64(pair_sep(rx, ry, rz, P), P) * div_f64(pj.w, vj.w);  // vol = m_j / rho_j
        const double gx = s * rx, gy = s * ry, gz = s * rz;
        const double vx = vi.x - (double)vj.x, vy = vi.y - (double)vj.y, vz = vi.z - (double)vj.z;
        if constexpr (SOLIDS) {
            v[0] = vx * gx; v[1] = vx * gy; v[2] = vx * gz;
            v[3] = vy * gx; v[4] = vy * gy; v[5] = vy * gz;
            v[6] = vz * gx; v[7] = vz * gy; v[8] = vz * gz;
        } else {
            if constexpr (BALS) {  // curl v, computeDerivatives.h:134
                v[0] = __builtin_fma(vy, gz, -(vz * gy));
                v[1] = __builtin_fma(vz, gx, -(vx * gz));
                v[2] = __builtin_fma(vx, gy, -(vy * gx));
            }
            if constexpr (BALS || INTD) v[NC - 1] = -__builtin_fma(vz, gz, __builtin_fma(vy, gy, vx * gx));  // :137
        }
        if constexpr (NC == 0) v[0] = 0.0;
    };
    for_each_neighbour<LPP == 4 ? kDeepStrain : 1, LPP, 2, 4>(
        (const vec4*)rec, xs, Ls, t, act, kmax, pi, m, P.H2, pending_of<LPP>(pending),
        [&](const vec4 (&q)[2], int rem) GRASPH_INLINE {
            double v[kTerms];
            term(q, v);
            R.add(v, rem, lt, lane);
        });
    double exx = 0, eyy = 0, ezz = 0, exy = 0, exz = 0, eyz = 0;  // strain rate (symmetric)
    double rxy = 0, rxz = 0, ryz = 0;                              // rotation rate (antisymmetric)
    double divv = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
    if constexpr (SOLIDS) {
        const double xy = R.value(1, lane), yx = R.value(3, lane), xz = R.value(2, lane), zx = R.value(6, lane),
                     yz = R.value(5, lane), zy = R.value(7, lane);
        exx = -R.value(0, lane); eyy = -R.value(4, lane); ezz = -R.value(8, lane);
        exy = -0.5 * (xy + yx); exz = -0.5 * (xz + zx); eyz = -0.5 * (yz + zy);
        rxy = -0.5 * (xy - yx); rxz = -0.5 * (xz - zx); ryz = -0.5 * (yz - zy);
        if (BALS || INTD) divv = exx + eyy + ezz;
    } else {
        if constexpr (BALS) { cx = R.value(0, lane); cy = R.value(1, lane); cz = R.value(2, lane); }
        if constexpr (BALS || INTD) divv = R.value(NC - 1, lane);
    }
    if (!act || lane % LPP != 0) return;

    // do_after, computeDerivatives.h:144-161
    Tens S = sym_to_full(st[0], st[1], st[2], st[3], st[4], st[5]);
    float sdt[6] = {0, 0, 0, 0, 0, 0};
    if (SOLIDS) {
        const Tens ed = sym_to_full((float)exx, (float)eyy, (float)ezz, (float)exy, (float)exz, (float)eyz);
        Tens rd;
        rd.m[0][0] = 0.0f; rd.m[1][1] = 0.0f; rd.m[2][2] = 0.0f;
        rd.m[0][1] = (float)rxy; rd.m[1][0] = -(float)rxy;
        rd.m[0][2] = (float)rxz; rd.m[2][0] = -(float)rxz;
        rd.m[1][2] = (float)ryz; rd.m[2][1] = -(float)ryz;
        sdt[0] = dsdt_entry(ed, rd, S, P.shear, 0, 0);
        sdt[1] = dsdt_entry(ed, rd, S, P.shear, 1, 1);
        sdt[2] = dsdt_entry(ed, rd, S, P.shear, 2, 2);
        sdt[3] = dsdt_entry(ed, rd, S, P.shear, 0, 1);
        sdt[4] = dsdt_entry(ed, rd, S, P.shear, 0, 2);
        sdt[5] = dsdt_entry(ed, rd, S, P.shear, 1, 2);
        // curl from the rotation rate, :150
        cx = -2.0 * ryz;
        cy = 2.0 * rxz;
        cz = -2.0 * rxy;
    }
    float bal = 0.0f;
    if (BALS) bal = balsara_switch_f64(divv, cx, cy, cz, P.c, P.H);
    if (balsara) balsara[i] = bal;
    if (density_dt) density_dt[i] = INTD ? (float)(-(double)rhoi * divv) : 0.0f;
    if (dstress_dt) {
#pragma unroll
        for (int c = 0; c < 6; ++c) dstress_dt[m.plane6(c, i)] = sdt[c];
    }

    // j-side record of the acceleration pass (its do_before, :193-219)
    if (SOLIDS) {
        const float pres = eos_murnaghan(rhoi, P.rho0, P.BULK, P.dBULKdP);
        const float d2 = rhoi * rhoi;
        rec[t].ra = make_float4((S.m[0][0] - pres) / d2, (S.m[1][1] - pres) / d2, (S.m[2][2] - pres) / d2,
                                S.m[0][1] / d2);
        rec[t].rb = make_float4(S.m[0][2] / d2, S.m[1][2] / d2, bal, rhoi);
    } else {
        const float sig = -eos_liquid(rhoi, P.rho0, P.c2);
        rec[t].ra = make_float4(sig / (rhoi * rhoi), 0.0f, 0.0f, 0.0f);
        rec[t].rb = make_float4(0.0f, 0.0f, bal, rhoi);
    }
}

// record only (no strain pass in this configuration)
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void prep_kernel(SlotRec* __restrict__ rec, const float* __restrict__ dstress,
                                                      const float* __restrict__ balsara, const int* __restrict__ perm,
                                                      const size_t nstride, const BlockTables T, const DevParams P0)
{
    const SlotMap m = slot_map<BATCH>(T, (int)nstride);
    const int t = m.slot0 + threadIdx.x;
    if (t >= m.slot_end) return;
    const DevParams P = BATCH ? T.prm[m.inst] : P0;
    const int i = perm ? perm[t] : t;
    const float rhoi = rec[t].vr.w;
    const float bal = balsara ? balsara[i] : 0.0f;
    if (P.flags & GRASPH_SOLIDS) {
        const float pres = eos_murnaghan(rhoi, P.rho0, P.BULK, P.dBULKdP);
        const float d2 = rhoi * rhoi;
        rec[t].ra = make_float4((dstress[m.plane6(0, i)] - pres) / d2, (dstress[m.plane6(1, i)] - pres) / d2,
                                (dstress[m.plane6(2, i)] - pres) / d2, dstress[m.plane6(3, i)] / d2);
        rec[t].rb = make_float4(dstress[m.plane6(4, i)] / d2, dstress[m.plane6(5, i)] / d2, bal, rhoi);
    } else {
        const float sig = -eos_liquid(rhoi, P.rho0, P.c2);
        rec[t].ra = make_float4(sig / (rhoi * rhoi), 0.0f, 0.0f, 0.0f);
        rec[t].rb = make_float4(0.0f, 0.0f, bal, rhoi);
    }
}

template <bool BATCH, int LPP, bool SOLIDS, bool BALS, bool AV, bool XSPH, bool ARTS>
__global__ __launch_bounds__(kBlock) void accel_kernel(
    const float4* __restrict__ xs, const SlotRec* __restrict__ rec, const int* __restrict__ perm, const Lists Ls,
    const size_t nstride,
    const int kmax, float4* __restrict__ acc, float4* __restrict__ xvel, float* __restrict__ maxvsig,
    const int acc_has_gravity, const BlockTables T, const DevParams P0)
{
    using Acc = ClassSums<LPP, 3, float, CSum>;
    using Xv = ClassSums<LPP, 3, float, float>;
    __shared__ __attribute__((aligned(16))) float terms[kWaves][(XSPH ? 2 : 1) * Acc::kLds];
    __shared__ int pending[kWaves][kPending];
    const SlotMap m = slot_map<BATCH>(T, (int)nstride, kBlock / LPP, xcd_run((int)nstride, kmax));
    const int t0 = pass_slot<LPP>(m), lane = threadIdx.x & 63, sub = lane % LPP;
    const bool act = t0 < m.slot_end;
    const int t = act ? t0 : m.slot_end - 1;  // lanes past the end only take part in the wavefront's exchanges
    float* const lt = terms[threadIdx.x >> 6];
    const DevParams P = BATCH ? T.prm[m.inst] : P0;
    const int i = perm ? perm[t] : t;
    const float4 pi = rec[t].pm;
    const float4 vi = rec[t].vr;
    const float4 ra = rec[t].ra, rb = rec[t].rb;
    const float rhoi = rb.w, bi = BALS ? rb.z : 1.0f;
    // sigma_i / rho_i^2 and, for liquids with artificial pressure, arts_i
    const float sxx = ra.x, syy = ra.y, szz = ra.z, sxy = ra.w, sxz = rb.x, syz = rb.y;
    const float arts_i = (ARTS && !SOLIDS) ? ((sxx > 0) ? (-P.mateps * sxx) : 0.0f) : 0.0f;

    Acc A{};
    Xv X{};
    if (acc_has_gravity) {
        const float4 g = acc[i];
        A.init(0, g.x, lane);
        A.init(1, g.y, lane);
        A.init(2, g.z, lane);
    }
    float mv = 0.0f;

    const auto term = [&](const vec4 (&q)[4], float (&f)[3], float (&x)[3], const bool counts) GRASPH_INLINE {
        const vec4 pj = q[0], vj = q[1], qa = q[2], qb = q[3];
        const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        // dW/r r_ij: FP64, rounded once (the pair terms cancel where the stresses are large)
        const PairSep sep = pair_sep(rx, ry, rz, P);
        const double s = dw_over_r_f64(sep, P);
        const float gx = (float)(s * (double)rx), gy = (float)(s * (double)ry), gz = (float)(s * (double)rz);
        const float rho2 = rhoi + qb.w;  // twice the mean density
        const float mj = pj.w;
        const float vx = vi.x - vj.x, vy = vi.y - vj.y, vz = vi.z - vj.z;
        float II = 0.0f;
        if (AV) {  // :277-289 (models.h:158-185)
            // unfused, as the reference rounds it: in a rigid rotation every v . r is rounding alone, and its sign
            // decides whether the pair counts for maxvsig
            const float wij = (rx * vx + ry * vy + rz * vz) * (float)sep.ir;
            const float vsig = __builtin_fmaf(-3.0f, wij, P.c + P.c);
            const float b = BALS ? bi + qb.z : 2.0f;
            const float II0 = -0.25f * b * P.alpha * wij * vsig / (0.5f * rho2);
            II = wij < 0.0f ? II0 : 0.0f;
            if (BALS && counts && wij < 0.0f) mv = fmaxf(mv, vsig);
        }
        if (SOLIDS) {  // acc += m_j (stress . gradw), stress = sOR_i + sOR_j  (:260, :275)
            const float txx = sxx + qa.x, tyy = syy + qa.y, tzz = szz + qa.z;
            const float txy = sxy + qa.w, txz = sxz + qb.x, tyz = syz + qb.y;
            f[0] = __builtin_fmaf(txz, gz, __builtin_fmaf(txy, gy, txx * gx));
            f[1] = __builtin_fmaf(tyz, gz, __builtin_fmaf(tyy, gy, txy * gx));
            f[2] = __builtin_fmaf(tzz, gz, __builtin_fmaf(tyz, gy, txz * gx));
        } else {
            float st = sxx + qa.x;
            if (ARTS) {  // :263-272 (liquid artificial pressure)
                const float r = sqrtf(dist2_exact(rx, ry, rz));
                const float fa = powf(w_spline(r, P.H, P.Wpref) / P.Wnorm, P.matexp);
                const float arts_j = (qa.x > 0) ? (-P.mateps * qa.x) : 0.0f;
                st += fa * (arts_i + arts_j);
            }
            f[0] = st * gx;
            f[1] = st * gy;
            f[2] = st * gz;
        }
        f[0] *= mj;
        f[1] *= mj;
        f[2] *= mj;
        if (AV) {  // the mass joins II first: II times the gradient can be below FP32's range where m II is not
            const float mII = mj * II;
            f[0] = __builtin_fmaf(-mII, gx, f[0]);
            f[1] = __builtin_fmaf(-mII, gy, f[1]);
            f[2] = __builtin_fmaf(-mII, gz, f[2]);
        }
        if (XSPH) {  // :291-294
            const float qf = (float)sep.q, om = 1.0f - qf;
            const float w = P.Wpref * (qf < 0.5f ? __builtin_fmaf(-6.0f * qf * qf, om, 1.0f) : 2.0f * om * om * om);
            const float fx = 2.0f * mj / rho2 * w;
            x[0] = -fx * vx;
            x[1] = -fx * vy;
            x[2] = -fx * vz;
        }
    };
    for_each_neighbour<kDeepAccel, LPP, 4, 4>(
        (const vec4*)rec, xs, Ls, t, act, kmax, pi, m, P.H2, pending_of<LPP>(pending),
        [&](const vec4 (&q)[4], int rem) GRASPH_INLINE {
            float f[3], x[3];
            term(q, f, x, sub < rem);
            A.add(f, rem, lt, lane);
            if constexpr (XSPH) X.add(x, rem, lt + Acc::kLds, lane);
        });
    float fx = A.value(0, lane), fy = A.value(1, lane), fz = A.value(2, lane);
    float xvx = 0.0f, xvy = 0.0f, xvz = 0.0f;
    if constexpr (XSPH) {
        xvx = X.value(0, lane); xvy = X.value(1, lane); xvz = X.value(2, lane);
    }
    if (BALS && AV) max_subs<LPP>(mv);
    if (!act || sub != 0) return;
    environment_acceleration(P, fx, fy, fz);
    acc[i] = make_float4(fx, fy, fz, 0.0f);
    if (maxvsig) maxvsig[i] = mv;
    if (xvel) xvel[i] = make_float4(xvx, xvy, xvz, 0.0f);
}

// Without SPH: environmentAcceleration on the gravity and the zero XVEL /
// MAXVSIG of calcAcceleration's store (computeDerivatives.h:171, 300-312).
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void finish_kernel(const float4* __restrict__ posm,
                                                        const float4* __restrict__ vel, float4* __restrict__ acc,
                                                        float4* __restrict__ xvel, float* __restrict__ maxvsig,
                                                        const int n, const BlockTables T, const DevParams P0)
{
    const SlotMap m = slot_map<BATCH>(T, n);
    const int i = m.slot0 + threadIdx.x;
    if (i >= m.slot_end) return;
    const DevParams P = BATCH ? T.prm[m.inst] : P0;
    const bool grav = P.flags & GRASPH_SELF_GRAVITY;
    if (!grav || (P.flags & GRASPH_CONSTANT_ACCELERATION)) {
        float4 a = grav ? acc[i] : make_float4(0.f, 0.f, 0.f, 0.f);  // no sweep ran without gravity
        environment_acceleration(P, a.x, a.y, a.z);
        acc[i] = make_float4(a.x, a.y, a.z, 0.0f);
    }
    if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (maxvsig) maxvsig[i] = 0.0f;
}

inline Lists lists_of(const NbrLaunch& L) { return Lists{L.nbr, L.nbr_cnt, L.coarse, L.mid}; }

inline dim3 grid_plain(const NbrLaunch& L)  // per-particle kernels without a list walk
{
    return dim3(L.T.nblocks > 0 ? L.T.nblocks : (L.n + kBlock - 1) / kBlock);
}
inline dim3 grid_of(const NbrLaunch& L)
{
    const int per = kBlock / L.lanes;  // particles per block
    return dim3(L.T.nblocks > 0 ? L.T.nblocks64 : (L.n + per - 1) / per);
}

template <bool BATCH, int LPP>
hipError_t strain_b(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    const bool so = P.flags & GRASPH_SOLIDS, ba = P.flags & GRASPH_BALSARA_SWITCH,
               in = P.flags & GRASPH_INTEGRATE_DENSITY;
#define GRASPH_STRAIN(A, B, C)                                                                                     \
    hipLaunchKernelGGL((strain_kernel<BATCH, LPP, A, B, C>), grid_of(L), dim3(kBlock), 0, s, L.xs, L.rec, L.dstress, \
                       L.perm, lists_of(L), (size_t)L.n, L.kmax, L.balsara, L.density_dt, L.dstress_dt, L.T, P)
    const int key = (so ? 4 : 0) | (ba ? 2 : 0) | (in ? 1 : 0);
    switch (key) {
        case 0: GRASPH_STRAIN(false, false, false); break;
        case 1: GRASPH_STRAIN(false, false, true); break;
        case 2: GRASPH_STRAIN(false, true, false); break;
        case 3: GRASPH_STRAIN(false, true, true); break;
        case 4: GRASPH_STRAIN(true, false, false); break;
        case 5: GRASPH_STRAIN(true, false, true); break;
        case 6: GRASPH_STRAIN(true, true, false); break;
        default: GRASPH_STRAIN(true, true, true); break;
    }
#undef GRASPH_STRAIN
    return hipGetLastError();
}

template <bool BATCH, int LPP>
hipError_t accel_b(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    const bool so = P.flags & GRASPH_SOLIDS, ba = P.flags & GRASPH_BALSARA_SWITCH,
               av = P.flags & GRASPH_ARTIFICIAL_VISCOSITY, xs = P.flags & GRASPH_XSPH,
               ar = P.flags & GRASPH_ARTIFICIAL_STRESS;
#define GRASPH_ACCEL(A, B, C, D, E)                                                                                  \
    hipLaunchKernelGGL((accel_kernel<BATCH, LPP, A, B, C, D, E>), grid_of(L), dim3(kBlock), 0, s, L.xs, L.rec,    \
                       L.perm,                                                                                     \
                       lists_of(L), (size_t)L.n, L.kmax, L.acc, L.xvel, L.maxvsig, L.acc_has_gravity ? 1 : 0,  \
                       L.T, P)
    // SOLIDS + ARTIFICIAL_STRESS is rejected before launch (the reference does not compile it).
    const int key = (so ? 16 : 0) | (ba ? 8 : 0) | (av ? 4 : 0) | (xs ? 2 : 0) | (ar ? 1 : 0);
    switch (key) {
        case 0: GRASPH_ACCEL(false, false, false, false, false); break;
        case 1: GRASPH_ACCEL(false, false, false, false, true); break;
        case 2: GRASPH_ACCEL(false, false, false, true, false); break;
        case 3: GRASPH_ACCEL(false, false, false, true, true); break;
        case 4: GRASPH_ACCEL(false, false, true, false, false); break;
        case 5: GRASPH_ACCEL(false, false, true, false, true); break;
        case 6: GRASPH_ACCEL(false, false, true, true, false); break;
        case 7: GRASPH_ACCEL(false, false, true, true, true); break;
        case 8: GRASPH_ACCEL(false, true, false, false, false); break;
        case 9: GRASPH_ACCEL(false, true, false, false, true); break;
        case 10: GRASPH_ACCEL(false, true, false, true, false); break;
        case 11: GRASPH_ACCEL(false, true, false, true, true); break;
        case 12: GRASPH_ACCEL(false, true, true, false, false); break;
        case 13: GRASPH_ACCEL(false, true, true, false, true); break;
        case 14: GRASPH_ACCEL(false, true, true, true, false); break;
        case 15: GRASPH_ACCEL(false, true, true, true, true); break;
        case 16: GRASPH_ACCEL(true, false, false, false, false); break;
        case 18: GRASPH_ACCEL(true, false, false, true, false); break;
        case 20: GRASPH_ACCEL(true, false, true, false, false); break;
        case 22: GRASPH_ACCEL(true, false, true, true, false); break;
        case 24: GRASPH_ACCEL(true, true, false, false, false); break;
        case 26: GRASPH_ACCEL(true, true, false, true, false); break;
        case 28: GRASPH_ACCEL(true, true, true, false, false); break;
        case 30: GRASPH_ACCEL(true, true, true, true, false); break;
        default: return hipErrorInvalidValue;
    }
#undef GRASPH_ACCEL
    return hipGetLastError();
}

}  // namespace

hipError_t launch_density(const NbrLaunch& L, float* density, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
#define GRASPH_DENSITY(BATCH, LPP)                                                                               \
    hipLaunchKernelGGL((density_kernel<BATCH, LPP>), grid_of(L), dim3(kBlock), 0, s, L.xs, L.rec, L.perm, lists_of(L), \
                       (size_t)L.n, L.kmax, density, L.T, P)
    if (L.T.nblocks > 0) GRASPH_DENSITY(true, 4);
    else if (L.lanes == 16) GRASPH_DENSITY(false, 16);
    else GRASPH_DENSITY(false, 4);
#undef GRASPH_DENSITY
    return hipGetLastError();
}

hipError_t launch_strain(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    if (L.T.nblocks > 0) return strain_b<true, 4>(L, P, s);
    return L.lanes == 16 ? strain_b<false, 16>(L, P, s) : strain_b<false, 4>(L, P, s);
}

hipError_t launch_prep(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    if (L.T.nblocks > 0)
        hipLaunchKernelGGL(prep_kernel<true>, grid_plain(L), dim3(kBlock), 0, s, L.rec, L.dstress, L.balsara_in, L.perm,
                           (size_t)L.n, L.T, P);
    else
        hipLaunchKernelGGL(prep_kernel<false>, grid_plain(L), dim3(kBlock), 0, s, L.rec, L.dstress, L.balsara_in,
                           L.perm, (size_t)L.n, L.T, P);
    return hipGetLastError();
}

hipError_t launch_accel(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    if (L.T.nblocks > 0) return accel_b<true, 4>(L, P, s);
    return L.lanes == 16 ? accel_b<false, 16>(L, P, s) : accel_b<false, 4>(L, P, s);
}

hipError_t launch_finish(const NbrLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    if (L.T.nblocks > 0)
        hipLaunchKernelGGL(finish_kernel<true>, grid_plain(L), dim3(kBlock), 0, s, L.posm, L.vel, L.acc, L.xvel,
                           L.maxvsig, L.n, L.T, P);
    else
        hipLaunchKernelGGL(finish_kernel<false>, grid_plain(L), dim3(kBlock), 0, s, L.posm, L.vel, L.acc, L.xvel,
                           L.maxvsig, L.n, L.T, P);
    return hipGetLastError();
}

}  // namespace grasph
