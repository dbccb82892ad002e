// sweep.hip -- the one-sided O(N^2) sweeps (gfx950): gravity, and the
// potential of the invariants.
//
// Gravity sums the softened gravity of calcAcceleration
// (src/computeDerivatives.h:229-235) over every pair, in place of the tiled
// device loop do_for_each_pair_fast_impl (src/particles/algorithms.h:270-309);
// it serves the particle counts below the symmetric sweep's (sym_sweep.hip),
// the allocation-free entry point and, persistently, the smaller instances
// of a batch.  The neighbour lists come from lists.hip.
//
// The particle stream xs is in slot order: with a curve order the positions
// gathered as xs[t] = posm[perm[t]], without one posm itself.  Results go to
// particle perm[t].  The pair loop is own_block.hpp's: up to 16 wavefronts of
// a workgroup share 64 or 256 own slots and add their sums in LDS; with more
// shares than that, planes of workgroups write partial sums that a second
// kernel adds.  Sums are plain FP32 over blocks of 64 partners, then
// compensated (TwoSum).
//
// The batched kernel runs the same code persistently over a queue of work
// items (instance, 64 NI slots) ordered longest instance first; each
// wavefront takes the next item with one atomic add.
#include <algorithm>

#include "own_block.hpp"

namespace grasph {
namespace {

constexpr int kBlock = 256;
constexpr int kMassBlocks = 256;  // blocks of the single-instance mass check (flags after umass[0..1])

// Workgroup (own block blockIdx.x, plane blockIdx.y): its wavefronts' shares
// of slice_len partners start at plane * waves * slice_len.  One plane: the
// accelerations; several: the plane's partial sums (2 float4 per particle).
// SPLIT > 1 (one plane): SPLIT lanes per slot (own_split_block).
template <int NI, bool SOFT, int SPLIT>
__global__ __launch_bounds__(64 * kOwnMaxWaves) void own_kernel(const float4* __restrict__ xs,
                                                                const int* __restrict__ perm, const int n,
                                                                float4* __restrict__ acc, const int finish,
                                                                float4* __restrict__ xvel,
                                                                float* __restrict__ maxvsig, const DevParams P,
                                                                const int slice_len, float4* __restrict__ part,
                                                                const float* __restrict__ umass)
{
    extern __shared__ float lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = blockDim.x >> 6;
    const int o0 = 64 / SPLIT * NI * blockIdx.x, j0 = (int)blockIdx.y * waves * slice_len;
    float4* const pp = part ? part + 2 * (size_t)blockIdx.y * n : nullptr;
    auto store = [&](const int t, const CSum& x, const CSum& y, const CSum& z) {
        const int i = perm ? perm[t] : t;
        if (pp) {
            pp[2 * (size_t)i] = make_float4(x.s, y.s, z.s, 0.0f);
            pp[2 * (size_t)i + 1] = make_float4(x.c, y.c, z.c, 0.0f);
            return;
        }
        float ax = x.value(), ay = y.value(), az = z.value();
        if (finish) {
            environment_acceleration(P, ax, ay, az);
            if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (maxvsig) maxvsig[i] = 0.0f;
        }
        acc[i] = make_float4(ax, ay, az, 0.0f);
    };
    if constexpr (SPLIT > 1)  // one plane, no mass check
        own_split_block<SPLIT, SOFT>(xs, o0, n, slice_len, P.H2, wave, waves, lds, store);
    else if (umass && umass[0] != 0.0f)  // {uniform, mass} of the particles
        own_block<NI, true, SOFT>(xs, o0, n, j0, n, slice_len, P.H2, umass[1], wave, waves, lds, store);
    else
        own_block<NI, false, SOFT>(xs, o0, n, j0, n, slice_len, P.H2, 1.0f, wave, waves, lds, store);
}

// Without gravity: what a sweep's finish leaves (environment, zero xvel / maxvsig).
__global__ __launch_bounds__(kBlock) void no_gravity_kernel(const int n, float4* __restrict__ acc,
                                                            float4* __restrict__ xvel, float* __restrict__ maxvsig,
                                                            const DevParams P)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    environment_acceleration(P, ax, ay, az);
    if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (maxvsig) maxvsig[i] = 0.0f;
    acc[i] = make_float4(ax, ay, az, 0.0f);
}

// pot[i] = -sum_{j != i} m_j / sqrt(r^2 + H^2), one particle per lane: all
// lanes visit the same j, read with scalar loads in chunks of 8, two buffers
// in ping-pong.  Softened, the self pair is in the sum and is taken back
// where r^2, as the oracle rounds it, is 0 (cand: softened squared distance
// that every such pair stays below).
constexpr int kChunk = 8, kPotFold = 128;  // partners per plain partial sum
template <bool SOFT>
__device__ __forceinline__ void pot_chunk(const float4 (&pj)[kChunk], const float xi, const float yi, const float zi,
                                          float& phi, const float H2, const float cand)
{
    float d2[kChunk];
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
        const float dx = pj[c].x - xi, dy = pj[c].y - yi, dz = pj[c].z - zi;
        d2[c] = SOFT ? fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, H2))) : fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const float inv = __builtin_amdgcn_rsqf(d2[c]);
        phi += SOFT ? pj[c].w * inv : ((d2[c] > 0.0f) ? pj[c].w * inv : 0.0f);
    }
    if (SOFT) {
        float mn = d2[0];
#pragma unroll
        for (int c = 0; c < kChunk; ++c) mn = fminf(mn, d2[c]);
        if (mn <= cand) {
#pragma unroll
            for (int c = 0; c < kChunk; ++c)
                if (d2[c] <= cand && dist2_exact(xi - pj[c].x, yi - pj[c].y, zi - pj[c].z) == 0.0f)
                    phi -= pj[c].w * __builtin_amdgcn_rsqf(d2[c]);
        }
    }
}

template <bool SOFT>
__global__ __launch_bounds__(kBlock) void pot_kernel(const float4* __restrict__ posm, const int n,
                                                     float* __restrict__ pot, const float H2, const float cand)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const float4 p = posm[min(i, n - 1)];
    float phi = 0.0f;
    CSum sum{0.0f, 0.0f};
    const int nchunks = n / kChunk, nfull = nchunks * kChunk;
    float4 A[kChunk], B[kChunk];
    if (nchunks > 0) {
#pragma unroll
        for (int c = 0; c < kChunk; ++c) A[c] = posm[c];
    }
    auto fold = [&]() {
        sum.add(phi);
        phi = 0.0f;
    };
    int k = 0;
    for (; k + 1 < nchunks; k += 2) {
        const int jb = k * kChunk;
#pragma unroll
        for (int c = 0; c < kChunk; ++c) B[c] = posm[jb + kChunk + c];
        pot_chunk<SOFT>(A, p.x, p.y, p.z, phi, H2, cand);
        // next A: chunk k + 2, or chunk k + 1 again when k + 2 is past the end
        const int ja = ((k + 2 < nchunks) ? (k + 2) : (k + 1)) * kChunk;
#pragma unroll
        for (int c = 0; c < kChunk; ++c) A[c] = posm[ja + c];
        pot_chunk<SOFT>(B, p.x, p.y, p.z, phi, H2, cand);
        if (((k + 1) % (kPotFold / kChunk)) == kPotFold / kChunk - 1) fold();
    }
    if (k < nchunks) pot_chunk<SOFT>(A, p.x, p.y, p.z, phi, H2, cand);
    if (nfull < n) {  // the last partial chunk, padded with far-away massless partners
#pragma unroll
        for (int c = 0; c < kChunk; ++c)
            A[c] = (nfull + c < n) ? posm[nfull + c] : make_float4(3.0e18f, 3.0e18f, 3.0e18f, 0.0f);
        pot_chunk<SOFT>(A, p.x, p.y, p.z, phi, H2, cand);
    }
    fold();
    if (i < n) pot[i] = -sum.value();
}

// {1, m} when every particle of [off, off + n) has mass m (bit for bit),
// else {0, m}; one block per instance (blockIdx.x; insts null: one instance
// [0, n)).  Written every evaluation, so no reset is needed.
__global__ __launch_bounds__(1024) void mass_check_kernel(const float4* __restrict__ posm,
                                                          const BatchInst* __restrict__ insts, const int n,
                                                          float* __restrict__ umass)
{
    const int k = blockIdx.x;
    const int off = insts ? insts[k].off : 0, cnt = insts ? insts[k].n : n;
    if (cnt <= 0) {
        if (threadIdx.x == 0) { umass[2 * k] = 0.0f; umass[2 * k + 1] = 0.0f; }
        return;  // the whole block leaves: no barrier below is reached
    }
    const float m0 = posm[off].w;
    int bad = 0;
    // eight loads in flight per thread (one at a time, each waited for
    // before the next, 16384 masses took 7 us)
    int i = threadIdx.x;
    for (; i + 7 * (int)blockDim.x < cnt; i += 8 * (int)blockDim.x) {
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) w[u] = posm[off + i + u * (int)blockDim.x].w;
#pragma unroll
        for (int u = 0; u < 8; ++u) bad |= __float_as_int(w[u]) != __float_as_int(m0);
    }
    for (; i < cnt; i += blockDim.x) bad |= __float_as_int(posm[off + i].w) != __float_as_int(m0);
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
        umass[2 * k] = bad ? 0.0f : 1.0f;
        umass[2 * k + 1] = m0;
    }
}

// The same check for one large instance: block b flags a mismatch in its
// grid-stride share, then one block folds the flags (every flag is written
// each time, so nothing needs clearing).
__global__ __launch_bounds__(kBlock) void mass_partial_kernel(const float4* __restrict__ posm, const int n,
                                                              int* __restrict__ partial)
{
    const float m0 = posm[0].w;
    int bad = 0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        bad |= __float_as_int(posm[i].w) != __float_as_int(m0);
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) partial[blockIdx.x] = bad;
}

__global__ __launch_bounds__(kBlock) void mass_final_kernel(const float4* __restrict__ posm,
                                                            const int* __restrict__ partial, const int nparts,
                                                            float* __restrict__ umass)
{
    int bad = 0;
    for (int b = threadIdx.x; b < nparts; b += kBlock) bad |= partial[b];
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
        umass[0] = bad ? 0.0f : 1.0f;
        umass[1] = posm[0].w;
    }
}

// Sum the planes' partial gravity in plane order (compensated) and finish
// the acceleration as a one-plane sweep would.
__global__ __launch_bounds__(64) void combine_kernel(const float4* __restrict__ part, const int nplanes, const int n,
                                                     float4* __restrict__ acc, const int finish,
                                                     float4* __restrict__ xvel, float* __restrict__ maxvsig,
                                                     const DevParams P)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
#pragma unroll 8
    for (int s = 0; s < nplanes; ++s) {
        const float4 a = part[2 * ((size_t)s * n + i)], c = part[2 * ((size_t)s * n + i) + 1];
        x.add(a.x); y.add(a.y); z.add(a.z);
        x.c += c.x; y.c += c.y; z.c += c.z;
    }
    float ax = x.value(), ay = y.value(), az = z.value();
    if (finish) {
        environment_acceleration(P, ax, ay, az);
        if (xvel) xvel[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (maxvsig) maxvsig[i] = 0.0f;
    }
    acc[i] = make_float4(ax, ay, az, 0.0f);
}

// Persistent sweep over a batch of independent instances.  Item w =
// (inst, slot0, ni) covers slots [slot0, slot0 + 64 ni) of instance inst
// with ni particles per lane (chosen per size bucket) against all of the
// instance's particles [off, off + n); its slots are the same range of perm.
// A wavefront's first item is its own number, the next come from the counter
// (2000 instances of 50: 134 us a derivative call with the first from there
// too); it leaves the loop past n_items.  NIMAX
// is the largest ni of the items.
template <int NIMAX, bool SOFT>
__global__ __launch_bounds__(kBlock) void batch_sweep_kernel(const float4* __restrict__ xs,
                                                             const int* __restrict__ perm,
                                                             const int4* __restrict__ items, const int n_items,
                                                             const BatchInst* __restrict__ insts,
                                                             int* __restrict__ queue, float4* __restrict__ acc,
                                                             const float* __restrict__ umass)
{
    __shared__ float lds[own_lds_floats(1, 1) * (kBlock / 64)];
    float* const tile = lds + own_lds_floats(1, 1) * (threadIdx.x >> 6);  // one wavefront's
    auto store = [&](const int t, const CSum& x, const CSum& y, const CSum& z) {
        acc[perm ? perm[t] : t] = make_float4(x.value(), y.value(), z.value(), 0.0f);
    };
    const int waves = (int)(gridDim.x * blockDim.x) >> 6;
    int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    while (w < n_items) {
        const int4 it = items[w];
        const BatchInst I = insts[it.x];
        const int e = I.off + I.n;
        const bool um = I.n >= kMassCheckMin && umass[2 * it.x] != 0.0f;  // as one instance
        const float m = umass[2 * it.x + 1];
        if (NIMAX == 2 && it.z == 2) {
            if (um)
                own_block<NIMAX, true, SOFT>(xs, it.y, e, I.off, e, I.n, I.H2, m, 0, 1, tile, store);
            else
                own_block<NIMAX, false, SOFT>(xs, it.y, e, I.off, e, I.n, I.H2, 1.0f, 0, 1, tile, store);
        } else if (um) {
            own_block<1, true, SOFT>(xs, it.y, e, I.off, e, I.n, I.H2, m, 0, 1, tile, store);
        } else {
            own_block<1, false, SOFT>(xs, it.y, e, I.off, e, I.n, I.H2, 1.0f, 0, 1, tile, store);
        }
        if (waves >= n_items) break;
        w = 0;
        if ((threadIdx.x & 63) == 0) w = atomicAdd(queue, 1);
        w = __builtin_amdgcn_readfirstlane(w) + waves;
    }
}

// Zero the work counters of the batched sweep (a kernel, so that a captured
// graph holds no memset node).
__global__ void reset_queue_kernel(int* __restrict__ queue, const int n)
{
    const int i = threadIdx.x;
    if (i < n) queue[i] = 0;
}

template <int NI, bool SOFT, int SPLIT = 1>
hipError_t launch_own(const SweepLaunch& L, const DevParams& P, hipStream_t s)
{
    constexpr int kSlots = 64 / SPLIT * NI;  // of a workgroup
    const dim3 grid((unsigned)((L.n + kSlots - 1) / kSlots), (unsigned)L.planes);
    const int lds = own_lds_floats(NI, SPLIT > 1 ? std::max(L.waves, 2) : L.waves);
    hipLaunchKernelGGL((own_kernel<NI, SOFT, SPLIT>), grid, dim3(64 * L.waves), sizeof(float) * lds, s, L.xs ? L.xs : L.posm, L.perm, L.n, L.acc, L.finish ? 1 : 0, L.xvel, L.maxvsig, P,
                       L.slice_len, L.planes > 1 ? L.part : nullptr, L.umass);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || L.planes == 1) return e;
    hipLaunchKernelGGL(combine_kernel, dim3((L.n + 63) / 64), dim3(64), 0, s, L.part, L.planes, L.n, L.acc,
                       L.finish ? 1 : 0, L.xvel, L.maxvsig, P);
    return hipGetLastError();
}

template <bool SOFT>
hipError_t launch_b(const BatchSweepLaunch& L, hipStream_t s)
{
    const int blocks = std::min(L.blocks, (L.n_items + L.waves_per_block - 1) / L.waves_per_block);
    if (L.ni_max == 2)
        hipLaunchKernelGGL((batch_sweep_kernel<2, SOFT>), dim3(blocks), dim3(64 * L.waves_per_block), 0, s, L.xs,
                           L.perm, L.items, L.n_items, L.insts, L.queue, L.acc, L.umass);
    else
        hipLaunchKernelGGL((batch_sweep_kernel<1, SOFT>), dim3(blocks), dim3(64 * L.waves_per_block), 0, s, L.xs,
                           L.perm, L.items, L.n_items, L.insts, L.queue, L.acc, L.umass);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_sweep(const SweepLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    const bool soft = P.H2 > 0.0f;
    if (L.want_pot) {
        const dim3 grid((L.n + kBlock - 1) / kBlock);
        if (soft)
            hipLaunchKernelGGL(pot_kernel<true>, grid, dim3(kBlock), 0, s, L.posm, L.n, L.pot, P.H2, P.cand);
        else
            hipLaunchKernelGGL(pot_kernel<false>, grid, dim3(kBlock), 0, s, L.posm, L.n, L.pot, P.H2, P.cand);
        return hipGetLastError();
    }
    if (!L.grav) {
        if (L.finish)
            hipLaunchKernelGGL(no_gravity_kernel, dim3((L.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, L.n, L.acc,
                               L.xvel, L.maxvsig, P);
        return hipGetLastError();
    }
    if (L.waves < 1 || L.waves > kOwnMaxWaves || L.planes < 1 || L.slice_len < 8 || L.slice_len % 8)
        return hipErrorInvalidValue;
    if (L.split != 1 && (L.split != kOwnSplit || L.ni != 1 || L.planes != 1 || L.umass)) return hipErrorInvalidValue;
    if (L.split != 1) return soft ? launch_own<1, true, kOwnSplit>(L, P, s) : launch_own<1, false, kOwnSplit>(L, P, s);
    switch (L.ni) {
        case 1: return soft ? launch_own<1, true>(L, P, s) : launch_own<1, false>(L, P, s);
        case 2: return soft ? launch_own<2, true>(L, P, s) : launch_own<2, false>(L, P, s);
        case 4: return soft ? launch_own<4, true>(L, P, s) : launch_own<4, false>(L, P, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_mass_check(const float4* posm, const BatchInst* insts, int n_inst, int n, float* umass,
                             hipStream_t s)
{
    if (n_inst <= 0) return hipSuccess;
    if (!insts && n > 16384) {  // one large instance: spread the scan over blocks, then fold their flags
        const int blocks = std::min(kMassBlocks, (n + 4095) / 4096);
        int* partial = (int*)(umass + 2);
        hipLaunchKernelGGL(mass_partial_kernel, dim3(blocks), dim3(kBlock), 0, s, posm, n, partial);
        hipLaunchKernelGGL(mass_final_kernel, dim3(1), dim3(kBlock), 0, s, posm, partial, blocks, umass);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(mass_check_kernel, dim3(n_inst), dim3(1024), 0, s, posm, insts, n, umass);
    return hipGetLastError();
}

hipError_t launch_mass_final(const float4* posm, const int* mass_flags, int nflags, float* umass, hipStream_t s)
{
    if (nflags <= 0) return hipSuccess;
    hipLaunchKernelGGL(mass_final_kernel, dim3(1), dim3(kBlock), 0, s, posm, mass_flags, nflags, umass);
    return hipGetLastError();
}

hipError_t launch_reset_queue(int* queue, int n, hipStream_t s)
{
    hipLaunchKernelGGL(reset_queue_kernel, dim3(1), dim3(64), 0, s, queue, n);
    return hipGetLastError();
}

hipError_t launch_batch_sweep(const BatchSweepLaunch& L, hipStream_t s)
{
    if (L.n_items <= 0) return hipSuccess;
    if (L.waves_per_block < 1 || L.waves_per_block > kBlock / 64) return hipErrorInvalidValue;
    if (L.ni_max != 1 && L.ni_max != 2) return hipErrorInvalidValue;
    return L.soft ? launch_b<true>(L, s) : launch_b<false>(L, s);
}

}  // namespace grasph
