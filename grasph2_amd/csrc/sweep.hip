// sweep.hip -- the one-sided O(N^2) gravity sweep (gfx950).
//
// It sums the softened gravity of calcAcceleration
// (src/computeDerivatives.h:229-235) over every pair, in place of the tiled
// device loop do_for_each_pair_fast_impl (src/particles/algorithms.h:270-309),
// or the potential.  The neighbour lists come from lists.hip.
//
// Mapping: NI i particles per lane (slots t and t + 64 for NI = 2).  The
// particle stream xs is in slot order: with a Morton order the positions
// gathered as xs[t] = posm[perm[t]], without one posm itself.  Results go to
// particle perm[t].  All lanes visit the same j at the same time, so the j
// stream (float4 x,y,z,m) is read with scalar loads into SGPRs -- no LDS, no
// barriers -- in chunks of 8, two SGPR buffers in ping-pong so the next
// chunk loads while this one computes.
// Per pair: 3 sub, 3 FMA for r^2 + H^2, one v_rsq_f32, 2 mul (3 with
// unequal masses), 3 FMA (a second transcendental per pair in place of a
// multiply, rsqrt * rcp, measured 12% slower).  Sums are plain FP32 over
// blocks of 128 j, then compensated (TwoSum) into the running total.
//
// The batched kernel runs the same code persistently over a queue of work
// items (instance, 64 NI slots) ordered longest instance first; each
// wavefront takes the next item with one atomic add.
#include <algorithm>

#include "sweep_core.hpp"

namespace grasph {
namespace {

constexpr int kMassBlocks = 256;  // blocks of the single-instance mass check (flags after umass[0..1])

template <int NI, bool GRAV, bool POT, bool SOFT>
__global__ __launch_bounds__(kBlock) void sweep_kernel(const float4* __restrict__ xs, const int* __restrict__ perm,
                                                       const int n, float4* __restrict__ acc,
                                                       float* __restrict__ pot, const int finish,
                                                       const float4* __restrict__ vel, float4* __restrict__ xvel,
                                                       float* __restrict__ maxvsig, const DevParams P,
                                                       const int slice_len, float4* __restrict__ part,
                                                       const float* __restrict__ umass)
{
    const int wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    const int s0 = wave * 64 * NI + lane;
    // slice blockIdx.y of the j range
    const int sl = blockIdx.y;
    const int j0 = sl * slice_len;
    int j1 = min(n, j0 + slice_len);
    if (!(GRAV || POT)) j1 = j0;  // nothing pairwise to do: skip the j loop
    float4* const pp = part ? part + 2 * (size_t)sl * n : nullptr;
    if constexpr (GRAV && !POT) {
        if (umass && umass[0] != 0.0f) {  // {uniform, mass} of the partners, wave-uniform
            sweep_slots<NI, GRAV, POT, SOFT, true>(xs, perm, s0, n, j0, j1, acc, pot, finish, vel, xvel, maxvsig, P,
                                                   P.H2, P.cand, umass[1], pp);
            return;
        }
    }
    sweep_slots<NI, GRAV, POT, SOFT, false>(xs, perm, s0, n, j0, j1, acc, pot, finish, vel, xvel, maxvsig, P, P.H2,
                                            P.cand, 1.0f, pp);
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

// Sum the slices' partial gravity in slice order (compensated) and finish
// the acceleration as a one-slice sweep would.
__global__ __launch_bounds__(kBlock) void combine_kernel(const float4* __restrict__ part, const int nslices,
                                                         const int n, const float4* __restrict__ posm,
                                                         float4* __restrict__ acc, const int finish,
                                                         const float4* __restrict__ vel, float4* __restrict__ xvel,
                                                         float* __restrict__ maxvsig, const DevParams P)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    CSum x{0.0f, 0.0f}, y{0.0f, 0.0f}, z{0.0f, 0.0f};
    for (int s = 0; s < nslices; ++s) {
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
// with ni particles per lane (chosen per size bucket); the instance's
// particles are [off, off + n) and its slots are the same range of perm.
// Every wavefront leaves the loop once the counter passes n_items.  NIMAX
// is the largest ni of the items: the two-per-lane code needs about twice
// the registers, so a batch without such items gets the leaner kernel.
template <int NIMAX, bool SOFT>
__global__ __launch_bounds__(kBlock) void batch_sweep_kernel(const float4* __restrict__ xs,
                                                             const int* __restrict__ perm,
                                                             const int4* __restrict__ items, const int n_items,
                                                             const BatchInst* __restrict__ insts,
                                                             int* __restrict__ queue, float4* __restrict__ acc,
                                                             const DevParams P, const float* __restrict__ umass)
{
    const int lane = threadIdx.x & 63;
    for (;;) {
        int w = 0;
        if (lane == 0) w = atomicAdd(queue, 1);
        w = __builtin_amdgcn_readfirstlane(w);
        if (w >= n_items) break;
        const int4 it = items[w];
        const BatchInst I = insts[it.x];
        const int s0 = it.y + lane, e = I.off + I.n;
        const bool um = umass && umass[2 * it.x] != 0.0f;
        const float m = um ? umass[2 * it.x + 1] : 1.0f;
        if (um) {
            if (NIMAX == 2 && it.z == 2)
                sweep_slots<NIMAX, true, false, SOFT, true>(xs, perm, s0, e, I.off, e, acc, nullptr, 0, nullptr,
                                                            nullptr, nullptr, P, I.H2, 0.0f, m);
            else
                sweep_slots<1, true, false, SOFT, true>(xs, perm, s0, e, I.off, e, acc, nullptr, 0, nullptr, nullptr,
                                                        nullptr, P, I.H2, 0.0f, m);
        } else if (NIMAX == 2 && it.z == 2) {
            sweep_slots<NIMAX, true, false, SOFT, false>(xs, perm, s0, e, I.off, e, acc, nullptr, 0, nullptr, nullptr,
                                                         nullptr, P, I.H2, 0.0f, m);
        } else {
            sweep_slots<1, true, false, SOFT, false>(xs, perm, s0, e, I.off, e, acc, nullptr, 0, nullptr, nullptr,
                                                     nullptr, P, I.H2, 0.0f, m);
        }
    }
}

// Zero the work counters of the batched sweep (a kernel, so that a captured
// graph holds no memset node).
__global__ void reset_queue_kernel(int* __restrict__ queue, const int n)
{
    const int i = threadIdx.x;
    if (i < n) queue[i] = 0;
}

template <int NI, bool GRAV, bool POT, bool SOFT>
hipError_t launch_t(const SweepLaunch& L, const DevParams& P, hipStream_t s)
{
    const int waves = (L.n + 64 * NI - 1) / (64 * NI);
    const int blocks = (waves + kBlock / 64 - 1) / (kBlock / 64);
    const int ns = L.nslices > 1 ? L.nslices : 1;
    hipLaunchKernelGGL((sweep_kernel<NI, GRAV, POT, SOFT>), dim3(blocks, ns), dim3(kBlock), 0, s,
                       L.xs ? L.xs : L.posm, L.perm, L.n, L.acc, L.pot, L.finish ? 1 : 0, L.vel, L.xvel, L.maxvsig, P,
                       ns > 1 ? L.slice_len : L.n, ns > 1 ? L.part : nullptr, L.umass);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ns == 1 || !(GRAV || L.finish)) return e;
    hipLaunchKernelGGL(combine_kernel, dim3((L.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, L.part, ns, L.n, L.posm,
                       L.acc, L.finish ? 1 : 0, L.vel, L.xvel, L.maxvsig, P);
    return hipGetLastError();
}

template <int NI>
hipError_t launch_ni(const SweepLaunch& L, const DevParams& P, hipStream_t s)
{
    const bool soft = P.H2 > 0.0f;
    const int key = (L.grav ? 4 : 0) | (L.want_pot ? 2 : 0) | (soft ? 1 : 0);
    switch (key) {
        case 0: return launch_t<NI, false, false, false>(L, P, s);
        case 1: return launch_t<NI, false, false, true>(L, P, s);
        case 2: return launch_t<NI, false, true, false>(L, P, s);
        case 3: return launch_t<NI, false, true, true>(L, P, s);
        case 4: return launch_t<NI, true, false, false>(L, P, s);
        case 5: return launch_t<NI, true, false, true>(L, P, s);
        default: return hipErrorInvalidValue;  // the potential sweep runs alone
    }
}

template <bool SOFT>
hipError_t launch_b(const BatchSweepLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.ni_max == 2)
        hipLaunchKernelGGL((batch_sweep_kernel<2, SOFT>), dim3(L.blocks), dim3(64 * L.waves_per_block), 0, s, L.xs,
                           L.perm, L.items, L.n_items, L.insts, L.queue, L.acc, P, L.umass);
    else
        hipLaunchKernelGGL((batch_sweep_kernel<1, SOFT>), dim3(L.blocks), dim3(64 * L.waves_per_block), 0, s, L.xs,
                           L.perm, L.items, L.n_items, L.insts, L.queue, L.acc, P, L.umass);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_sweep(const SweepLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n <= 0) return hipSuccess;
    return L.ni == 2 ? launch_ni<2>(L, P, s) : launch_ni<1>(L, P, s);
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

hipError_t launch_batch_sweep(const BatchSweepLaunch& L, const DevParams& P, hipStream_t s)
{
    if (L.n_items <= 0) return hipSuccess;
    if (L.waves_per_block < 1 || L.waves_per_block > kBlock / 64) return hipErrorInvalidValue;
    if (L.ni_max != 1 && L.ni_max != 2) return hipErrorInvalidValue;
    return L.soft ? launch_b<true>(L, P, s) : launch_b<false>(L, P, s);
}

}  // namespace grasph
