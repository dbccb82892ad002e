// reorder.hip -- Hilbert-curve ordering of the particles (gfx950).
//
// The list kernel and the neighbour passes map slot t to particle perm[t] and
// read the particles through slot-ordered copies (gather_kernel: positions,
// velocities, densities).  Along a space-filling curve consecutive slots are
// spatial neighbours, so the 64 lanes of a wavefront share most of their SPH
// partners, the boxes of consecutive slots are small (lists.hip), and the
// list passes' gathers of neighbour data hit the same cache lines.  The order
// changes the summation order of the (compensated) sums, not which pairs are
// summed.
//
// Hilbert's curve, on cubic cells, rather than Morton's on the bounding box's
// own proportions: it has no jumps inside the particles.  Two spheres of 8192,
// H = 2.5 spacings: a box of 8 slots comes within H of 51 others instead of
// 90, and 1.5% of them instead of 10% are longer than 2 H.
#include <rocprim/device/device_radix_sort.hpp>

#include "internal.hpp"

namespace grasph {
namespace {

constexpr int kBlock = 256;
constexpr int kBoxBlocks = 256;
// counts up to this are ordered by rank (rank_kernel), larger ones by a sort
constexpr int kRankMax = 16384;

__global__ __launch_bounds__(kBlock) void bbox_partial(const float4* __restrict__ posm, const int n,
                                                       float* __restrict__ part)
{
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const float4 p = posm[i];
        mn[0] = fminf(mn[0], p.x); mn[1] = fminf(mn[1], p.y); mn[2] = fminf(mn[2], p.z);
        mx[0] = fmaxf(mx[0], p.x); mx[1] = fmaxf(mx[1], p.y); mx[2] = fmaxf(mx[2], p.z);
    }
    __shared__ float sh[6][kBlock];
    for (int d = 0; d < 3; ++d) {
        sh[d][threadIdx.x] = mn[d];
        sh[3 + d][threadIdx.x] = mx[d];
    }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int d = 0; d < 3; ++d) {
                sh[d][threadIdx.x] = fminf(sh[d][threadIdx.x], sh[d][threadIdx.x + s]);
                sh[3 + d][threadIdx.x] = fmaxf(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = sh[threadIdx.x][0];
}

// the boxes of a block's threads folded into one, in every thread
template <int THREADS>
__device__ __forceinline__ void bbox_fold(float (&box)[6])
{
    __shared__ float sh[6][THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            const float o = __shfl_xor(box[d], off, 64);
            box[d] = (d < 3) ? fminf(box[d], o) : fmaxf(box[d], o);
        }
    if (lane == 0)
#pragma unroll
        for (int d = 0; d < 6; ++d) sh[d][w] = box[d];
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 6; ++d)
        for (int q = 0; q < THREADS / 64; ++q) box[d] = (d < 3) ? fminf(box[d], sh[d][q]) : fmaxf(box[d], sh[d][q]);
}

__device__ inline uint32_t spread10(uint32_t v)
{
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// place along the Hilbert curve of a cell of the 1024^3 grid (J. Skilling,
// "Programming the Hilbert curve", AIP Conf. Proc. 707 (2004) 381: from the
// axes to the transposed index, whose bits then interleave)
__device__ inline uint32_t hilbert_index(uint32_t x, uint32_t y, uint32_t z)
{
    uint32_t c[3] = {x, y, z};
    for (uint32_t q = 512; q > 1; q >>= 1) {
        const uint32_t low = q - 1;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const uint32_t t = (c[0] ^ c[d]) & low;
            if (c[d] & q) {
                c[0] ^= low;
            } else {
                c[0] ^= t;
                c[d] ^= t;
            }
        }
    }
    c[1] ^= c[0];
    c[2] ^= c[1];
    uint32_t t = 0;
    for (uint32_t q = 512; q > 1; q >>= 1)
        if (c[2] & q) t ^= q - 1;
    return (spread10(c[0] ^ t) << 2) | (spread10(c[1] ^ t) << 1) | spread10(c[2] ^ t);
}

// p's place along the curve through the box {lo xyz, hi xyz}.  The cells are
// cubes of a 1024th of the longest side; across a side less than an eighth of
// it they are finer (bodies far apart keep their resolution across the line
// between them).
__device__ inline uint32_t curve_key(const float4 p, const float* box)
{
    const float c[3] = {p.x, p.y, p.z};
    float ext[3], longest = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        ext[d] = box[3 + d] - box[d];
        longest = fmaxf(longest, ext[d]);
    }
    uint32_t q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float side = fminf(longest, 8.0f * ext[d]);
        float u = (side > 0.0f) ? (c[d] - box[d]) / side : 0.0f;
        if (!(u >= 0.0f)) u = 0.0f;  // NaN and negatives
        if (u > 1.0f) u = 1.0f;
        q[d] = (uint32_t)(u * 1023.0f);
    }
    return hilbert_index(q[0], q[1], q[2]);
}

// keys of the particles from the nparts (<= kBlock) block boxes
__global__ __launch_bounds__(kBlock) void curve_keys(const float4* __restrict__ posm, const int n,
                                                     const float* __restrict__ part, const int nparts,
                                                     uint32_t* __restrict__ keys, int* __restrict__ vals)
{
    const int i = blockIdx.x * kBlock + threadIdx.x, b = threadIdx.x;
    const float4 p = posm[min(i, n - 1)];
    float box[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) box[d] = (b < nparts) ? part[b * 6 + d] : ((d < 3) ? INFINITY : -INFINITY);
    bbox_fold<kBlock>(box);
    if (i >= n) return;
    keys[i] = curve_key(p, box);
    vals[i] = i;
}

// keys of up to kRankMax particles in one launch: every workgroup finds the
// whole bounding box for itself (256 KiB of positions from L2 at most)
constexpr int kRankThreads = 1024;
__global__ __launch_bounds__(kRankThreads) void rank_keys(const float4* __restrict__ posm, const int n,
                                                          uint32_t* __restrict__ keys)
{
    const int i = blockIdx.x * kRankThreads + threadIdx.x;
    float box[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll 4
    for (int j = threadIdx.x; j < n; j += kRankThreads) {
        const float4 p = posm[j];
        box[0] = fminf(box[0], p.x); box[1] = fminf(box[1], p.y); box[2] = fminf(box[2], p.z);
        box[3] = fmaxf(box[3], p.x); box[4] = fmaxf(box[4], p.y); box[5] = fmaxf(box[5], p.z);
    }
    const float4 p = posm[min(i, n - 1)];
    bbox_fold<kRankThreads>(box);
    if (i < n) keys[i] = curve_key(p, box);
}

// The order of up to kRankMax particles, without a sort: particle i's slot is
// the number of particles before it on the curve, those with a smaller key
// and, of its own key, those with a smaller index.  A workgroup counts for 32
// particles: its half wavefronts 1/32 of the keys each, a particle per lane,
// all lanes of a half reading the same keys from LDS, four at a time.  The
// sign of (key j - limit) is shifted into a word that a population count
// adds up every 32 keys: two plain vector instructions a pair (a compare and
// an add with its carry take twice the clocks).  Rank, keys and bounding box
// in two launches: allocation-free SPH step at 1000 particles 61.9 -> 56.2 us,
// 8192 108 -> 92, 16384 167 -> 164; past kRankMax the sort is the faster one.
constexpr int kRankWaves = 16, kRankOwn = 32;              // particles of a workgroup
constexpr int kRankShares = 64 / kRankOwn * kRankWaves;    // shares of the keys
__global__ __launch_bounds__(64 * kRankWaves) void rank_kernel(const uint32_t* __restrict__ keys, const int n,
                                                               int* __restrict__ perm)
{
    __shared__ __attribute__((aligned(16))) uint32_t all[kRankMax];
    __shared__ int part[kRankShares][kRankOwn];
    const int own = threadIdx.x % kRankOwn, share = threadIdx.x / kRankOwn;
    const int i0 = kRankOwn * blockIdx.x, i = i0 + own;
    const uint32_t key = keys[min(i, n - 1)];
    const int blocks = (n + kRankOwn - 1) / kRankOwn;  // of as many keys; the shares take whole ones
    for (int j = threadIdx.x; j < blocks * kRankOwn; j += 64 * kRankWaves)
        all[j] = j < n ? keys[j] : 0x40000000u;  // past the end: after every key of 30 bits
    __syncthreads();
    const int b0 = blocks * share / kRankShares, b1 = blocks * (share + 1) / kRankShares;
    int before = 0;
    for (int b = b0; b < b1; ++b) {
        uint32_t less = 0;
        const uint4* const k4 = reinterpret_cast<const uint4*>(all + kRankOwn * b);
        if (b == (int)blockIdx.x) {  // its own block
#pragma unroll
            for (int u = 0; u < kRankOwn / 4; ++u) {
                const uint4 k = k4[u];
                less = __builtin_amdgcn_alignbit(less, k.x - key - (4 * u + 0 < own ? 1u : 0u), 31);
                less = __builtin_amdgcn_alignbit(less, k.y - key - (4 * u + 1 < own ? 1u : 0u), 31);
                less = __builtin_amdgcn_alignbit(less, k.z - key - (4 * u + 2 < own ? 1u : 0u), 31);
                less = __builtin_amdgcn_alignbit(less, k.w - key - (4 * u + 3 < own ? 1u : 0u), 31);
            }
        } else {
            const uint32_t limit = key + (b < (int)blockIdx.x ? 1u : 0u);
#pragma unroll
            for (int u = 0; u < kRankOwn / 4; ++u) {
                const uint4 k = k4[u];
                less = __builtin_amdgcn_alignbit(less, k.x - limit, 31);
                less = __builtin_amdgcn_alignbit(less, k.y - limit, 31);
                less = __builtin_amdgcn_alignbit(less, k.z - limit, 31);
                less = __builtin_amdgcn_alignbit(less, k.w - limit, 31);
            }
        }
        before += __builtin_popcount(less);
    }
    part[share][own] = before;
    __syncthreads();
    if (share != 0 || i >= n) return;
#pragma unroll
    for (int w = 1; w < kRankShares; ++w) before += part[w][own];
    perm[before] = i;
}

// one block per instance: bounding box of its particles
__global__ __launch_bounds__(kBlock) void batch_bbox(const float4* __restrict__ posm,
                                                     const BatchInst* __restrict__ insts, float* __restrict__ box)
{
    const BatchInst I = insts[blockIdx.x];
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = I.off + threadIdx.x; i < I.off + I.n; i += kBlock) {
        const float4 p = posm[i];
        mn[0] = fminf(mn[0], p.x); mn[1] = fminf(mn[1], p.y); mn[2] = fminf(mn[2], p.z);
        mx[0] = fmaxf(mx[0], p.x); mx[1] = fmaxf(mx[1], p.y); mx[2] = fmaxf(mx[2], p.z);
    }
    __shared__ float sh[6][kBlock];
    for (int d = 0; d < 3; ++d) {
        sh[d][threadIdx.x] = mn[d];
        sh[3 + d][threadIdx.x] = mx[d];
    }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int d = 0; d < 3; ++d) {
                sh[d][threadIdx.x] = fminf(sh[d][threadIdx.x], sh[d][threadIdx.x + s]);
                sh[3 + d][threadIdx.x] = fmaxf(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) box[blockIdx.x * 6 + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(kBlock) void batch_keys(const float4* __restrict__ posm, const int* __restrict__ inst_of,
                                                     const int n, const float* __restrict__ box,
                                                     uint64_t* __restrict__ keys, int* __restrict__ vals)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int k = inst_of[i];
    keys[i] = ((uint64_t)k << 30) | (uint64_t)curve_key(posm[i], box + 6 * k);
    vals[i] = i;
}

// slot-ordered copies: xs[t] = posm[perm[t]] (when xs is given) and the
// slot records' {x y z m} and {vx vy vz rho}; with mass_flags, also the
// first half of the equal-mass check: flag b is set when a mass of block b
// differs from particle 0's, bit for bit; with fine, also the lists' boxes
// (in a kernel of their own they took 5 us at any size); with ts_next, the
// variable step's next dt := ts_max (a launch of its own: default solids at
// 16384 particles 99.3 us a step, now 97.7)
__global__ __launch_bounds__(kGatherBlock) void gather_kernel(
    const int* __restrict__ perm, const int n, const float4* __restrict__ posm, const float4* __restrict__ vel,
    const float* __restrict__ density, float4* __restrict__ xs, SlotRec* __restrict__ rec,
    int* __restrict__ mass_flags, float4* __restrict__ fine, float4* __restrict__ mid,
    float4* __restrict__ coarse, int* __restrict__ list_max, float* __restrict__ ts_next, const float ts_max)
{
    const int t = blockIdx.x * kGatherBlock + threadIdx.x;
    int bad = 0;
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t < n) {
        const int i = perm ? perm[t] : t;
        p = posm[i];
        if (xs) xs[t] = p;
        if (rec) {
            const float4 v = vel ? vel[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            rec[t].pm = p;
            rec[t].vr = make_float4(v.x, v.y, v.z, density ? density[i] : 0.0f);
        }
        if (mass_flags) bad = __float_as_int(p.w) != __float_as_int(posm[0].w);
    }
    if (list_max && t == 0) *list_max = 0;
    if (ts_next && t == 0) *ts_next = ts_max;
    if (mass_flags) {  // uniform: the whole workgroup reaches the barrier
        bad = __syncthreads_or(bad);
        if (threadIdx.x == 0) mass_flags[blockIdx.x] = bad;
    }
    if (fine) block_boxes(p, t < n, blockIdx.x * kGatherBlock, n, fine, mid, coarse);
}

}  // namespace

hipError_t launch_gather(const int* perm, int n, const float4* posm, const float4* vel, const float* density,
                         float4* xs, SlotRec* rec, hipStream_t s, int* mass_flags, float4* fine, float4* mid,
                         float4* coarse, int* list_max, float* ts_next, float ts_max)
{
    if (n <= 0) return hipSuccess;
    if (!posm || (xs && !perm) || (fine && !(mid && coarse))) return hipErrorInvalidValue;
    static_assert(kGatherBlock == kBoxCoarse, "a workgroup of the gather makes one coarse box");
    hipLaunchKernelGGL(gather_kernel, dim3((n + kGatherBlock - 1) / kGatherBlock), dim3(kGatherBlock), 0, s, perm, n,
                       posm, vel, density, xs, rec, mass_flags, fine, mid, coarse, list_max, ts_next, ts_max);
    return hipGetLastError();
}

size_t batch_order_tmp_bytes(int ntotal, int key_bits)
{
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (int*)nullptr,
                                    (int*)nullptr, ntotal, 0u, (unsigned)key_bits, (hipStream_t)0);
    return bytes;
}

hipError_t launch_batch_order(const BatchOrder& B, hipStream_t s)
{
    if (B.ntotal <= 0 || B.n_inst <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_bbox, dim3(B.n_inst), dim3(kBlock), 0, s, B.posm, B.insts, B.bbox);
    hipLaunchKernelGGL(batch_keys, dim3((B.ntotal + kBlock - 1) / kBlock), dim3(kBlock), 0, s, B.posm, B.inst_of,
                       B.ntotal, B.bbox, B.keys, B.vals);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t bytes = B.sort_tmp_bytes;
    return rocprim::radix_sort_pairs(B.sort_tmp, bytes, B.keys, B.keys_alt, B.vals, B.perm, B.ntotal, 0u,
                                     (unsigned)B.key_bits, s);
}

size_t reorder_tmp_bytes(int n)
{
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, (uint32_t*)nullptr, (uint32_t*)nullptr, (int*)nullptr,
                                    (int*)nullptr, n, 0u, 30u, (hipStream_t)0);
    return bytes;
}

hipError_t launch_reorder(const float4* posm, int n, Ctx& c, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (n <= kRankMax) {
        hipLaunchKernelGGL(rank_keys, dim3((n + kRankThreads - 1) / kRankThreads), dim3(kRankThreads), 0, s, posm, n,
                           c.keys);
        hipLaunchKernelGGL(rank_kernel, dim3((n + kRankOwn - 1) / kRankOwn), dim3(64 * kRankWaves), 0, s, c.keys, n,
                           c.perm);
        return hipGetLastError();
    }
    const int blocks = (n + kBlock - 1) / kBlock, parts = std::min(blocks, kBoxBlocks);
    static_assert(kBoxBlocks <= kBlock, "curve_keys folds at most one box per thread");
    hipLaunchKernelGGL(bbox_partial, dim3(parts), dim3(kBlock), 0, s, posm, n, c.bbox);
    hipLaunchKernelGGL(curve_keys, dim3(blocks), dim3(kBlock), 0, s, posm, n, c.bbox, parts, c.keys, c.vals);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t bytes = c.sort_tmp_bytes;
    return rocprim::radix_sort_pairs(c.sort_tmp, bytes, c.keys, c.keys_alt, c.vals, c.perm, n, 0u, 30u, s);
}

}  // namespace grasph
