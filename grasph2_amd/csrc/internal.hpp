// internal.hpp -- library-internal declarations shared by the .hip units.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string>
#include <vector>

#include "physics.hpp"

namespace grasph {

// Neighbour lists come in tiles of 64 slots, contiguous (as planes [k][slot]
// each entry of a long list lay in another part of a gigabyte-sized array, and
// the page-table walks made walking them several times slower); in a tile four
// entries of a slot side by side, then the next slot's four, then all slots'
// next four (single entries if kmax is no multiple of 4): entry k of slot t lies
// at list_entry(t, k, kmax).  So a 128-byte line holds four entries of 8 slots, which
// is what one wavefront of the list kernel fills within a few steps, and 4 lanes
// of a pass read a slot's next four together.  With a row of 64 slots per entry
// the lines left the L2 half written: collision after impact (1e8 neighbours,
// 131072 particles) lists 0.85 ms, now 0.36, passes 0.42 + 0.65 + 0.75, now 0.30 +
// 0.54 + 0.61; 65537 squeezed particles 1229 -> 1115 us, SPH without gravity at
// 100000 149 -> 142.  A plane holds list_plane(n, kmax) entries.
__host__ __device__ inline int list_chunk(int kmax) { return kmax % 4 ? 1 : 4; }
__host__ __device__ inline uint32_t list_mask(int kmax) { return ~(uint32_t)(list_chunk(kmax) - 1); }
// of entry k from the list's entry 0; increases with k
__host__ __device__ inline uint32_t list_offset(uint32_t k, uint32_t mask) { return k + 63u * (k & mask); }
__host__ __device__ inline size_t list_entry(int t, int k, int kmax)
{
    return (size_t)(t >> 6) * (size_t)kmax * 64 + (size_t)(t & 63) * (size_t)list_chunk(kmax) + list_offset(k, list_mask(kmax));
}
__host__ __device__ inline size_t list_plane(int64_t n, int kmax) { return (size_t)((n + 63) / 64) * 64 * (size_t)kmax; }

enum KernelClass {
    KC_SWEEP = 0,
    KC_DENSITY = 1,
    KC_STRAIN = 2,
    KC_ACCEL = 3,
    KC_INTEGRATE = 4,
    KC_REORDER = 5,
    KC_OTHER = 6,
    KC_FAR = 7  // far field of the symmetric sweep
};

// Per-device library state.  Scratch grows on demand and is reused.
struct Ctx {
    int device = 0;
    std::string err;

    // options
    int max_neighbours = 160;      // list capacity of this context's single-instance evaluations (grows)
    int max_neighbours_set = 160;  // the capacity last set: batches and their launch-loop contexts start from it
    // grow max_neighbours after an evaluation whose lists overflowed: the
    // list kernel stores its largest count in pinned host memory, and a later
    // call reads what has landed there (no wait)
    int max_neighbours_grow = 1;
    int* list_max_dev = nullptr;   // of the evaluation under way (the gather clears it)
    int* list_max_host = nullptr;
    int reorder_interval = 8;  // particles move little in 8 steps: the order only affects speed
    int sweep_ni = 1;  // i particles per lane in the single-instance sweep
    int sweep_slices = 0;  // j-split of the single-instance sweep (0: chosen from the occupancy)
    int sweep_symmetric = 2;  // single instance, far pairs once for both sides (sym_sweep.hip): 0 off, 1 on, 2 from kSymAutoMin particles
    int sym_workgroups = 0;   // workgroups of its far kernel (0: 2 wavefronts per SIMD)
    int sym_near_shares = 0;  // wavefronts per 64 slots of its in-group gravity (0: chosen from the count)
    // bytes of partner-side partials one column batch of its far field may take (6 n^2 / 1024 in all)
    int64_t sym_partial_bytes = int64_t(12) << 30;
    int sym_list_priority = 2;  // kept for callers that set it; without effect
    int batch_symmetric = 1;  // batches: the symmetric sweep for instances of batch_symmetric_min particles or more
    int batch_symmetric_min = 0;
    int cus = 256;         // compute units of the device
    bool profile = false;
    // batched sweep tuning: i per lane per size bucket, persistent launch shape
    int batch_ni[4] = {1, 1, 1, 1};
    int batch_wpb = 4;
    int batch_bpc = 8;

    // variable-step leapfrog state {current dt, next dt}, zero at creation
    float* ts = nullptr;
    // {uniform, mass} of the particles, written before each gravity sweep,
    // then the per-block flags of the check (2 + 256 floats)
    float* umass = nullptr;
    int* mass_flags = nullptr;  // per-256-slot flags of the check when the gather makes them
    int64_t mass_flags_cap = 0;

    // Hilbert order of the i side (slot t -> particle perm[t])
    int* perm = nullptr;
    int64_t perm_n = 0;
    const void* perm_src = nullptr;  // posm pointer the order was computed for
    int64_t evals_since_reorder = 0;
    uint32_t* keys = nullptr;
    uint32_t* keys_alt = nullptr;
    int* vals = nullptr;
    void* sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    float* bbox = nullptr;  // [nblocks][6] partial bounds then final [6]
    int64_t reorder_cap = 0;

    // neighbour lists: entry k of slot t at list_entry(t, k, kmax), counts nbr_cnt[slot]
    int* nbr = nullptr;
    int* nbr_cnt = nullptr;
    int64_t nbr_cap_n = 0;
    int nbr_cap_k = 0;
    float4* box = nullptr;  // the lists' boxes: fine, then coarse, then mid
    int64_t box_cap = 0;
    int64_t last_list_n = 0;  // particles of the last neighbour list built
    float4* part = nullptr;   // partial sums of a j-split sweep
    int64_t part_cap = 0;
    // work arrays of the symmetric sweep
    float4* sym_near = nullptr;
    int64_t sym_near_cap = 0;
    float4* sym_apart = nullptr;
    int64_t sym_apart_cap = 0;
    float* sym_bpart = nullptr;
    int64_t sym_bpart_cap = 0;
    float4* sym_accsum = nullptr;  // running sums between the far field's column batches
    int64_t sym_accsum_cap = 0;

    // slot-ordered positions for the sweep, and the slot records of the passes
    float4* xs = nullptr;
    int64_t xs_cap = 0;
    struct SlotRec* rec = nullptr;
    int64_t rec_cap = 0;

    // potential and reduction partials
    float* pot = nullptr;
    int64_t pot_cap = 0;
    double* red = nullptr;
    int64_t red_cap = 0;

    // timing
    struct Ev {
        hipEvent_t a, b;
        int cls;
    };
    std::vector<Ev> ev_pending;
    std::vector<hipEvent_t> ev_free;
    double ms[GRASPH_NKERNEL_CLASSES] = {};
    int64_t launches[GRASPH_NKERNEL_CLASSES] = {};
    bool capturing = false;  // no timing events while a graph is being captured

    struct BatchState* batch = nullptr;

    // The allocation-free entry point runs the derivative path on a
    // stand-in context whose buffers are cut from the device's static
    // scratch array; there no_alloc turns every allocation the path would
    // make into an error.  scratch: that array's device address on this
    // context's device (null, with the reason in scratch_err, when the
    // runtime could not resolve it).
    bool no_alloc = false;
    void* scratch = nullptr;
    std::string scratch_err;
    int noalloc_slices = 0;  // j-slices of the last allocation-free call
};

// Bracket a kernel launch with events when profiling is on.
struct ProfScope {
    Ctx* c;
    hipStream_t s;
    int cls;
    hipEvent_t a = nullptr, b = nullptr;
    ProfScope(Ctx* ctx, hipStream_t st, int k);
    ~ProfScope();
};

// ---- launchers (return hipError_t of the launch) -------------------------
struct SweepLaunch {
    const float4* posm;  // particles (index order)
    const float4* xs;    // the same in slot order (xs[t] = posm[perm[t]]), or null when perm is null
    const int* perm;
    int n;
    float4* acc;        // gravity (written when grav)
    float* pot;         // written when want_pot
    bool grav, want_pot;
    bool finish;        // apply environmentAcceleration, zero xvel / maxvsig (SPH off)
    float4* xvel;
    float* maxvsig;
    // one-sided gravity: ni particles per lane (1, 2 or 4); `waves` wavefronts
    // of a workgroup and `planes` workgroups share their particles' partners,
    // slice_len (a multiple of 8) each; split: lanes per particle (1, or with
    // ni 1 and one plane kOwnSplit, which take a share each)
    int ni, waves, planes, slice_len, split;
    float4* part;       // [planes][n][2] partial sums when planes > 1
    const float* umass; // {uniform, mass} from launch_mass_check, or null
};
hipError_t launch_sweep(const SweepLaunch& L, const DevParams& P, hipStream_t s);

// The symmetric single-instance gravity sweep (sym_sweep.hip): groups of
// 1024 slots; inside a group one-sided, between groups once per unordered
// pair.  Sizes of its work arrays, in elements.
struct SymGeom {
    int groups, wgs;
    int64_t nsb, units;   // super-blocks; far work units
    int split;            // pieces a partner group is cut into for the far work's split
    int64_t near_elems;   // float4: in-group sums and their corrections per slot
    int64_t apart_elems;  // float4: far own-side fragments (kFragElems each)
    bool plain;           // no far workgroup flushes a fragment twice: no correction planes
    int64_t bpart_elems;  // float: far partner-side partials (of the widest column batch)
    int ncols;            // column batches of the far field (1: the whole far field at once)
};
SymGeom sym_geometry(int64_t n, int wgs, int64_t col_elems = INT64_MAX);
// one column batch [c0, c1) of the far field's partner groups
struct SymCol {
    int c0, c1;
    int64_t units;
    int wgs;
    bool plain;
};
SymCol sym_column(int split, int fold, int wanted, int c0, int c1);
int sym_default_workgroups(int cus);  // far-field workgroups for 2 wavefronts per SIMD
struct SymLaunch {
    const float4* xs;   // slot-ordered positions + masses
    const int* perm;    // slot -> particle, or null
    int n;
    bool finish;        // as SweepLaunch::finish
    bool add_acc;       // acc already holds the SPH terms: the combine adds the gravity to them
    int near_waves;     // in-group gravity: wavefronts sharing 64 slots
    float4* acc;
    float4* xvel;
    float* maxvsig;
    const float* umass; // {uniform, mass}, or null
    int wgs;            // workgroups of the far kernel
    float4* near_part;
    float4* apart;        // own-side fragments (kFragElems each)
    float* bpart;
    int64_t col_elems;    // partner-side partials (floats) a column batch of the far field may take
    float4* accsum;       // running sums between column batches: 2 float4 per slot (column-batched far field)
};
// the symmetric sweep in three launches: the in-group gravity, the far
// field, then the combine
hipError_t launch_sym_ingroup(const SymLaunch& L, const DevParams& P, hipStream_t s);
hipError_t launch_sym_far(const SymLaunch& L, const DevParams& P, hipStream_t s);
bool sym_fused(const SymLaunch& L);
hipError_t launch_sym_near_combine(const SymLaunch& L, const DevParams& P, hipStream_t s);
hipError_t launch_sym_combine(const SymLaunch& L, const DevParams& P, hipStream_t s);
bool sym_has_far(const SymLaunch& L);

// The symmetric sweep over a batch (slot indices are the batch's).
struct BatchInst;
struct SymInst {
    int off, n;         // slots [off, off + n)
    int nsb, nrows;     // groups; far rows (groups with later ones)
    int row0;           // its first far row in the batch's arrays
    int64_t bpart0;     // first float of its partner-side partials
};
struct SymRow {
    int inst, g, piece, units;  // piece `piece` of far row g of instance inst: units partner groups
};
// [begin, end) of instance k in blocks of `slots`
inline void append_blocks(std::vector<int4>& blk, int k, int64_t begin, int64_t end, int slots)
{
    for (int64_t s = begin; s < end; s += slots) blk.push_back(make_int4(k, (int)s, (int)std::min(s + slots, end), 0));
}
struct SymBatchTables {
    std::vector<SymInst> insts;  // every instance; those below min_n have n = 0
    std::vector<SymRow> rows;    // longest first
    std::vector<int4> blk, blk64;  // 256-slot and 64-slot blocks (instance, first, end) of the instances in the sweep
    int64_t apart_elems = 0, bpart_elems = 0;
    int most = 4;       // pieces of a row at most (kBatchPieces to kBatchPiecesMost)
    bool plain = true;  // no row piece flushes its fragment twice
};
// instances of at least min_n particles take the symmetric sweep; wgs: wavefronts of the far field that run at once
SymBatchTables sym_batch_tables(const std::vector<int64_t>& offsets, int64_t min_n, int64_t wgs);
struct SymBatchLaunch {
    const float4* xs;     // slot-ordered positions + masses of the batch
    const int* perm;      // slot -> particle, or null
    int ntotal, n_inst;
    bool soft;
    bool add_acc;         // acc already holds the SPH terms: the combine adds the gravity to them
    const SymInst* sinst;
    const BatchInst* insts;
    const int4* blk;      // 256-slot and 64-slot blocks of the instances in the sweep
    int n_blk;
    const int4* blk64;
    int n_blk64;
    const SymRow* rows;
    int nrows;
    int most;             // SymBatchTables::most
    int* queue;           // one work counter
    int wgs;
    bool plain;           // SymBatchTables::plain
    const float* umass;   // {uniform, mass} per instance
    float4* acc;
    float4* near_part;
    float4* apart;        // own-side fragments (kFragElems each)
    float* bpart;
};
// the batched symmetric sweep in three launches, as the single-instance one
hipError_t launch_sym_batch_ingroup(const SymBatchLaunch& L, hipStream_t s);
hipError_t launch_sym_batch_far(const SymBatchLaunch& L, hipStream_t s);
hipError_t launch_sym_batch_combine(const SymBatchLaunch& L, hipStream_t s);
inline bool sym_batch_has_far(const SymBatchLaunch& L) { return L.ntotal > 0 && L.n_blk > 0 && L.nrows > 0; }

// Neighbour lists (lists.hip): bounding boxes of every kBoxFine, kBoxMid and
// kBoxCoarse consecutive slots of an instance, two float4 (lo, hi) each, then
// one list per slot.  A box array holds all fine ones, all coarse ones, then
// the mid ones (a batch's: kBoxCoarse / kBoxMid per coarse box).
constexpr int kBoxFine = 8, kBoxMid = 64, kBoxCoarse = 512;
inline int64_t fine_boxes(int64_t n) { return (n + kBoxFine - 1) / kBoxFine; }
inline int64_t mid_boxes(int64_t n) { return (n + kBoxMid - 1) / kBoxMid; }
inline int64_t coarse_boxes(int64_t n) { return (n + kBoxCoarse - 1) / kBoxCoarse; }
inline int64_t all_boxes(int64_t n) { return fine_boxes(n) + coarse_boxes(n) + mid_boxes(n); }
struct BatchInst;
struct ListLaunch {
    const float4* xs;  // slot-ordered positions
    int n;
    float H2;          // one instance
    float4* fine;      // boxes: one instance's come from the gather, a batch's are made here
    float4* coarse;
    float4* mid;
    int* nbr;
    int* nbr_cnt;
    int kmax;
    int* max_dev;      // largest count of an overflowed list: of this evaluation (0 before it), and
    int* max_host;     // the host's copy; null: not reported
    const int4* blk;   // batch: 256-slot and 32-slot blocks of all instances
    int n_blk;
    const int4* blk32;
    int n_blk32;
    const BatchInst* insts;
};
hipError_t launch_lists(const ListLaunch& L, hipStream_t s);
hipError_t launch_batch_lists(const ListLaunch& L, hipStream_t s);

// Per-slot record of the neighbour passes (64 bytes, slot order): position
// and mass; velocity and density; the acceleration pass's j-side terms
// sigma/rho^2 (xx yy zz xy | xz yz), balsara, density.
struct SlotRec {
    float4 pm, vr, ra, rb;
};

// One instance of a batch, as the device kernels see it.
struct BatchInst {
    int off;     // first particle
    int n;       // particle count
    float H2;    // smoothing length squared
    int fine0, coarse0;  // its first fine and coarse box in the batch's arrays
};

// Block descriptors of the per-particle passes over a batch: block b covers
// slots [blk[b].y, blk[b].z) of instance blk[b].x (never two instances).
struct BlockTables {
    const int4* blk;
    const BatchInst* insts;
    const DevParams* prm;  // per-instance parameters
    int nblocks;           // 0: one instance, the grid covers all slots
    // the same cut into blocks of 64 slots, one list pass workgroup each (with four
    // to a block of 256, most of them empty, 2000 instances of 50 took 55 us in the
    // strain and the acceleration pass, now 19)
    const int4* blk64;
    int nblocks64;
};

// Workgroups are dealt to the GPU's 8 XCDs in turn (workgroup b to XCD
// b mod 8), and each XCD has an L2 of its own.  xcd_block gives XCD x the
// x-th contiguous eighth of the nb blocks: consecutive slots are spatial
// neighbours, so a block's neighbour gathers then hit the L2 that its
// neighbouring blocks filled (dealt round-robin, every record of the
// ensemble's strain pass was fetched into several L2s: 11 GB per pass for
// 10 GB of gathers).  A bijection of [0, nb): the work and the results do
// not change, only where they run.
__device__ inline int xcd_block(int b, int nb)
{
    constexpr int kXcds = 8;
    const int x = b % kXcds, i = b / kXcds, q = nb / kXcds, r = nb % kXcds;
    return x * q + min(x, r) + i;
}

// The same in runs of c blocks: 8 c blocks after another are dealt to the XCDs
// c to each, what is left at the end as xcd_block deals it.
__device__ inline int xcd_runs(int b, int nb, int c)
{
    constexpr int kXcds = 8;
    const int run = kXcds * c, full = nb / run * run;
    if (b >= full) return full + xcd_block(b - full, nb - full);
    const int r = b % run;
    return b - r + r % kXcds * c + r / kXcds;
}

// A single instance's lists have grown long (capacity past this, bodies crushed
// together): dense parts, contiguous in slot order, hold most neighbours.
// Whole eighths then leave most of the work to an XCD or two, and 4 lanes per
// particle wait for the longest list of 16: the passes take runs of kXcdRun
// slots and 16 lanes.  131072 particles after impact (1e8 neighbours, up to
// 3021 each), density, strain and acceleration: 0.40 + 0.79 + 0.92 ms with 4 lanes and
// runs, 0.37 + 0.67 + 0.78 with 16 and whole eighths, 0.30 + 0.54 + 0.61 with both (a
// step 4.90, 4.48 and 4.13 ms).  Runs read more halo than eighths: evenly squeezed
// spheres, whose eighths hold the same work, lose by them (131072 particles 3094
// against 3193 us, 90000 1678 against 1754, 65537 1058 against 1115; to 65536 an
// eighth is 8192 slots at most and stays), and with short lists 200003 particles
// 274 against 278.
constexpr int kLongLists = 512, kXcdRun = 4096, kXcdRunMin = 65536;
__device__ inline int xcd_run(int n, int kmax) { return kmax > kLongLists && n > kXcdRunMin ? kXcdRun : 0; }

// What one block of a per-particle pass works on (run: slots per XCD in turn, 0
// for whole eighths).
struct SlotMap {
    int slot0, slot_end, off, n, inst, coarse0;
    // element c of particle i in an array of 6 (resp. 3) planes per instance
    __device__ size_t plane6(int c, int i) const { return 6 * (size_t)off + (size_t)c * n + (size_t)(i - off); }
    __device__ size_t plane3(int c, int i) const { return 3 * (size_t)off + (size_t)c * n + (size_t)(i - off); }
};

template <bool BATCH>
__device__ inline SlotMap slot_map(const BlockTables& T, int n, int slots_per_block = 256, int run = 0)
{
    SlotMap m;
    const int blk = BATCH || run == 0 ? xcd_block((int)blockIdx.x, (int)gridDim.x)
                                      : xcd_runs((int)blockIdx.x, (int)gridDim.x, run / slots_per_block);
    if (BATCH) {
        const int4 b = slots_per_block == 64 ? T.blk64[blk] : T.blk[blk];  // 64 or 256
        const BatchInst I = T.insts[b.x];
        m.inst = b.x;
        m.slot0 = b.y;
        m.slot_end = b.z;
        m.off = I.off;
        m.n = I.n;
        m.coarse0 = I.coarse0;
    } else {
        m.inst = 0;
        m.slot0 = blk * slots_per_block;
        m.slot_end = n;
        m.off = 0;
        m.n = n;
        m.coarse0 = 0;
    }
    return m;
}

// The boxes of the kBoxCoarse slots first + threadIdx.x of an instance of n
// (a workgroup of as many threads; p: this thread's slot, act: below n) into
// the instance's fine, mid and coarse arrays.
__device__ inline void block_boxes(const float4 p, const bool act, const int first, const int n,
                                   float4* __restrict__ fine, float4* __restrict__ mid, float4* __restrict__ coarse)
{
    constexpr int kWaves = kBoxCoarse / 64;
    __shared__ float red[6][kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float v[6] = {act ? p.x : INFINITY,  act ? p.y : INFINITY,  act ? p.z : INFINITY,
                  act ? p.x : -INFINITY, act ? p.y : -INFINITY, act ? p.z : -INFINITY};
    if (__any(act)) {  // else the wavefront's slots are past the end
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[c] = fminf(v[c], __shfl_xor(v[c], o, 64));
                v[c + 3] = fmaxf(v[c + 3], __shfl_xor(v[c + 3], o, 64));
            }
            if (o == kBoxFine / 2 && (lane & (kBoxFine - 1)) == 0 && act) {
                const int f = (first + (int)threadIdx.x) / kBoxFine;
                fine[2 * f] = make_float4(v[0], v[1], v[2], 0.0f);
                fine[2 * f + 1] = make_float4(v[3], v[4], v[5], 0.0f);
            }
        }
    }
    if (lane == 0) {
        if (act) {
            const int f = (first + (int)threadIdx.x) / kBoxMid;
            mid[2 * f] = make_float4(v[0], v[1], v[2], 0.0f);
            mid[2 * f + 1] = make_float4(v[3], v[4], v[5], 0.0f);
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) red[c][wave] = v[c];
    }
    __syncthreads();  // every thread of the workgroup gets here
    if (threadIdx.x == 0 && first < n) {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            v[c] = red[c][0];
            for (int w = 1; w < kWaves; ++w) v[c] = c < 3 ? fminf(v[c], red[c][w]) : fmaxf(v[c], red[c][w]);
        }
        coarse[2 * (first / kBoxCoarse)] = make_float4(v[0], v[1], v[2], 0.0f);
        coarse[2 * (first / kBoxCoarse) + 1] = make_float4(v[3], v[4], v[5], 0.0f);
    }
}

struct BatchSweepLaunch {
    const float4* xs;   // particles in slot order (posm itself when perm is null)
    const int* perm;
    const int4* items;  // (instance, first slot, i per lane, 0) per work item, longest instance first
    int n_items;
    const BatchInst* insts;
    int* queue;         // work counter, zero before the launch
    float4* acc;
    int blocks;           // persistent grid
    int waves_per_block;  // 1, 2 or 4
    bool soft;
    const float* umass;   // {uniform, mass} per instance
    int ni_max;           // largest ni of the items (1 or 2)
};
hipError_t launch_batch_sweep(const BatchSweepLaunch& L, hipStream_t s);
// umass[2k] = 1 when every particle of instance k (insts null: the n
// particles of one instance) has the same mass, umass[2k + 1] = that mass.
// With insts null, umass must hold 2 + 256 floats (per-block flags follow).
hipError_t launch_mass_check(const float4* posm, const BatchInst* insts, int n_inst, int n, float* umass,
                             hipStream_t s);
hipError_t launch_reset_queue(int* queue, int n, hipStream_t s);

// Batched Hilbert order: per-instance bounding boxes, keys (instance, cell
// along the curve), one radix sort; perm maps each instance's slots into its own range.
struct BatchOrder {
    const float4* posm;
    const int* inst_of;      // instance of every particle
    const BatchInst* insts;
    int n_inst;
    int ntotal;
    float* bbox;             // [n_inst][6]
    uint64_t* keys;
    uint64_t* keys_alt;
    int* vals;
    int* perm;
    void* sort_tmp;
    size_t sort_tmp_bytes;
    int key_bits;
};
size_t batch_order_tmp_bytes(int ntotal, int key_bits);
hipError_t launch_batch_order(const BatchOrder& B, hipStream_t s);

// Neighbour passes.  Slot t is particle perm[t] (perm null: t); inputs of
// the lists' partners come from the slot records, per-particle outputs go
// to particle perm[t] of the caller's arrays, and the lists hold slot
// indices (one list per particle).  posm / vel (index order) serve the
// finish kernel of configurations without SPH.
struct NbrLaunch {
    const float4* posm;
    const float4* vel;
    const float4* xs;  // positions in slot order (posm itself when perm is null)
    SlotRec* rec;
    const float* dstress;
    const float* balsara_in;
    const int* perm;
    const int* nbr;
    const int* nbr_cnt;
    const float4* coarse;  // the lists' boxes of 512 slots
    const float4* mid;     // and of 64
    int n;
    int kmax;
    float* balsara;
    float* density_dt;
    float* dstress_dt;
    float4* acc;
    float4* xvel;
    float* maxvsig;
    bool acc_has_gravity;
    int lanes;      // lanes per particle in the list passes: 4 or, in one instance, 16
    BlockTables T;  // batch tables (T.nblocks == 0 for one instance)
};
hipError_t launch_density(const NbrLaunch& L, float* density, const DevParams& P, hipStream_t s);
hipError_t launch_strain(const NbrLaunch& L, const DevParams& P, hipStream_t s);
hipError_t launch_prep(const NbrLaunch& L, const DevParams& P, hipStream_t s);
hipError_t launch_accel(const NbrLaunch& L, const DevParams& P, hipStream_t s);

struct IntegLaunch {
    float4* posm;
    double* pos64;
    float4* vel;
    const float4* acc;
    const float4* xvel;
    float* density;
    const float* density_dt;
    float* dstress;
    const float* dstress_dt;
    int n;
    int not_first_step;
    BlockTables T;  // batch tables (T.nblocks == 0 for one instance)
    // variable-step leapfrog: per instance {current dt, next dt}; null for the fixed step
    float* ts;
    const float* maxvsig;  // read by the velocity criterion
    int n_instances;
};
// Fixed step: fixedTsLeapfrog.  With L.ts: the second kernel of the
// variable step (kick + drift with dt = max(next dt, min_timestep)).
hipError_t launch_integrate(const IntegLaunch& L, const DevParams& P, hipStream_t s);
// First kernel of the variable step: half kick with the current dt and the
// dt criteria folded into the next dt (atomic minimum per block).
hipError_t launch_vts_kick(const IntegLaunch& L, const DevParams& P, hipStream_t s);
// next dt of every instance := initial_timestep (which 0) or max_timestep
// (which 1); per-instance parameters from prm (null: P for one instance)
hipError_t launch_vts_set_next(float* ts, int n_instances, const DevParams* prm, const DevParams& P, int which,
                               hipStream_t s);
// Both stages of one integrate(pb, notFirstStep) call.
hipError_t launch_integrate_step(const IntegLaunch& L, const DevParams& P, hipStream_t s);

struct InvLaunch {
    const float4* posm;
    const double* pos64;
    const float4* vel;
    const float4* acc;
    const float* density;
    const float* dstress;
    const float* pot;  // may be null
    int n;
    double half_kick;
    double* partials;  // [nblocks][GRASPH_NINV] then final [GRASPH_NINV]
    int nblocks;
};
int inv_blocks(int n);
hipError_t launch_invariants(const InvLaunch& L, const grasph_params& prm, hipStream_t s);

// Slot order: perm[t] = particle index of the t-th particle along a
// Hilbert curve over the bounding box of posm.
size_t reorder_tmp_bytes(int n);
hipError_t launch_reorder(const float4* posm, int n, Ctx& c, hipStream_t s);
// Slot-ordered copies for the sweep and the list passes (perm null: the
// identity): xs[t] = posm[perm[t]] when xs is given, and the slot records'
// position/mass and velocity/density (vel or density null: zeros there).
// With mass_flags (one int per kGatherBlock slots) also the per-block half of
// the equal-mass check, which launch_mass_final completes; with fine, mid and
// coarse the lists' boxes (one instance), and list_max cleared;
// with ts_next that set to ts_max.
constexpr int kGatherBlock = kBoxCoarse;
hipError_t launch_gather(const int* perm, int n, const float4* posm, const float4* vel, const float* density,
                         float4* xs, SlotRec* rec, hipStream_t s, int* mass_flags = nullptr,
                         float4* fine = nullptr, float4* mid = nullptr, float4* coarse = nullptr,
                         int* list_max = nullptr, float* ts_next = nullptr, float ts_max = 0.0f);
hipError_t launch_mass_final(const float4* posm, const int* mass_flags, int nflags, float* umass, hipStream_t s);

// environmentAcceleration and the zero XVEL / MAXVSIG stores of
// calcAcceleration for configurations without SPH (batched form).
hipError_t launch_finish(const NbrLaunch& L, const DevParams& P, hipStream_t s);

// ---- host helpers shared by the C-ABI units -------------------------------
inline int fail(Ctx& c, int code, const std::string& msg)
{
    c.err = msg;
    return code;
}

inline int hip_fail(Ctx& c, hipError_t e, const char* where)
{
    c.err = std::string(where) + ": " + hipGetErrorString(e);
    (void)hipGetLastError();
    return GRASPH_E_HIP;
}

template <typename T>
int grow(Ctx& c, T*& ptr, int64_t& cap, int64_t need, const char* what)
{
    if (need <= cap && ptr) return 0;
    if (c.no_alloc) return fail(c, GRASPH_E_NOMEM, std::string(what) + " would need a device allocation");
    if (ptr) {
        (void)hipFree(ptr);
        ptr = nullptr;
        cap = 0;
    }
    hipError_t e = hipMalloc((void**)&ptr, (size_t)(need > 0 ? need : 1) * sizeof(T));
    if (e != hipSuccess) {
        ptr = nullptr;
        (void)hipGetLastError();
        return fail(c, GRASPH_E_NOMEM, std::string("device allocation of ") + what + " failed");
    }
    cap = need;
    return 0;
}

inline int check_params(Ctx& c, const grasph_params* prm)
{
    if (!prm) return fail(c, GRASPH_E_INVALID, "params is NULL");
    if (prm->flags & ~GRASPH_ALL_FLAGS) return fail(c, GRASPH_E_INVALID, "unknown flag bits");
    if (prm->dimension < 1 || prm->dimension > 3) return fail(c, GRASPH_E_INVALID, "dimension must be 1, 2 or 3");
    if (!(prm->H >= 0.0f) || !(prm->H < 3.0e38f)) return fail(c, GRASPH_E_INVALID, "H must be finite and >= 0");
    if ((prm->flags & GRASPH_SPH) && !(prm->H > 0.0f)) return fail(c, GRASPH_E_INVALID, "SPH needs H > 0");
    if (prm->flags & GRASPH_CLOHESSY_WILTSHIRE)
        return fail(c, GRASPH_E_UNSUPPORTED,
                    "CLOHESSY_WILTSHIRE is not supported: src/computeDerivatives.h:37-39 adds a scalar to a "
                    "float3 through an mpUtils operator whose meaning no available source fixes");
    if ((prm->flags & GRASPH_SOLIDS) && (prm->flags & GRASPH_ARTIFICIAL_STRESS))
        return fail(c, GRASPH_E_UNSUPPORTED,
                    "SOLIDS with ARTIFICIAL_STRESS is not supported (the reference does not compile it, "
                    "src/computeDerivatives.h:267)");
    if ((prm->flags & GRASPH_PLASTICITY_MIESE) && (prm->flags & GRASPH_PLASTICITY_MC))
        return fail(c, GRASPH_E_INVALID, "choose up to one plasticity model (settings.h:203-205)");
    if (prm->flags & GRASPH_VARIABLE_TIMESTEP) {
        const float v[5] = {prm->initial_timestep, prm->min_timestep, prm->max_timestep, prm->accel_accuracy,
                            prm->velocity_accuracy};
        for (float x : v)
            if (!(x >= 0.0f) || !(x < 3.0e38f))
                return fail(c, GRASPH_E_INVALID, "variable time-step settings must be finite and >= 0");
    }
    return 0;
}

inline int check_particles(Ctx& c, const grasph_particles* p)
{
    if (!p) return fail(c, GRASPH_E_INVALID, "particles is NULL");
    if (p->n < 0) return fail(c, GRASPH_E_INVALID, "negative particle count");
    if (p->n > 0x7ffffff0LL) return fail(c, GRASPH_E_INVALID, "particle count exceeds 2^31 - 16");
    if (p->n > 0 && !p->posm) return fail(c, GRASPH_E_INVALID, "posm is NULL");
    return 0;
}

// How the one-sided gravity sweep of n particles is cut: `slices` (0:
// chosen from the count) shares of the partners, as many wavefronts of a
// workgroup as take them, the rest in planes.
constexpr int kOwnSplit = 4;
struct OwnPlan {
    int ni, waves, planes, len, split;
    int slices() const { return waves * planes * split; }
};
// slices: the option sweep_slices, 0 for the automatic choice (of at most
// max_planes planes)
OwnPlan own_plan(const Ctx& c, int64_t n, int slices, int max_planes);
// particles from which the one-sided sweep looks whether all masses are equal
// (the check's launch costs more than the multiply per pair it saves: without
// it Plummer 1000 14.2 -> 10 us per step, 9500 42.4 -> 38, allocation-free SPH
// at 20000 240 -> 236; at 24000 271 -> 274)
constexpr int64_t kMassCheckMin = 24576;
// and from which the symmetric sweep looks at all masses first (below, the far
// field's wavefronts look at their own, far_work, and the in-group gravity
// takes them as they come: Plummer 16384 66.6 -> 61.5 us per step, 50021
// 434 -> 423)
constexpr int64_t kMassCheckMinSym = 65536;
// below so many particles the symmetric sweep keeps what the one-sided sweep gives:
// unequal masses in any units, and gravity that the SPH terms join, not the reverse
constexpr int64_t kSymOneSided = 16384;

// arrays each pass needs, by configuration; 0 or a GRASPH_E_INVALID code
int check_derivative_arrays(Ctx& c, const grasph_particles* p, uint32_t f, int which);
int check_integrate_arrays(Ctx& c, const grasph_particles* p, uint32_t f);

struct BatchState;
void destroy_batch_state(BatchState* b);

}  // namespace grasph

struct grasph_ctx {
    grasph::Ctx c;
};

#define GRASPH_NEED(ptr, name)                                                                                \
    do {                                                                                                      \
        if (!(ptr)) return grasph::fail(c, GRASPH_E_INVALID, std::string(name) + " is NULL but the flags need it"); \
    } while (0)
