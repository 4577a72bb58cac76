// particle_kernels.hip -- particle side of the PM step on gfx950:
//   * tile binning (counting sort by deposit tile, wave-aggregated atomics),
//   * deterministic CIC deposit (AssignDensity: NyxParticleContainer.H:90-97 ->
//     amrex_deposit_cic + SumBoundary + 1/vol),
//   * fold of tile halos + RHS preparation (Gravity.cpp:1207-1244, 283, 290),
//   * fused central-difference gradient + CIC gather + kick(-drift)
//     (get_new_grav_vector Gravity.cpp:817-850 + update_dm_particle_single,
//     DarkMatterParticleContainer.cpp:249-306), with the periodic shift of
//     Redistribute fused into the kick.
//
// Deposit determinism.  Each tile's particles are accumulated in LDS as exact
// fixed-point integers (two unsigned 64-bit words per cell: units 2^(E-31) and
// 2^(E-63) with 2^E <= max particle mass), so the sum does not depend on the order
// in which particles arrive; the per-tile sums are then converted to FP64 and the
// tile halos folded in a fixed order.  Runs are bitwise reproducible although the
// binning itself uses atomics.
#include "nyxpm_internal.h"

namespace nyxpm {

// ---------------------------------------------------------------------------
// shared helpers
// ---------------------------------------------------------------------------

// Cell index i = floor((x - plo)*dxi + 0.5) of a coordinate, as both the deposit
// and the interpolation compute it, plus the fractional weight.
__device__ __forceinline__ int cic_index(double x, double plo, double dxi, double* frac) {
    const double l = (x - plo) * dxi + 0.5;
    const int i = (int)floor(l);
    *frac = l - i;
    return i;
}

// Error flags 1, 2, 4, 8: a word each in pinned host memory, set by plain stores (rarely
// any), so that the host reads them behind its wait for the stream without a copy.
constexpr int kErrFlags = 4;
__device__ __forceinline__ void raise_err(int* err, int flags) {
    for (int i = 0; i < kErrFlags; ++i)
        if (flags >> i & 1) __hip_atomic_store(&err[i], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Wave-aggregated atomicAdd: lanes with equal keys share one atomic.  Returns, for
// each valid lane, the counter's previous value plus the lane's rank among the
// lanes with its key.  Must be called by every lane of the wave.
__device__ __forceinline__ int agg_atomic_add(int* counters, int key, bool valid) {
    const int lane = threadIdx.x & (kWave - 1);
    const unsigned long long below = (lane == 0) ? 0ull : ((~0ull) >> (kWave - lane));
    int result = 0;
    bool todo = valid;
    for (;;) {
        const unsigned long long act = __ballot(todo);
        if (act == 0ull) break;
        const int leader = __ffsll((unsigned long long)act) - 1;
        const int lkey = __shfl(key, leader);
        const bool mine = todo && key == lkey;
        const unsigned long long mm = __ballot(mine);
        int base = 0;
        if (lane == leader) base = atomicAdd(&counters[lkey], (int)__popcll(mm));
        base = __shfl(base, leader);
        if (mine) {
            result = base + (int)__popcll(mm & below);
            todo = false;
        }
    }
    return result;
}

// Appends v to list (length counter n) for the active lanes with pred set: one
// atomic per wave, safe in divergent code (only active lanes take part).
__device__ __forceinline__ void wave_append(long long* list, int* n, long long v, bool pred) {
    const unsigned long long mask = __ballot(pred);
    if (mask == 0ull) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int leader = __ffsll((unsigned long long)mask) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(n, (int)__popcll(mask));
    base = __shfl(base, leader);
    if (pred) list[base + (int)__popcll(mask & ((1ull << lane) - 1ull))] = v;
}

// x of an empty particle slot.
__device__ __forceinline__ double empty_slot() { return __longlong_as_double(0x7ff8000000000000LL); }

// Slots above which a tile's deposit block is launched ahead of the others.
constexpr int kHeavyTile = 2048;
// A tile with more than kSplitTile slots and more than 1/kSplitShare of all particles
// is deposited by several blocks, which add their fixed-point sums in global memory: a
// CU holds seven blocks of 16x8x8 tiles, so one with more than 1/1792 of the work
// outlasts the others.  Parts of at least kSplitPart slots and 1/kSplitParts of all
// particles: the additions are at most 2754 64-bit atomics a part, ~30 per ns in all.
// 1/256 and 1/1024 -> 1/2048 and 1/2048, us: 128^3 with 2 10^6 clustered particles,
// density and velocities, 250 -> 236; 256^3 with 2 10^7, density, 465 -> 382 (parts of
// 1/4096 and tiles above 1/4096 the same within 2%).
constexpr int kSplitTile = 4096, kSplitPart = 2048, kSplitShare = 2048, kSplitParts = 2048;

// One block of the deposit ahead of the ordinary tiles: `len` slots from `off` of a
// heavy tile, one of nparts pieces (1: the whole tile); split: the tile's accumulator.
struct HeavyItem {
    int tile, off, len, nparts, split;
};

// i / T for 0 <= i < 2^17 and T <= 32 with magic = ceil(2^31 / T) (exact over that
// range; the bound is checked when a context is created).
__device__ __forceinline__ int tile_div(int i, unsigned magic) {
    return (int)(((unsigned long long)(unsigned)i * magic) >> 31);
}

__device__ __forceinline__ int tile_of(const BoxDev& B, double x, double y, double z, int* err) {
    double f;
    const int ci = cic_index(x, B.plo[0], B.dxi[0], &f);
    const int cj = cic_index(y, B.plo[1], B.dxi[1], &f);
    const int ck = cic_index(z, B.plo[2], B.dxi[2], &f);
    // an index more than one period out: one flag branch for the three (rare)
    if ((unsigned)(ci + B.n[0]) >= (unsigned)(3 * B.n[0]) || (unsigned)(cj + B.n[1]) >= (unsigned)(3 * B.n[1]) ||
        (unsigned)(ck + B.n[2]) >= (unsigned)(3 * B.n[2]))
        raise_err(err, 1);
    const int i = wrap1(ci, B.n[0]), j = wrap1(cj, B.n[1]), k = wrap1(ck, B.n[2]);
    const int tx = tile_div(i, B.tdiv[0]), ty = tile_div(j, B.tdiv[1]), tz = tile_div(k, B.tdiv[2]);
    return (int)(B.tile_off + ((long long)tz * B.ntile[1] + ty) * B.ntile[0] + tx);
}

// ---------------------------------------------------------------------------
// binning: keys + counts, exclusive scan, scatter
// ---------------------------------------------------------------------------

// Block blk's slots: keys and tile counts; empty_x (may be null): their x in the other
// buffer emptied.
__device__ __forceinline__ void keys_block(int blk, const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                           const double* __restrict__ x, const double* __restrict__ y,
                                           const double* __restrict__ z, int* __restrict__ key, int* counts, int* err,
                                           double* __restrict__ empty_x) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blk)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blk - sg.blk0) * kBlock + threadIdx.x;
    bool valid = false;
    int t = 0;
    if (q < B.span) {
        const long long p = B.part_off + q;
        const double px = x[p];
        valid = !isnan(px);  // NaN: an empty slot, keyed -1
        if (valid) t = tile_of(B, px, y[p], z[p], err);
        key[p] = valid ? t : -1;
        if (empty_x) empty_x[p] = empty_slot();
    }
    agg_atomic_add(counts, t, valid);
}

__global__ void __launch_bounds__(kBlock) k_keys(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                 const double* __restrict__ x, const double* __restrict__ y,
                                                 const double* __restrict__ z, int* __restrict__ key,
                                                 int* counts, int* err) {
    keys_block(blockIdx.x, segs, nseg, boxes, x, y, z, key, counts, err, nullptr);
}

// Slot capacity of each tile for a sort with slack: cnt + floor(cnt * num / 1024)
// + pad (integer arithmetic, so a box's capacities never exceed its slots).
__global__ void __launch_bounds__(kBlock) k_tile_caps(const int* __restrict__ counts, long long n, int num,
                                                      int pad, int* __restrict__ cap) {
    const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (t < n) {
        const long long c = counts[t];
        cap[t] = (int)(c + ((c * num) >> 10) + pad);
    }
}

// First slot of each tile: the scan of the capacities restarted at each box's
// first slot (boxes keep fixed slot ranges).
__global__ void __launch_bounds__(kBlock) k_tile_base(const BoxSeg* tsegs, int ntseg, const BoxDev* boxes,
                                                      const long long* __restrict__ start, long long n,
                                                      long long* __restrict__ tbase) {
    const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (t >= n) return;
    const BoxDev& B = boxes[tsegs[find_seg(tsegs, ntseg, (int)t)].box];
    tbase[t] = start[t] - start[B.tile_off] + B.part_off;
}

constexpr int kScanItems = 16;  // entries per thread in the scan passes

__global__ void __launch_bounds__(kBlock) k_scan_reduce(const int* __restrict__ counts, long long n,
                                                        long long* __restrict__ bsum) {
    const long long base = (long long)blockIdx.x * kBlock * kScanItems;
    long long s = 0;
    for (int it = 0; it < kScanItems; ++it) {
        const long long q = base + (long long)it * kBlock + threadIdx.x;
        if (q < n) s += counts[q];
    }
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    __shared__ long long ws[kBlock / kWave];
    if ((threadIdx.x & (kWave - 1)) == 0) ws[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        for (int w = 0; w < kBlock / kWave; ++w) t += ws[w];
        bsum[blockIdx.x] = t;
    }
}

// Exclusive scan of the block sums in place (one block), total in bsum[nb].
__global__ void __launch_bounds__(1024) k_scan_top(long long* bsum, int nb) {
    __shared__ long long sh[1024];
    long long carry = 0;
    for (int base = 0; base < nb; base += 1024) {
        const int q = base + threadIdx.x;
        const long long v = q < nb ? bsum[q] : 0;
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            long long t = threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
            __syncthreads();
            sh[threadIdx.x] += t;
            __syncthreads();
        }
        if (q < nb) bsum[q] = carry + sh[threadIdx.x] - v;
        const long long tot = sh[1023];
        __syncthreads();
        carry += tot;
    }
    if (threadIdx.x == 0) bsum[nb] = carry;
}

// start[q] = exclusive prefix of counts; cursor[q] = 0; start[n] = total.
__global__ void __launch_bounds__(kBlock) k_scan_down(const int* __restrict__ counts, long long n,
                                                      const long long* __restrict__ bsum,
                                                      long long* __restrict__ start, int* __restrict__ cursor) {
    __shared__ long long sh[kBlock];
    const long long base = (long long)blockIdx.x * kBlock * kScanItems;
    // each thread owns kScanItems consecutive entries
    long long vals[kScanItems];
    long long s = 0;
    for (int it = 0; it < kScanItems; ++it) {
        const long long q = base + (long long)threadIdx.x * kScanItems + it;
        vals[it] = q < n ? counts[q] : 0;
        s += vals[it];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 1; o < kBlock; o <<= 1) {
        long long t = threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    long long run = bsum[blockIdx.x] + sh[threadIdx.x] - s;
    for (int it = 0; it < kScanItems; ++it) {
        const long long q = base + (long long)threadIdx.x * kScanItems + it;
        if (q < n) {
            start[q] = run;
            cursor[q] = 0;
        }
        run += vals[it];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) start[n] = bsum[gridDim.x];
}

// One particle buffer: arrays of one allocation that starts at x (`bytes` long), or, with
// bytes = 0, of their own (or none).
struct PartPtrs {
    double *x, *y, *z, *vx, *vy, *vz, *m;
    int* id;
    size_t bytes;
};

// Move block blk's particles to their tiles' slot ranges (order inside a tile is
// arbitrary); cursor[t] ends as the tile's particle count.
__device__ __forceinline__ void scatter_block(int blk, const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                              const int* __restrict__ key, const long long* __restrict__ tbase,
                                              int* cursor, const PartPtrs& src, const PartPtrs& dst) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blk)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blk - sg.blk0) * kBlock + threadIdx.x;
    const long long p = B.part_off + q;
    // occupied slots only (a kick-drift keys the slots it visits, not the free ones)
    bool valid = false;
    int t = 0;
    if (q < B.span) {
        const int k = key[p];
        valid = k >= 0 && !isnan(src.x[p]);
        t = valid ? k : 0;
    }
    const int r = agg_atomic_add(cursor, t, valid);
    if (valid) {
        const long long d = tbase[t] + r;
        dst.x[d] = src.x[p];
        dst.y[d] = src.y[p];
        dst.z[d] = src.z[p];
        dst.vx[d] = src.vx[p];
        dst.vy[d] = src.vy[p];
        dst.vz[d] = src.vz[p];
        if (src.m) dst.m[d] = src.m[p];
        dst.id[d] = src.id[p];
    }
}

__global__ void __launch_bounds__(kBlock) k_scatter(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                    const int* __restrict__ key,
                                                    const long long* __restrict__ tbase, int* cursor,
                                                    PartPtrs src, PartPtrs dst) {
    scatter_block(blockIdx.x, segs, nseg, boxes, key, tbase, cursor, src, dst);
}

// The full sort of a captured step, decided on the device: a replay cannot read
// k_migrate's flags back, so it records the incremental re-sort and behind it these
// kernels, which do nothing unless a tile ran out of slack or the emptied slots pass
// their limit.  They sort into the idle buffer and copy back (the buffers' roles are
// baked into the recorded launches).  Few, persistent blocks: skipped, the four cost ~2 us
// each; a full sort per captured step took 1.6 ms for 5.2 10^7 particles.
struct Resort {
    const int* mig;    // of k_migrate: overflow, particles moved
    long long* state;  // [0] emptied slots, [1] full sorts, [2] incremental ones, [3] particles moved
    long long np;      // particles and the share (of 1024) of emptied slots that asks for a full sort
    int hole_num;
};
__device__ __forceinline__ bool resort_full(const Resort& r) {
    return r.mig[0] != 0 || (r.state[0] + r.mig[1]) * 1024 > r.np * r.hole_num;
}

__global__ void __launch_bounds__(kBlock) k_resort_keys(Resort r, int nblk, const BoxSeg* segs, int nseg,
                                                        const BoxDev* boxes, PartPtrs A, int* __restrict__ key,
                                                        int* counts, int* err, PartPtrs idle) {
    if (!resort_full(r)) return;
    for (int b = blockIdx.x; b < nblk; b += gridDim.x)
        keys_block(b, segs, nseg, boxes, A.x, A.y, A.z, key, counts, err, idle.x);
}

// Capacities, slot ranges (per box from its first slot) and empty cursors of all tiles,
// one block.
__global__ void __launch_bounds__(1024) k_resort_scan(Resort r, const BoxSeg* tsegs, int ntseg, const BoxDev* boxes,
                                                      const int* __restrict__ counts, long long ntiles, int num,
                                                      int pad, int* __restrict__ cap, long long* start,
                                                      long long* __restrict__ tbase, int* __restrict__ cursor) {
    if (!resort_full(r)) return;
    __shared__ long long sh[1024];
    long long carry = 0;
    for (long long base = 0; base < ntiles; base += 1024) {
        const long long t = base + threadIdx.x;
        long long v = 0;
        if (t < ntiles) {
            const long long c = counts[t];
            v = c + ((c * num) >> 10) + pad;
            cap[t] = (int)v;
            cursor[t] = 0;
        }
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const long long u = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
            __syncthreads();
            sh[threadIdx.x] += u;
            __syncthreads();
        }
        if (t < ntiles) start[t] = carry + sh[threadIdx.x] - v;
        carry += sh[1023];
        __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
    for (long long t = threadIdx.x; t < ntiles; t += 1024) {
        const BoxDev& B = boxes[tsegs[find_seg(tsegs, ntseg, (int)t)].box];
        tbase[t] = start[t] - start[B.tile_off] + B.part_off;
    }
}

__global__ void __launch_bounds__(kBlock) k_resort_scatter(Resort r, int nblk, const BoxSeg* segs, int nseg,
                                                           const BoxDev* boxes, const int* __restrict__ key,
                                                           const long long* __restrict__ tbase, int* cursor,
                                                           PartPtrs src, PartPtrs dst) {
    if (!resort_full(r)) return;
    for (int b = blockIdx.x; b < nblk; b += gridDim.x)
        scatter_block(b, segs, nseg, boxes, key, tbase, cursor, src, dst);
}

__global__ void __launch_bounds__(kBlock) k_resort_copy(Resort r, long long slots, PartPtrs src, PartPtrs dst) {
    if (!resort_full(r)) return;
    for (long long p = (long long)blockIdx.x * kBlock + threadIdx.x; p < slots; p += (long long)gridDim.x * kBlock) {
        const double px = src.x[p];
        dst.x[p] = px;
        if (isnan(px)) continue;  // an empty slot
        dst.y[p] = src.y[p];
        dst.z[p] = src.z[p];
        dst.vx[p] = src.vx[p];
        dst.vy[p] = src.vy[p];
        dst.vz[p] = src.vz[p];
        if (src.m) dst.m[p] = src.m[p];
        dst.id[p] = src.id[p];
    }
}

// A recorded full sort that is not k_resort_*'s: no emptied slots, counted.
__global__ void k_resort_full(long long* state, long long* h_state) {
    state[0] = 0;
    state[1] += 1;
    for (int q = 0; q < 4; ++q)
        __hip_atomic_store(&h_state[q], state[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The state a replay starts from.
__global__ void k_resort_state(long long* state, long long holes) {
    state[0] = holes;
    state[1] = state[2] = state[3] = 0;
}

// ---------------------------------------------------------------------------
// deposit
// ---------------------------------------------------------------------------

// Index of a low-halo cell (lx==0 || ly==0 || lz==0) of a tile whose LDS block is
// (bx+1) x (by+1) x (bz+1): the x face first (y fastest), then the y face without
// its x=0 column, then the z face without x=0 and y=0 (both x fastest).  The fold
// walks cells row-major, so the y- and z-face entries it reads for a row of a
// tile's top face are consecutive (a strided face order fetched a separate
// memory sector per entry).
__device__ __forceinline__ int halo_index(int lx, int ly, int lz, int bx, int by, int bz) {
    if (lx == 0) return lz * (by + 1) + ly;
    const int fx = (by + 1) * (bz + 1);
    if (ly == 0) return fx + lz * bx + (lx - 1);
    const int fy = bx * (bz + 1);
    return fx + fy + (ly - 1) * bx + (lx - 1);
}

// A non-negative FP32 value w < 2^(E+1) in units 2^(E-31), rounded to nearest:
// w * 2^(31-E) < 2^32 is exact in FP32 (a power-of-two scale, `scale`), and the
// native f32 -> u32 conversion (truncating) of it plus one half rounds it (ties
// as FP32 rounds the sum; a value that rounds up to 2^32 saturates at 2^32 - 1).
// Four instructions per contribution.
__device__ __forceinline__ unsigned fx32_units(float w, float scale) {
    return __float2uint_rz(w * scale + 0.5f);
}

// The parts of a split tile: adds the block's LDS words to the tile's accumulator
// (integers: exact in any order); the last part to arrive takes the sums back into
// LDS, leaving the accumulator and its counter at zero for the next deposit, and
// returns true.  Everything shared between the parts is touched by device-scope atomics
// alone, which are performed where all XCDs see them: a part waits for its additions to
// be performed, then arrives.  (A fence instead of the wait writes back the XCD's whole
// L2 for each part: with it 128^3 with 2 10^6 clustered particles took 121 us instead of
// 43, the three momenta 376 instead of 86, 10^6 in 112x96x144 FP32 66 instead of 19.)
__device__ __forceinline__ bool split_combine(unsigned long long* acc, int words, const HeavyItem& hv,
                                              unsigned long long* split_acc, int split_words, int* split_done) {
    __shared__ int s_last;
    unsigned long long* g = split_acc + (size_t)hv.split * split_words;
    for (int c = threadIdx.x; c < words; c += kBlock)
        if (acc[c]) atomicAdd(&g[c], acc[c]);
    __builtin_amdgcn_s_waitcnt(0);  // every addition before the arrival
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(&split_done[hv.split], 1) == hv.nparts - 1;
    __syncthreads();
    if (!s_last) return false;
    // several exchanges in flight per thread: each is a round trip past the L2
    constexpr int U = 6;
    for (int c0 = threadIdx.x; c0 < words; c0 += U * kBlock) {
        unsigned long long v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u * kBlock < words) v[u] = atomicExch(&g[c0 + u * kBlock], 0ull);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u * kBlock < words) acc[c0 + u * kBlock] = v[u];
    }
    if (threadIdx.x == 0) atomicExch(&split_done[hv.split], 0);
    __syncthreads();
    return true;
}

// One block per tile.  Contributions m*sx[ii]*sy[jj]*sz[kk] (amrex_deposit_cic
// weights, product left to right) of the tile's particles go to LDS as fixed
// point; interior cells are written to `own`, the low halo layer to `halo`.
//
// F32 (the mixed-precision step): the fractional weights and the product are
// FP32 (the cell index and the fraction come from the FP64 position as in FP64
// mode), and each contribution is one 32-bit count of units 2^(E-31)
// (fx32_units) added into the cell's 64-bit word, so the LDS sum is still exact
// and order independent, with half the atomics: a cell's sum of at most 2^32
// contributions below 2^32 units each stays below 2^64.  Per contribution the
// FP32 rounding (~6e-8 relative) dominates the unit (2^-31 of the largest mass).
//
// MOM (AssignDensityAndVels, FP64): velocity component blockIdx.y, contributions
// (sx*sy*sz*m) * v_d as signed fixed point (two's complement in the u64 words, hi in
// units 2^(E-30) converted through int32, lo in 2^(E-62), 2^E <= max |m v_d| of the
// box, from maxbits), exact and order independent like the mass deposit's.  The
// three components are one launch (a launch each, one block per tile: 3 x 287 us for
// 2 10^6 clustered particles, held by the heaviest tile).
struct DepositMom {
    const double* v[3];                 // vx, vy, vz
    const unsigned long long* maxbits;  // max |m v_d| per box and component
    double* own[3];                     // per component
    double* halo[3];
};
// FP64: compiled for the seven waves per SIMD that the LDS of seven 16x8x8 tiles admits.
// Without a bound / for eight / for seven waves, deposit, us: 512^3 cells with 2 10^7
// particles 567 / 538 / 523, with 10^6 555 / 527 / 521, with 2^27 1200 / 1190 / 1170, 256^3
// with 2 10^6 78 / 74.5 / 72.6 (517, 515, 1150 and 71.2 before tiles were deposited in
// parts); the momenta, whole call, 512^3 with 2 10^7, none / seven: 4860 / 4680.  FP32: no
// difference.
template <bool F32, bool MOM = false>
__global__ void __launch_bounds__(kBlock, F32 ? 1 : 7)
    k_deposit(const BoxSeg* segs, int nseg, const BoxDev* boxes, const long long* __restrict__ tbase,
              const int* __restrict__ thw, const HeavyItem* __restrict__ heavy, const int* nheavy, int heavy_cap,
              unsigned long long* split_acc, int split_words, int* split_done, int split_cap,
              const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
              const double* __restrict__ m, double* __restrict__ own, double* __restrict__ halo, int* err,
              DepositMom mom = {}) {
    static_assert(!(F32 && MOM), "momenta are deposited in FP64");
    extern __shared__ unsigned long long acc[];
    const int comp = MOM ? (int)blockIdx.y : 0;
    const double* __restrict__ vel = MOM ? mom.v[comp] : nullptr;
    if (MOM) {
        own = mom.own[comp];
        halo = mom.halo[comp];
    }
    // the first heavy_cap blocks take the heavy tiles or their parts (listed by
    // k_make_items), so the longest blocks start first; the rest take every other
    // tile in order
    int tile;
    HeavyItem hv{0, 0, 0, 1, -1};
    if ((int)blockIdx.x < heavy_cap) {
        if ((int)blockIdx.x >= *nheavy) return;
        hv = heavy[blockIdx.x];
        tile = hv.tile;
    } else {
        tile = blockIdx.x - heavy_cap;
        if (thw[tile] > kHeavyTile) return;
    }
    const BoxSeg sg = segs[find_seg(segs, nseg, tile)];
    // the box's fields as block-uniform values in registers: read through a
    // reference they would be re-read from memory after every possible store
    // or atomic (the error flag) of the particle loop
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const int lt = tile - sg.blk0;
    const int tx = lt % B.ntile[0], ty = (lt / B.ntile[0]) % B.ntile[1], tz = lt / (B.ntile[0] * B.ntile[1]);
    const int o0 = tx * B.tile[0], o1 = ty * B.tile[1], o2 = tz * B.tile[2];
    const int bx = min(B.tile[0], B.n[0] - o0), by = min(B.tile[1], B.n[1] - o1), bz = min(B.tile[2], B.n[2] - o2);
    const int Lx = bx + 1, Ly = by + 1, Lz = bz + 1;
    const int LC = Lx * Ly * Lz;
    const long long gt = B.tile_off + lt;
    long long p0 = tbase[gt], p1 = p0 + thw[gt];
    if (hv.nparts > 1) {
        p0 += hv.off;
        p1 = p0 + hv.len;
    }
    // the thread's first two particles are loaded before the accumulator is
    // cleared, so their latency overlaps the clearing
    double xa = 0.0, ya = 0.0, za = 0.0, ma = 0.0, xb = 0.0, yb = 0.0, zb = 0.0, mb = 0.0;
    double va = 0.0, vb = 0.0;
    auto load2 = [&](long long pa) {
        const long long pb = pa + kBlock;
        if (pa < p1) {
            xa = x[pa]; ya = y[pa]; za = z[pa];
            ma = B.has_mass ? m[pa] : B.m_const;
            if (MOM) va = vel[pa];
        }
        if (pb < p1) {
            xb = x[pb]; yb = y[pb]; zb = z[pb];
            mb = B.has_mass ? m[pb] : B.m_const;
            if (MOM) vb = vel[pb];
        }
    };
    load2(p0 + threadIdx.x);
    for (int c = threadIdx.x; c < (F32 ? LC : 2 * LC); c += kBlock) acc[c] = 0ull;
    __syncthreads();
    int E = B.fx_exp;
    if (MOM) {
        const double vmax = __longlong_as_double((long long)mom.maxbits[3 * sg.box + comp]);
        E = vmax > 0.0 ? ilogb(vmax) : 0;
    }
    // one particle's CIC contributions as two fixed-point words: w * 2^(31-E) =
    // hi + lo * 2^-32 (hi < 2^32 since w < 2^(E+1); lo rounded, a rounding up to
    // 2^32 carried into hi), both converted with the native f64 -> u32 instruction
    auto dep = [&](double px, double py, double pz, double mp, double vp) {
        if (isnan(px)) return;  // empty slot
        double xint, yint, zint;
        const int i = cic_index(px, B.plo[0], B.dxi[0], &xint);
        const int j = cic_index(py, B.plo[1], B.dxi[1], &yint);
        const int k = cic_index(pz, B.plo[2], B.dxi[2], &zint);
        // an index more than one period out (flag 1) or a cell outside the tile
        // the particle is binned in (flag 2): one branch for both, rarely taken
        const bool far = (unsigned)(i + B.n[0]) >= (unsigned)(3 * B.n[0]) ||
                         (unsigned)(j + B.n[1]) >= (unsigned)(3 * B.n[1]) ||
                         (unsigned)(k + B.n[2]) >= (unsigned)(3 * B.n[2]);
        const int iw = wrap1(i, B.n[0]) - o0;
        const int jw = wrap1(j, B.n[1]) - o1;
        const int kw = wrap1(k, B.n[2]) - o2;
        const bool outside = (unsigned)iw >= (unsigned)bx || (unsigned)jw >= (unsigned)by ||
                             (unsigned)kw >= (unsigned)bz;
        if (far || outside) {
            raise_err(err, (far ? 1 : 0) | (outside ? 2 : 0));
            return;
        }
        if (F32) {
            const float scale = ldexpf(1.0f, 31 - E);
            const float fx = (float)xint, fy = (float)yint, fz = (float)zint, fm = (float)mp;
            const float sx[2] = {1.0f - fx, fx};
            const float sy[2] = {1.0f - fy, fy};
            const float sz[2] = {1.0f - fz, fz};
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int ii = 0; ii < 2; ++ii) {
                        const float w = sx[ii] * sy[jj] * sz[kk] * fm;
                        const int idx = ((kw + kk) * Ly + (jw + jj)) * Lx + (iw + ii);
                        atomicAdd(&acc[idx], (unsigned long long)fx32_units(w, scale));
                    }
            return;
        }
        const double sx[2] = {1.0 - xint, xint};
        const double sy[2] = {1.0 - yint, yint};
        const double sz[2] = {1.0 - zint, zint};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int ii = 0; ii < 2; ++ii) {
                    const double w = sx[ii] * sy[jj] * sz[kk] * mp;
                    const double s = MOM ? ldexp(w * vp, 30 - E) : ldexp(w, 31 - E);  // MOM: |s| < 2^31
                    const double hf = floor(s);
                    const double lr = rint(ldexp(s - hf, 32));
                    const bool carry = lr >= 4294967296.0;
                    const unsigned long long hi =
                        MOM ? (unsigned long long)((long long)(int)hf + (carry ? 1 : 0))
                            : (unsigned long long)(unsigned)hf + (carry ? 1ull : 0ull);
                    const unsigned long long lo = carry ? 0ull : (unsigned long long)(unsigned)lr;
                    const int idx = ((kw + kk) * Ly + (jw + jj)) * Lx + (iw + ii);
                    atomicAdd(&acc[idx], hi);
                    atomicAdd(&acc[LC + idx], lo);
                }
    };
    // two particles per thread, both loaded before either is deposited
    for (long long pa = p0 + threadIdx.x; pa < p1; pa += 2 * kBlock) {
        if (pa != p0 + threadIdx.x) load2(pa);
        dep(xa, ya, za, ma, va);
        if (pa + kBlock < p1) dep(xb, yb, zb, mb, vb);
    }
    __syncthreads();
    if (MOM && hv.split >= 0) hv.split += comp * split_cap;
    if (hv.nparts > 1 && !split_combine(acc, F32 ? LC : 2 * LC, hv, split_acc, split_words, split_done)) return;
    // write-out by rows of Lx cells (Lx <= 33 < 64): a wave takes rpw rows per
    // pass, so no cell needs a division for its coordinates
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int rpw = kWave / Lx;
    const int lrow = lane / Lx, lx = lane - lrow * Lx;
    if (lrow < rpw) {
        const int step = (kBlock / kWave) * rpw;
        const int r0 = wave * rpw + lrow;
        int ly = r0 % Ly, lz = r0 / Ly;
        const int dly = step % Ly, dlz = step / Ly;
        while (lz < Lz) {
            const int c = (lz * Ly + ly) * Lx + lx;
            const double v = F32   ? ldexp((double)acc[c], E - 31)
                             : MOM ? ldexp((double)(long long)acc[c], E - 30) + ldexp((double)acc[LC + c], E - 62)
                                   : ldexp((double)acc[c], E - 31) + ldexp((double)acc[LC + c], E - 63);
            if (lx > 0 && ly > 0 && lz > 0)
                own[B.cell_off + cidx(o0 + lx - 1, o1 + ly - 1, o2 + lz - 1, B.n[0], B.n[1])] = v;
            else
                halo[gt * B.halo_stride + halo_index(lx, ly, lz, bx, by, bz)] = v;
            ly += dly;
            lz += dlz;
            if (ly >= Ly) {
                ly -= Ly;
                ++lz;
            }
        }
    }
}

// atomicMax of a block's largest value (bit patterns), skipped where the slot already
// holds as much: the slot only grows, so a stale read costs an atomic at most (one
// atomic per block on one word took ~12 ns each, one per particle 1.2 ms in all).
__device__ __forceinline__ void block_max_to(unsigned long long v, unsigned long long* slot) {
    for (int o = kWave / 2; o > 0; o >>= 1) v = max(v, (unsigned long long)__shfl_xor((long long)v, o));
    __shared__ unsigned long long wmax[kBlock / kWave];
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) wmax[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / kWave; ++w) v = max(v, wmax[w]);
        if (v > __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(slot, v);
    }
}

// max |m v_d| per box and component (bit patterns) for the momentum deposit.
__global__ void __launch_bounds__(kBlock) k_max_mom(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                    const double* __restrict__ x, const double* __restrict__ m,
                                                    const double* __restrict__ vx, const double* __restrict__ vy,
                                                    const double* __restrict__ vz, unsigned long long* maxbits) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blockIdx.x - sg.blk0) * kBlock + threadIdx.x;
    const long long p = B.part_off + q;
    unsigned long long b0 = 0, b1 = 0, b2 = 0;
    if (q < B.span && !isnan(x[p])) {
        const double mp = B.has_mass ? m[p] : B.m_const;
        b0 = dbits(fabs(mp * vx[p]));
        b1 = dbits(fabs(mp * vy[p]));
        b2 = dbits(fabs(mp * vz[p]));
    }
    block_max_to(b0, maxbits + 3 * sg.box + 0);
    block_max_to(b1, maxbits + 3 * sg.box + 1);
    block_max_to(b2, maxbits + 3 * sg.box + 2);
}

// Sum of a block's values in a fixed order (wave butterfly, then waves in order).
__device__ __forceinline__ double block_sum_fixed(double v) {
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __shared__ double ws[kBlock / kWave];
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) ws[threadIdx.x / kWave] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) t += ws[w];
    return t;
}

// The edge and corner terms of cell (i, j, k) after SumBoundary: the low-halo
// entries of the upper neighbour tiles across two or three of the tile's top
// faces (neighbour in xy, xz, yz, xyz, in that order), added to v.
__device__ __forceinline__ double fold_edges(const BoxDev& B, const double* __restrict__ halo, double v, int tx,
                                             int ty, int tz, int li, int lj, int lk, bool topx, bool topy,
                                             bool topz) {
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int T0 = B.tile[0], T1 = B.tile[1], T2 = B.tile[2];
    const int nt0 = B.ntile[0], nt1 = B.ntile[1], nt2 = B.ntile[2];
    const int sel[4] = {3, 5, 6, 7};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int S = sel[s];
        const bool sx = S & 1, sy = S & 2, sz = S & 4;
        if ((sx && !topx) || (sy && !topy) || (sz && !topz)) continue;
        int ntx = tx + (sx ? 1 : 0), nty = ty + (sy ? 1 : 0), ntz = tz + (sz ? 1 : 0);
        if (ntx == nt0) ntx = 0;
        if (nty == nt1) nty = 0;
        if (ntz == nt2) ntz = 0;
        const int nbx = min(T0, nx - ntx * T0), nby = min(T1, ny - nty * T1), nbz = min(T2, nz - ntz * T2);
        const int hx = sx ? 0 : li + 1, hy = sy ? 0 : lj + 1, hz = sz ? 0 : lk + 1;
        const long long nt = B.tile_off + ((long long)ntz * nt1 + nty) * nt0 + ntx;
        v += halo[nt * B.halo_stride + halo_index(hx, hy, hz, nbx, nby, nbz)];
    }
    return v;
}

// Row-major walk over a block's share of a box's cells: block b of the piece takes
// cells [b*per, (b+1)*per) (per a multiple of kBlock, so whole cache lines), each
// thread every kBlock-th of them in order; body(i, j, k, c) per cell.  The cell
// order of each thread is fixed, so per-thread sums are reproducible.
template <class F>
__device__ __forceinline__ void for_block_cells(const CellSeg& sg, const BoxDev& B, F body) {
    const int nx = B.n[0], ny = B.n[1];
    const long long N = (long long)nx * ny * B.n[2];
    long long per = (N + sg.nblk - 1) / sg.nblk;
    per = (per + kBlock - 1) / kBlock * kBlock;
    const long long c0 = (long long)(blockIdx.x - sg.blk0) * per;
    const long long c1 = min(N, c0 + per);
    long long c = c0 + threadIdx.x;
    if (c >= c1) return;
    const long long plane = (long long)nx * ny;
    int k = (int)(c / plane);
    const long long rem = c - (long long)k * plane;
    int j = (int)(rem / nx);
    int i = (int)(rem - (long long)j * nx);
    for (; c < c1; c += kBlock) {
        body(i, j, k, c);
        i += kBlock;
        if (i >= nx) {
            const int t = i / nx;
            i -= t * nx;
            j += t;
            if (j >= ny) {
                const int u = j / ny;
                j -= u * ny;
                k += u;
            }
        }
    }
}

// The folded deposit (SumBoundary) of a block's share of a box's cells, in
// for_block_cells' order (the same cells per thread, in the same sequence):
// own deposit plus the low-halo entries of the up-to-7 upper neighbour tiles
// that hold the cell, added in a fixed order (neighbour in x, y, z, xy, xz, yz,
// xyz); emit(q, v) per cell in order.  U cells per thread at a time: their own
// values and face terms (x, y, z) are loaded before any is used, so a thread
// has up to 4U loads in flight; the edge and corner terms (cells on two or
// three top faces of a tile) follow them.  Coordinates advance by kBlock cells
// with block-uniform carries instead of divisions.  C fields of the same tiles at
// once (their addresses derived once): emit(q, v, u) gets the C values of a cell, the
// u-th of the thread's U in flight.  V consecutive shares of the piece's nv in one block
// (its block b takes shares b*V ..): with shares of kBlock cells and V <= U, the u-th
// cell of a thread is its one cell of share b*V + u.
template <int C>
struct FoldFields {
    const double* own[C];
    const double* halo[C];
};
template <int U, int C, class F>
__device__ __forceinline__ void fold_walk(const CellSeg& sg, int nv, int V, const BoxDev& B,
                                          const FoldFields<C>& fields, F emit) {
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int T0 = B.tile[0], T1 = B.tile[1], T2 = B.tile[2];
    const int nt0 = B.ntile[0], nt1 = B.ntile[1], nt2 = B.ntile[2];
    const long long N = (long long)nx * ny * nz;
    long long per = (N + nv - 1) / nv;
    per = (per + kBlock - 1) / kBlock * kBlock;
    const long long c0 = (long long)(blockIdx.x - sg.blk0) * V * per;
    const long long c1 = min(N, c0 + V * per);
    long long c = c0 + threadIdx.x;
    if (c >= c1) return;
    const long long plane = (long long)nx * ny;
    int k = (int)(c / plane);
    const long long rem = c - (long long)k * plane;
    int j = (int)(rem / nx);
    int i = (int)(rem - (long long)j * nx);
    // kBlock cells = dk planes + dj rows + di cells (block-uniform)
    const int di = kBlock % nx, dq = kBlock / nx;
    const int dj = dq % ny, dk = dq / ny;
    const long long hbase = B.tile_off;
    const long long hs = B.halo_stride;
    for (; c < c1; c += (long long)U * kBlock) {
        double v[U][C], hx[U][C], hy[U][C], hz[U][C];
        int cx[U], cy[U], cz[U];
        int fl[U];  // bit 0, 1, 2: on the tile's top x, y, z face; -1: past the block's cells
#pragma unroll
        for (int u = 0; u < U; ++u) {
            cx[u] = i;
            cy[u] = j;
            cz[u] = k;
            fl[u] = -1;
#pragma unroll
            for (int f = 0; f < C; ++f) hx[u][f] = hy[u][f] = hz[u][f] = 0.0;
            if (c + (long long)u * kBlock < c1) {
#pragma unroll
                for (int f = 0; f < C; ++f) v[u][f] = fields.own[f][B.cell_off + c + (long long)u * kBlock];
                const int tx = tile_div(i, B.tdiv[0]), ty = tile_div(j, B.tdiv[1]), tz = tile_div(k, B.tdiv[2]);
                const int li = i - tx * T0, lj = j - ty * T1, lk = k - tz * T2;
                const int bx = min(T0, nx - tx * T0), by = min(T1, ny - ty * T1), bz = min(T2, nz - tz * T2);
                const int lt = (tz * nt1 + ty) * nt0 + tx;
                fl[u] = (li == bx - 1 ? 1 : 0) | (lj == by - 1 ? 2 : 0) | (lk == bz - 1 ? 4 : 0);
                if (li == bx - 1) {  // x face of tile tx + 1 (same rows and planes)
                    const int nlt = tx + 1 == nt0 ? lt - tx : lt + 1;
                    const long long o = (hbase + nlt) * hs + (lk + 1) * (by + 1) + (lj + 1);
#pragma unroll
                    for (int f = 0; f < C; ++f) hx[u][f] = fields.halo[f][o];
                }
                if (lj == by - 1) {  // y face of tile ty + 1
                    const int nty = ty + 1 == nt1 ? 0 : ty + 1;
                    const int nby = min(T1, ny - nty * T1);
                    const int nlt = lt + (nty - ty) * nt0;
                    const long long o = (hbase + nlt) * hs + (nby + 1) * (bz + 1) + (lk + 1) * bx + li;
#pragma unroll
                    for (int f = 0; f < C; ++f) hy[u][f] = fields.halo[f][o];
                }
                if (lk == bz - 1) {  // z face of tile tz + 1
                    const int ntz = tz + 1 == nt2 ? 0 : tz + 1;
                    const int nbz = min(T2, nz - ntz * T2);
                    const int nlt = lt + (ntz - tz) * nt0 * nt1;
                    const long long o = (hbase + nlt) * hs + (by + 1) * (nbz + 1) + bx * (nbz + 1) + lj * bx + li;
#pragma unroll
                    for (int f = 0; f < C; ++f) hz[u][f] = fields.halo[f][o];
                }
            }
            i += di;
            j += dj;
            k += dk;
            if (i >= nx) {
                i -= nx;
                ++j;
            }
            if (j >= ny) {
                j -= ny;
                ++k;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int top = fl[u];
            if (top < 0) continue;
            double w[C];
#pragma unroll
            for (int f = 0; f < C; ++f) {
                w[f] = v[u][f];
                if (top & 1) w[f] += hx[u][f];
                if (top & 2) w[f] += hy[u][f];
                if (top & 4) w[f] += hz[u][f];
            }
            if (__builtin_popcount(top) >= 2) {
                const int tx = tile_div(cx[u], B.tdiv[0]), ty = tile_div(cy[u], B.tdiv[1]),
                          tz = tile_div(cz[u], B.tdiv[2]);
#pragma unroll
                for (int f = 0; f < C; ++f)
                    w[f] = fold_edges(B, fields.halo[f], w[f], tx, ty, tz, cx[u] - tx * T0, cy[u] - ty * T1,
                                      cz[u] - tz * T2, top & 1, top & 2, top & 4);
            }
            emit(B.cell_off + (size_t)(c + (long long)u * kBlock), w, u);
        }
    }
}

// Cells per thread in flight in the fold.
constexpr int kFoldU = 4;

// rho = (own + halos, fold_walk) * 1/vol; f = rho + (-mass_offset); sum of f per share
// for the solvability correction.  Cells in row-major order (coalesced reads of own and
// writes of f, whole cache lines).  rho itself is written only when the caller wants the
// density (AssignDensity); the step needs only f.
// The shares (and so the order of the sums) are the reducing table's blocks: piece s has
// s.ebuf of them from partial[s.coff] on, s.zchunk per block of this launch.  In boxes
// of up to 2^21 cells a share is one cell per thread, too little to have loads in
// flight: four shares per block took 52M cells of 64^3-128^3 boxes from 0.54 to 0.31 ms.
// Without such pieces (SHARES false) the shares' sums are not carried along: 256^3 72 us
// instead of 78.
template <bool WRITE_RHO, bool SHARES>
__global__ void __launch_bounds__(kBlock) k_fold(const CellSeg* segs, int nseg, const BoxDev* boxes,
                                                 const double* own, const double* __restrict__ halo,
                                                 double* rho, double* __restrict__ f,
                                                 double* __restrict__ partial) {
    // rho may be own itself (each cell is read, then written, by one thread)
    const CellSeg& sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const FoldFields<1> fields{{own}, {halo}};
    if (!SHARES) {
        double acc = 0.0;  // this thread's cells, in a fixed order
        fold_walk<kFoldU, 1>(sg, sg.nblk, 1, B, fields, [&](size_t q, const double (&v)[1], int) {
            const double rv = v[0] * B.inv_vol;
            if (WRITE_RHO) rho[q] = rv;
            const double fv = rv + (-B.mass_offset);
            f[q] = fv;
            acc += fv;
        });
        const double bs = block_sum_fixed(acc);
        if (threadIdx.x == 0) partial[sg.coff + (blockIdx.x - sg.blk0)] = bs;
        return;
    }
    const int V = sg.zchunk, nv = sg.ebuf;
    double acc[kFoldU];  // this thread's cells of each share, in a fixed order
#pragma unroll
    for (int u = 0; u < kFoldU; ++u) acc[u] = 0.0;
    fold_walk<kFoldU, 1>(sg, nv, V, B, fields, [&](size_t q, const double (&v)[1], int u) {
        const double rv = v[0] * B.inv_vol;
        if (WRITE_RHO) rho[q] = rv;
        const double fv = rv + (-B.mass_offset);
        f[q] = fv;
        if (V == 1)
            acc[0] += fv;
        else
            acc[u] += fv;
    });
    const int b0 = (int)(blockIdx.x - sg.blk0) * V;
    // each share's sum as block_sum_fixed forms it: a butterfly per wave, then the waves
    // in order
    __shared__ double ws[kFoldU][kBlock / kWave];
#pragma unroll
    for (int u = 0; u < kFoldU; ++u) {
        if (u >= V) break;
        for (int o = kWave / 2; o > 0; o >>= 1) acc[u] += __shfl_xor(acc[u], o);
        if ((threadIdx.x & (kWave - 1)) == 0) ws[u][threadIdx.x / kWave] = acc[u];
    }
    __syncthreads();
    if ((int)threadIdx.x < V && b0 + (int)threadIdx.x < nv) {
        double t = 0.0;
        for (int w = 0; w < kBlock / kWave; ++w) t += ws[threadIdx.x][w];
        partial[sg.coff + b0 + threadIdx.x] = t;
    }
}

// AssignDensityAndVels for one box (segs: its piece): the folded mass and momenta,
// rho = mass * 1/vol, v_d = mom_d / mass (0 without mass), written as 4 fields of the
// box's cells.  One pass over the four deposits (a fold per field into its own sums
// and a pass to divide them before: 5 launches, 80 B more per cell).
__global__ void __launch_bounds__(kBlock) k_fold_vels(const CellSeg* segs, const BoxDev* boxes, FoldFields<4> fields,
                                                      double* __restrict__ out) {
    CellSeg sg = segs[0];
    sg.blk0 = 0;
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const size_t nc = (size_t)B.n[0] * B.n[1] * B.n[2];
    fold_walk<2, 4>(sg, sg.nblk, 1, B, fields, [&](size_t q, const double (&v)[4], int) {
        double* o = out + (q - B.cell_off);
        const double ms = v[0];
        o[0] = ms * B.inv_vol;
#pragma unroll
        for (int d = 1; d < 4; ++d) o[d * nc] = ms != 0.0 ? v[d] / ms : 0.0;
    });
}

// sum = (S*dV)/ProbSize, as vol_weight_sum computes it (sum_utils.cpp:85-93).
__global__ void __launch_bounds__(kBlock) k_rhs_sum(const CellSeg* segs, const double* __restrict__ partial,
                                                    const double* __restrict__ dv_size, double* __restrict__ solv) {
    const CellSeg& sg = segs[blockIdx.x];
    double s = 0.0;
    // eight loads in flight, added in order (a load at a time: 12 us for 8192 shares)
    constexpr int U = 8;
    for (int b = threadIdx.x; b < sg.nblk; b += U * kBlock) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = partial[sg.blk0 + min(b + u * kBlock, sg.nblk - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * kBlock < sg.nblk) s += v[u];
    }
    const double S = block_sum_fixed(s);
    if (threadIdx.x == 0) {
        double sum = S * dv_size[2 * sg.box];
        sum = sum / dv_size[2 * sg.box + 1];
        solv[sg.box] = sum;
    }
}

// f = ((f + (-sum)) * Ggravity) * (1/a), Ggravity = -4 pi G.
__global__ void __launch_bounds__(kBlock) k_rhs_final(const CellSeg* segs, int nseg, const BoxDev* boxes,
                                                      const double* __restrict__ solv, double* __restrict__ f,
                                                      double Ggravity, double inv_a) {
    const CellSeg& sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long n = (long long)B.n[0] * B.n[1] * B.n[2];
    const long long q = (long long)(blockIdx.x - sg.blk0) * kBlock + threadIdx.x;
    if (q >= n) return;
    const double ns = -solv[sg.box];
    double v = f[B.cell_off + q] + ns;
    f[B.cell_off + q] = (v * Ggravity) * inv_a;
}

// ---------------------------------------------------------------------------
// gradient + CIC gather + kick (+ drift)
// ---------------------------------------------------------------------------

// Periodic position shift (Redistribute): above rhi -> subtract the length until
// not (clamp to lo on undershoot); below lo -> add until not (clamp to rhi).
// A coordinate more than two periods away (or not finite) is clamped and flagged
// instead of looping.
__device__ __forceinline__ double periodic_shift(double v, double lo, double rhi, double len, int* err) {
    if (!(v >= lo - 2.0 * len && v <= rhi + 2.0 * len)) {
        if (err) raise_err(err, 8);
        return (v < lo) ? lo : rhi;  // NaN compares false: goes to rhi
    }
    if (v > rhi) {
        while (v > rhi) v = v - len;
        if (v < lo) v = lo;
    } else if (v < lo) {
        while (v < lo) v = v + len;
        if (v > rhi) v = rhi;
    }
    return v;
}

// val[d] = sum_{kk,jj,ii} sx[1-ii]*sy[1-jj]*sz[1-kk] * g_d(i-ii, j-jj, k-kk) with
// g_d(c) = 0.5*(dxi*(phi(c) - phi(c-e_d)) + dxi*(phi(c+e_d) - phi(c))).
// G is the interpolation arithmetic: double (the drop-in) or float (the
// mixed-precision step: g of each corner cell formed in FP64 and rounded to
// FP32, the fractions rounded to FP32, the weights and the sum in FP32, in the
// order of the staged kick, so the two agree bit for bit).  Forming g in FP64
// first keeps the difference of neighbouring phi values exact: phi rounded to
// FP32 first would lose ~n/2pi times more of g's digits to cancellation.
template <typename G>
__device__ __forceinline__ void gather_grad(const BoxDev& B, const double* __restrict__ P, double x, double y,
                                            double z, double val[3], int* err) {
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    double xint, yint, zint;
    const int i = cic_index(x, B.plo[0], B.dxi[0], &xint);
    const int j = cic_index(y, B.plo[1], B.dxi[1], &yint);
    const int k = cic_index(z, B.plo[2], B.dxi[2], &zint);
    if (i < -nx + 2 || i >= 2 * nx - 1 || j < -ny + 2 || j >= 2 * ny - 1 || k < -nz + 2 || k >= 2 * nz - 1)
        raise_err(err, 4);
    int ix[4], iy[4], iz[4];
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) {
        ix[mm] = wrap1(i - 2 + mm, nx);
        iy[mm] = wrap1(j - 2 + mm, ny);
        iz[mm] = wrap1(k - 2 + mm, nz);
    }
    const G sx[2] = {G(1) - G(xint), G(xint)};
    const G sy[2] = {G(1) - G(yint), G(yint)};
    const G sz[2] = {G(1) - G(zint), G(zint)};
    auto ld = [&](int a, int b, int c) -> double { return P[cidx(ix[a], iy[b], iz[c], nx, ny)]; };
    const double dxi0 = B.dxi[0], dxi1 = B.dxi[1], dxi2 = B.dxi[2];
    G v0 = G(0), v1 = G(0), v2 = G(0);
#pragma unroll
    for (int kk = 0; kk <= 1; ++kk)
#pragma unroll
        for (int jj = 0; jj <= 1; ++jj)
#pragma unroll
            for (int ii = 0; ii <= 1; ++ii) {
                const int a = 2 - ii, b = 2 - jj, c = 2 - kk;
                const double pc = ld(a, b, c);
                const G gx = G(0.5 * (dxi0 * (pc - ld(a - 1, b, c)) + dxi0 * (ld(a + 1, b, c) - pc)));
                const G gy = G(0.5 * (dxi1 * (pc - ld(a, b - 1, c)) + dxi1 * (ld(a, b + 1, c) - pc)));
                const G gz = G(0.5 * (dxi2 * (pc - ld(a, b, c - 1)) + dxi2 * (ld(a, b, c + 1) - pc)));
                const G w = sx[1 - ii] * sy[1 - jj] * sz[1 - kk];
                v0 += w * gx;
                v1 += w * gy;
                v2 += w * gz;
            }
    val[0] = double(v0);
    val[1] = double(v1);
    val[2] = double(v2);
}

// moveKickDrift (DO_MOVE) or moveKick (!DO_MOVE) of update_dm_particle_single:
//   v = (a_prev*v + (0.5*dt)*val) * (1/a_cur);  DO_MOVE: x += (dt*(1/a_cur))*v
// DO_MOVE also bins the drifted particle (key + count for the next deposit);
// !DO_MOVE applies the periodic shift of Redistribute.
template <bool DO_MOVE, typename G>
__global__ void __launch_bounds__(kBlock) k_kick(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                 const double* __restrict__ phi, double* __restrict__ x,
                                                 double* __restrict__ y, double* __restrict__ z,
                                                 double* __restrict__ vx, double* __restrict__ vy,
                                                 double* __restrict__ vz, double dt, double a_prev, double a_cur,
                                                 int* __restrict__ key, int* counts, int* err) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blockIdx.x - sg.blk0) * kBlock + threadIdx.x;
    const long long p = B.part_off + q;
    double px = 0.0;
    if (q < B.span) {
        px = x[p];
        if (DO_MOVE && isnan(px)) key[p] = -1;  // empty slot
    }
    const bool valid = q < B.span && !isnan(px);
    int t = 0;
    if (valid) {
        const double half_dt = 0.5 * dt;
        const double a_cur_inv = 1.0 / a_cur;
        const double dt_a_cur_inv = dt * a_cur_inv;
        double py = y[p], pz = z[p];
        double val[3];
        gather_grad<G>(B, phi + B.cell_off, px, py, pz, val, err);
        double ux = a_prev * vx[p] + half_dt * val[0];
        ux = ux * a_cur_inv;
        double uy = a_prev * vy[p] + half_dt * val[1];
        uy = uy * a_cur_inv;
        double uz = a_prev * vz[p] + half_dt * val[2];
        uz = uz * a_cur_inv;
        vx[p] = ux;
        vy[p] = uy;
        vz[p] = uz;
        if (DO_MOVE) {
            px = px + dt_a_cur_inv * ux;
            py = py + dt_a_cur_inv * uy;
            pz = pz + dt_a_cur_inv * uz;
            x[p] = px;
            y[p] = py;
            z[p] = pz;
            t = tile_of(B, px, py, pz, err);
            key[p] = t;
        } else {
            const double sxp = periodic_shift(px, B.plo[0], B.rhi[0], B.len[0], err);
            const double syp = periodic_shift(py, B.plo[1], B.rhi[1], B.len[1], err);
            const double szp = periodic_shift(pz, B.plo[2], B.rhi[2], B.len[2], err);
            if (sxp != px) x[p] = sxp;
            if (syp != py) y[p] = syp;
            if (szp != pz) z[p] = szp;
        }
    }
    if (DO_MOVE) agg_atomic_add(counts, t, valid);
}

// Work items for the tile-staged particle kernels: each tile's occupied slot
// range [tbase, tbase + thw) cut into chunks of at most kChunk slots (empty
// tiles give none).  Slots are
// reserved with one atomic per wave, so the item order varies between runs; every
// item is processed independently, so results do not.
constexpr int kChunk = 16 * kBlock;  // default particles per work item (fewer items: less phi staging)

// Entries of a tile above which a wave writes them together: one thread takes ~50 ns an
// entry, and a clump's tile has up to 2048 parts and np / chunk items (4 10^6 particles in
// one cell of 64^3: 146 -> 12 us, half of 2^24 in one cell of 256^3: 149 -> 15 us).
constexpr int kItemsByThread = 8;

struct TileItem {
    long long p0;   // first particle
    int np;         // particles in this chunk
    int tile;       // global tile id
};

__global__ void __launch_bounds__(kBlock) k_make_items(const long long* __restrict__ tbase,
                                                       const int* __restrict__ thw, long long ntiles,
                                                       TileItem* __restrict__ items, int* nitems, int chunk,
                                                       HeavyItem* __restrict__ heavy, int* nheavy, int* nsplit,
                                                       long long split_min, int split_part, int split_cap,
                                                       const int* mig, int* h_mig, Resort resort,
                                                       long long* h_resort) {
    const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
    // the migration's flags to the host's mirror (pinned memory) along the way, or in a
    // captured step the outcome of the re-sort
    if (mig && t < 2) __hip_atomic_store(&h_mig[t], mig[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (resort.state && t == 0) {
        long long* st = resort.state;
        const bool full = resort_full(resort);
        st[0] = full ? 0 : st[0] + resort.mig[1];
        st[full ? 1 : 2] += 1;
        st[3] += resort.mig[1];
        for (int q = 0; q < 4; ++q)
            __hip_atomic_store(&h_resort[q], st[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // a migration that ran out of slack has counted the particles it could not place in
    // thw, whose sum then passes the slots that the lists are sized for: no lists (the
    // full sort that follows makes them)
    const bool overflow = mig && mig[0] != 0;
    int nc = 0, parts = 0, len = 0, split = -1, h = 0;
    long long p0 = 0, cnt = 0;
    if (t < ntiles && !overflow) {
        p0 = tbase[t];
        cnt = thw[t];
        nc = (int)((cnt + chunk - 1) / chunk);
    }
    // wave-inclusive prefix of nc, one atomic per wave, before the atomics of the heavy
    // tiles: the kicks want the items in tile order (each XCD a run of neighbouring tiles),
    // and waves that reach it a round trip or two late scatter their items (512^3 particles,
    // half of them in clumps, FP64: kick 2.72 -> 2.51 ms, paired kick 6.97 -> 6.77)
    const int lane = threadIdx.x & (kWave - 1);
    int incl = nc;
    for (int o = 1; o < kWave; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    const int total = __shfl(incl, kWave - 1);
    int base = 0;
    if (lane == kWave - 1 && total > 0) base = atomicAdd(nitems, total);
    base = __shfl(base, kWave - 1);
    int slot = base + incl - nc;
    // tiles the deposit starts first (the longest blocks), the heaviest in parts
    if (cnt > kHeavyTile) {
        parts = 1;
        len = (int)cnt;
        if (cnt > split_min) split = atomicAdd(nsplit, 1);
        if (split >= split_cap) split = -1;
        if (split >= 0) {
            len = split_part;
            parts = (int)((cnt + len - 1) / len);
        }
        h = atomicAdd(nheavy, parts);
    }
    auto put_item = [&](int at, int c, long long p, long long n, int tile) {
        TileItem it;
        it.p0 = p + (long long)c * chunk;
        it.np = (int)min((long long)chunk, n - (long long)c * chunk);
        it.tile = tile;
        items[at + c] = it;
    };
    auto put_heavy = [&](int at, int q, int l, long long n, int np, int sp, int tile) {
        heavy[at + q] = HeavyItem{tile, q * l, (int)min((long long)l, n - (long long)q * l), np, sp};
    };
    // a tile of few entries by its thread, one of many by the whole wave
    const bool wide = max(nc, parts) > kItemsByThread;
    if (!wide) {
        for (int c = 0; c < nc; ++c) put_item(slot, c, p0, cnt, (int)t);
        for (int q = 0; q < parts; ++q) put_heavy(h, q, len, cnt, parts, split, (int)t);
    }
    for (unsigned long long m = __ballot(wide); m; m &= m - 1) {
        const int src = __ffsll((long long)m) - 1;
        const long long wp = __shfl(p0, src), wn = __shfl(cnt, src);
        const int wt = __shfl((int)t, src), wc = __shfl(nc, src), ws = __shfl(slot, src);
        const int wparts = __shfl(parts, src), wh = __shfl(h, src), wl = __shfl(len, src), wsp = __shfl(split, src);
        for (int c = lane; c < wc; c += kWave) put_item(ws, c, wp, wn, wt);
        for (int q = lane; q < wparts; q += kWave) put_heavy(wh, q, wl, wn, wparts, wsp, wt);
    }
}

// NyxParticleContainer::estTimestep (NyxParticleContainer.H:327-410) for one
// particle: cfl / max_d(|v_d| dxi_d / a), capped by 1 / sqrt(|g| dxi_x) with g the
// cell-centred gravity of the particle's cell (cell = floor((x - plo) dxi)).
__device__ __forceinline__ double particle_dt(double ux, double uy, double uz, double adxi0, double adxi1,
                                              double adxi2, double ax, double ay, double az, double dxi0,
                                              double cfl) {
    const double mx = fabs(ux) * adxi0;
    const double my = fabs(uy) * adxi1;
    const double mz = fabs(uz) * adxi2;
    double m = mx > my ? mx : my;
    m = m > mz ? m : mz;
    double dtp = (m > 0) ? (cfl / m) : 1e50;
    const double mag = sqrt(ax * ax + ay * ay + az * az);
    if (mag > 0) {
        const double da = 1 / sqrt(mag * dxi0);
        dtp = dtp < da ? dtp : da;
    }
    return dtp;
}

// Cell-centred gravity (k_grav_vector's arithmetic, rounded to G as the staged
// kick keeps it) at cell (i, j, k) of a box.
template <typename G>
__device__ __forceinline__ void grav_at(const BoxDev& B, const double* __restrict__ P, int i, int j, int k,
                                        double& gx, double& gy, double& gz) {
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int im = i == 0 ? nx - 1 : i - 1, ip = i == nx - 1 ? 0 : i + 1;
    const int jm = j == 0 ? ny - 1 : j - 1, jp = j == ny - 1 ? 0 : j + 1;
    const int km = k == 0 ? nz - 1 : k - 1, kp = k == nz - 1 ? 0 : k + 1;
    const double pc = P[cidx(i, j, k, nx, ny)];
    gx = double(G(0.5 * (B.dxi[0] * (pc - P[cidx(im, j, k, nx, ny)]) + B.dxi[0] * (P[cidx(ip, j, k, nx, ny)] - pc))));
    gy = double(G(0.5 * (B.dxi[1] * (pc - P[cidx(i, jm, k, nx, ny)]) + B.dxi[1] * (P[cidx(i, jp, k, nx, ny)] - pc))));
    gz = double(G(0.5 * (B.dxi[2] * (pc - P[cidx(i, j, km, nx, ny)]) + B.dxi[2] * (P[cidx(i, j, kp, nx, ny)] - pc))));
}

// The estimate from global phi (any position; cells wrapped periodically).
template <typename G>
__device__ __forceinline__ double particle_dt_global(const BoxDev& B, const double* __restrict__ P, double px,
                                                     double py, double pz, double ux, double uy, double uz,
                                                     double a, double cfl) {
    const int i = wrap1((int)floor((px - B.plo[0]) * B.dxi[0]), B.n[0]);
    const int j = wrap1((int)floor((py - B.plo[1]) * B.dxi[1]), B.n[1]);
    const int k = wrap1((int)floor((pz - B.plo[2]) * B.dxi[2]), B.n[2]);
    double gx, gy, gz;
    grav_at<G>(B, P, i, j, k, gx, gy, gz);
    return particle_dt(ux, uy, uz, B.dxi[0] / a, B.dxi[1] / a, B.dxi[2] / a, gx, gy, gz, B.dxi[0], cfl);
}

// Minimum over a block into a per-box slot (bit pattern of a positive double:
// atomicMin is exact and order independent).
__device__ __forceinline__ void block_min_to(double v, unsigned long long* slot) {
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double w = __shfl_xor(v, o);
        v = w < v ? w : v;
    }
    __shared__ double wmin[kBlock / kWave];
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) wmin[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = wmin[0];
        for (int w = 1; w < kBlock / kWave; ++w) m = wmin[w] < m ? wmin[w] : m;
        // (the slot only falls: see block_max_to)
        const unsigned long long b = dbits(m);
        if (m < 1e50 && b < __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(slot, b);
    }
}

// Standalone estimate over every particle (nyxpm_est_time_step when no fused
// estimate of the current state is kept).
template <typename G>
__global__ void __launch_bounds__(kBlock) k_est_dt(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                   const double* __restrict__ phi, const double* __restrict__ x,
                                                   const double* __restrict__ y, const double* __restrict__ z,
                                                   const double* __restrict__ vx, const double* __restrict__ vy,
                                                   const double* __restrict__ vz, double a, double cfl,
                                                   unsigned long long* dtmin) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blockIdx.x - sg.blk0) * kBlock + threadIdx.x;
    double d = 1e50;
    if (q < B.span) {
        const long long p = B.part_off + q;
        const double px = x[p];
        if (!isnan(px)) d = particle_dt_global<G>(B, phi + B.cell_off, px, y[p], z[p], vx[p], vy[p], vz[p], a, cfl);
    }
    block_min_to(d, dtmin + sg.box);
}

// Kick variants of the tile-staged particle kernel.
// Cells of g per thread that the tile-staged kernel keeps in registers to
// write g over the staged phi (tiles of up to kBlock * kKickG g cells).
constexpr int kKickG = 8;
constexpr int kKick = 0;       // moveKick: kick, then the periodic shift of Redistribute
constexpr int kKickDrift = 1;  // moveKickDrift: kick, drift, new tile key
constexpr int kKickPair = 2;   // moveKick of one step followed by moveKickDrift of the next

// Particles the tile-staged kernel hands over to k_kick_deferred: index (bits
// 0-39), box (bits 40-59) and what is left to do (bit 62: the kick-drift half of
// a pair whose kick is already stored; bit 61: only the time-step estimate of
// the stored state; neither: the whole update of the launch).
constexpr long long kDeferPairKD = 1LL << 62;
constexpr long long kDeferDtOnly = 1LL << 61;  // update done; only the time-step estimate is left
__device__ __forceinline__ long long defer_entry(long long p, int box) {
    return p | ((long long)box << 40);
}

// g (the average of the face gradients) on the (tile+1)^3 cells that the particles of
// the tile at (o0, o1, o2), bx x by x bz cells, interpolate from, in LDS: phi of the tile
// and a halo of 2 staged at sphi, then the three components of a cell side by side.
// Returns g's place (over the staged phi or behind it); the caller's barrier follows.
template <typename G>
__device__ __forceinline__ const G* stage_g(const BoxDev& B, const double* __restrict__ P, double* sphi, int o0, int o1,
                                            int o2, int bx, int by, int bz) {
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int SX = bx + 3, SY = by + 3, SZ = bz + 3;
    const int GX = bx + 1, GY = by + 1, GZ = bz + 1;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    {
        // rows of SX cells: a wave takes rpw rows per pass (SX <= 35 < 64).  The
        // passes go in batches of kStageBatch: every load of a batch is issued
        // before any of them is stored, so their latencies overlap (one load,
        // wait, store per pass left 8 serial latencies per lane and tile).  Rows
        // past the last are clamped onto it (the extra lanes store the owner's
        // value to the same LDS word), so no branch separates the loads.
        constexpr int kStageBatch = 8;
        const int rpw = kWave / SX;
        const int lrow = lane / SX, lx = lane - lrow * SX;
        if (lrow < rpw) {
            const size_t gx = (size_t)wrap1(o0 - 2 + lx, nx);
            const int step = (kBlock / kWave) * rpw;
            const int r0 = wave * rpw + lrow;
            int ly = r0 % SY, lz = r0 / SY;
            const int dly = step % SY, dlz = step / SY;
            while (lz < SZ) {
                double v[kStageBatch];
                int o[kStageBatch];
#pragma unroll
                for (int u = 0; u < kStageBatch; ++u) {
                    const bool in = lz < SZ;
                    const int cy = in ? ly : SY - 1, cz = in ? lz : SZ - 1;
                    const int gy = wrap1(o1 - 2 + cy, ny), gz = wrap1(o2 - 2 + cz, nz);
                    v[u] = P[((size_t)gz * ny + gy) * nx + gx];
                    o[u] = (cz * SY + cy) * SX + lx;
                    ly += dly;
                    lz += dlz;
                    if (ly >= SY) {
                        ly -= SY;
                        ++lz;
                    }
                }
#pragma unroll
                for (int u = 0; u < kStageBatch; ++u) sphi[o[u]] = v[u];
            }
        }
    }
    __syncthreads();
    const double dxi0 = B.dxi[0], dxi1 = B.dxi[1], dxi2 = B.dxi[2];
    // g at the cells the tile's particles interpolate from (local -1 .. b-1 per
    // dimension), components of a cell adjacent; formed in FP64, kept as G.
    // Where every thread's share fits in registers (kKickG cells) g is formed
    // there and, after a barrier, written over the staged phi, which it no
    // longer needs: the block holds the larger of the two arrays instead of both
    // (more blocks per CU); otherwise g goes beside the staged phi.
    const int ng = GX * GY * GZ;
    const bool alias = ng <= kBlock * kKickG;
    G* sg = reinterpret_cast<G*>(alias ? sphi : sphi + SX * SY * SZ);
    if (alias) {
        G gv[kKickG][3];
        // cell index q = tid + u * kBlock, as (cx, cy, cz), advanced incrementally
        int cx = threadIdx.x % GX, cy = (threadIdx.x / GX) % GY, cz = threadIdx.x / (GX * GY);
        const int dcx = kBlock % GX, dcy = (kBlock / GX) % GY, dcz = kBlock / (GX * GY);
#pragma unroll
        for (int u = 0; u < kKickG; ++u) {
            if ((int)threadIdx.x + u * kBlock < ng) {
                const int o = ((cz + 1) * SY + (cy + 1)) * SX + (cx + 1);  // staged index of the cell
                const double pc = sphi[o];
                gv[u][0] = G(0.5 * (dxi0 * (pc - sphi[o - 1]) + dxi0 * (sphi[o + 1] - pc)));
                gv[u][1] = G(0.5 * (dxi1 * (pc - sphi[o - SX]) + dxi1 * (sphi[o + SX] - pc)));
                gv[u][2] = G(0.5 * (dxi2 * (pc - sphi[o - SX * SY]) + dxi2 * (sphi[o + SX * SY] - pc)));
            }
            cx += dcx;
            cy += dcy;
            cz += dcz;
            if (cx >= GX) {
                cx -= GX;
                ++cy;
            }
            if (cy >= GY) {
                cy -= GY;
                ++cz;
            }
        }
        __syncthreads();  // every read of the staged phi is done
#pragma unroll
        for (int u = 0; u < kKickG; ++u) {
            const int q = (int)threadIdx.x + u * kBlock;
            if (q < ng) {
                sg[3 * q] = gv[u][0];
                sg[3 * q + 1] = gv[u][1];
                sg[3 * q + 2] = gv[u][2];
            }
        }
    } else {
        const int rpw = kWave / GX;
        const int lrow = lane / GX, cx = lane - lrow * GX;
        if (lrow < rpw) {
            const int step = (kBlock / kWave) * rpw;
            const int r0 = wave * rpw + lrow;
            int cy = r0 % GY, cz = r0 / GY;
            const int dcy = step % GY, dcz = step / GY;
            while (cz < GZ) {
                const int o = ((cz + 1) * SY + (cy + 1)) * SX + (cx + 1);  // staged index of the cell
                const double pc = sphi[o];
                G* g = sg + 3 * ((cz * GY + cy) * GX + cx);
                g[0] = G(0.5 * (dxi0 * (pc - sphi[o - 1]) + dxi0 * (sphi[o + 1] - pc)));
                g[1] = G(0.5 * (dxi1 * (pc - sphi[o - SX]) + dxi1 * (sphi[o + SX] - pc)));
                g[2] = G(0.5 * (dxi2 * (pc - sphi[o - SX * SY]) + dxi2 * (sphi[o + SX * SY] - pc)));
                cy += dcy;
                cz += dcz;
                if (cy >= GY) {
                    cy -= GY;
                    ++cz;
                }
            }
        }
    }
    return sg;
}

// Tile-staged gather + kick(-drift).  phi over the tile plus a halo of 2 is
// staged in LDS once per item (rows of the staged box spread over the lanes of a
// wave, so the index arithmetic is per row), and g (the average of the face
// gradients, the three components of a cell side by side) is formed there on the
// (tile+1)^3 cells the CIC stencils of the tile's particles touch.  Same
// arithmetic as k_kick, bit for bit.
//
// kKickPair runs the closing kick of step n (a_prev, a_cur) and the opening
// kick-drift of step n+1 (a_prev2, a_cur2) in one pass: both use g from the same
// phi at the same position.  A particle moved by the periodic shift in between
// has its kick stored and its kick-drift deferred (to be interpolated again at
// the shifted position, as the separate kernels would); so is any particle whose
// cell falls outside the item's tile (binning older than a shift).  Deferral
// keeps those rare paths out of this kernel's registers.
//
// Binning for the next deposit (kick-drifts): with inc, the particles whose new
// tile differs from the item's are listed for k_migrate; otherwise every
// particle gets its key, and the tile counts are summed per block for the
// particles that stay in the item's tile (one atomic), counted individually
// for the others.
//
// EST (closing kicks only): also NyxParticleContainer::estTimestep of the kicked
// particles (cfl, a = a_cur) into dtmin, from the staged g; a compile-time
// variant so that the kernels without it keep their register budget.
template <int MODE, bool EST, typename G>
__global__ void __launch_bounds__(kBlock) k_kick_tiled(const BoxSeg* tsegs, int ntseg, const BoxDev* boxes,
                                                       const TileItem* __restrict__ items, const int* nitems,
                                                       const double* __restrict__ phi, double* __restrict__ x,
                                                       double* __restrict__ y, double* __restrict__ z,
                                                       double* __restrict__ vx, double* __restrict__ vy,
                                                       double* __restrict__ vz, double dt, double a_prev,
                                                       double a_cur, double a_prev2, double a_cur2,
                                                       int* __restrict__ key, int* counts,
                                                       long long* __restrict__ defer, int* ndefer, double cfl,
                                                       unsigned long long* dtmin, int inc,
                                                       long long* __restrict__ moves, int* nmove, int* err) {
    extern __shared__ __align__(16) unsigned char kick_smem[];
    double* sphi = reinterpret_cast<double*>(kick_smem);
    __shared__ int s_same[kBlock / kWave];
    // items are in (roughly) tile order; giving each XCD a contiguous range of them
    // lets neighbouring tiles share the phi halo lines in that XCD's L2
    const int n_items = *nitems;
    if ((int)blockIdx.x >= n_items) return;
    const TileItem it = items[xcd_block(blockIdx.x, n_items)];
    const int sgi = find_seg(tsegs, ntseg, it.tile);
    const int box = __builtin_amdgcn_readfirstlane(tsegs[sgi].box);
    // the box's fields as block-uniform values in registers: read through a
    // reference they would be re-read from memory (and waited for, behind the
    // particle stores) after every store or atomic of the particle loop
    const BoxDev B = boxes[box];
    const int lt = it.tile - tsegs[sgi].blk0;
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const int tx = lt % B.ntile[0], ty = (lt / B.ntile[0]) % B.ntile[1], tz = lt / (B.ntile[0] * B.ntile[1]);
    const int o0 = tx * B.tile[0], o1 = ty * B.tile[1], o2 = tz * B.tile[2];
    const int bx = min(B.tile[0], nx - o0), by = min(B.tile[1], ny - o1), bz = min(B.tile[2], nz - o2);
    const double* P = phi + B.cell_off;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    // the item's particles through block-uniform base pointers and 32-bit
    // indices (scalar base + vector offset addressing)
    double* __restrict__ X = x + it.p0;
    double* __restrict__ Y = y + it.p0;
    double* __restrict__ Z = z + it.p0;
    double* __restrict__ VX = vx + it.p0;
    double* __restrict__ VY = vy + it.p0;
    double* __restrict__ VZ = vz + it.p0;
    int* __restrict__ KEY = key + it.p0;
    // one particle per thread at a time, the first loaded before the staging of
    // phi so that its latency overlaps the staging.  (Two per thread in flight
    // need 12-27 more VGPRs, one wave per SIMD fewer: 2% slower in mixed
    // precision, 14% in FP64.)
    double ax = 0.0, ay = 0.0, az = 0.0, aux = 0.0, auy = 0.0, auz = 0.0;
    auto load1 = [&](int q) {
        ax = X[q]; ay = Y[q]; az = Z[q];
        aux = VX[q]; auy = VY[q]; auz = VZ[q];
    };
    if ((int)threadIdx.x < it.np) load1(threadIdx.x);
    const int GX = bx + 1, GY = by + 1;
    const double dxi0 = B.dxi[0], dxi1 = B.dxi[1], dxi2 = B.dxi[2];
    const G* sg = stage_g<G>(B, P, sphi, o0, o1, o2, bx, by, bz);
    __syncthreads();
    const double half_dt = 0.5 * dt;
    const double a_cur_inv = 1.0 / a_cur;
    const double dt_a_cur_inv = dt * a_cur_inv;
    const double a_cur2_inv = 1.0 / a_cur2;
    const double dt_a_cur2_inv = dt * a_cur2_inv;
    int same = 0;
    // time-step estimate of the state after the (closing) kick, a = a_cur
    constexpr bool est = EST && MODE != kKickDrift;
    const double adxi0 = dxi0 / a_cur, adxi1 = dxi1 / a_cur, adxi2 = dxi2 / a_cur;
    double dtmin_t = 1e50;
    // one particle: position (px, py, pz), velocity (qx, qy, qz), index q in the item
    auto one = [&](int q, double px, double py, double pz, double qx, double qy, double qz) {
        if (isnan(px)) return;  // empty slot
        double xint, yint, zint;
        const int i = cic_index(px, B.plo[0], dxi0, &xint);
        const int j = cic_index(py, B.plo[1], dxi1, &yint);
        const int k = cic_index(pz, B.plo[2], dxi2, &zint);
        const int li = wrap1(i, nx) - o0, lj = wrap1(j, ny) - o1, lk = wrap1(k, nz) - o2;
        if (li >= 0 && li < bx && lj >= 0 && lj < by && lk >= 0 && lk < bz) {
            // val_d = sum_{kk,jj,ii} sx[1-ii]*sy[1-jj]*sz[1-kk] * g_d(i-ii, j-jj, k-kk);
            // cell i-ii has g index li+1-ii
            const G fx = G(xint), fy = G(yint), fz = G(zint);
            const G mx = G(1) - fx, my = G(1) - fy, mz = G(1) - fz;
            G g0 = G(0), g1 = G(0), g2 = G(0);
#pragma unroll
            for (int kk = 0; kk <= 1; ++kk) {
                const G wz = kk ? mz : fz;
#pragma unroll
                for (int jj = 0; jj <= 1; ++jj) {
                    const G wy = jj ? my : fy;
                    const G* g = sg + 3 * (((lk + 1 - kk) * GY + (lj + 1 - jj)) * GX + li);
                    const G w0 = fx * wy * wz;  // ii = 0: cell i
                    g0 += w0 * g[3];
                    g1 += w0 * g[4];
                    g2 += w0 * g[5];
                    const G w1 = mx * wy * wz;  // ii = 1: cell i-1
                    g0 += w1 * g[0];
                    g1 += w1 * g[1];
                    g2 += w1 * g[2];
                }
            }
            const double v0 = double(g0), v1 = double(g1), v2 = double(g2);
            double ux = a_prev * qx + half_dt * v0;
            ux = ux * a_cur_inv;
            double uy = a_prev * qy + half_dt * v1;
            uy = uy * a_cur_inv;
            double uz = a_prev * qz + half_dt * v2;
            uz = uz * a_cur_inv;
            bool stay = true;  // the update of this launch completes here
            if (MODE == kKickDrift) {
                px = px + dt_a_cur_inv * ux;
                py = py + dt_a_cur_inv * uy;
                pz = pz + dt_a_cur_inv * uz;
            } else {
                // periodic_shift changes exactly the coordinates outside [plo, rhi]
                // (and flags the non-finite ones): the shifted values are formed
                // only on that rare path, so they hold no registers on the other
                const bool moved = !(px >= B.plo[0] && px <= B.rhi[0]) || !(py >= B.plo[1] && py <= B.rhi[1]) ||
                                   !(pz >= B.plo[2] && pz <= B.rhi[2]);
                if (est && !moved) {
                    // cell = floor((x - plo) dxi) is i or i-1 of the CIC index: in the staged g
                    const int ci = (int)floor((px - B.plo[0]) * dxi0) - (i - (li + o0));
                    const int cj = (int)floor((py - B.plo[1]) * dxi1) - (j - (lj + o1));
                    const int ck = (int)floor((pz - B.plo[2]) * dxi2) - (k - (lk + o2));
                    const G* gc = sg + 3 * (((ck - o2 + 1) * GY + (cj - o1 + 1)) * GX + (ci - o0 + 1));
                    const double d = particle_dt(ux, uy, uz, adxi0, adxi1, adxi2, double(gc[0]), double(gc[1]),
                                                 double(gc[2]), dxi0, cfl);
                    dtmin_t = d < dtmin_t ? d : dtmin_t;
                }
                if (moved) {
                    const double sxp = periodic_shift(px, B.plo[0], B.rhi[0], B.len[0], err);
                    const double syp = periodic_shift(py, B.plo[1], B.rhi[1], B.len[1], err);
                    const double szp = periodic_shift(pz, B.plo[2], B.rhi[2], B.len[2], err);
                    if (MODE == kKick) {
                        if (sxp != px) X[q] = sxp;
                        if (syp != py) Y[q] = syp;
                        if (szp != pz) Z[q] = szp;
                        if (est) defer[atomicAdd(ndefer, 1)] = defer_entry(it.p0 + q, box) | kDeferDtOnly;
                    } else {
                        // store the kick; the kick-drift follows in k_kick_deferred
                        X[q] = sxp;
                        Y[q] = syp;
                        Z[q] = szp;
                        stay = false;
                        defer[atomicAdd(ndefer, 1)] = defer_entry(it.p0 + q, box) | kDeferPairKD;
                    }
                } else if (MODE != kKick) {
                    double wx = a_prev2 * ux + half_dt * v0;
                    ux = wx * a_cur2_inv;
                    double wy = a_prev2 * uy + half_dt * v1;
                    uy = wy * a_cur2_inv;
                    double wz = a_prev2 * uz + half_dt * v2;
                    uz = wz * a_cur2_inv;
                    px = px + dt_a_cur2_inv * ux;
                    py = py + dt_a_cur2_inv * uy;
                    pz = pz + dt_a_cur2_inv * uz;
                }
            }
            // streaming stores (each particle is written once per pass; the
            // L2 keeps the phi lines the neighbouring tiles stage)
            __builtin_nontemporal_store(ux, &VX[q]);
            __builtin_nontemporal_store(uy, &VY[q]);
            __builtin_nontemporal_store(uz, &VZ[q]);
            if (MODE != kKick && stay) {
                __builtin_nontemporal_store(px, &X[q]);
                __builtin_nontemporal_store(py, &Y[q]);
                __builtin_nontemporal_store(pz, &Z[q]);
                const int t = tile_of(B, px, py, pz, err);
                if (inc) {
                    // incremental re-sort: only the particles that left the tile
                    wave_append(moves, nmove, defer_entry(it.p0 + q, box), t != it.tile);
                } else {
                    KEY[q] = t;
                    if (t == it.tile)
                        ++same;
                    else
                        atomicAdd(&counts[t], 1);
                }
            }
        } else {
            // binned in another tile: the whole update in k_kick_deferred
            defer[atomicAdd(ndefer, 1)] = defer_entry(it.p0 + q, box);
        }
    };
    for (int q = threadIdx.x; q < it.np; q += kBlock) {
        if (q != (int)threadIdx.x) load1(q);
        one(q, ax, ay, az, aux, auy, auz);
    }
    if (est) block_min_to(dtmin_t, dtmin + box);
    if (MODE != kKick) {
        for (int o = kWave / 2; o > 0; o >>= 1) same += __shfl_xor(same, o);
        if (lane == 0) s_same[wave] = same;
        __syncthreads();
        if (threadIdx.x == 0) {
            int tot = 0;
            for (int w = 0; w < kBlock / kWave; ++w) tot += s_same[w];
            if (tot) atomicAdd(&counts[it.tile], tot);
        }
    }
}

// The particles k_kick_tiled deferred, one thread each, phi read from global
// memory (gather_grad: same arithmetic as the staged path).
template <int MODE, typename G>
__global__ void __launch_bounds__(kBlock) k_kick_deferred(const long long* __restrict__ defer, const int* ndefer,
                                                          const BoxDev* boxes, const double* __restrict__ phi,
                                                          double* __restrict__ x, double* __restrict__ y,
                                                          double* __restrict__ z, double* __restrict__ vx,
                                                          double* __restrict__ vy, double* __restrict__ vz,
                                                          double dt, double a_prev, double a_cur, double a_prev2,
                                                          double a_cur2, int* __restrict__ key, int* counts,
                                                          double cfl, unsigned long long* dtmin, int inc,
                                                          long long* __restrict__ moves, int* nmove, int* err) {
    const int n = *ndefer;
    const bool est = MODE != kKickDrift && cfl > 0;
    const double half_dt = 0.5 * dt;
    // binning of a drifted particle (k_kick_tiled's rule; k_migrate finds out
    // whether a listed particle changed tile)
    auto bin = [&](long long p, int box, const BoxDev& B, double px, double py, double pz) {
        if (inc) {
            wave_append(moves, nmove, defer_entry(p, box), true);
        } else {
            const int t = tile_of(B, px, py, pz, err);
            key[p] = t;
            atomicAdd(&counts[t], 1);
        }
    };
    for (int q = blockIdx.x * kBlock + threadIdx.x; q < n; q += gridDim.x * kBlock) {
        const long long e = defer[q];
        const long long p = e & ((1LL << 40) - 1);
        const int box = (int)((e >> 40) & 0xFFFFF);
        const BoxDev& B = boxes[box];
        const double* P = phi + B.cell_off;
        double px = x[p], py = y[p], pz = z[p];
        double ux = vx[p], uy = vy[p], uz = vz[p];
        double val[3];
        if (e & kDeferDtOnly) {
            atomicMin(dtmin + box, dbits(particle_dt_global<G>(B, P, px, py, pz, ux, uy, uz, a_cur, cfl)));
            continue;
        }
        if (!(e & kDeferPairKD)) {
            const double a_cur_inv = 1.0 / a_cur;
            gather_grad<G>(B, P, px, py, pz, val, err);
            ux = a_prev * ux + half_dt * val[0];
            ux = ux * a_cur_inv;
            uy = a_prev * uy + half_dt * val[1];
            uy = uy * a_cur_inv;
            uz = a_prev * uz + half_dt * val[2];
            uz = uz * a_cur_inv;
            if (MODE == kKickDrift) {
                const double dt_a_cur_inv = dt * a_cur_inv;
                px = px + dt_a_cur_inv * ux;
                py = py + dt_a_cur_inv * uy;
                pz = pz + dt_a_cur_inv * uz;
                vx[p] = ux; vy[p] = uy; vz[p] = uz;
                x[p] = px; y[p] = py; z[p] = pz;
                bin(p, box, B, px, py, pz);
                continue;
            }
            const double sxp = periodic_shift(px, B.plo[0], B.rhi[0], B.len[0], err);
            const double syp = periodic_shift(py, B.plo[1], B.rhi[1], B.len[1], err);
            const double szp = periodic_shift(pz, B.plo[2], B.rhi[2], B.len[2], err);
            if (est)
                atomicMin(dtmin + box, dbits(particle_dt_global<G>(B, P, sxp, syp, szp, ux, uy, uz, a_cur, cfl)));
            if (MODE == kKick) {
                vx[p] = ux; vy[p] = uy; vz[p] = uz;
                if (sxp != px) x[p] = sxp;
                if (syp != py) y[p] = syp;
                if (szp != pz) z[p] = szp;
                continue;
            }
            const bool moved = sxp != px || syp != py || szp != pz;
            px = sxp;
            py = syp;
            pz = szp;
            if (moved) gather_grad<G>(B, P, px, py, pz, val, err);
        } else {
            // pair whose kick is stored: its estimate, then the kick-drift at the
            // shifted position
            if (est) atomicMin(dtmin + box, dbits(particle_dt_global<G>(B, P, px, py, pz, ux, uy, uz, a_cur, cfl)));
            gather_grad<G>(B, P, px, py, pz, val, err);
        }
        const double a_cur2_inv = 1.0 / a_cur2;
        const double dt_a_cur2_inv = dt * a_cur2_inv;
        double wx = a_prev2 * ux + half_dt * val[0];
        ux = wx * a_cur2_inv;
        double wy = a_prev2 * uy + half_dt * val[1];
        uy = wy * a_cur2_inv;
        double wz = a_prev2 * uz + half_dt * val[2];
        uz = wz * a_cur2_inv;
        px = px + dt_a_cur2_inv * ux;
        py = py + dt_a_cur2_inv * uy;
        pz = pz + dt_a_cur2_inv * uz;
        vx[p] = ux; vy[p] = uy; vz[p] = uz;
        x[p] = px; y[p] = py; z[p] = pz;
        bin(p, box, B, px, py, pz);
    }
}

// Incremental re-sort.  Each listed particle whose position now lies in another
// tile than the one whose slot range holds it is copied into the free slack of
// its new tile (slot thw[t]++), and its old slot is emptied (x = NaN).  A tile
// with no free slot sets flags[0]: the particle stays where it is and the
// caller sorts in full.  flags[1] counts the particles moved (= slots emptied).
// Destinations lie at or above every tile's high-water mark at launch, so no
// destination is a listed source.
__global__ void __launch_bounds__(kBlock) k_migrate(const long long* __restrict__ moves, const int* nmove,
                                                    const BoxDev* boxes, const long long* __restrict__ tbase,
                                                    const int* __restrict__ tcap, int* thw, PartPtrs P, int* flags,
                                                    int* err) {
    const int n = *nmove;
    int moved = 0;
    for (int q = blockIdx.x * kBlock + threadIdx.x; q < n; q += gridDim.x * kBlock) {
        const long long e = moves[q];
        const long long p = e & ((1LL << 40) - 1);
        const BoxDev& B = boxes[(int)((e >> 40) & 0xFFFFF)];
        const double px = P.x[p];
        if (isnan(px)) continue;
        const double py = P.y[p], pz = P.z[p];
        const int t = tile_of(B, px, py, pz, err);
        // the tile holding slot p: the last of the box whose range starts at or before p
        int lo = (int)B.tile_off, hi = (int)B.tile_off + B.ntile[0] * B.ntile[1] * B.ntile[2] - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (tbase[mid] <= p) lo = mid; else hi = mid - 1;
        }
        if (lo == t) continue;
        const int slot = atomicAdd(&thw[t], 1);
        if (slot >= tcap[t]) {
            atomicOr(&flags[0], 1);
            continue;
        }
        const long long d = tbase[t] + slot;
        P.x[d] = px;
        P.y[d] = py;
        P.z[d] = pz;
        P.vx[d] = P.vx[p];
        P.vy[d] = P.vy[p];
        P.vz[d] = P.vz[p];
        if (P.m) P.m[d] = P.m[p];
        P.id[d] = P.id[p];
        P.x[p] = empty_slot();
        ++moved;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) moved += __shfl_xor(moved, o);
    if ((threadIdx.x & (kWave - 1)) == 0 && moved) atomicAdd(&flags[1], moved);
}

// Periodic shift alone (nyxpm_redistribute).
__global__ void __launch_bounds__(kBlock) k_wrap(const BoxSeg* segs, int nseg, const BoxDev* boxes,
                                                 double* __restrict__ x, double* __restrict__ y,
                                                 double* __restrict__ z, int* err) {
    const BoxSeg sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    const long long q = (long long)(blockIdx.x - sg.blk0) * kBlock + threadIdx.x;
    if (q >= B.span) return;
    const long long p = B.part_off + q;
    if (isnan(x[p])) return;
    x[p] = periodic_shift(x[p], B.plo[0], B.rhi[0], B.len[0], err);
    y[p] = periodic_shift(y[p], B.plo[1], B.rhi[1], B.len[1], err);
    z[p] = periodic_shift(z[p], B.plo[2], B.rhi[2], B.len[2], err);
}

// Cell-centred gravity field of one box (get_new_grav_vector), 3 components.
__global__ void __launch_bounds__(kBlock) k_grav_vector(const BoxDev* boxes, int box, const double* __restrict__ phi,
                                                        double* __restrict__ g) {
    const BoxDev B = boxes[box];
    const int nx = B.n[0], ny = B.n[1], nz = B.n[2];
    const long long nc = (long long)nx * ny * nz;
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= nc) return;
    const int i = (int)(q % nx);
    const long long t = q / nx;
    const int j = (int)(t % ny), k = (int)(t / ny);
    const double* P = phi + B.cell_off;
    const int im = i == 0 ? nx - 1 : i - 1, ip = i == nx - 1 ? 0 : i + 1;
    const int jm = j == 0 ? ny - 1 : j - 1, jp = j == ny - 1 ? 0 : j + 1;
    const int km = k == 0 ? nz - 1 : k - 1, kp = k == nz - 1 ? 0 : k + 1;
    const double pc = P[q];
    const double fxl = B.dxi[0] * (pc - P[cidx(im, j, k, nx, ny)]);
    const double fxh = B.dxi[0] * (P[cidx(ip, j, k, nx, ny)] - pc);
    const double fyl = B.dxi[1] * (pc - P[cidx(i, jm, k, nx, ny)]);
    const double fyh = B.dxi[1] * (P[cidx(i, jp, k, nx, ny)] - pc);
    const double fzl = B.dxi[2] * (pc - P[cidx(i, j, km, nx, ny)]);
    const double fzh = B.dxi[2] * (P[cidx(i, j, kp, nx, ny)] - pc);
    g[q] = 0.5 * (fxl + fxh);
    g[nc + q] = 0.5 * (fyl + fyh);
    g[2 * nc + q] = 0.5 * (fzl + fzh);
}

// out[id] = in[p] for the occupied slots of one box (undo the tile order for
// download).
__global__ void __launch_bounds__(kBlock) k_unsort(long long p0, long long span, const double* __restrict__ x,
                                                   const int* __restrict__ id, const double* __restrict__ in,
                                                   double* __restrict__ out) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= span || isnan(x[p0 + q])) return;
    out[id[p0 + q]] = in[p0 + q];
}

// The wanted components of a download (n of x y z vx vy vz): the particles' arrays and
// their destinations in upload order.
struct UnsortCols {
    const double* in[6];
    double* out[6];
    int n;
};

// The wanted components of a box's particles to their destinations in upload order, one
// thread per slot: what the caches hold of the scattered 8-byte writes merges into
// whole lines while the output is small.
__global__ void __launch_bounds__(kBlock) k_unsort_all(long long p0, long long span, const double* __restrict__ x,
                                                       const int* __restrict__ id, UnsortCols cols) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= span) return;
    const long long p = p0 + q;
    if (isnan(x[p])) return;
    const int d = id[p];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (k < cols.n) cols.out[k][d] = cols.in[k][p];
}

// The same in two passes for outputs the caches do not hold: k_pack_records writes
// each particle's components as one record of RD doubles at its upload index (whole
// lines, or fewer pieces of them, instead of scattered 8-byte writes, each of which
// costs a line), and k_unpack_records spreads the records over the component arrays in
// order.  RD is the smallest of 2, 4 and 8 that holds the wanted components.  Both go
// through LDS so that RD / 2 lanes move a record as 16-byte pieces (a record of one
// piece needs none).  Bound by HBM: 60 + 64 B and 64 + 48 B per particle for all six.
// Measured: see kUnsortDirect.
template <int RD>
__global__ void __launch_bounds__(kBlock) k_pack_records(long long p0, long long span, const double* __restrict__ x,
                                                         const int* __restrict__ id, UnsortCols cols,
                                                         double* __restrict__ rec) {
    constexpr int L = RD / 2, ST = RD + 2;  // pieces; LDS stride (16-byte aligned, spread over the banks)
    __shared__ __align__(16) double sh[L > 1 ? kBlock * ST : 2];
    __shared__ int sid[L > 1 ? kBlock : 1];
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    const long long p = p0 + q;
    const bool valid = q < span && !isnan(x[p]);
    double v[RD] = {};
    int d = -1;
    if (valid) {
        d = id[p];
#pragma unroll
        for (int k = 0; k < (RD < 6 ? RD : 6); ++k)
            if (k < cols.n) v[k] = cols.in[k][p];
    }
    double2* out = reinterpret_cast<double2*>(rec);
    if (L == 1) {
        if (valid) out[d] = make_double2(v[0], v[1]);
        return;
    }
    double2* s = reinterpret_cast<double2*>(sh + threadIdx.x * ST);
#pragma unroll
    for (int c = 0; c < L; ++c) s[c] = make_double2(v[2 * c], v[2 * c + 1]);
    sid[threadIdx.x] = d;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < L; ++it) {
        const int r = it * (kBlock / L) + threadIdx.x / L, c = threadIdx.x & (L - 1);
        const int dr = sid[r];
        if (dr >= 0) out[(size_t)dr * L + c] = reinterpret_cast<const double2*>(sh + r * ST)[c];
    }
}

template <int RD>
__global__ void __launch_bounds__(kBlock) k_unpack_records(long long np, const double* __restrict__ rec,
                                                           UnsortCols cols) {
    constexpr int L = RD / 2, ST = RD + 2, LU = RD < 6 ? L : 3;  // LU: pieces that can hold a component
    __shared__ __align__(16) double sh[L > 1 ? kBlock * ST : 2];
    const long long base = (long long)blockIdx.x * kBlock;
    const long long d = base + threadIdx.x;
    const double2* in = reinterpret_cast<const double2*>(rec);
    double2 v[LU];
    if (L == 1) {
        if (d < np) v[0] = in[d];
    } else {
#pragma unroll
        for (int it = 0; it < L; ++it) {
            const int r = it * (kBlock / L) + threadIdx.x / L, c = threadIdx.x & (L - 1);
            if (base + r < np && c < LU)
                reinterpret_cast<double2*>(sh + r * ST)[c] = in[(size_t)(base + r) * L + c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < LU; ++c) v[c] = reinterpret_cast<const double2*>(sh + threadIdx.x * ST)[c];
    }
    if (d >= np) return;
#pragma unroll
    for (int c = 0; c < LU; ++c) {
        if (2 * c < cols.n) cols.out[2 * c][d] = v[c].x;
        if (2 * c + 1 < cols.n) cols.out[2 * c + 1][d] = v[c].y;
    }
}

__global__ void __launch_bounds__(kBlock) k_iota(long long p0, long long np, int* __restrict__ id) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q < np) id[p0 + q] = (int)q;
}

__global__ void __launch_bounds__(kBlock) k_fill_int(int* a, long long n, int v) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q < n) a[q] = v;
}

// Initial guess of a step's solve: *ok ? phi = 2 phi - prev : phi unchanged;
// prev = the old phi either way.
__global__ void __launch_bounds__(kBlock) k_phi_guess(double* __restrict__ phi, double* __restrict__ prev,
                                                      long long n, const int* ok) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= n) return;
    const double p = phi[q];
    if (*ok) phi[q] = 2.0 * p - prev[q];
    prev[q] = p;
}

__global__ void __launch_bounds__(kBlock) k_fill_dbl(double* a, long long n, double v) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q < n) a[q] = v;
}

// f = rho + (-mass_offset) with per-block sums (used when the density was set
// from outside rather than by the fold).  Cells are visited exactly as k_fold
// visits them (same cells per block and per thread, same order), so the
// solvability sum of a density does not depend on which of the two produced f.
__global__ void __launch_bounds__(kBlock) k_rhs1(const CellSeg* segs, int nseg, const BoxDev* boxes,
                                                 const double* __restrict__ rho, double* __restrict__ f,
                                                 double* __restrict__ partial) {
    const CellSeg& sg = segs[find_seg(segs, nseg, blockIdx.x)];
    const BoxDev B = boxes[__builtin_amdgcn_readfirstlane(sg.box)];
    double acc = 0.0;
    for_block_cells(sg, B, [&](int, int, int, long long c) {
        const size_t q = B.cell_off + (size_t)c;
        const double fv = rho[q] + (-B.mass_offset);
        f[q] = fv;
        acc += fv;
    });
    const double bs = block_sum_fixed(acc);
    if (threadIdx.x == 0) partial[blockIdx.x] = bs;
}

// Accelerations at the particles of one box (the val of update_dm_particle_single)
// without touching the particles; written in upload (id) order, component-major.
template <typename G>
__global__ void __launch_bounds__(kBlock) k_gather(const BoxDev* boxes, int box, const double* __restrict__ phi,
                                                   const double* __restrict__ x, const double* __restrict__ y,
                                                   const double* __restrict__ z, const int* __restrict__ id,
                                                   double* __restrict__ out, int* err) {
    const BoxDev B = boxes[box];
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= B.span) return;
    const long long p = B.part_off + q;
    const double px = x[p];
    if (isnan(px)) return;
    double val[3];
    gather_grad<G>(B, phi + B.cell_off, px, y[p], z[p], val, err);
    const long long o = id[p];
    out[o] = val[0];
    out[B.np + o] = val[1];
    out[2 * B.np + o] = val[2];
}

// The same from the tiles' staged g (k_kick_tiled's items and arithmetic: the values of
// k_gather bit for bit), for one box of a context: a block stages g of an item's tile
// once where k_gather reads 32 phi values per particle through the caches.  A particle
// whose cell is not one of the tile's (the binning is older than its position) is
// interpolated from global phi.  REC: the values go out as records of kAccelRec doubles
// at the upload index (rec, spread over the components by k_unpack_accel), for outputs
// the caches do not hold: a scattered 8-byte write costs a line.  A wave passes its
// values through LDS so that adjacent lanes write a record.  With G = float the values
// are FP32 numbers, and a record is four of those, written by the particle's own lane.
// Measured, whole call: 9 10^6 clustered particles in random upload order 1144 -> 552 us
// mixed, 1047 -> 555 us FP64; 2^24 in lattice order 674 -> 529 us (records of 64 bytes
// 604, 622 and 733 us; 32-byte records written by one lane each 605 us, the first).
// FP32 records of 16 bytes, the first again: 616 -> 492 us.
constexpr int kAccelRec = 4;
template <typename G, bool REC>
__global__ void __launch_bounds__(kBlock) k_gather_tiled(const BoxSeg* tsegs, int ntseg, const BoxDev* boxes, int box,
                                                         const TileItem* __restrict__ items, const int* nitems,
                                                         const double* __restrict__ phi,
                                                         const double* __restrict__ x, const double* __restrict__ y,
                                                         const double* __restrict__ z, const int* __restrict__ id,
                                                         double* __restrict__ out, int* err) {
    extern __shared__ __align__(16) unsigned char gather_smem[];
    const int n_items = *nitems;
    if ((int)blockIdx.x >= n_items) return;
    const TileItem it = items[xcd_block(blockIdx.x, n_items)];
    const int sgi = find_seg(tsegs, ntseg, it.tile);
    if (tsegs[sgi].box != box) return;
    const BoxDev B = boxes[box];
    const int lt = it.tile - tsegs[sgi].blk0;
    const int tx = lt % B.ntile[0], ty = (lt / B.ntile[0]) % B.ntile[1], tz = lt / (B.ntile[0] * B.ntile[1]);
    const int o0 = tx * B.tile[0], o1 = ty * B.tile[1], o2 = tz * B.tile[2];
    const int bx = min(B.tile[0], B.n[0] - o0), by = min(B.tile[1], B.n[1] - o1), bz = min(B.tile[2], B.n[2] - o2);
    const double* __restrict__ X = x + it.p0;
    const double* __restrict__ Y = y + it.p0;
    const double* __restrict__ Z = z + it.p0;
    const int* __restrict__ ID = id + it.p0;
    // one particle per thread at a time, the next one loaded before this one's value
    double ax = 0.0, ay = 0.0, az = 0.0;
    int aid = 0;
    auto load = [&](int q) {
        ax = X[q];
        ay = Y[q];
        az = Z[q];
        aid = ID[q];
    };
    if ((int)threadIdx.x < it.np) load(threadIdx.x);
    const int GX = bx + 1, GY = by + 1;
    const G* sg = stage_g<G>(B, phi + B.cell_off, reinterpret_cast<double*>(gather_smem), o0, o1, o2, bx, by, bz);
    __syncthreads();
    constexpr bool F32 = std::is_same<G, float>::value;
    constexpr bool EXCH = REC && !F32;
    constexpr int RL = kAccelRec / 2;  // lanes per record
    __shared__ __align__(16) double sval[EXCH ? kBlock * 4 : 2];
    __shared__ int sid[EXCH ? kBlock : 1];
    const int lane = threadIdx.x & (kWave - 1), w0 = threadIdx.x - lane;
    // whole waves together (the lanes past the item's particles hold none)
    for (int q = threadIdx.x; q - lane < it.np; q += kBlock) {
        const double px = q < it.np ? ax : empty_slot(), py = ay, pz = az;
        const long long o = aid;
        if (q + kBlock < it.np) load(q + kBlock);
        const bool valid = !isnan(px);
        if (EXCH) sid[threadIdx.x] = valid ? (int)o : -1;
        if (valid) {
        double xint, yint, zint;
        const int li = cic_index(px, B.plo[0], B.dxi[0], &xint) - o0;
        const int lj = cic_index(py, B.plo[1], B.dxi[1], &yint) - o1;
        const int lk = cic_index(pz, B.plo[2], B.dxi[2], &zint) - o2;
        double val[3];
        if ((unsigned)li < (unsigned)bx && (unsigned)lj < (unsigned)by && (unsigned)lk < (unsigned)bz) {
            const G fx = G(xint), fy = G(yint), fz = G(zint);
            const G mx = G(1) - fx, my = G(1) - fy, mz = G(1) - fz;
            G g0 = G(0), g1 = G(0), g2 = G(0);
#pragma unroll
            for (int kk = 0; kk <= 1; ++kk) {
                const G wz = kk ? mz : fz;
#pragma unroll
                for (int jj = 0; jj <= 1; ++jj) {
                    const G wy = jj ? my : fy;
                    const G* g = sg + 3 * (((lk + 1 - kk) * GY + (lj + 1 - jj)) * GX + li);
                    const G w0 = fx * wy * wz;  // cell i
                    g0 += w0 * g[3];
                    g1 += w0 * g[4];
                    g2 += w0 * g[5];
                    const G w1 = mx * wy * wz;  // cell i-1
                    g0 += w1 * g[0];
                    g1 += w1 * g[1];
                    g2 += w1 * g[2];
                }
            }
            val[0] = double(g0);
            val[1] = double(g1);
            val[2] = double(g2);
        } else {
            gather_grad<G>(B, phi + B.cell_off, px, py, pz, val, err);
        }
        if (REC && F32) {
            reinterpret_cast<float4*>(out)[o] = make_float4((float)val[0], (float)val[1], (float)val[2], 0.0f);
        } else if (REC) {
            double2* sv = reinterpret_cast<double2*>(sval + 4 * threadIdx.x);
            sv[0] = make_double2(val[0], val[1]);
            sv[1] = make_double2(val[2], 0.0);
        } else {
            out[o] = val[0];
            out[B.np + o] = val[1];
            out[2 * B.np + o] = val[2];
        }
        }
        if (EXCH) {
            // LDS operations of one wave complete in order: no barrier
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int k = 0; k < RL; ++k) {
                const int rr = w0 + k * (kWave / RL) + lane / RL, part = lane % RL;
                const int d = sid[rr];
                if (d >= 0)
                    reinterpret_cast<double2*>(out)[(size_t)d * RL + part] =
                        reinterpret_cast<const double2*>(sval + 4 * rr)[part & 1];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

template <typename G>
__global__ void __launch_bounds__(kBlock) k_unpack_accel(long long np, const double* __restrict__ rec,
                                                         double* __restrict__ out) {
    const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (q >= np) return;
    if (std::is_same<G, float>::value) {
        const float4 a = reinterpret_cast<const float4*>(rec)[q];
        out[q] = (double)a.x;
        out[np + q] = (double)a.y;
        out[2 * np + q] = (double)a.z;
        return;
    }
    const double2* r = reinterpret_cast<const double2*>(rec) + (kAccelRec / 2) * q;
    const double2 a = r[0], b = r[1];
    out[q] = a.x;
    out[np + q] = a.y;
    out[2 * np + q] = b.x;
}

}  // namespace nyxpm
