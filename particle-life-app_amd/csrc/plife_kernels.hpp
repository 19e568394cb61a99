// plife_kernels.hpp -- gfx950 kernels of the particle-life physics step.
//
// One step (reference: backend/Physics.java:112-134):
//   k_bin                    cell key per particle (Physics.java:362-375), cell histogram, and
//                            each particle's place among its cell's arrivals
//   k_scan_*                 scan of the cell counts -> cell_start / cell_end
//                            (cell_end is the reference's `containers` array, Physics.java:329-348)
//   k_place, k_rank          the reference's stable counting-sort permutation
//                            (Physics.java:342-353): particles placed in their cell in
//                            arrival order, then ranked by index inside it
//   k_force (plife_force.hpp) velocity phase + position phase fused (Physics.java:397-450);
//                            legal because the update is Jacobi: velocities read only the
//                            sorted step-start positions, new positions go to another buffer.
//
// Positions are 32-bit fixed point (x = k * 2^-32, unit box), so the periodic
// minimum image of Range.wrapConnection (Range.java:68-81) is the exact int32
// difference k_q - k_p, and converting a position to FP64 is exact.  Cell keys
// use the same FP64 division and truncation as the reference.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace plife {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr double kFix = 4294967296.0;       // 2^32
constexpr double kInvFix = 1.0 / 4294967296.0;

// ---------------------------------------------------------------------------
// wave64 / block helpers
// ---------------------------------------------------------------------------
// Inclusive scan over a wave64 in registers (DPP, no LDS round trips):
// Hillis-Steele steps of 1, 2, 4, 8 lanes inside each row of 16 (lanes
// shifted in from outside the row read 0), then row 0's total added to row 1
// and row 2's to row 3 (row_bcast:15), and the first two rows' total to rows
// 2 and 3 (row_bcast:31).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    constexpr int kRowShr = 0x110, kBcast15 = 0x142, kBcast31 = 0x143;
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowShr + 1, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowShr + 2, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowShr + 4, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowShr + 8, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kBcast15, 0xa, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kBcast31, 0xc, 0xf, false);
    return v;
}

// Exclusive scan over a block of NT threads.  s_w: NT / 64 words of LDS.
template <int NT = kBlock>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *s_w, uint32_t &total)
{
    const uint32_t inc = wave_incl_scan(v);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) s_w[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < NT / kWave; ++k) {
        uint32_t t = s_w[k];
        off += (k < w) ? t : 0u;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

// Sum over a block of NT threads; every thread gets the total.  s_w: NT / 64 words of LDS.
template <int NT = kBlock>
__device__ __forceinline__ unsigned long long block_sum_u64(unsigned long long v,
                                                            unsigned long long *s_w)
{
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) s_w[w] = v;
    __syncthreads();
    unsigned long long tot = 0;
#pragma unroll
    for (int k = 0; k < NT / kWave; ++k) tot += s_w[k];
    __syncthreads();
    return tot;
}

// Block ids are dealt round-robin to the 8 XCDs; remap so each XCD works on a
// contiguous run of tiles and neighbouring tiles share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int b, int nb)
{
    const int q = nb >> 3, rem = nb & 7;
    const int xcd = b & 7, k = b >> 3;
    return xcd < rem ? xcd * (q + 1) + k : rem * (q + 1) + (xcd - rem) * q + k;
}

// ---------------------------------------------------------------------------
// fill
// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t *p, uint32_t v, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// The last step's counters to the host's pinned copy (the step after copies
// them itself, in k_bin).
__global__ void k_copy_u64(const unsigned long long *__restrict__ src, unsigned long long *__restrict__ dst,
                           int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ void k_zero_u64(unsigned long long *p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// ---------------------------------------------------------------------------
// cell keys (Physics.java:362-375): cx = trunc(x / cs) in FP64, clamped to nx-1.
// ---------------------------------------------------------------------------
// One world of a batch (a single-world handle is a batch of one).  Worlds
// occupy consecutive particle slots [off, off + n) in both the pre-sort and the
// sorted order, and consecutive cells [cell_base, cell_base + nx^DIM) of the
// batch's cell arrays, so one stable sort of the batch's cell keys sorts every
// world exactly as stepping it alone would.
struct WorldDev {
    int off, n;                      // particle slots
    int nx, all_global;              // cells per axis; 1: literal stencil and force law (home_global)
    uint32_t cell_base;              // first batch cell of this world
    int ntypes, moff;                // matrix size and offset (doubles) in the batch matrix
    int wrap;
    float r2hi;                      // screen bound, units 2^-64: (rmax 2^32)^2 (1 + 2^-20)
    int exact_d2;                    // 1: squared distances in range are exact (pair_d2_of)
    int sbias;                       // screen bound on 16-bit coordinates: -(bq + 1) (screen_hi)
    double cs, ics;                  // cell size = rmax (Physics.java:312), and 1 / cs
    double r2u;                      // fl(rmax*rmax) * 2^64: the reference's bound in units 2^-64
    double S;                        // 2^-32 / rmax: |rel| = |D| S with D in units 2^-32
    double R;                        // rmax * 2^32:  1/|rel| = R / |D|
    double beta, one_plus_beta, inv_1mb, inv_beta;
    double m2S;                      // -2 S
    double betaR;                    // beta R: |D| below it is the repulsion zone
    double ff;                       // friction^(60 dt) (host FP64 pow, Physics.java:401)
    double kdt;                      // force * dt * 2^-32
    double ka;                       // force * 2^-32: acceleration per unit of accumulated D (f/dist)
    double dt;
};

// World index of every slot of a batch: the last world whose first slot is
// at or before the slot (worlds are laid out in order; an empty world shares
// its offset with the next one, so the last such world is the non-empty one).
__global__ void k_world_of(int n, const WorldDev *__restrict__ worlds, int nworlds,
                           uint16_t *__restrict__ world_of)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int lo = 0, hi = nworlds;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (worlds[mid].off <= i) lo = mid;
        else hi = mid;
    }
    world_of[i] = (uint16_t)lo;
}

// trunc(x / cs) (IEEE FP64 division, x >= 0: trunc == floor) for x = k 2^-32
// without the division where that is safe:
// x * (1 / cs) is within 3 ulp of the rounded quotient, i.e. within 2^-35
// for quotients below 2^16 cells, so its integer part is the division's
// unless the product lies within 1e-9 of an integer -- then divide.
__device__ __forceinline__ int trunc_div_fast(uint32_t k, double cs, double ics)
{
    const double x = (double)k * kInvFix;
    const double q = x * ics;
    int c = (int)q;
    const double f = q - (double)c;
    if (f < 1e-9 || f > 1.0 - 1e-9) c = (int)(x / cs);
    return c;
}

__device__ __forceinline__ int key_axis_fast(uint32_t k, double cs, double ics, int nx)
{
    const int c = trunc_div_fast(k, cs, ics);
    return c == nx ? nx - 1 : c;
}

// Cell counts are accumulated with one atomic per run of equal keys inside a
// wave: the input is the previous step's cell order, so most lanes of a wave
// share a few keys and per-lane atomics would serialise on the same address.
// Returns the lane's place among the cell's arrivals: what the run's atomic
// found plus the lane's position in the run.
__device__ __forceinline__ uint32_t count_runs(uint32_t key, bool valid, uint32_t *__restrict__ cell_count)
{
    const int lane = __lane_id();
    const uint32_t prev = __shfl_up(key, 1, kWave);
    const bool head = valid && (lane == 0 || prev != key);
    const uint64_t heads = __ballot(head);
    const int nvalid = (int)__popcll(__ballot(valid));   // valid lanes are a prefix
    uint32_t base = 0;
    if (head) {
        const uint64_t later = lane == 63 ? 0ull : (heads & (~0ull << (lane + 1)));
        const int next = later ? (int)__ffsll((long long)later) - 1 : nvalid;
        base = atomicAdd(&cell_count[key], (uint32_t)(next - lane));
    }
    const uint64_t upto = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
    const int first = upto ? 63 - (int)__clzll((long long)upto) : 0;
    return __shfl(base, first, kWave) + (uint32_t)(lane - first);
}

// Binning: cell keys, the cell histogram (run-aggregated atomics) and each
// particle's place among its cell's arrivals.  Block 0 also clears the step's
// counters.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_bin(const uint32_t *__restrict__ px, const uint32_t *__restrict__ py,
                                                const uint32_t *__restrict__ pz, int n,
                                                const WorldDev *__restrict__ worlds,
                                                const uint16_t *__restrict__ world_of,
                                                uint32_t *__restrict__ keys, uint32_t *__restrict__ arrival,
                                                uint32_t *__restrict__ cell_count,
                                                unsigned long long *__restrict__ counters, int ncounters,
                                                unsigned long long tag, unsigned long long *__restrict__ stat_out)
{
    // the step's counters (pairs, sum of squares, per-world pairs) start at
    // zero, after the previous step's final values (and its layout tag) have
    // gone to the host's pinned copy (stat_out, when given)
    if (blockIdx.x == 0) {
        for (int t = threadIdx.x; t <= ncounters; t += kBlock) {
            if (stat_out) stat_out[t] = counters[t];
            counters[t] = t < ncounters ? 0ull : tag;   // [ncounters]: which layout the counts belong to
        }
    }
    double cs = worlds[0].cs, ics = worlds[0].ics;
    int nx = worlds[0].nx;
    uint32_t cb = worlds[0].cell_base;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = i < n;
    uint32_t key = 0xFFFFFFFFu;
    if (valid) {
        if (world_of) {                                // several worlds: this slot's world
            const WorldDev *w = worlds + world_of[i];
            cs = w->cs;
            ics = w->ics;
            nx = w->nx;
            cb = w->cell_base;
        }
        key = (uint32_t)key_axis_fast(px[i], cs, ics, nx) + (uint32_t)key_axis_fast(py[i], cs, ics, nx) * (uint32_t)nx;
        if constexpr (DIM == 3) key += (uint32_t)key_axis_fast(pz[i], cs, ics, nx) * (uint32_t)nx * (uint32_t)nx;
        key += cb;
        keys[i] = key;
    }
    const uint32_t at = count_runs(key, valid, cell_count);
    if (valid) arrival[i] = at;
}

// Particle i to its cell's slots in arrival order.
__global__ __launch_bounds__(kBlock) void k_place(int n, const uint32_t *__restrict__ keys,
                                                  const uint32_t *__restrict__ arrival,
                                                  const uint32_t *__restrict__ cell_start,
                                                  uint32_t *__restrict__ order)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) order[cell_start[keys[i]] + arrival[i]] = (uint32_t)i;
}

// Stable order: each particle's rank among its cell's by index gives its
// sorted slot, which gets the permutation, the key and the particle's record
// (x, y, z, type), so that the force kernels read neighbours as contiguous
// 16-byte entries.  The comparisons are the sum of count^2 over cells; the
// force phase evaluates at least as many candidates at several times the cost
// each, so that dense cells need no other sort.  Bound by the latency of its
// dependent reads: threads go by pre-sort slot (coalesced keys and state, and
// a wave's lanes share a few cells), and a cell is read sixteen indices at a
// time, past its end too (`order` has kRankPad spare entries).
constexpr int kRankPad = 16;

template <int DIM>
__global__ __launch_bounds__(kBlock) void k_rank(int n, const uint32_t *__restrict__ keys,
                                                 const uint32_t *__restrict__ order,
                                                 const uint32_t *__restrict__ cell_start,
                                                 const uint32_t *__restrict__ cell_end,
                                                 const uint32_t *__restrict__ px, const uint32_t *__restrict__ py,
                                                 const uint32_t *__restrict__ pz, const int32_t *__restrict__ type,
                                                 uint32_t *__restrict__ perm, uint32_t *__restrict__ skeys,
                                                 uint4 *__restrict__ rec)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= (uint32_t)n) return;
    const uint32_t key = keys[i];
    const uint32_t s = cell_start[key], e = cell_end[key];
    const uint4 p = make_uint4(px[i], py[i], DIM == 3 ? pz[i] : 0u, (uint32_t)type[i]);
    uint32_t r = s;
    for (uint32_t k = s; k < e; k += 16) {
        uint32_t v[16];
        __builtin_memcpy(v, order + k, sizeof v);
        const int m = (int)min(e - k, 16u);
#pragma unroll
        for (int u = 0; u < 16; ++u) r += ((v[u] < i) & (u < m)) ? 1u : 0u;
    }
    perm[r] = i;
    skeys[r] = key;
    rec[r] = p;
}

// ---------------------------------------------------------------------------
// device-wide scan of u32 (reduce -> scan block sums -> downsweep)
// ---------------------------------------------------------------------------
constexpr int kScanItems = 4;
constexpr int kScanTile = kBlock * kScanItems;

// Exclusive scan of n cell counts into excl and inclusive into incl; the
// counts are cleared once read, which leaves them ready for the next step's
// histogram.  The sum of their squares (the number of (particle, cell-mate)
// pairs, a clustering measure) is added to *sq: the reduce pass stores each
// block's sum in sqb and one block adds them up, so the device-wide total
// costs one atomic rather than one per block.
struct ScanJob {
    uint32_t *in;
    int n;
    uint32_t *excl, *incl;
    unsigned long long *sq;
    uint32_t *bsum;           // ceil(n / kScanTile) block sums
    unsigned long long *sqb;  // ceil(n / kScanTile) per-block sums of squares
};

__device__ __forceinline__ void scan_load(const ScanJob &j, int i0, uint32_t (&v)[kScanItems], uint32_t &s)
{
    s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = (i0 + k < j.n) ? j.in[i0 + k] : 0u;
        s += v[k];
    }
}

__device__ __forceinline__ void scan_store(const ScanJob &j, int i0, const uint32_t (&v)[kScanItems], uint32_t off)
{
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (i0 + k < j.n) {
            j.in[i0 + k] = 0u;
            j.excl[i0 + k] = off;
            off += v[k];
            j.incl[i0 + k] = off;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_scan_reduce(ScanJob j)
{
    __shared__ uint32_t s_w[4];
    __shared__ unsigned long long s_q[kBlock / kWave];
    uint32_t v[kScanItems], s;
    scan_load(j, blockIdx.x * kScanTile + threadIdx.x * kScanItems, v, s);
    unsigned long long q = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) q += (unsigned long long)v[k] * v[k];
    uint32_t total;
    block_excl_scan(s, s_w, total);
    q = block_sum_u64(q, s_q);
    if (threadIdx.x == 0) {
        j.bsum[blockIdx.x] = total;
        j.sqb[blockIdx.x] = q;
    }
}

// The block sums of jobs of more than kFoldBlocks blocks.
__global__ __launch_bounds__(kBlock) void k_scan_single(ScanJob j)
{
    __shared__ uint32_t s_w[4];
    __shared__ unsigned long long s_q[kBlock / kWave];
    const int n = (j.n + kScanTile - 1) / kScanTile;
    uint32_t carry = 0;
    unsigned long long q = 0;
    for (int base = 0; base < n; base += kScanTile) {
        const int i0 = base + threadIdx.x * kScanItems;
        uint32_t v[kScanItems];
        uint32_t s = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            v[k] = (i0 + k < n) ? j.bsum[i0 + k] : 0u;
            s += v[k];
            if (i0 + k < n) q += j.sqb[i0 + k];
        }
        uint32_t total;
        uint32_t off = block_excl_scan(s, s_w, total) + carry;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (i0 + k < n) j.bsum[i0 + k] = off;
            off += v[k];
        }
        carry += total;
    }
    q = block_sum_u64(q, s_q);
    if (threadIdx.x == 0 && q) atomicAdd(j.sq, q);
}

__global__ __launch_bounds__(kBlock) void k_scan_down(ScanJob j)
{
    __shared__ uint32_t s_w[4];
    const int i0 = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems], s, total;
    scan_load(j, i0, v, s);
    const uint32_t off = block_excl_scan(s, s_w, total) + j.bsum[blockIdx.x];
    scan_store(j, i0, v, off);
}

// Down-sweep for jobs of at most kFoldBlocks blocks, with the block-sum scan
// folded in: each block adds up the sums of the blocks before it (at most
// kFoldBlocks / kBlock loads per thread), and block 0 adds the sum of
// squares -- two launches instead of three, same outputs.
constexpr int kFoldBlocks = 1024;

__global__ __launch_bounds__(kBlock) void k_scan_down_fold(ScanJob j)
{
    __shared__ uint32_t s_w[4];
    __shared__ unsigned long long s_q[kBlock / kWave];
    const int blk = blockIdx.x;
    uint32_t pre = 0;
    for (int b = threadIdx.x; b < blk; b += kBlock) pre += j.bsum[b];
    uint32_t before;
    block_excl_scan(pre, s_w, before);             // `before` = the sum over all threads
    const int i0 = blk * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems], s, total;
    scan_load(j, i0, v, s);
    const uint32_t off = block_excl_scan(s, s_w, total) + before;
    scan_store(j, i0, v, off);
    if (blk == 0) {
        const int nb = (j.n + kScanTile - 1) / kScanTile;
        unsigned long long q = 0;
        for (int b = threadIdx.x; b < nb; b += kBlock) q += j.sqb[b];
        q = block_sum_u64(q, s_q);
        if (threadIdx.x == 0 && q) atomicAdd(j.sq, q);
    }
}

// The whole scan by one workgroup when the job is small (at most kSmallScan
// entries, at most two passes), carrying the running sum -- one launch instead
// of two, for arrays whose scan time is launch latency.  Same outputs.
constexpr int kSmallBlock = 1024;
constexpr int kSmallScan = 8192;

__global__ __launch_bounds__(kSmallBlock) void k_scan_small(ScanJob j)
{
    __shared__ uint32_t s_w[kSmallBlock / kWave];
    __shared__ unsigned long long s_q[kSmallBlock / kWave];
    uint32_t carry = 0;
    unsigned long long q = 0;
    for (int base = 0; base < j.n; base += kSmallBlock * kScanItems) {
        const int i0 = base + threadIdx.x * kScanItems;
        uint32_t v[kScanItems], s, total;
        scan_load(j, i0, v, s);
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) q += (unsigned long long)v[k] * v[k];
        const uint32_t off = block_excl_scan<kSmallBlock>(s, s_w, total) + carry;
        scan_store(j, i0, v, off);
        carry += total;
    }
    q = block_sum_u64<kSmallBlock>(q, s_q);
    if (threadIdx.x == 0 && q) atomicAdd(j.sq, q);
}

// ---------------------------------------------------------------------------
// SoA state
// ---------------------------------------------------------------------------
// Compaction of a batch after worlds left: destination slot i of world w
// (worlds[w].off <= i < worlds[w].off + worlds[w].n in the new layout) takes
// the particle at src_off[w] + (i - worlds[w].off) of the old layout.
__global__ __launch_bounds__(kBlock) void k_compact(int n, const WorldDev *__restrict__ worlds,
                                                   const uint16_t *__restrict__ world_of,
                                                   const int *__restrict__ src_off,
                                                   const uint32_t *__restrict__ sx,
                                                   const uint32_t *__restrict__ sy,
                                                   const uint32_t *__restrict__ sz,
                                                   const float *__restrict__ svx,
                                                   const float *__restrict__ svy,
                                                   const float *__restrict__ svz,
                                                   const int32_t *__restrict__ stype,
                                                   const int32_t *__restrict__ sid,
                                                   uint32_t *__restrict__ dx, uint32_t *__restrict__ dy,
                                                   uint32_t *__restrict__ dz, float *__restrict__ dvx,
                                                   float *__restrict__ dvy, float *__restrict__ dvz,
                                                   int32_t *__restrict__ dtype, int32_t *__restrict__ did)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int w = world_of ? (int)world_of[i] : 0;
    const int j = src_off[w] + (i - worlds[w].off);
    dx[i] = sx[j];
    dy[i] = sy[j];
    dz[i] = sz[j];
    dvx[i] = svx[j];
    dvy[i] = svy[j];
    dvz[i] = svz[j];
    dtype[i] = stype[j];
    did[i] = sid[j];
}

// Seeded world generation, the device side of the default presets
// (backend/DefaultPositionSetter.java: uniform positions; backend/
// DefaultTypeSetter.java: uniform types; velocities 0, Physics.java:297-303).
// Counter-based SplitMix64 (Vigna's published generator): draw k of stream s
// of `seed` is mix(base_s + (k + 1) * gamma), base_s = mix(seed + s * kStream).
// Uniforms are the top 24 bits (a 2^-24 grid, exact in FP32, FP64 and the
// 32-bit fixed point); streams 1..3 are x, y, z and 4 the type.
constexpr uint64_t kGamma = 0x9E3779B97F4A7C15ull;
constexpr uint64_t kStream = 0xD1B54A32D192ED03ull;

__host__ __device__ inline uint64_t splitmix_mix(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

struct GenArgs {
    uint64_t base[4];                  // stream bases for x, y, z, type
    int n, off, ntypes, dim;
    uint32_t *px, *py, *pz;
    float *vx, *vy, *vz;
    int32_t *type, *id;
};

__global__ __launch_bounds__(kBlock) void k_gen_uniform(GenArgs g)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= g.n) return;
    const uint64_t step = (uint64_t)(k + 1) * kGamma;
    const int i = g.off + k;
    g.px[i] = (uint32_t)(splitmix_mix(g.base[0] + step) >> 40) << 8;      // u24 * 2^-24 in 2^-32 units
    g.py[i] = (uint32_t)(splitmix_mix(g.base[1] + step) >> 40) << 8;
    g.pz[i] = g.dim == 3 ? (uint32_t)(splitmix_mix(g.base[2] + step) >> 40) << 8 : 0u;
    const uint64_t m = splitmix_mix(g.base[3] + step) >> 40;            // floor(u24 * T) exactly
    g.type[i] = (int32_t)((m * (uint64_t)g.ntypes) >> 24);
    g.vx[i] = 0.0f;
    g.vy[i] = 0.0f;
    g.vz[i] = 0.0f;
    g.id[i] = k;
}

// Physics.ensurePosition (Physics.java:499-505) of an FP64 coordinate, then
// rounding to the 2^-32 grid.  Periodic: the fractional part (a result of
// 1.0, reference quirk Q3, is the same torus point as 0).  Clamped: [0, 1],
// with 1.0 stored as 1 - 2^-32.  NaN becomes 0.
__host__ __device__ inline uint32_t fixed_of(double x, bool wrap)
{
    if (!(x == x)) return 0u;
    if (wrap) {
        x = x - floor(x);
        return (uint32_t)(unsigned long long)rint(x * kFix);
    }
    x = x < 0 ? 0 : (x > 1 ? 1 : x);
    const double s = rint(x * kFix);
    return s >= 4294967295.0 ? 0xFFFFFFFFu : (uint32_t)(unsigned long long)s;
}

// ---------------------------------------------------------------------------
// The app's position and type presets (app/PositionSetterProvider.java:17-119,
// app/TypeSetterProvider.java:12-45) over a range of slots, with the
// counter-based SplitMix64 draws above in place of the reference's unseeded
// java.util.Random: uniform u = (draw >> 11) * 2^-53, Gaussians by Box-Muller
// from two streams, sqrt(-2 ln(1 - u1)) cos(2 pi u2).  Shapes are computed in
// the reference's side-2 frame with its float constants and evaluation order,
// mapped to the unit box by x * 0.5 + 0.5 as each preset does, then placed
// by fixed_of.  The uniform preset is the generator above (2^-24 grid,
// streams 1-3).  3D worlds (no reference counterpart) take z from stream 3.
// ---------------------------------------------------------------------------
enum PositionPreset {
    kPosCentered, kPosUniform, kPosUniformCircle, kPosCenteredCircle, kPosRing, kPosRainbowRing,
    kPosColorBattle, kPosColorWheel, kPosLine, kPosSpiral, kPosRainbowSpiral, kPosPresets
};
enum TypePreset {
    kTypeRandom, kTypeRandomize10, kTypeSlices, kTypeOnion, kTypeRotate, kTypeFlip,
    kTypeMoreOfFirst, kTypeKillStill, kTypePresets
};
constexpr int kPresetStream = 40;      // preset draws use streams 40..43 (positions), 44..45 (types)
constexpr double kPi = 3.141592653589793;     // java.lang.Math.PI

struct PresetArgs {
    uint64_t base[6];                  // streams 40..45
    uint64_t ubase[4];                 // streams 1..4 (the uniform generator's)
    int n, off, ntypes, dim, preset, wrap;
    uint32_t *px, *py, *pz;
    float *vx, *vy, *vz;
    int32_t *type;
    unsigned long long *tag;           // positions: the step counters' layout tag, cleared (may be null)
};

__device__ __forceinline__ double preset_u(uint64_t base, uint64_t step)
{
    return (double)(splitmix_mix(base + step) >> 11) * 0x1p-53;
}

__device__ __forceinline__ double preset_gauss(uint64_t b1, uint64_t b2, uint64_t step)
{
#pragma clang fp contract(off)
    const double u1 = ((double)(splitmix_mix(b1 + step) >> 11) + 1.0) * 0x1p-53;   // (0, 1]
    const double u2 = (double)(splitmix_mix(b2 + step) >> 11) * 0x1p-53;
    return sqrt(-2.0 * log(u1)) * cos(2.0 * kPi * u2);
}

// mapType of TypeSetterProvider.java:46-52
__device__ __forceinline__ int preset_map_type(double v, int nt)
{
    return max(0, min(nt - 1, (int)floor(v * nt)));
}

__global__ __launch_bounds__(kBlock) void k_set_positions(PresetArgs g)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= g.n) return;
    if (k == 0 && g.tag) *g.tag = 0ull;
    const int i = g.off + k;
    const uint64_t s = (uint64_t)(k + 1) * kGamma;
    const int t = g.type[i];
    const double T = (double)g.ntypes;
    double x = 0.0, y = 0.0;
    switch (g.preset) {
        case kPosCentered: {
            const double scale = (double)0.3f;
            x = preset_gauss(g.base[0], g.base[1], s) * scale;
            y = preset_gauss(g.base[2], g.base[3], s) * scale;
            break;
        }
        case kPosUniformCircle: {
            const double angle = preset_u(g.base[0], s) * 2 * kPi;
            const double radius = 0.5 * sqrt(preset_u(g.base[1], s));
            x = cos(angle) * radius;
            y = sin(angle) * radius;
            break;
        }
        case kPosCenteredCircle: {
            const double angle = preset_u(g.base[0], s) * 2 * kPi;
            const double radius = (double)0.5f * preset_u(g.base[1], s);
            x = cos(angle) * radius;
            y = sin(angle) * radius;
            break;
        }
        case kPosRing: {
            const double angle = preset_u(g.base[0], s) * 2 * kPi;
            const double radius = 0.7 + 0.02 * preset_gauss(g.base[2], g.base[3], s);
            x = cos(angle) * radius;
            y = sin(angle) * radius;
            break;
        }
        case kPosRainbowRing: {
            const double angle = (0.3 * preset_gauss(g.base[0], g.base[1], s) + t) / T * 2 * kPi;
            const double radius = 0.7 + 0.02 * preset_gauss(g.base[2], g.base[3], s);
            x = cos(angle) * radius;
            y = sin(angle) * radius;
            break;
        }
        case kPosColorBattle: {
            const double ca = t / T * 2 * kPi;
            const double cr = (double)0.5f;
            const double angle = preset_u(g.base[0], s) * 2 * kPi;
            const double radius = preset_u(g.base[1], s) * (double)0.1f;
            x = cr * cos(ca) + cos(angle) * radius;
            y = cr * sin(ca) + sin(angle) * radius;
            break;
        }
        case kPosColorWheel: {
            const double ca = t / T * 2 * kPi;
            const double cr = (double)0.3f, ir = (double)0.2f;
            x = cr * cos(ca) + preset_gauss(g.base[0], g.base[1], s) * ir;
            y = cr * sin(ca) + preset_gauss(g.base[2], g.base[3], s) * ir;
            break;
        }
        case kPosLine:
            x = 2 * preset_u(g.base[0], s) - 1;
            y = (2 * preset_u(g.base[1], s) - 1) * (double)0.15f;
            break;
        case kPosSpiral:
        case kPosRainbowSpiral: {
            double f;
            if (g.preset == kPosSpiral) {
                f = preset_u(g.base[0], s);
            } else {
                const double spread_t = 0.3 / g.ntypes;
                f = (t + 1) / (double)(g.ntypes + 2) + spread_t * preset_gauss(g.base[0], g.base[1], s);
                f = f < 0 ? 0 : (f > 1 ? 1 : f);
            }
            const double angle = 2.0 * 2 * kPi * f;
            const double spread = 0.5 * fmin(f, 0.2);
            const double radius = 0.9 * f + spread * preset_gauss(g.base[2], g.base[3], s) * spread;
            x = radius * cos(angle);
            y = radius * sin(angle);
            break;
        }
        default:    // kPosUniform: the uniform generator's grid values
            x = (double)(splitmix_mix(g.ubase[0] + s) >> 40) * 0x1p-24;
            y = (double)(splitmix_mix(g.ubase[1] + s) >> 40) * 0x1p-24;
            break;
    }
    if (g.preset != kPosUniform) {
        x = x * 0.5 + 0.5;
        y = y * 0.5 + 0.5;
    }
    const bool wrap = g.wrap != 0;
    g.px[i] = fixed_of(x, wrap);
    g.py[i] = fixed_of(y, wrap);
    g.pz[i] = g.dim == 3 ? (uint32_t)(splitmix_mix(g.ubase[2] + s) >> 40) << 8 : 0u;
    g.vx[i] = 0.0f;     // Physics.setPosition (Physics.java:297-303)
    g.vy[i] = 0.0f;
    g.vz[i] = 0.0f;
}

__global__ __launch_bounds__(kBlock) void k_set_types(PresetArgs g)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= g.n) return;
    const int i = g.off + k;
    const uint64_t s = (uint64_t)(k + 1) * kGamma;
    const int nt = g.ntypes;
    int t = g.type[i];
    switch (g.preset) {
        case kTypeRandomize10:
            if (preset_u(g.base[4], s) < 0.1) t = preset_map_type(preset_u(g.base[5], s), nt);
            break;
        case kTypeSlices:
            t = preset_map_type((double)g.px[i] * kInvFix, nt);
            break;
        case kTypeOnion: {
            const double dx = (double)g.px[i] * kInvFix - 0.5, dy = (double)g.py[i] * kInvFix - 0.5;
            const double dz = g.dim == 3 ? (double)g.pz[i] * kInvFix : 0.0;
            t = preset_map_type(sqrt(dx * dx + (dy * dy + dz * dz)) * 2, nt);
            break;
        }
        case kTypeRotate:
            t = (t + 1) % nt;
            break;
        case kTypeFlip:
            t = nt - 1 - t;
            break;
        case kTypeMoreOfFirst:
            t = preset_map_type(preset_u(g.base[4], s) * preset_u(g.base[5], s), nt);
            break;
        case kTypeKillStill: {
            const double vx = g.vx[i], vy = g.vy[i], vz = g.dim == 3 ? (double)g.vz[i] : 0.0;
            if (sqrt(vx * vx + (vy * vy + vz * vz)) < 0.01) t = nt - 1;
            break;
        }
        default: {  // kTypeRandom: the uniform generator's type draw
            const uint64_t m = splitmix_mix(g.ubase[3] + s) >> 40;
            t = (int32_t)((m * (uint64_t)nt) >> 24);
            break;
        }
    }
    g.type[i] = t;
}

// One in-place edit of a particle between steps (positions already wrapped or
// clamped and rounded to the 2^-32 grid); ids are kept.
struct SlotEdit {
    int32_t slot;
    uint32_t x, y, z;
    float vx, vy, vz;
    int32_t type;
};

__global__ __launch_bounds__(kBlock) void k_set_slots(const SlotEdit *__restrict__ e, int k, int off,
                                                      uint32_t *px, uint32_t *py, uint32_t *pz,
                                                      float *vx, float *vy, float *vz, int32_t *type)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= k) return;
    const SlotEdit r = e[i];
    const int s = off + r.slot;
    px[s] = r.x;
    py[s] = r.y;
    pz[s] = r.z;
    vx[s] = r.vx;
    vy[s] = r.vy;
    vz[s] = r.vz;
    type[s] = r.type;
}

struct PosBuf {
    uint32_t *x, *y, *z;
};
struct AuxBuf {
    float *vx, *vy, *vz;
    int32_t *type, *id;
};

// Slots [off, off + n) of up to kPackMax device arrays of 32-bit words,
// gathered chunk-major for a chunked download: chunk c (slots c*chunk ...)
// holds each array's len_c words in turn, so one DMA moves one chunk.
constexpr int kPackMax = 8;
struct PackArgs {
    const uint32_t *src[kPackMax];
    int na, off, n, chunk;
};

__global__ __launch_bounds__(kBlock) void k_pack(PackArgs p, uint32_t *dst)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= p.n) return;
    const int c = i / p.chunk, j = i - c * p.chunk;
    const int len = min(p.chunk, p.n - c * p.chunk);
    uint32_t *d = dst + (size_t)c * p.chunk * p.na + j;
#pragma unroll
    for (int a = 0; a < kPackMax; ++a)
        if (a < p.na) d[(size_t)a * len] = p.src[a][p.off + i];
}

// The inverse for uploads: staged arrays x, y, [z], vx, vy, [vz], type (each
// n words, FP32 velocities as their bits) into slots [off, off + n) of the
// SoA buffers, ids 0..n-1, z and vz zero in 2D.
struct UnpackArgs {
    uint32_t *px, *py, *pz;
    float *vx, *vy, *vz;
    int32_t *type, *id;
    int off, n, dim;
};

__global__ __launch_bounds__(kBlock) void k_unpack(UnpackArgs u, const uint32_t *__restrict__ src)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= u.n) return;
    const size_t n = (size_t)u.n;
    const bool d3 = u.dim == 3;
    const uint32_t *v = src + (d3 ? 3 : 2) * n;      // velocities
    const int s = u.off + i;
    u.px[s] = src[i];
    u.py[s] = src[n + i];
    u.pz[s] = d3 ? src[2 * n + i] : 0u;
    u.vx[s] = __uint_as_float(v[i]);
    u.vy[s] = __uint_as_float(v[n + i]);
    u.vz[s] = d3 ? __uint_as_float(v[2 * n + i]) : 0.0f;
    u.type[s] = (int32_t)v[(d3 ? 3 : 2) * n + i];
    u.id[s] = i;
}

}  // namespace plife
