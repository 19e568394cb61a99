// plife_force.hpp -- the fused velocity + position kernel of the particle-life step.
//
// Reference: backend/Physics.java:397-450 (updateVelocity, updatePosition),
// the accelerator lambda app/Main.java:275-280, Range.java:40-96.
//
// Work decomposition: a workgroup of BS threads owns BS consecutive home
// particles of the cell-sorted order, so every wave is full.  It stages, for
// each grid row it touches (2D: row = cy, 3D: row = cy + cz*nx), the
// 3^(DIM-1) neighbour rows x (span + 2) cells of the sorted SoA in LDS; each
// thread owns one home and, per stencil row, scans the three staged cells
// around its own column -- exactly the cells the reference's 3x3 (3x3x3)
// stencil visits.
//
// Each home particle runs two phases over its candidates:
//   A  integer screen on the high 16 bits of the coordinates (screen_hi).  Kept
//      candidates become bits of mask words in LDS.
//   B  For kept candidates only: the reference's predicate in FP64
//      (d2 = dx*dx + dy*dy, d2 != 0 && d2 <= rmax*rmax; Physics.java:430-432) and
//      the force law in FP64 (FP64 FMA issues at the non-packed FP32 rate on
//      CDNA4), accumulated in FP64.
// The screen is a strict superset of the FP64 predicate, so neighbour sets are
// exactly the reference's.
#pragma once

#include <type_traits>

#include "plife_kernels.hpp"

namespace plife {

struct ForceArgs {
    const uint4 *rec;                // x, y, z, type of each sorted slot (multi-launch path)
    // step-start state in the pre-sort order, read through the permutation
    const uint32_t *perm;            // sorted slot -> pre-sort index
    const uint32_t *sx, *sy, *sz;    // (one-launch step)
    const float *vx, *vy, *vz;
    const int32_t *type, *id;
    // the new state, written in the sorted order (Physics.particles after the swap)
    uint32_t *ox, *oy, *oz;
    float *ovx, *ovy, *ovz;
    int32_t *otype, *oid;
    const uint32_t *skeys;           // batch cell key of each sorted slot
    const uint32_t *cell_start, *cell_end;
    const double *matrix;            // per world ntypes*ntypes at moff, row = acted-on type
    const WorldDev *worlds;
    const uint2 *blocks;             // per workgroup: (world, first home slot)
    int block_base;                  // this launch's first entry of blocks
    int ntypes_max, m_in_lds;
    int cap, max_cells;
    int wpool;                       // mask words of a workgroup with one window (0: always several)
    int wpool2;                      // and of one that streams several
    unsigned long long *pair_total;  // interacting pairs of the step, all worlds
    unsigned long long *pair_world;  // per world
    uint32_t *block_work;            // pinned host memory: per table entry its pairs (saturated); [nb_total] = tag
    uint32_t work_tag;               // identifies the block table the counts belong to
    int nb_total;
    int32_t *dbg_count;
    unsigned long long *dbg_hash;
    float *dbg_acc;                  // debug: the step's acceleration per sorted slot, (x, y, z)
};

struct Acc {
    double x, y, z;
    int cnt;
    unsigned long long hash;
};

__device__ __forceinline__ unsigned long long id_hash(uint32_t id)
{
    unsigned long long z = (unsigned long long)id + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// One pair in FP64, in units of 2^-32 (the fixed-point grid), where scaling
// by powers of two is exact: with D = x_q - x_p, rel = D/rmax, dist = |rel|,
// the reference adds rel*(f/dist)*(rmax*force*dt) = D*(f/dist)*(force*dt) where
//   f/dist = 1/beta - 1/dist                             (dist <  beta)
//          = a*(1 - |1 + beta - 2 dist|/(1 - beta))/dist (dist >= beta)
// (app/Main.java:275-280).  acc accumulates D*(f/dist) in units of 2^-32.
// With u = |D| = dist R (R = rmax 2^32) and y = 1/|D|: 1/dist = R y, and the
// attractive branch is (a R) (1 - |1 + beta - 2 S u|/(1 - beta)) y, so the
// caller passes mR = a * R (staged that way with the matrix).
template <int DIM>
__device__ __forceinline__ double pair_d2(double dx, double dy, double dz)
{
#pragma clang fp contract(off)
    // JOML lengthSquared without FMA: x*x + (y*y + z*z) (exact 2^64 scaling)
    return DIM == 3 ? dx * dx + (dy * dy + dz * dz) : dx * dx + dy * dy;
}

// 1/|D|: one Newton step from FP32, low by up to 2^-44 of itself.  (NaN where d2 = 0.)
__device__ __forceinline__ double pair_recip(double d2)
{
    const double y0 = (double)__builtin_amdgcn_rsqf((float)d2);
    const double e = d2 * y0;
    const double h = fma(-e, y0, 1.0);
    return fma(0.5 * y0, h, y0);
}

// pair_d2 where every square of a pair in range is below 2^52 (rmax <= 2^-6,
// WorldDev::exact_d2): squares and sums of integers below 2^53 are exact, so
// FMAs give the same value in one instruction less per axis; a pair whose sum
// is past 2^53 is out of range either way.
template <int DIM, bool EXACT>
__device__ __forceinline__ double pair_d2_of(double dx, double dy, double dz)
{
    if constexpr (!EXACT) return pair_d2<DIM>(dx, dy, dz);
    else return DIM == 3 ? fma(dx, dx, fma(dy, dy, dz * dz)) : fma(dx, dx, dy * dy);
}

// f/dist of the force law for a pair in range (0 < d2 <= rmax^2), y =
// pair_recip(d2), its branches summed in place of selected: below beta g is
// negative, at and above it 1/beta - 1/dist is not, so that of max(g, 0) and
// min(1/beta - 1/dist, 0) one is zero and the FMA adds an exact zero to the other
// branch's value -- two instructions where a compare, two selects and a multiply
// take four.  (g <= 1, so the clamp to [0, 1], free on its FMA, is max(g, 0).
// Within 2^-44 of beta both terms are zero.)  ANY: mR need not be finite -- its
// term is taken where g is not zero or dist not below beta; for a finite mR the
// bits are the same, so they do not depend on the kernel that steps a world.
template <bool ANY>
__device__ __forceinline__ double pair_coef(double d2, double y, double mR, const WorldDev &a)
{
    const double u = d2 * y;                       // |D| = dist R
    const double t = fabs(fma(u, a.m2S, a.one_plus_beta));
    const double g = fmin(fmax(fma(t, -a.inv_1mb, 1.0), 0.0), 1.0);
    const double rep = fmin(fma(-a.R, y, a.inv_beta), 0.0);   // 1/beta - 1/dist
    const double att = !ANY || g > 0.0 || !(u < a.betaR) ? mR * g : 0.0;
    return fma(att, y, rep);
}

// A coefficient, or (almost) zero for a pair out of range: its high word goes,
// and the 2^-1042 that may be left, times any difference and count, stays below
// 2^-980, which no velocity, position or exported acceleration shows (world_dev
// keeps force and dt within 2^400).  Clearing both words, 1.3% more
// instructions: 512-world batch 1655 us a launch, 1640 so; clearing 1/|D| in FP32
// instead lengthens the chain, dense 196k 2D world 1870 -> 1975.
__device__ __forceinline__ double clear_high(double c, bool in)
{
    uint2 b = __builtin_bit_cast(uint2, c);
    b.y = in ? b.y : 0u;
    return __builtin_bit_cast(double, b);
}

template <int DIM, bool DEBUG>
__device__ __forceinline__ void pair64(Acc &acc, int dxi, int dyi, int dzi, double mR, uint32_t qid,
                                       const WorldDev &a)
{
    const double dx = (double)dxi, dy = (double)dyi, dz = (double)dzi;
    const double d2 = pair_d2<DIM>(dx, dy, dz);
    const bool in = (d2 != 0.0) & (d2 <= a.r2u);     // Physics.java:432
    if (in) {
        const double c = pair_coef<true>(d2, pair_recip(d2), mR, a);
        acc.x = fma(c, dx, acc.x);
        acc.y = fma(c, dy, acc.y);
        if constexpr (DIM == 3) acc.z = fma(c, dz, acc.z);
        acc.cnt += 1;
        if constexpr (DEBUG) acc.hash += id_hash(qid);
    }
}

// G lanes share a home (G = 4: a quad of lanes; G = 16: a row of 16): lane k of
// the group holds candidate k's coefficient and difference, and every lane adds
// the G terms in candidate order, acc = fma(c_k, D_k, acc) for k = 0 .. G-1,
// each lane's values broadcast across the group by DPP -- the operations and
// the order of one lane stepping them all (a term with c = 0 leaves a sum
// unchanged: a sum that starts at +0 is never -0).
template <int G, int K>
__device__ __forceinline__ uint32_t group_bcast(uint32_t v)
{
    static_assert(G == 4 || G == 16, "groups are DPP quads or rows");
    if constexpr (G == 4) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, K * 0x55, 0xf, 0xf, false);  // quad_perm:[K,K,K,K]
    else return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + K, 0xf, 0xf, false);  // row_newbcast:K
}

template <int DIM, int G, int K = 0>
__device__ __forceinline__ void group_terms(Acc &acc, double c, int dx, int dy, int dz)
{
    if constexpr (K < G) {
        const unsigned long long cb = (unsigned long long)__double_as_longlong(c);
        const unsigned long long kb = (unsigned long long)group_bcast<G, K>((uint32_t)cb) |
                                      ((unsigned long long)group_bcast<G, K>((uint32_t)(cb >> 32)) << 32);
        const double ck = __longlong_as_double((long long)kb);
        acc.x = fma(ck, (double)(int)group_bcast<G, K>((uint32_t)dx), acc.x);
        acc.y = fma(ck, (double)(int)group_bcast<G, K>((uint32_t)dy), acc.y);
        if constexpr (DIM == 3) acc.z = fma(ck, (double)(int)group_bcast<G, K>((uint32_t)dz), acc.z);
        group_terms<DIM, G, K + 1>(acc, c, dx, dy, dz);
    }
}

// The block's pairs, for the host to order the next updates' blocks
// heaviest first; entry nb_total tags the table they belong to.
__device__ __forceinline__ void record_block_work(const ForceArgs &a, int blk,
                                                  unsigned long long pairs)
{
    const int e = a.block_base + blk;
    a.block_work[e] = (uint32_t)min(pairs, 0xFFFFFFFFull);
    if (e == 0) a.block_work[a.nb_total] = a.work_tag;
}

// Largest of the wave's values (each >= 0), the same in every lane: the DPP
// steps of wave_incl_scan with max in place of add, read from lane 63 into a
// scalar register, so that loops bounded by it branch on scalars.
__device__ __forceinline__ int wave_max(int v)
{
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));    // row_shr:1
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));    // row_bcast:15
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));    // row_bcast:31
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

// Phase A screen on exact fixed-point deltas.  In a clamped world the int32
// difference may wrap across the box (|D| >= 1/2 > rmax); phase B's exact
// sign test drops those, so the screen stays a superset.
template <int DIM>
__device__ __forceinline__ bool screen(uint32_t hx, uint32_t hy, uint32_t hz, uint32_t qx,
                                       uint32_t qy, uint32_t qz, float r2hi)
{
    const float dx = (float)(int)(qx - hx), dy = (float)(int)(qy - hy);
    float d2 = dx * dx;
    d2 = fmaf(dy, dy, d2);
    if constexpr (DIM == 3) {
        const float dz = (float)(int)(qz - hz);
        d2 = fmaf(dz, dz, d2);
    }
    // d2 == 0 (the home itself, coincident particles) passes the screen; the
    // FP64 predicate of phase B drops it
    return d2 <= r2hi;
}

// The staged kernel keeps each candidate's x and y as two words, the high
// halves (x >> 16 | y & 0xFFFF0000) and the low halves (x & 0xFFFF | y << 16):
// phase A reads the first alone, phase B rebuilds the exact coordinates from
// both (one v_perm_b32 each).
__device__ __forceinline__ uint32_t high_halves(uint32_t x, uint32_t y)
{
    return __builtin_amdgcn_perm(y, x, 0x07060302u);
}
__device__ __forceinline__ uint32_t low_halves(uint32_t x, uint32_t y)
{
    return __builtin_amdgcn_perm(y, x, 0x05040100u);
}
__device__ __forceinline__ uint32_t join_x(uint2 hl) { return __builtin_amdgcn_perm(hl.x, hl.y, 0x05040100u); }
__device__ __forceinline__ uint32_t join_y(uint2 hl) { return __builtin_amdgcn_perm(hl.x, hl.y, 0x07060302u); }

typedef short short2v __attribute__((ext_vector_type(2)));

// Phase A screen on the high 16 bits of each coordinate (65,536 steps per
// box, so differences modulo 2^16 are minimum-image differences): negative
// when the candidate is kept.  One 32-bit subtract takes both differences: a
// borrow out of the low half takes one more step off the high one, so x is
// less than 1 step off the exact difference, y less than 2, z less than 1, and
// `bias` = -(bq + 1), bq = (rmax / step + sqrt(DIM + 3))^2 (WorldDev::sbias),
// keeps every pair with |D| <= rmax (1 + 2^-20).  Issue cycles per wave and
// candidate, measured: subtract 2, dot product with the bias as accumulator
// 4, the caller's v_alignbit_b32 4 -- against 26 for exact differences in
// FP32 (two subtracts, two conversions, mul, fma, compare, select, or).  The
// clamped dot product is the three-operand form (no copy of the bias).
template <int DIM>
__device__ __forceinline__ int screen_hi(uint32_t q, uint32_t h, uint32_t qz, uint32_t hz, int bias)
{
    const short2v d = __builtin_bit_cast(short2v, q - h);
    int c = bias;
    if constexpr (DIM == 3) {
        const uint32_t dz = qz - hz;      // its high half: z's difference in steps
        asm("v_mad_i32_i16 %0, %1, %1, %2 op_sel:[1,1,0,0]" : "=v"(c) : "v"(dz), "s"(bias));
    }
    return __builtin_amdgcn_sdot2(d, d, c, true);
}

__device__ __forceinline__ int wrap_cell(int c, int n)
{
    return c < 0 ? c + n : (c >= n ? c - n : c);
}

// FP64 stencil origin floor(x / cs) (Physics.java:404-405), not clamped.
__device__ __forceinline__ int stencil_origin(uint32_t k, double cs)
{
    return (int)floor(((double)k * kInvFix) / cs);
}

// Physics.java:443-450 + Range.wrap / Range.clamp in FP64, rounded to 2^-32.
__device__ __forceinline__ uint32_t integrate_axis(uint32_t k, double v, double dt, bool wrap)
{
#pragma clang fp contract(off)
    double x = v * dt + (double)k * kInvFix;    // JOML mulAdd: v*dt + x
    if (!(x == x)) return 0u;
    if (wrap) {
        x = x - floor(x);                       // equals Range.wrap's repeated +-1
        const double s = rint(x * kFix);        // [0, 2^32]; 2^32 (x == 1.0) wraps to 0
        return (uint32_t)(unsigned long long)s;
    }
    x = x < 0.0 ? 0.0 : (x > 1.0 ? 1.0 : x);
    const double s = rint(x * kFix);
    return s >= 4294967295.0 ? 0xFFFFFFFFu : (uint32_t)(unsigned long long)s;
}

template <int DIM, bool WRAP, bool DEBUG>
__device__ __forceinline__ void finish_home(const ForceArgs &a, const WorldDev &w, const Acc &acc,
                                            uint32_t hx, uint32_t hy, uint32_t hz, int htype,
                                            uint32_t o, int g)
{
    const double nvx = w.ff * (double)a.vx[o] + w.kdt * acc.x;
    const double nvy = w.ff * (double)a.vy[o] + w.kdt * acc.y;
    a.ovx[g] = (float)nvx;
    a.ovy[g] = (float)nvy;
    a.ox[g] = integrate_axis(hx, nvx, w.dt, WRAP);
    a.oy[g] = integrate_axis(hy, nvy, w.dt, WRAP);
    if constexpr (DIM == 3) {
        const double nvz = w.ff * (double)a.vz[o] + w.kdt * acc.z;
        a.ovz[g] = (float)nvz;
        a.oz[g] = integrate_axis(hz, nvz, w.dt, WRAP);
    }
    a.otype[g] = htype;
    a.oid[g] = a.id[o];
    if constexpr (DEBUG) {
        a.dbg_count[g] = acc.cnt;
        a.dbg_hash[g] = acc.hash;
        // the force law's acceleration (Physics.java:437 summed, over dt) in FP32
        a.dbg_acc[3 * (size_t)g + 0] = (float)(w.ka * acc.x);
        a.dbg_acc[3 * (size_t)g + 1] = (float)(w.ka * acc.y);
        a.dbg_acc[3 * (size_t)g + 2] = DIM == 3 ? (float)(w.ka * acc.z) : 0.0f;
    }
}

// Candidates lo..hi-1 of the cell-sorted order for home g (slot), FP64
// throughout: the body of the reference's per-cell loop (Physics.java:413-424).
template <int DIM, bool WRAP, bool DEBUG, bool MLDS>
__device__ __forceinline__ void visit_run(const ForceArgs &a, const WorldDev &w, const double *Mlds,
                                          int g, uint32_t hx, uint32_t hy, uint32_t hz, int row,
                                          Acc &acc, int lo, int hi)
{
    constexpr int G = 4;               // records read together
#pragma unroll 1
    for (int j0 = lo; j0 < hi; j0 += G) {
        uint4 q[G];
#pragma unroll
        for (int u = 0; u < G; ++u) q[u] = a.rec[min(j0 + u, hi - 1)];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int j = j0 + u;
            const uint32_t qx = q[u].x, qy = q[u].y, qz = DIM == 3 ? q[u].z : 0u;
            const int dxi = (int)(qx - hx), dyi = (int)(qy - hy);
            const int dzi = DIM == 3 ? (int)(qz - hz) : 0;
            bool ok = (j < hi) & (j != g);
            if (!WRAP) {
                // plain difference of the clamped world: skip |D| >= 1/2
                ok &= ((dxi >= 0) == (qx >= hx)) & ((dyi >= 0) == (qy >= hy));
                if (DIM == 3) ok &= ((dzi >= 0) == (qz >= hz));
            }
            if (!ok) continue;
            const int idx = row + (int)q[u].w;
            const double m = MLDS ? Mlds[idx] : a.matrix[w.moff + idx] * w.R;
            pair64<DIM, DEBUG>(acc, dxi, dyi, dzi, m, DEBUG ? (uint32_t)a.id[a.perm[j]] : 0u, w);
        }
    }
}

// Literal reference stencil over 3^DIM cells straight from global memory
// (Physics.java:404-424), FP64 throughout.  Used for strips whose staged
// neighbourhood does not fit in LDS, for sparse worlds and for grids with
// fewer than 3 cells per axis (where the reference visits repeated cells).
// Where a stencil row does not wrap in x its three cells are consecutive keys,
// so the row is one run of the cell-sorted order: the same candidates in the
// same order as the per-cell loop, from two bound loads instead of six, all
// issued before the first candidate is visited.
template <int DIM, bool WRAP, bool DEBUG, bool MLDS>
__device__ void home_global(const ForceArgs &a, const WorldDev &w, const double *Mlds, int g,
                            uint32_t hx, uint32_t hy, uint32_t hz, int row, Acc &acc)
{
    constexpr int NR = DIM == 3 ? 9 : 3;
    const int nx = w.nx;
    const int cx0 = stencil_origin(hx, w.cs);
    const int cy0 = stencil_origin(hy, w.cs);
    const int cz0 = DIM == 3 ? stencil_origin(hz, w.cs) : 0;
    if (cx0 >= 1 && cx0 <= nx - 2) {
        int lo[NR], hi[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int cy = wrap_cell(cy0 + r % 3 - 1, nx);
            const int cz = DIM == 3 ? wrap_cell(cz0 + r / 3 - 1, nx) : 0;
            const uint32_t ci = w.cell_base + (uint32_t)(cx0 - 1 + cy * nx + cz * nx * nx);
            lo[r] = (int)a.cell_start[ci];
            hi[r] = (int)a.cell_end[ci + 2];
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            visit_run<DIM, WRAP, DEBUG, MLDS>(a, w, Mlds, g, hx, hy, hz, row, acc, lo[r], hi[r]);
        return;
    }
    const int zlo = DIM == 3 ? -1 : 0, zhi = DIM == 3 ? 1 : 0;
    for (int oz = zlo; oz <= zhi; ++oz)
        for (int oy = -1; oy <= 1; ++oy)
            for (int ox = -1; ox <= 1; ++ox) {
                int cx = wrap_cell(cx0 + ox, nx), cy = wrap_cell(cy0 + oy, nx);
                int cz = DIM == 3 ? wrap_cell(cz0 + oz, nx) : 0;
                if (WRAP) {
                    cx = wrap_cell(cx, nx);
                    cy = wrap_cell(cy, nx);
                    if (DIM == 3) cz = wrap_cell(cz, nx);
                } else if (cx < 0 || cx >= nx || cy < 0 || cy >= nx ||
                           (DIM == 3 && (cz < 0 || cz >= nx))) {
                    continue;
                }
                const uint32_t ci = w.cell_base + (uint32_t)(cx + cy * nx + cz * nx * nx);
                visit_run<DIM, WRAP, DEBUG, MLDS>(a, w, Mlds, g, hx, hy, hz, row, acc,
                                                  (int)a.cell_start[ci], (int)a.cell_end[ci]);
            }
}

// Staged columns of the parts: part q holds rows x p_w[q] cells from
// p_base[q] on.  A workgroup's homes span a few consecutive cells of one grid
// row, or (at row ends) of a few rows; each distinct row is a part.
constexpr int kMaxParts = 4;
constexpr int kScreenPad = 40;   // candidates a screen step reads from one base, at most

// A staged row's columns are consecutive cells, one run of the sorted order,
// except where they wrap around the box in x: up to three runs (segments).
constexpr int kMaxSegs = kMaxParts * 3;      // per stencil row

// Exclusive prefix of the NC staged cells' counts (off, NC + 1 entries) for a
// workgroup of T threads, and the segment table: entry k of segs holds the
// first staged entry of segment k and the sorted slot minus the staged entry
// of its particles.  An unused segment starts where the next one does.
// Returns the staged particle count, the same in every thread.  Ends with a
// barrier.
template <int DIM, int T>
__device__ __forceinline__ uint32_t stage_cells(const ForceArgs &a, const int (&p_base)[kMaxParts + 1],
                                                const int (&p_w)[kMaxParts], const int (&p_row)[kMaxParts],
                                                const int (&p_ca)[kMaxParts], int nx, uint32_t cb,
                                                uint32_t *off, uint2 *segs, uint32_t *s_cnt)
{
    constexpr int NW = T / kWave, NR = DIM == 3 ? 9 : 3;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int NC = p_base[kMaxParts];
    uint32_t carry = 0;
    for (int f0 = 0; f0 < NC; f0 += T) {
        const int f = f0 + tid;
        uint32_t c = 0, s0 = 0;
        int seg = 0, j = 0, pw = p_w[0], pc = p_ca[0];
        if (f < NC) {
            int pb = p_base[0], pr = p_row[0], part = 0;
#pragma unroll
            for (int q = 1; q < kMaxParts; ++q)
                if (f >= p_base[q] && p_w[q] > 0) { pb = p_base[q]; pw = p_w[q]; pr = p_row[q]; pc = p_ca[q]; part = q; }
            const int r = (f - pb) / pw;
            j = (f - pb) - r * pw;
            const int oy = (r % 3) - 1, oz = DIM == 3 ? (r / 3) - 1 : 0;
            const int cy = pr % nx, cz = DIM == 3 ? pr / nx : 0;
            const int x = wrap_cell(pc - 1 + j, nx);
            const int y = wrap_cell(cy + oy, nx);
            const int z = DIM == 3 ? wrap_cell(cz + oz, nx) : 0;
            const uint32_t ci = cb + (uint32_t)(x + y * nx + z * nx * nx);
            s0 = a.cell_start[ci];
            c = a.cell_end[ci] - s0;
            seg = (part * NR + r) * 3;
        }
        const uint32_t inc = wave_incl_scan(c);
        if (lane == kWave - 1) s_cnt[wv] = inc;
        __syncthreads();
        uint32_t wbase0 = carry, tot = 0;
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            wbase0 += v < wv ? s_cnt[v] : 0u;
            tot += s_cnt[v];
        }
        if (f < NC) {
            const uint32_t o = wbase0 + inc - c;
            const uint2 here = make_uint2(o, s0 - o);
            off[f] = o;
            // column 0 (wrapped or not), column 1 (a run of its own only after a
            // wrapped column 0), the last column (only when it wraps)
            const bool lw = pc == 0, rw = pc - 1 + pw - 1 == nx;
            if (j == 0) {
                segs[seg] = here;
                if (!lw) segs[seg + 1] = here;
            }
            if (j == 1 && lw) segs[seg + 1] = here;
            if (j == pw - 1) segs[seg + 2] = rw ? here : make_uint2(o + c, 0u);
        }
        carry += tot;
        __syncthreads();
    }
    if (tid == 0) off[NC] = carry;
    __syncthreads();
    return carry;
}

// A staged coordinate, and the difference of two.  Periodic worlds: the
// coordinate itself; its differences modulo 2^32 are minimum-image differences.
// Clamped worlds: with the top bit flipped, so that a saturating signed
// subtraction gives the plain difference where |D| < 1/2 and +-2^31 where it is
// not: past any rmax that has a staged grid (at most 1/3), with no sign test.
template <bool WRAP>
__device__ __forceinline__ uint32_t staged_axis(uint32_t x)
{
    return WRAP ? x : x ^ 0x80000000u;
}
template <bool WRAP>
__device__ __forceinline__ int staged_diff(uint32_t q, uint32_t h)
{
    if constexpr (WRAP) return (int)(q - h);
    else return __builtin_elementwise_sub_sat((int)q, (int)h);
}

// Staged candidates in LDS: high and low halves of x and y, z, type and
// (debug) id.
struct StagedAt {                    // LDS addresses of entry 0, less 8 (xy) or 4 (z) times the types'
    uint32_t type, xy, z;
};
struct Staged {
    uint2 *xy;
    uint32_t *z, *id;
    uint8_t *type;
    StagedAt at;
};

#define PLIFE_LDS __attribute__((address_space(3)))
template <typename T>
__device__ __forceinline__ uint32_t lds_address(T *p)
{
    return (uint32_t)(uintptr_t)(PLIFE_LDS unsigned char *)(unsigned char *)p;
}
template <typename T>
__device__ __forceinline__ T lds_read(uint32_t at)
{
    return *(PLIFE_LDS const T *)(uintptr_t)at;
}

__device__ __forceinline__ Staged staged_at(uint2 *xy, uint32_t *z, uint32_t *id, uint8_t *type)
{
    const uint32_t t = lds_address(type);
    return Staged{xy, z, id, type, StagedAt{t, lds_address(xy) - 8u * t, lds_address(z) - 4u * t}};
}

// Stages entries [w0, w0 + wn) of the neighbourhood (nsegs segments) with T
// threads: one 16-byte record read per entry.
template <int DIM, bool WRAP, bool DEBUG, int T>
__device__ __forceinline__ void stage_window(const ForceArgs &a, const Staged &s, const uint2 *segs, int nsegs,
                                             int w0, int wn)
{
    for (int t = threadIdx.x; t < wn; t += T) {
        const uint32_t sg = (uint32_t)(w0 + t);
        int lo = 0, hi = nsegs;        // the last segment that starts at or before sg
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (segs[mid].x <= sg) lo = mid;
            else hi = mid;
        }
        const uint32_t slot = sg + segs[lo].y;
        const uint4 q = a.rec[slot];
        const uint32_t x = staged_axis<WRAP>(q.x), y = staged_axis<WRAP>(q.y);
        s.xy[t] = make_uint2(high_halves(x, y), low_halves(x, y));
        if constexpr (DIM == 3) s.z[t] = staged_axis<WRAP>(q.z);
        if constexpr (DEBUG) s.id[t] = (uint32_t)a.id[a.perm[slot]];
        s.type[t] = (uint8_t)q.w;
    }
}

// U candidates from entry kb against one home: word << U, bit u set when
// candidate kb + u passes the phase-A screen.  Built from the last candidate
// down, each result's sign bit shifted in by one v_alignbit_b32.
template <int DIM, int U>
__device__ __forceinline__ uint32_t screen_group(const Staged &s, int kb, uint32_t hq, uint32_t hz, int bias,
                                                 uint32_t word)
{
    const uint2 *qp = s.xy + kb;
    const uint32_t *qzp = s.z + kb;
    int t[U];
#pragma unroll
    for (int u = U - 1; u >= 0; --u) t[u] = screen_hi<DIM>(qp[u].x, hq, DIM == 3 ? qzp[u] : 0u, hz, bias);
#pragma unroll
    for (int u = U - 1; u >= 0; --u) word = __builtin_amdgcn_alignbit(word, (uint32_t)t[u], 31);
    return word;
}

// The low n bits set (n clamped to [0, 32]).
__device__ __forceinline__ uint32_t low_bits(int n)
{
    return n >= 32 ? ~0u : n <= 0 ? 0u : (1u << n) - 1u;
}

// Staged candidate at place k (the LDS address of its type, from which the
// others follow in one instruction each) against a home at (px, py, pz)
// (staged_axis) with matrix row mrow: its matrix entry times R, the difference
// and its square.
template <int DIM, bool WRAP, bool MLDS, bool EXACT>
__device__ __forceinline__ double staged_pair(const ForceArgs &a, const WorldDev &w, const Staged &s,
                                              const double *M, uint32_t k, uint32_t px, uint32_t py, uint32_t pz,
                                              int mrow, int &dxi, int &dyi, int &dzi, double &d2)
{
    const uint64_t xy = lds_read<uint64_t>(8u * k + s.at.xy);
    const uint2 hl = make_uint2((uint32_t)xy, (uint32_t)(xy >> 32));
    dxi = staged_diff<WRAP>(join_x(hl), px);
    dyi = staged_diff<WRAP>(join_y(hl), py);
    dzi = DIM == 3 ? staged_diff<WRAP>(lds_read<uint32_t>(4u * k + s.at.z), pz) : 0;
    const int idx = mrow + (int)lds_read<uint8_t>(k);
    d2 = pair_d2_of<DIM, EXACT>((double)dxi, (double)dyi, (double)dzi);
    return MLDS ? M[idx] : a.matrix[w.moff + idx] * w.R;
}

// Mask words: the top kWordCands bits one candidate each, first at the top, the
// rest the first candidate's place.  Phase B needs a new word for some lane
// nearly every candidate: one 4-byte read at a running address, where 32-bit
// masks with a table of their bases took two reads at computed ones and 6 bytes
// (force kernel, 1M 2D world 173 -> 165 us, 512-world batch 1740 -> 1619; with
// 16-bit bases, 22% more LDS and a workgroup less on a CU, 1M 175).
constexpr int kWordCands = 20, kPlaceBits = 32 - kWordCands;
// Places are below it: the types are at LDS address 0, as long as k_force has no
// static LDS (which is checked in the built library).
constexpr int kMaxStaged = (1 << kPlaceBits) - 64;

// Phase B of one home at (px, py, pz) with matrix row mrow: its `left` kept
// candidates, word by word from `at` in candidate order, two per iteration (half
// the loop's bookkeeping; their force laws overlap).  ab.cnt counts the lane's
// interacting pairs in debug mode; else, on the scalar unit, `loop` those of all
// the wave's lanes while this lane is in the loop (the wave's total is its
// largest) and ab.cnt the lane's odd last one.
template <int DIM, bool WRAP, bool DEBUG, bool MLDS, bool EXACT>
__device__ __forceinline__ void walk_home_of(const ForceArgs &a, const WorldDev &w, const Staged &s,
                                             const double *M, Acc &ab, int &loop, int left, const uint32_t *at,
                                             uint32_t px, uint32_t py, uint32_t pz, int mrow)
{
    auto visit = [&](uint32_t k, bool last) {
        int dxi, dyi, dzi;
        double d2;
        const double m = staged_pair<DIM, WRAP, MLDS, EXACT>(a, w, s, M, k, px, py, pz, mrow, dxi, dyi, dzi, d2);
        const uint64_t in = __ballot(d2 != 0.0) & __ballot(d2 <= w.r2u);       // Physics.java:432
        double y = pair_recip(d2);
        // (the mask is complete by here, off the chain that ends in its use)
        asm("" : "+v"(y) : "s"(in));
        const bool mine = __builtin_amdgcn_inverse_ballot_w64(in);
        const double c = clear_high(pair_coef<false>(d2, y, m, w), mine);
        ab.x = fma(c, (double)dxi, ab.x);
        ab.y = fma(c, (double)dyi, ab.y);
        if constexpr (DIM == 3) ab.z = fma(c, (double)dzi, ab.z);
        if (DEBUG || last) {
            ab.cnt += mine ? 1 : 0;
            if constexpr (DEBUG)
                if (mine) ab.hash += id_hash(s.id[k - s.at.type]);
        } else {
            loop += __popcll(in);
        }
    };
    uint32_t m = 0;
    auto next = [&]() {
        if (m < (1u << kPlaceBits)) m = *at++;
        const int b = __builtin_clz(m);
        m ^= 0x80000000u >> b;
        return (m & ((1u << kPlaceBits) - 1u)) + (uint32_t)b;
    };
#pragma unroll 1
    for (; left >= 2; left -= 2) {
        const uint32_t k1 = next();
        const uint32_t k2 = next();
        visit(k1, false);
        visit(k2, false);
    }
    if (left > 0) visit(next(), true);
}

template <int DIM, bool WRAP, bool DEBUG, bool MLDS>
__device__ __forceinline__ void walk_home(const ForceArgs &a, const WorldDev &w, const Staged &s,
                                          const double *M, Acc &ab, int &loop, int left, const uint32_t *at,
                                          uint32_t px, uint32_t py, uint32_t pz, int mrow)
{
    if (w.exact_d2) walk_home_of<DIM, WRAP, DEBUG, MLDS, true>(a, w, s, M, ab, loop, left, at, px, py, pz, mrow);
    else walk_home_of<DIM, WRAP, DEBUG, MLDS, false>(a, w, s, M, ab, loop, left, at, px, py, pz, mrow);
}

// Counting sort of the HPT * T homes of a workgroup by their kept-candidate
// counts (thread tid holds the counts of slots tid, tid + T, ..., in bins of
// 2^shift; the order inside a bin does not matter): s_deal[rank] = slot.
// Synchronises before it reads anything the homes' threads wrote, and after.
template <int T, int HPT>
__device__ __forceinline__ void deal_homes(const int (&count)[HPT], int shift, uint32_t *s_bin,
                                           uint16_t *s_deal, uint32_t *s_cnt)
{
    constexpr int PER = 256 / T;              // bins per thread
    const int tid = threadIdx.x;
    for (int t = tid; t < 256; t += T) s_bin[t] = 0u;
    __syncthreads();
    int bin[HPT];
    uint32_t local[HPT];
#pragma unroll
    for (int q = 0; q < HPT; ++q) {
        bin[q] = min(count[q] >> shift, 255);
        local[q] = atomicAdd(&s_bin[bin[q]], 1u);
    }
    __syncthreads();
    {
        uint32_t v[PER], sum = 0, total = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            v[q] = s_bin[tid * PER + q];
            sum += v[q];
        }
        uint32_t ex = block_excl_scan<T>(sum, s_cnt, total);
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            s_bin[tid * PER + q] = ex;
            ex += v[q];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < HPT; ++q) s_deal[s_bin[bin[q]] + local[q]] = (uint16_t)(tid + q * T);
    __syncthreads();
}

// The LDS of a staged workgroup: `cap` staged entries at most; the windowed
// path streams a denser neighbourhood through it.
struct ForceLds {
    size_t st, m, sxy, words, ax, ay, az, dhash, hxy, hz, dcnt, words2, ht, sz, sid, off, fixed, total;
};

// Bytes per home that several windows keep in LDS besides the mask words: the
// sums, the home's position and type, and (debug) its count and hash.
constexpr int force_home_bytes(int dim, bool debug) { return dim * 8 + (dim == 3 ? 12 : 8) + 1 + (debug ? 12 : 0); }

// LDS of a workgroup of BS homes whose size does not depend on the plan.
template <int BS, int NR>
struct ForceFixed {
    uint2 seg[kMaxSegs * NR];
    unsigned long long pairs[BS / kWave];
    uint32_t bin[256];
    uint32_t cnt[BS / kWave + 1];
    int part[kMaxParts][3];            // row, first column, last column
    uint16_t deal[BS];
    uint16_t si[BS], hc[BS], wo[BS];   // per home: its staged index, kept candidates and first mask word
};
constexpr size_t force_fixed_bytes(int dim, int bs)
{
    return dim == 3 ? (bs == 64 ? sizeof(ForceFixed<64, 9>) : bs == 128 ? sizeof(ForceFixed<128, 9>) : sizeof(ForceFixed<256, 9>))
                    : (bs == 64 ? sizeof(ForceFixed<64, 3>) : bs == 128 ? sizeof(ForceFixed<128, 3>) : sizeof(ForceFixed<256, 3>));
}

// A workgroup whose neighbourhood is one window has a pool of wpool mask words;
// one that streams several windows keeps the per-home data in the same region
// and a pool of wpool2 words.
__host__ __device__ inline ForceLds force_lds_layout(int dim, bool debug, int ntypes, bool m_in_lds,
                                                     int cap, int bs, int max_cells, int wpool, int wpool2)
{
    ForceLds L;
    size_t o = 0;
    // the types first: a candidate's place is its type's address (kMaxStaged)
    L.st = o;    o += ((size_t)cap + 7) & ~(size_t)7;
    L.m = o;     o += m_in_lds ? (size_t)ntypes * ntypes * 8 : 0;
    // the screened arrays carry kScreenPad spare entries: a screen step reads
    // up to that many candidates from one base, all but one past a lane's range
    L.sxy = o;   o += (size_t)(cap + kScreenPad) * 8;
    L.words = o;
    const size_t wend = o + (size_t)wpool * 4;
    L.ax = o;    o += (size_t)bs * 8;
    L.ay = o;    o += (size_t)bs * 8;
    L.az = o;    o += dim == 3 ? (size_t)bs * 8 : 0;
    L.dhash = o; o += debug ? (size_t)bs * 8 : 0;
    L.hxy = o;   o += (size_t)bs * 8;
    L.hz = o;    o += dim == 3 ? (size_t)bs * 4 : 0;
    L.dcnt = o;  o += debug ? (size_t)bs * 4 : 0;
    L.words2 = o; o += (size_t)wpool2 * 4;
    L.ht = o;    o += (size_t)bs;
    o = o > wend ? o : wend;
    o = (o + 3) & ~(size_t)3;
    L.sz = o;    o += dim == 3 ? (size_t)(cap + kScreenPad) * 4 : 0;
    L.sid = o;   o += debug ? (size_t)cap * 4 : 0;
    L.off = o;   o += (size_t)(max_cells + 1) * 4;
    o = (o + 7) & ~(size_t)7;
    L.fixed = o; o += force_fixed_bytes(dim, bs);
    L.total = (o + 15) & ~(size_t)15;
    return L;
}

// MLDS: the type matrix is staged in LDS (ntypes <= 32); otherwise it is read
// from global memory.  A compile-time switch, so the hot loop's matrix load is
// a plain ds_read and never a generic (flat) load.
//
// A workgroup of BS threads (BS/64 waves) owns BS consecutive home particles
// of the cell-sorted order, so every wave is full.  The parts' 3^(DIM-1)
// stencil rows x (span + 2) cells are staged in LDS for the whole workgroup.
// Workgroups with more parts or staged cells than the cell table holds take
// the global path.
template <int DIM, bool WRAP, bool DEBUG, bool MLDS, int BS>
__global__ __launch_bounds__(BS) void k_force(ForceArgs a)
{
    constexpr int NR = DIM == 3 ? 9 : 3;      // stencil rows per part
    constexpr int RMID = DIM == 3 ? 4 : 1;    // the stencil row of the home's own row (oy = oz = 0)
    constexpr int U = 8;                      // candidates per screen group
    constexpr int NW = BS / kWave;
    extern __shared__ __align__(16) unsigned char smem[];
    const ForceLds L = force_lds_layout(DIM, DEBUG, a.ntypes_max, MLDS, a.cap, BS, a.max_cells,
                                        a.wpool, a.wpool2);
    double *M = reinterpret_cast<double *>(smem + L.m);
    uint2 *sxy = reinterpret_cast<uint2 *>(smem + L.sxy);
    uint32_t *szz = reinterpret_cast<uint32_t *>(smem + L.sz);
    uint32_t *sid = reinterpret_cast<uint32_t *>(smem + L.sid);
    uint32_t *off = reinterpret_cast<uint32_t *>(smem + L.off);
    uint8_t *st = smem;                       // L.st
    auto &fix = *reinterpret_cast<ForceFixed<BS, NR> *>(smem + L.fixed);
    auto &s_part = fix.part;
    uint32_t *const s_cnt = fix.cnt, *const s_bin = fix.bin;
    unsigned long long *const s_pairs = fix.pairs;
    uint16_t *const s_deal = fix.deal, *const s_si = fix.si, *const s_hc = fix.hc, *const s_wo = fix.wo;
    uint2 *const s_seg = fix.seg;

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const uint2 bw = a.blocks[a.block_base + blk];
    const WorldDev w = a.worlds[bw.x];
    const int nx = w.nx;
    const uint32_t cb = w.cell_base;
    const int g0 = (int)bw.y;
    const int nact = min(BS, w.off + w.n - g0);

    if constexpr (MLDS)
        for (int t = tid; t < w.ntypes * w.ntypes; t += BS) M[t] = a.matrix[w.moff + t] * w.R;

    // Thread tid stands for home g0 + tid (sorted order).  Parts: grid rows (2D:
    // cy; 3D: cy + cz*nx) and columns of the homes.
    // Its position and type are read up front: independent loads whose
    // latency overlaps the setup.
    const bool active = tid < nact;
    const int g = g0 + (active ? tid : nact - 1);
    const uint32_t ho = a.perm[g];
    const uint4 hr = a.rec[g];
    const uint32_t hx = hr.x, hy = hr.y, hz = DIM == 3 ? hr.z : 0u;
    const int htype = (int)hr.w;
    const uint32_t hkey = a.skeys[g] - cb;
    const int hrow = (int)(hkey / (uint32_t)nx);
    const int hcx = (int)(hkey - (uint32_t)hrow * (uint32_t)nx);

    // parts = distinct rows among the homes (rows are non-decreasing with tid);
    // only active threads past the first read the previous home's key, so the
    // read stays inside [g0, g0 + nact)
    const int prow = (tid > 0 && active) ? (int)((a.skeys[g - 1] - cb) / (uint32_t)nx) : -1;
    const bool pstart = active && (tid == 0 || prow != hrow);
    const int nrow_next = (tid + 1 < nact) ? (int)((a.skeys[g + 1] - cb) / (uint32_t)nx) : -1;
    const bool pend = active && (tid + 1 == nact || nrow_next != hrow);
    const uint64_t wstarts = __ballot(pstart);
    if (lane == 0) s_cnt[wv] = (uint32_t)__popcll(wstarts);
    __syncthreads();
    uint32_t before = 0, nparts = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        before += w < wv ? s_cnt[w] : 0u;
        nparts += s_cnt[w];
    }
    const uint64_t le = lane == 63 ? ~0ull : ((2ull << lane) - 1);
    const int mypart = (int)(before + __popcll(wstarts & le)) - 1;
    if (pstart && mypart < kMaxParts) {
        s_part[mypart][0] = hrow;
        s_part[mypart][1] = hcx;
    }
    if (pend && mypart < kMaxParts) s_part[mypart][2] = hcx;
    __syncthreads();

    int p_row[kMaxParts], p_ca[kMaxParts], p_w[kMaxParts], p_base[kMaxParts + 1];
    p_base[0] = 0;
#pragma unroll
    for (int p = 0; p < kMaxParts; ++p) {
        const bool have = p < (int)nparts;
        p_row[p] = have ? s_part[p][0] : 0;
        p_ca[p] = have ? s_part[p][1] : 0;
        p_w[p] = have ? s_part[p][2] - p_ca[p] + 3 : 0;     // span + 2 staged columns
        p_base[p + 1] = p_base[p] + NR * p_w[p];
    }
    const int NC = p_base[kMaxParts];
    const bool use_lds = !w.all_global && a.cap > 0 && nparts <= (uint32_t)kMaxParts && NC <= a.max_cells;

    uint32_t carry = 0;
    if (use_lds) carry = stage_cells<DIM, BS>(a, p_base, p_w, p_row, p_ca, nx, cb, off, s_seg, s_cnt);
    else __syncthreads();

    const int mrow = htype * w.ntypes;

    // The force law's two additive constants held in VGPRs: each meets
    // another scalar operand in an FMA, which reads one scalar at most.
    WorldDev wf = w;
    asm volatile("" : "+v"(wf.one_plus_beta));
    asm volatile("" : "+v"(wf.inv_beta));
    const Staged stg = staged_at(sxy, szz, sid, st);

    Acc acc;
    acc.x = acc.y = acc.z = 0.0;
    acc.cnt = 0;
    acc.hash = 0ull;
    unsigned long long mycnt = 0;      // interacting pairs this thread stepped
    if (use_lds) {
        int pb = p_base[0], pw = p_w[0], pc = p_ca[0];
#pragma unroll
        for (int q = 1; q < kMaxParts; ++q)
            if (mypart == q) { pb = p_base[q]; pw = p_w[q]; pc = p_ca[q]; }
        const int jh = hcx - pc + 1;           // staged column of the home cell
        // Reference quirk: the stencil origin floor(x/cs) may be nx while the
        // key is clamped to nx-1 (Physics.java:367-372 vs 404-405).  The
        // reference then scans columns {nx-1, 0, 1}: skip staged column nx-2
        // (column 1 is always farther than rmax).  Same for rows / layers.
        const int cy = hrow % nx, cz = DIM == 3 ? hrow / nx : 0;
        // (the FP64 division only for homes in a last column, row or layer)
        bool q2x = false, q2y = false, q2z = false;
        if (hcx == nx - 1) q2x = stencil_origin(hx, w.cs) == nx;
        if (cy == nx - 1) q2y = stencil_origin(hy, w.cs) == nx;
        if (DIM == 3 && cz == nx - 1) q2z = stencil_origin(hz, w.cs) == nx;
        const int j_lo = jh - 1 + (q2x ? 1 : 0);
        const uint32_t bx = staged_axis<WRAP>(hx), by = staged_axis<WRAP>(hy), bz = staged_axis<WRAP>(hz);
        const uint32_t hq = high_halves(bx, by);

        // The home's run of stencil row r inside the window [w0, w0 + wn),
        // window-relative: returns its length, its first entry in lo.
        auto run_of = [&](int r, int w0, int wn, int &lo) -> int {
            const int oyr = (r % 3) - 1, ozr = DIM == 3 ? (r / 3) - 1 : 0;
            const bool skip = !active || (q2y && oyr == -1) || (q2z && ozr == -1);
            const int rb = pb + r * pw;
            lo = max((int)off[rb + j_lo] - w0, 0);
            const int hi = min((int)off[rb + jh + 2] - w0, wn);
            return skip ? 0 : max(0, hi - lo);
        };
        // First mask word of each home in the pool (s_wo) for a window, a run of
        // len candidates taking ceil(len / kWordCands) words; returns the words
        // needed.
        auto place_words = [&](int w0, int wn) -> uint32_t {
            int need = 0;
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                int lo;
                need += (run_of(r, w0, wn, lo) + kWordCands - 1) / kWordCands;
            }
            uint32_t total = 0;
            s_wo[tid] = (uint16_t)block_excl_scan<BS>((uint32_t)need, s_cnt, total);
            return total;
        };
        // Phase A: thread tid screens home tid; each 20 candidates of a row run
        // give one mask word, stored when any candidate passed.  Returns the kept
        // candidates.
        auto screen_home = [&](int w0, int wn, uint32_t *wmask) -> int {
            int at = s_wo[tid], npass = 0;
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                int klo;
                const int len = run_of(r, w0, wn, klo);
                const int K = wave_max(len);
#pragma unroll 1
                for (int i = 0; i < K; i += 2 * kWordCands) {
                    // a lane past its run reads the window's first entries
                    // (and keeps none of them)
                    const int kb = i < len ? klo + i : 0;
                    auto put = [&](uint32_t word, int c) {
                        word &= low_bits(len - i - c);
                        if (word) {
                            wmask[at] = __builtin_bitreverse32(word) | ((uint32_t)(kb + c) + stg.at.type);
                            ++at;
                            npass += __popc(word);
                        }
                    };
                    uint32_t word = 0;
                    if (i + 16 < K) word = screen_group<DIM, 4>(stg, kb + 16, hq, bz, w.sbias, word);
                    if (i + 8 < K) word = screen_group<DIM, U>(stg, kb + 8, hq, bz, w.sbias, word);
                    put(screen_group<DIM, U>(stg, kb, hq, bz, w.sbias, word), 0);
                    if (i + 20 < K) {
                        word = 0;
                        if (i + 36 < K) word = screen_group<DIM, 4>(stg, kb + 36, hq, bz, w.sbias, word);
                        if (i + 28 < K) word = screen_group<DIM, U>(stg, kb + 28, hq, bz, w.sbias, word);
                        put(screen_group<DIM, U>(stg, kb + 20, hq, bz, w.sbias, word), kWordCands);
                    }
                }
            }
            return npass;
        };

        // this thread's share of the pairs walk_home counted
        auto wave_pairs = [&](int loop, int cnt) -> unsigned long long {
            const int most = wave_max(loop);
            return (unsigned long long)cnt + (lane == 0 ? (unsigned long long)most : 0ull);
        };

        const int S = (int)carry, nsegs = (int)nparts * NR * 3;
        if (a.wpool > 0 && S <= a.cap && place_words(0, S) <= (uint32_t)a.wpool) {
            // ---- one window ----------------------------------------------
            uint32_t *const wmask = reinterpret_cast<uint32_t *>(smem + L.words);
            stage_window<DIM, WRAP, DEBUG, BS>(a, stg, s_seg, nsegs, 0, S);
            __syncthreads();
            const int count[1] = {screen_home(0, S, wmask)};
            int si = 0;
            if (active) {
                const int f = pb + RMID * pw + jh;
                si = (int)off[f] + (g - (int)a.cell_start[cb + hkey]);
            }
            s_si[tid] = (uint16_t)si;
            s_hc[tid] = (uint16_t)count[0];
            // Phase B: lane tid steps the home of count rank tid whole, in its
            // scan order, so its sums do not depend on the windows.
            deal_homes<BS, 1>(count, 0, s_bin, s_deal, s_cnt);
            const int h = (int)s_deal[tid];
            int wloop = 0, wcnt = 0;
            if (h < nact) {
                const int hsi = s_si[h];
                const uint2 hhl = sxy[hsi];
                const uint2 hp = make_uint2(join_x(hhl), join_y(hhl));
                const uint32_t bhz = DIM == 3 ? szz[hsi] : 0u;
                const int btype = (int)st[hsi];
                Acc ab;
                ab.x = ab.y = ab.z = 0.0;
                ab.cnt = 0;
                ab.hash = 0ull;
                walk_home<DIM, WRAP, DEBUG, MLDS>(a, wf, stg, M, ab, wloop, (int)s_hc[h], wmask + s_wo[h], hp.x, hp.y,
                                                  bhz, btype * w.ntypes);
                const int gh = g0 + h;
                finish_home<DIM, WRAP, DEBUG>(a, w, ab, staged_axis<WRAP>(hp.x), staged_axis<WRAP>(hp.y),
                                              staged_axis<WRAP>(bhz), btype, a.perm[gh], gh);
                wcnt = ab.cnt;
            }
            mycnt = wave_pairs(wloop, wcnt);
        } else {
            // ---- several windows -----------------------------------------
            // The staged neighbourhood streams through LDS in windows of at most
            // cap entries and wpool2 mask words.  Each window's homes are dealt to
            // lanes by their counts of that window; a home's sums travel in LDS
            // from the lane that stepped it in one window to the lane that steps
            // it in the next, so its candidates are added in staged order
            // whatever the windows are.  (Per-thread candidate lists, flushed when
            // one lane's list filled, kept a third to a half of phase B's lanes
            // busy.)
            double *const ax = reinterpret_cast<double *>(smem + L.ax);
            double *const ay = reinterpret_cast<double *>(smem + L.ay);
            double *const az = reinterpret_cast<double *>(smem + L.az);
            unsigned long long *const dhash = reinterpret_cast<unsigned long long *>(smem + L.dhash);
            int *const dcnt = reinterpret_cast<int *>(smem + L.dcnt);
            uint2 *const hxy = reinterpret_cast<uint2 *>(smem + L.hxy);
            uint32_t *const hzz = reinterpret_cast<uint32_t *>(smem + L.hz);
            uint8_t *const ht = smem + L.ht;
            uint32_t *const wmask = reinterpret_cast<uint32_t *>(smem + L.words2);
            ax[tid] = ay[tid] = 0.0;
            hxy[tid] = make_uint2(bx, by);
            ht[tid] = (uint8_t)htype;
            if constexpr (DIM == 3) {
                az[tid] = 0.0;
                hzz[tid] = bz;
            }
            if constexpr (DEBUG) {
                dhash[tid] = 0ull;
                dcnt[tid] = 0;
            }
            for (int w0 = 0; w0 < S;) {
                // one entry needs a word per home at most, and wpool2 >= BS
                int wn = min(a.cap, S - w0);
                while (place_words(w0, wn) > (uint32_t)a.wpool2) wn = (wn + 1) >> 1;
                stage_window<DIM, WRAP, DEBUG, BS>(a, stg, s_seg, nsegs, w0, wn);
                __syncthreads();
                const int count[1] = {screen_home(w0, wn, wmask)};
                s_hc[tid] = (uint16_t)count[0];
                int shift = 0;
                while ((wn >> shift) > 256) ++shift;
                deal_homes<BS, 1>(count, shift, s_bin, s_deal, s_cnt);
                const int h = (int)s_deal[tid];
                const int left = (int)s_hc[h];
                int wloop = 0, wcnt = 0;
                if (left > 0) {
                    Acc ab;
                    ab.x = ax[h];
                    ab.y = ay[h];
                    ab.z = DIM == 3 ? az[h] : 0.0;
                    ab.cnt = 0;
                    ab.hash = 0ull;
                    const uint2 hp = hxy[h];
                    walk_home<DIM, WRAP, DEBUG, MLDS>(a, wf, stg, M, ab, wloop, left, wmask + s_wo[h], hp.x, hp.y,
                                                      DIM == 3 ? hzz[h] : 0u, (int)ht[h] * w.ntypes);
                    ax[h] = ab.x;
                    ay[h] = ab.y;
                    if constexpr (DIM == 3) az[h] = ab.z;
                    if constexpr (DEBUG) {
                        dcnt[h] += ab.cnt;
                        dhash[h] += ab.hash;
                    }
                    wcnt = ab.cnt;
                }
                mycnt += wave_pairs(wloop, wcnt);
                __syncthreads();
                w0 += wn;
            }
            if (active) {
                acc.x = ax[tid];
                acc.y = ay[tid];
                if constexpr (DIM == 3) acc.z = az[tid];
                if constexpr (DEBUG) {
                    acc.cnt = dcnt[tid];
                    acc.hash = dhash[tid];
                }
                finish_home<DIM, WRAP, DEBUG>(a, w, acc, hx, hy, hz, htype, ho, g);
            }
        }
    } else if (active) {
        home_global<DIM, WRAP, DEBUG, MLDS>(a, w, M, g, hx, hy, hz, mrow, acc);
        finish_home<DIM, WRAP, DEBUG>(a, w, acc, hx, hy, hz, htype, ho, g);
        mycnt = (unsigned long long)acc.cnt;
    }

    // interacting pairs, one 64-bit atomic per workgroup
    unsigned long long tot = mycnt;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) tot += __shfl_xor(tot, d, kWave);
    if (lane == 0) s_pairs[wv] = tot;
    __syncthreads();
    if (tid == 0) {
        unsigned long long sum = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += s_pairs[w];
        if (sum) {
            atomicAdd(a.pair_total, sum);
            atomicAdd(a.pair_world + bw.x, sum);
        }
        record_block_work(a, blk, sum);
    }
}

// Worlds whose workgroups would span more grid rows than the staged layout
// holds (a particle or less per cell): one thread per home of the cell-sorted
// order, each running home_global, with no LDS but the type matrix, so that
// many waves per CU hide the latency of the cell bounds and the gathers.
// Results are those of k_force for the same homes, bit for bit (k_force's
// global path is this code, and its staged path visits the same candidates in
// the same order).
constexpr int kSparseBlock = 256;

template <int DIM, bool WRAP, bool DEBUG, bool MLDS>
__global__ __launch_bounds__(kSparseBlock) void k_force_sparse(ForceArgs a)
{
    constexpr int NW = kSparseBlock / kWave;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ unsigned long long s_pairs[NW];
    double *M = reinterpret_cast<double *>(smem);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const uint2 bw = a.blocks[a.block_base + blk];
    const WorldDev w = a.worlds[bw.x];
    if constexpr (MLDS) {
        for (int t = tid; t < w.ntypes * w.ntypes; t += kSparseBlock) M[t] = a.matrix[w.moff + t] * w.R;
        __syncthreads();
    }
    const int g = (int)bw.y + tid;
    const bool active = g < w.off + w.n;
    Acc acc;
    acc.x = acc.y = acc.z = 0.0;
    acc.cnt = 0;
    acc.hash = 0ull;
    if (active) {
        const uint32_t ho = a.perm[g];
        const uint4 hr = a.rec[g];
        const uint32_t hx = hr.x, hy = hr.y, hz = DIM == 3 ? hr.z : 0u;
        const int htype = (int)hr.w;
        home_global<DIM, WRAP, DEBUG, MLDS>(a, w, M, g, hx, hy, hz, htype * w.ntypes, acc);
        finish_home<DIM, WRAP, DEBUG>(a, w, acc, hx, hy, hz, htype, ho, g);
    }
    // interacting pairs, one 64-bit atomic per workgroup
    unsigned long long tot = active ? (unsigned long long)acc.cnt : 0ull;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) tot += __shfl_xor(tot, d, kWave);
    if (lane == 0) s_pairs[wv] = tot;
    __syncthreads();
    if (tid == 0) {
        unsigned long long sum = 0;
#pragma unroll
        for (int k = 0; k < NW; ++k) sum += s_pairs[k];
        if (sum) {
            atomicAdd(a.pair_total, sum);
            atomicAdd(a.pair_world + bw.x, sum);
        }
        record_block_work(a, blk, sum);
    }
}

}  // namespace plife
