// plife_split.hpp -- the fused velocity + position kernel for worlds whose
// densest homes outlast the rest of the launch.
//
// Reference: backend/Physics.java:397-450 (updateVelocity, updatePosition).
//
// A home's candidates are added in order, so one lane steps them as a chain:
// about 0.28 us a neighbour on k_force.  Where a launch holds few particles
// with thousands of neighbours (a small world that has clustered), that chain
// and not the device's rate is the step's time.  Here four lanes share a home:
// a workgroup of 256 threads owns 64 homes and streams their neighbourhood
// through LDS in windows of `cap` candidates.
//   A  lane `sub` of a home's quad screens every fourth 32-candidate word of
//      its runs, and the quad's lanes write the kept indices, in candidate
//      order, to the home's list (a prefix sum of their counts across the quad);
//   B  the quad evaluates four kept candidates at a time, two steps in flight,
//      and every lane adds their terms in candidate order (group_terms).
// The sums stay in registers from window to window.  These are k_force's
// operations in its order: the bits do not change.  The instructions per pair
// are 2.1 times k_force's, which a launch that leaves most of the device idle
// does not notice (classify_worlds).
#pragma once

#include "plife_force.hpp"

namespace plife {

constexpr int kSplitThreads = 256;
constexpr int kSplitLanes = 4;
constexpr int kSplitHomes = kSplitThreads / kSplitLanes;

struct SplitLds {
    size_t m, xy, list, z, id, off, type, total;
};

// List entries per home: a window's worth, plus two so that the homes' lists
// start in different banks.  An entry is the LDS address of a candidate's type
// in 16 bits: static and dynamic LDS together stay within 64 KB (plan_split_for).
__host__ __device__ constexpr int split_list_stride(int cap) { return cap + 2; }

__host__ __device__ inline SplitLds split_lds_layout(int dim, bool debug, int ntypes, bool m_in_lds, int cap,
                                                     int max_cells)
{
    SplitLds L;
    size_t o = 0;
    L.m = o;     o += m_in_lds ? (size_t)ntypes * ntypes * 8 : 0;
    L.xy = o;    o += (size_t)(cap + kScreenPad) * 8;
    L.list = o;  o += (size_t)kSplitHomes * split_list_stride(cap) * 2;
    L.z = o;     o += dim == 3 ? (size_t)(cap + kScreenPad) * 4 : 0;
    L.id = o;    o += debug ? (size_t)cap * 4 : 0;
    L.off = o;   o += (size_t)(max_cells + 1) * 4;
    L.type = o;  o += (size_t)cap;
    L.total = (o + 15) & ~(size_t)15;
    return L;
}

template <int DIM, bool WRAP, bool DEBUG, bool MLDS>
__global__ __launch_bounds__(kSplitThreads) void k_force_split(ForceArgs a)
{
    constexpr int NR = DIM == 3 ? 9 : 3;      // stencil rows per part
    constexpr int T = kSplitThreads, G = kSplitLanes, NW = T / kWave;
    constexpr int U = 8;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_part[kMaxParts][3];      // row, first column, last column
    __shared__ uint32_t s_cnt[NW + 1];
    __shared__ unsigned long long s_pairs[NW];
    __shared__ uint2 s_seg[kMaxSegs * NR];

    const SplitLds L = split_lds_layout(DIM, DEBUG, a.ntypes_max, MLDS, a.cap, a.max_cells);
    double *const M = reinterpret_cast<double *>(smem + L.m);
    const Staged stg = staged_at(reinterpret_cast<uint2 *>(smem + L.xy), reinterpret_cast<uint32_t *>(smem + L.z),
                                 reinterpret_cast<uint32_t *>(smem + L.id), smem + L.type);
    uint32_t *const off = reinterpret_cast<uint32_t *>(smem + L.off);

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int home = tid / G, sub = tid % G;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const uint2 bw = a.blocks[a.block_base + blk];
    const WorldDev w = a.worlds[bw.x];
    const int nx = w.nx;
    const uint32_t cb = w.cell_base;
    const int g0 = (int)bw.y;
    const int nact = min(kSplitHomes, w.off + w.n - g0);
    uint16_t *const list = reinterpret_cast<uint16_t *>(smem + L.list) + home * split_list_stride(a.cap);

    if constexpr (MLDS)
        for (int t = tid; t < w.ntypes * w.ntypes; t += T) M[t] = a.matrix[w.moff + t] * w.R;

    const bool active = home < nact;
    const int g = g0 + (active ? home : nact - 1);
    const uint4 hr = a.rec[g];
    const uint32_t hx = hr.x, hy = hr.y, hz = DIM == 3 ? hr.z : 0u;
    const int mrow = (int)hr.w * w.ntypes;
    const uint32_t key = a.skeys[g] - cb;
    const int hrow = (int)(key / (uint32_t)nx);
    const int hcx = (int)(key - (uint32_t)hrow * (uint32_t)nx);

    // parts = distinct rows among the homes (each quad's first lane speaks for it)
    const bool first = active && sub == 0;
    const int prow = (home > 0 && active) ? (int)((a.skeys[g - 1] - cb) / (uint32_t)nx) : -1;
    const int nrow = (home + 1 < nact) ? (int)((a.skeys[g + 1] - cb) / (uint32_t)nx) : -1;
    const bool pstart = first && (home == 0 || prow != hrow);
    const bool pend = first && (home + 1 == nact || nrow != hrow);
    const uint64_t starts = __ballot(pstart);
    if (lane == 0) s_cnt[wv] = (uint32_t)__popcll(starts);
    __syncthreads();
    uint32_t before = 0, nparts = 0;
#pragma unroll
    for (int v = 0; v < NW; ++v) {
        before += v < wv ? s_cnt[v] : 0u;
        nparts += s_cnt[v];
    }
    const uint64_t le = lane == 63 ? ~0ull : ((2ull << lane) - 1);
    const int mypart = (int)(before + __popcll(starts & le)) - 1;
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
    const bool use_lds = !w.all_global && nparts <= (uint32_t)kMaxParts && p_base[kMaxParts] <= a.max_cells;

    Acc acc;
    acc.x = acc.y = acc.z = 0.0;
    acc.cnt = 0;                       // interacting pairs this lane evaluated
    acc.hash = 0ull;
    if (use_lds) {
        const int S = (int)stage_cells<DIM, T>(a, p_base, p_w, p_row, p_ca, nx, cb, off, s_seg, s_cnt);
        const int nsegs = (int)nparts * NR * 3;
        int pb = p_base[0], pw = p_w[0], pc = p_ca[0];
#pragma unroll
        for (int q = 1; q < kMaxParts; ++q)
            if (mypart == q) { pb = p_base[q]; pw = p_w[q]; pc = p_ca[q]; }
        const int jh = hcx - pc + 1;
        // the stencil-origin quirk's skipped column, row and layer (see k_force)
        const int cy = hrow % nx, cz = DIM == 3 ? hrow / nx : 0;
        bool q2x = false, q2y = false, q2z = false;
        if (hcx == nx - 1) q2x = stencil_origin(hx, w.cs) == nx;
        if (cy == nx - 1) q2y = stencil_origin(hy, w.cs) == nx;
        if (DIM == 3 && cz == nx - 1) q2z = stencil_origin(hz, w.cs) == nx;
        const int j_lo = jh - 1 + (q2x ? 1 : 0);
        const uint32_t bx = staged_axis<WRAP>(hx), by = staged_axis<WRAP>(hy), bz = staged_axis<WRAP>(hz);
        const uint32_t hq = high_halves(bx, by);
        WorldDev wf = w;
        asm volatile("" : "+v"(wf.one_plus_beta));
        asm volatile("" : "+v"(wf.inv_beta));

        auto step_list = [&](auto exact, int n) {
            constexpr bool EXACT = decltype(exact)::value;
            auto coef = [&](int p, int &dx, int &dy, int &dz) -> double {
                const uint32_t k = list[min(p, n - 1)];
                double d2;
                const double m = staged_pair<DIM, WRAP, MLDS, EXACT>(a, wf, stg, M, k, bx, by, bz, mrow, dx, dy, dz, d2);
                const double c = pair_coef<false>(d2, pair_recip(d2), m, wf);
                const bool in = (p < n) & (d2 != 0.0) & (d2 <= w.r2u);      // Physics.java:432
                acc.cnt += in ? 1 : 0;
                if constexpr (DEBUG)
                    if (in) acc.hash += id_hash(stg.id[k - stg.at.type]);
                return in ? c : 0.0;
            };
#pragma unroll 1
            for (int s = 0; s < n; s += 2 * G) {
                int x1, y1, z1, x2, y2, z2;
                const double c1 = coef(s + sub, x1, y1, z1);
                const double c2 = coef(s + G + sub, x2, y2, z2);
                group_terms<DIM, G>(acc, c1, x1, y1, z1);
                group_terms<DIM, G>(acc, c2, x2, y2, z2);
            }
        };

        for (int w0 = 0; w0 < S; w0 += a.cap) {
            const int wn = min(a.cap, S - w0);
            stage_window<DIM, WRAP, DEBUG, T>(a, stg, s_seg, nsegs, w0, wn);
            __syncthreads();
            // ---- phase A: the home's kept candidates, in order, into its list
            int n = 0;
#pragma unroll 1
            for (int r = 0; r < NR; ++r) {
                const int oyr = (r % 3) - 1, ozr = DIM == 3 ? (r / 3) - 1 : 0;
                const bool skip = !active || (q2y && oyr == -1) || (q2z && ozr == -1);
                const int rb = pb + r * pw;
                const int klo = max((int)off[rb + j_lo] - w0, 0);
                const int len = skip ? 0 : max(0, min((int)off[rb + jh + 2] - w0, wn) - klo);
                const int K = wave_max(len);
#pragma unroll 1
                for (int i0 = 0; i0 < K; i0 += 32 * G) {
                    const int i = i0 + 32 * sub;
                    const int kb = i < len ? klo + i : 0;
                    uint32_t word = 0;
#pragma unroll
                    for (int gq = 3; gq >= 0; --gq)
                        if (i0 + gq * U < K) word = screen_group<DIM, U>(stg, kb + gq * U, hq, bz, w.sbias, word);
                    word &= low_bits(len - i);
                    const uint32_t c = (uint32_t)__popc(word);
                    const uint32_t c0 = group_bcast<G, 0>(c), c1 = group_bcast<G, 1>(c), c2 = group_bcast<G, 2>(c),
                                   c3 = group_bcast<G, 3>(c);
                    int at = n + (int)((sub > 0 ? c0 : 0u) + (sub > 1 ? c1 : 0u) + (sub > 2 ? c2 : 0u));
                    const uint32_t ka = (uint32_t)kb + stg.at.type;
                    while (word) {
                        list[at++] = (uint16_t)(ka + (uint32_t)__builtin_ctz(word));
                        word &= word - 1u;
                    }
                    n += (int)(c0 + c1 + c2 + c3);
                }
            }
            // the quad's lanes are in one wave, whose LDS accesses are in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            // ---- phase B
            if (w.exact_d2) step_list(std::true_type{}, n);
            else step_list(std::false_type{}, n);
            __syncthreads();
        }
    } else if (first) {
        home_global<DIM, WRAP, DEBUG, MLDS>(a, w, M, g, hx, hy, hz, mrow, acc);
    }
    unsigned long long tot = (unsigned long long)acc.cnt;
    if constexpr (DEBUG)
        for (int d = 1; d < G; d <<= 1) {
            acc.cnt += __shfl_xor(acc.cnt, d, kWave);
            acc.hash += __shfl_xor(acc.hash, d, kWave);
        }
    if (first) finish_home<DIM, WRAP, DEBUG>(a, w, acc, hx, hy, hz, (int)hr.w, a.perm[g], g);

    // interacting pairs, one 64-bit atomic per workgroup
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) tot += __shfl_xor(tot, d, kWave);
    if (lane == 0) s_pairs[wv] = tot;
    __syncthreads();
    if (tid == 0) {
        unsigned long long sum = 0;
#pragma unroll
        for (int v = 0; v < NW; ++v) sum += s_pairs[v];
        if (sum) {
            atomicAdd(a.pair_total, sum);
            atomicAdd(a.pair_world + bw.x, sum);
        }
        record_block_work(a, blk, sum);
    }
}

}  // namespace plife
