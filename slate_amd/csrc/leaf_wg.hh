// Panel LU in one workgroup, rows in registers (gfx950).
#pragma once
#include "common.hh"
#include <limits>

namespace sa {

// One-workgroup LU of a panel of at most NT * RPT rows of W columns, rows in
// registers: v[q][c] of a thread holds column (j + c) mod W of its q-th row at
// step j, so every register index is a constant.  Used by the panel leaf
// (panel.hip) and by the batched solver's panels (batched.hip).
// Bound: the serial chain of a column, two barriers long, so everything that
// can is taken off it:
//  - rows never move: an interchange swaps the two owners' row labels, and a
//    row is stored at its label at the end;
//  - the next column is updated first and its candidates are searched (DPP
//    maxima) while the other columns' updates issue; each wave's candidate is
//    inverted on that side, too;
//  - only the live part of the pivot row goes through LDS, from its owner,
//    between the two barriers.
// The update writes v[q][c - 1] from v[q][c], which is the rotation; the
// columns still to update shrink by W / 4 per stage.  Finished columns of a
// stage and finished rows meet a zero factor (a wave that sees a non-finite
// factor puts them aside meanwhile).
// FP64, 32 columns of 100 rows: 140 us per leaf with the exchange through
// memory that one workgroup does not need, 50 us here, and 500 rows as much;
// with two rows per thread 1000 rows 69 us, where the exchange now takes 64.
// A column of that is about 3000 cycles, of which the two barriers and the LDS round trips
// between them are a third.
template <class T>
struct LeafEntry { T abs, val, inv; uint32_t idx; };       // a wave's candidate

template <class T, int W, int NT>
struct LeafWg {
    static_assert(NT / 64 <= 8, "one entry per lane of a group of eight");
    LeafEntry<T> ent[NT / 64];
    T ajj;                                                 // row j of the column being searched
    __attribute__((aligned(16))) T prow[W];
    int pivs[W];
};

// Candidates of column j (rows labelled >= j), published per wave; `between`
// is issued between the maxima's start and their use.
template <class T, int W, int RPT, int NT, class F>
__device__ __forceinline__ void leaf_wg_publish(LeafWg<T, W, NT>& s, const T (&col)[RPT], const int (&lab)[RPT], int j,
                                                int m, F&& between)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    T babs = T(-1), bval = T(0);
    uint32_t bidx = 0xFFFFFFFFu;
    #pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const T a = fabs(col[q]);
        // a thread's rows are not in label order after interchanges
        const bool take = lab[q] >= j && lab[q] < m && (a > babs || (a == babs && uint32_t(lab[q]) < bidx));
        babs = take ? a : babs;
        bval = take ? col[q] : bval;
        bidx = take ? uint32_t(lab[q]) : bidx;
    }
    const uint32_t key = argmax_key(babs);
    const uint32_t mk = wave_max_u32(key);
    const T binv = T(1) / bval;
    between();
    const int wl = wave_argmax_lane(babs, bidx, key, mk);
    if (lane == wl) s.ent[wave] = LeafEntry<T>{babs, bval, binv, bidx};
    #pragma unroll
    for (int q = 0; q < RPT; ++q)
        if (lab[q] == j) s.ajj = col[q];
}

// Columns [j, jend) with rotated columns 1 .. C - 1 live (C >= W - j).
template <class T, int W, int RPT, int NT, int C, class I>
__device__ __forceinline__ void leaf_wg_steps(LeafWg<T, W, NT>& s, T (&v)[RPT][W], int (&lab)[RPT], int& j, int jend,
                                              int w, int m, T* __restrict__ A, int64_t ld, int64_t r0, int64_t c0,
                                              I* info, T threshold)
{
    constexpr int NW = NT / 64;
    // entries of the pivot row in flight per wait: what the registers allow
    constexpr int XCH = RPT * W * int(sizeof(T)) >= 512 ? 16 : W;
    const int tid = threadIdx.x, lane = tid & 63;
    const T safe_min = std::numeric_limits<T>::min();
    #pragma unroll 1
    for (; j < jend; ++j) {
        __syncthreads();                                   // candidates of column j published
        // the winner among the waves: lane k holds wave k's candidate
        const LeafEntry<T> e = s.ent[lane < NW ? lane : 0];
        const T ajj = s.ajj;
        const uint32_t key = lane < NW ? argmax_key(e.abs) : 0u;
        const uint32_t mk = max8_u32(key);
        const int bw = wave_argmax_lane(e.abs, e.idx, key, mk);
        // Tile_getrf.hh:283-289: keep the diagonal if it is large enough
        const uint64_t keep = __ballot(!(e.abs >= T(0)) || fabs(ajj) >= threshold * e.abs);
        int p = __builtin_amdgcn_readlane(int(e.idx), bw);
        T inv = lane_val(e.inv, bw), pv = lane_val(e.val, bw);
        if (((keep >> bw) & 1) && p != j) {                // the diagonal, and it is not the winner itself
            p = j;
            pv = ajj;
            inv = T(1) / ajj;
        }
        const bool zero = pv == T(0), tiny = fabs(pv) < safe_min;
        #pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (lab[q] == p) {
                #pragma unroll
                for (int c = 1; c < C; ++c) s.prow[c] = v[q][c];
            }
        // rows j and p change places: their labels do
        T l[RPT];
        bool odd = false;                                  // a non-finite factor seen by this wave
        #pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int lb = lab[q];
            lab[q] = lb == p ? j : (lb == j ? p : lb);
            const bool act = lab[q] > j && lab[q] < m;
            T t = v[q][0] * inv;
            if (zero || tiny) t = zero ? v[q][0] : v[q][0] / pv;
            l[q] = act ? t : T(0);
            v[q][0] = act ? t : v[q][0];
            odd = odd || !isfinite(l[q]);
        }
        if (tid == 0) {
            s.pivs[j] = p;
            if (zero && *info == 0) *info = I(c0 + j + 1);
        }
        __syncthreads();                                   // row p published
        const int lim = W - j;                             // rotated columns lim .. W - 1 are finished
        odd = odd || (lane >= 1 && lane < lim && lane < W && !isfinite(s.prow[lane & (W - 1)]));
        const bool sel = __ballot(odd) != 0;
        // 0 * inf would reach finished columns and rows: park them in the
        // leaf's own memory, which is free until the end, and take them back
        auto park = [&](bool back) {
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int i = tid + NT * q;
                const bool act = lab[q] > j && lab[q] < m;
                T* rowp = A + (r0 + (i < m ? i : 0)) * ld + c0;
                #pragma unroll
                for (int c = 1; c < W; ++c) {
                    const int col = (j + c) & (W - 1);
                    if (!back) { if (i < m && col < w) rowp[col] = v[q][c]; }
                    else if (!(act && c < lim)) v[q][c - 1] = i < m && col < w ? rowp[col] : T(0);
                }
            }
        };
        if (sel) park(false);
        T t0[RPT], nxt[RPT];
        {
            const T x1 = s.prow[1];
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                t0[q] = v[q][0];
                nxt[q] = (lab[q] > j && 1 < lim) ? v[q][1] - l[q] * x1 : v[q][1];
            }
        }
        // the other columns: update and move down by one
        auto rest = [&] {
            #pragma unroll
            for (int q = 0; q < RPT; ++q) v[q][0] = nxt[q];
            #pragma unroll
            for (int c = 2; c < C; ++c) {
                if (c % XCH == 0) asm volatile("" ::: "memory");
                const T xr = s.prow[c];
                const T x = c > C - W / 4 ? (c < lim ? xr : T(0)) : xr;
                #pragma unroll
                for (int q = 0; q < RPT; ++q) v[q][c - 1] = v[q][c] - l[q] * x;
            }
            #pragma unroll
            for (int c = C; c < W; ++c)
                #pragma unroll
                for (int q = 0; q < RPT; ++q) v[q][c - 1] = v[q][c];
            #pragma unroll
            for (int q = 0; q < RPT; ++q) v[q][W - 1] = t0[q];
            if (sel) park(true);
        };
        leaf_wg_publish<T, W, RPT, NT>(s, nxt, lab, j + 1, m, rest);   // after the last column: not read
    }
}

// All w columns (the candidates of column 0 are published here).
template <class T, int W, int RPT, int NT, class I>
__device__ __forceinline__ void leaf_wg_factor(LeafWg<T, W, NT>& s, T (&v)[RPT][W], int (&lab)[RPT], int w, int m,
                                               T* __restrict__ A, int64_t ld, int64_t r0, int64_t c0, I* info,
                                               T threshold)
{
    T col[RPT];
    #pragma unroll
    for (int q = 0; q < RPT; ++q) col[q] = v[q][0];
    leaf_wg_publish<T, W, RPT, NT>(s, col, lab, 0, m, [] {});
    int j = 0;
    leaf_wg_steps<T, W, RPT, NT, W>(s, v, lab, j, w < W / 4 ? w : W / 4, w, m, A, ld, r0, c0, info, threshold);
    leaf_wg_steps<T, W, RPT, NT, 3 * W / 4>(s, v, lab, j, w < W / 2 ? w : W / 2, w, m, A, ld, r0, c0, info, threshold);
    leaf_wg_steps<T, W, RPT, NT, W / 2>(s, v, lab, j, w < 3 * W / 4 ? w : 3 * W / 4, w, m, A, ld, r0, c0, info, threshold);
    leaf_wg_steps<T, W, RPT, NT, W / 4>(s, v, lab, j, w, w, m, A, ld, r0, c0, info, threshold);
    __syncthreads();                                       // every wave is done with its parking rows
}

} // namespace sa
