// Panel LU leaf and row interchanges (gfx950).
//
// The leaf kernel factors a tall, narrow block (up to 65536+ rows x W columns)
// with partial pivoting.  It replaces SLATE's host panel (internal::getrf_panel
// <HostTask>, src/internal/internal_getrf.cc:20-121, which pulls the panel to
// the CPU every step) by a GPU kernel in which G workgroups each keep a slice
// of rows in registers.  Per column, each workgroup publishes its pivot
// candidate as tagged words to a double-buffered exchange area; every
// workgroup reads the G candidates (one memory round trip once they have
// landed, with no grid barrier and no fences), picks the winner itself and
// finishes the next column with it; the rest of the pivot row follows while
// the next candidates travel.
// Pivot rules follow src/internal/Tile_getrf.hh:197-366: largest |a_ij| with
// the smallest row winning exact ties, the diagonal kept when
// |a_jj| >= threshold * max, scaling by the reciprocal unless the pivot is
// below the smallest normal number, and info = first exactly-zero pivot.
#include "common.hh"
#include "kernels.hh"
#include "leaf_wg.hh"
#include <limits>

namespace sa {

template <class T> struct LeafW;
template <> struct LeafW<double> { static constexpr int W = 32; };
template <> struct LeafW<float> { static constexpr int W = 32; };

int panel_leaf_width(int elem_bytes) { return elem_bytes == 8 ? LeafW<double>::W : LeafW<float>::W; }

// Exchange area (64-bit tagged words, see tw_store in common.hh).  Heads, one
// area per column parity: G + 1 entries of HW words, the candidates and row j
// (value, factor of the last column, entry of the next column, row index; a
// value is two words, the low one first, in FP64).  Pivot rows, one area per column parity:
// REP copies of W values in rotated order, workgroup g reads copy g mod REP
// (all of them polling one copy would queue up on its few cache lines).
// Column j of a launch carries tag tag0 + j.  Areas are reused only when every
// reader is through: a workgroup publishes its head j + 2 after it has read
// every head j + 1, which the others publish after they have read the heads
// j; and row j + 2 goes out after every head j + 2, which a workgroup
// publishes when its waves have read row j.
template <class T, int W>
struct LeafSlots {
    static constexpr int NWV = int(sizeof(T)) / 4;         // words per value
    static constexpr int HW = 4 * NWV;
    static constexpr int RW = W * NWV;
    static constexpr int REP = 8;
    __host__ __device__ static int64_t heads(int G) { return (int64_t(G) + 1) * HW; }
    __host__ __device__ static int64_t words(int G) { return 2 * heads(G) + 2 * REP * RW; }
};

//------------------------------------------------------------------------------
// The leaf's w interchanges (row j <-> row piv[j], sequentially, rows local to
// r0) applied to the other columns of the enclosing panel, [xp0, c0) and
// [c0 + w, xp0 + xpw), so that the recursive panel needs no row-swap launches
// of its own.  Both ranges are untouched while the leaf runs: the right part
// is only read by the solves that follow the leaf, the left part (finished
// columns of L) only needs the interchanges brought back.  Every workgroup
// builds the same list of at most 2w (dst <- src) row moves: a touched row
// r receives the original row t_0(t_1(...t_{w-1}(r))), t_j the j-th
// transposition; then it moves its share of the columns through LDS
// (gather, barrier, scatter), so sources are read before any is overwritten.
template <class T, int W, int NT, int CH = 32>
__device__ void leaf_swap_others(T* __restrict__ A, int64_t ld, int64_t r0, int64_t c0, int w, int64_t xp0,
                                 int64_t xpw, const int* s_pivs, int G, int g)
{
    // CH: columns per chunk
    __shared__ int s_dst[2 * W], s_src[2 * W];
    __shared__ int s_nmv;
    __shared__ T s_stage[2 * W * CH];
    const int tid = threadIdx.x;
    if (tid == 0) s_nmv = 0;
    __syncthreads();                            // s_pivs complete, counter cleared
    if (tid < 2 * W) {
        const int t = tid < W ? tid : tid - W;
        int dst = -1;
        if (t < w) {
            if (tid < W) {
                dst = t;
            }
            else {
                const int pt = s_pivs[t];
                bool first = pt >= w;
                for (int u = 0; u < t; ++u) first = first && s_pivs[u] != pt;
                if (first) dst = pt;
            }
        }
        if (dst >= 0) {
            int x = dst;
            for (int jj = w - 1; jj >= 0; --jj) {
                const int pj = s_pivs[jj];
                x = (x == jj) ? pj : (x == pj ? jj : x);
            }
            if (x != dst) {
                const int slot = atomicAdd(&s_nmv, 1);
                s_dst[slot] = dst;
                s_src[slot] = x;
            }
        }
    }
    __syncthreads();
    const int nmv = s_nmv;
    if (nmv == 0) return;
    const int64_t nother = xpw - w, left = c0 - xp0;
    const int64_t share = (nother + G - 1) / G;
    const int64_t q0 = int64_t(g) * share;
    const int64_t q1 = q0 + share < nother ? q0 + share : nother;
    for (int64_t qc = q0; qc < q1; qc += CH) {
        const int nc = int(q1 - qc < CH ? q1 - qc : CH);
        for (int e = tid; e < nmv * CH; e += NT) {
            const int mv = e / CH, cc = e % CH;
            if (cc < nc) {
                const int64_t q = qc + cc;
                const int64_t col = q < left ? xp0 + q : c0 + w + (q - left);
                s_stage[e] = A[(r0 + s_src[mv]) * ld + col];
            }
        }
        __syncthreads();
        for (int e = tid; e < nmv * CH; e += NT) {
            const int mv = e / CH, cc = e % CH;
            if (cc < nc) {
                const int64_t q = qc + cc;
                const int64_t col = q < left ? xp0 + q : c0 + w + (q - left);
                A[(r0 + s_dst[mv]) * ld + col] = s_stage[e];
            }
        }
        __syncthreads();
    }
}

//------------------------------------------------------------------------------
// A candidate in the form in which it travels, one word per lane: its value,
// its factor of the column before, its entry of the column after, its row (no
// candidate: value 0 and the largest row number, which loses to every other).
template <class T>
struct alignas(4 * sizeof(T)) LeafHead { T val, fac, nxt; uint32_t idx; };
// A column's decision: the winner's head and the last pivot row's entry of the
// column after.
template <class T>
struct LeafDec { LeafHead<T> h; T u2; };

// Of E candidates in LDS, the largest magnitude, then the smallest row.
template <class T>
__device__ __forceinline__ int leaf_best(const LeafHead<T>* h, int E)
{
    const int lane = threadIdx.x & 63;
    T ba = T(-1);
    uint32_t bi = 0xFFFFFFFFu;
    int be = 0;
    for (int e = lane; e < E; e += 64) {
        const T a = fabs(h[e].val);
        const uint32_t x = h[e].idx;
        const bool take = a > ba || (a == ba && x < bi);
        ba = take ? a : ba;
        bi = take ? x : bi;
        be = take ? e : be;
    }
    const uint32_t key = argmax_key(ba);
    const int l = wave_argmax_lane(ba, bi, key, wave_max_u32(key));
    return __builtin_amdgcn_readlane(be, l);
}

// The exchange of a leaf, by one wave of each workgroup: per column, between
// two barriers, it publishes the workgroup's candidate, gathers the heads of
// all workgroups, 64 words per load, and picks the winner out of its
// registers.  One wave issues an instruction about every five cycles, so the
// words stay on the lanes that loaded them: magnitudes order like their
// leading words, six DPP maxima find the largest, and its lanes store the head
// on.  Several of the same leading word are compared in LDS (s_tie).
template <class T, int W, int NW, int GMAX>
__device__ __forceinline__ void leaf_exchange(int w, int m, int64_t r0, int64_t c0, int64_t* __restrict__ ipiv,
                                              int64_t* __restrict__ info, T threshold, uint32_t tag0, uint64_t* slots,
                                              int* error, const LeafHead<T>* s_cand, LeafHead<T>* s_tie,
                                              LeafDec<T>* s_dec, int* s_pivs)
{
    using SL = LeafSlots<T, W>;
    typedef uint32_t __attribute__((may_alias)) word_t;
    constexpr int NWV = SL::NWV, HW = SL::HW, RW = SL::RW;
    constexpr int EPL = 64 / HW;                           // entries per load
    constexpr int NU = GMAX / EPL;
    constexpr int IDX = 3 * NWV, USED = IDX + 1;
    constexpr int LEAD = NWV - 1;                          // the leading word of the value
    const int G = gridDim.x, g = blockIdx.x;
    const int lane = threadIdx.x & 63, k = lane % HW;
    // load NU: row j's head on the first lanes, then the words of the last
    // pivot row that belong to column j + 1, tagged one step earlier; lanes
    // without a word of their own read another's
    const bool isu = lane >= HW && lane < HW + NWV;
    const int ku = k < USED ? k : 0;
    uint32_t off[NU], mask[NU];
    #pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = u * EPL + lane / HW;
        off[u] = uint32_t((e < G ? e : G) * HW + ku);
        mask[u] = (e < G && k == LEAD) ? 0x7FFFFFFFu : 0u;
    }
    const uint32_t cmask = (lane / HW < NW && k == LEAD) ? 0x7FFFFFFFu : 0u;
    #pragma unroll 1
    for (int j = 0; j < w; ++j) {
        uint64_t* const head = slots + (j & 1) * SL::heads(G);
        const uint64_t* const urow = slots + 2 * SL::heads(G) + (((j + 1) & 1) * SL::REP + (g & (SL::REP - 1))) * RW;
        const uint32_t tag = tag0 + uint32_t(j);
        __syncthreads();                                   // the waves' candidates
        {
            // lane e HW + k holds word k of wave e's candidate
            const uint32_t x = reinterpret_cast<const word_t*>(s_cand + (lane / HW < NW ? lane / HW : NW - 1))[ku];
            const uint32_t xj = reinterpret_cast<const word_t*>(s_cand + NW)[ku];
            const uint32_t key = x & cmask;
            const uint64_t eq = __builtin_amdgcn_ballot_w64(key == wave_max_u32(key));
            int b = int(__builtin_ctzll(eq)) / HW;
            if (eq & (eq - 1)) b = leaf_best(s_cand, NW);
            if (lane / HW == b && k < USED) tw_store(head + int64_t(g) * HW + k, x, tag);
            if (__builtin_amdgcn_readlane(int(xj), IDX) == j && lane < USED)
                tw_store(head + int64_t(G) * HW + lane, xj, tag);
        }
        uint32_t got[NU + 1];
        {
            const bool wantu = isu && j > 0 && j + 1 < w;
            const uint64_t* const px = wantu ? urow + 2 * NWV + (lane - HW) : head + int64_t(G) * HW + ku;
            const uint32_t tagx = wantu ? tag - 1 : tag;
            uint64_t t0 = 0;
            bool first = true;
            while (true) {
                uint64_t x[NU + 1];
                #pragma unroll
                for (int u = 0; u < NU; ++u) x[u] = tw_load(head + off[u]);
                x[NU] = tw_load(px);
                const int err = __hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                uint32_t bad = uint32_t(x[NU] >> 32) ^ tagx;
                got[NU] = uint32_t(x[NU]);
                #pragma unroll
                for (int u = 0; u < NU; ++u) {
                    bad |= uint32_t(x[u] >> 32) ^ tag;
                    got[u] = uint32_t(x[u]);
                }
                if (__builtin_amdgcn_ballot_w64(bad != 0) == 0 || err != 0) break;
                if (first) { t0 = wall_clock64(); first = false; }
                else if (wall_clock64() - t0 > 400000000ull) {
                    __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
        }
        uint32_t km = 0;
        #pragma unroll
        for (int u = 0; u < NU; ++u) {
            const uint32_t key = got[u] & mask[u];
            km = key > km ? key : km;
        }
        km = wave_max_u32(km);
        uint32_t bw = got[NU];                             // the winner's words, on lanes bl ...
        uint64_t any = 0, twice = 0;
        #pragma unroll
        for (int u = 0; u < NU; ++u) {
            const uint64_t eq = __builtin_amdgcn_ballot_w64((got[u] & mask[u]) == km);
            twice |= any & eq;
            any |= eq;
            bw = eq ? got[u] : bw;
        }
        int bl = __builtin_ctzll(any) & ~(HW - 1);
        if (twice | (any & (any - 1))) {
            #pragma unroll
            for (int u = 0; u < NU; ++u) reinterpret_cast<word_t*>(s_tie)[u * 64 + lane] = got[u];
            __builtin_amdgcn_wave_barrier();
            bw = reinterpret_cast<const word_t*>(s_tie + leaf_best(s_tie, G))[ku];
            bl = 0;
            __builtin_amdgcn_wave_barrier();
        }
        // Tile_getrf.hh:283-289: keep the diagonal if it is large enough (a
        // threshold of 1 keeps it where it is the first of the largest, the
        // winner); never take a row outside the leaf
        const uint32_t bi = uint32_t(__builtin_amdgcn_readlane(int(bw), bl + IDX));
        bool keep = bi < uint32_t(j) || bi >= uint32_t(m);
        if (threshold < T(1)) {
            if (lane / HW == bl / HW) reinterpret_cast<word_t*>(s_tie)[k] = bw;
            if (lane < HW) reinterpret_cast<word_t*>(s_tie + 1)[k] = got[NU];
            __builtin_amdgcn_wave_barrier();
            keep = keep || fabs(s_tie[1].val) >= threshold * fabs(s_tie[0].val);
            keep = __builtin_amdgcn_ballot_w64(keep) != 0;
            __builtin_amdgcn_wave_barrier();
        }
        bw = keep ? (k == IDX ? uint32_t(j) : got[NU]) : bw;
        bl = keep ? 0 : bl;
        if (lane / HW == bl / HW && k < USED) reinterpret_cast<word_t*>(&s_dec->h)[k] = bw;
        if (isu) reinterpret_cast<word_t*>(&s_dec->u2)[lane - HW] = got[NU];
        if (lane == bl + IDX) s_pivs[j] = int(bw);
        __syncthreads();                                   // the decision
        if (g == 0) {
            if (lane == bl + IDX) ipiv[c0 + j] = r0 + int64_t(bw);
            if (lane == 0 && s_dec->h.val == T(0) && *info == 0) *info = c0 + j + 1;
        }
    }
}

// Leaf over G workgroups of NT / 64 waves with rows and one for the exchange.
// v[q][c] of a thread holds column (j + c) mod W of its q-th row at step j, so
// every register index is a constant; rows never move, an interchange swaps
// their labels, and a row is stored at its label.
// Bound: the exchange between workgroups, one publication and one read per
// column, so little else stays on that chain:
//  - The pivot row travels beside it.  A head carries the candidate's value,
//    its factor l of the column before, and its entry of the column after as
//    it was before that column's update; with the pivot row of the column
//    before, which has arrived by then, every workgroup forms the one entry
//    u1 = next - l u that the next search needs, by the operation that the
//    row's owner applies.  The other entries are read and used while the next
//    heads travel.
//  - The exchanging wave has no rows, so updates and exchange overlap.
// Us per column, before (heads, then the row, then everything) and now: FP64,
// 8192 rows 4.6 and 2.3; FP32, 16384 rows 5.1 and 2.4, 65536 rows 7.1 and 2.8.
// Of 4900 cycles (FP64, 8192 rows) the heads' way through memory is 2300, the
// search 700, picking the winner 700, scaling 570, publishing 500; the pivot
// row arrives 2700 cycles after its column's search.
template <class T, int W, int RPT, int NT, int GMAX>
__global__ __launch_bounds__(NT + 64, RPT * W * sizeof(T) <= 256 ? 4 : 1)
void panel_leaf_rot_kernel(T* __restrict__ A, int64_t ld, int64_t r0, int64_t m_total, int64_t c0,
                           int w, int64_t* __restrict__ ipiv, int64_t* __restrict__ info, T threshold,
                           uint32_t tag0, uint64_t* slots, int* error, int64_t xp0, int64_t xpw, bool vec)
{
    using SL = LeafSlots<T, W>;
    constexpr int NWV = SL::NWV, RW = SL::RW;
    constexpr int NW = NT / 64;
    constexpr int VE = 16 / int(sizeof(T));
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    static_assert((W & (W - 1)) == 0 && RW <= 64 && W % VE == 0, "a row is one word per lane");
    static_assert(NW <= 8, "one candidate per lane of a group of eight");
    typedef T vec_t __attribute__((ext_vector_type(VE)));
    typedef uint32_t __attribute__((may_alias)) word_t;
    const int G = gridDim.x;
    const int g = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = int(m_total - r0);
    const T safe_min = std::numeric_limits<T>::min();

    __shared__ LeafHead<T> s_cand[NW + 1];                     // the waves', and row j if it is here
    __shared__ LeafHead<T> s_tie[GMAX];
    __shared__ LeafDec<T> s_dec;
    __shared__ __attribute__((aligned(16))) T s_row[NW][W];    // each wave's copy of the pivot row
    __shared__ T s_raw[NW][W];                                 // the same with what is not finite
    __shared__ int s_pivs[W];                                  // local pivot row of each column

    if (wave == NW) {
        if (lane == 0) s_cand[NW].idx = NONE;                  // before the first barrier
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    if (wave == NW) {
        leaf_exchange<T, W, NW, GMAX>(w, m, r0, c0, ipiv, info, threshold, tag0, slots, error, s_cand, s_tie,
                                      &s_dec, s_pivs);
    }
    else {
        const int gbase = g * NT * RPT;
        uint64_t* const rows = slots + 2 * SL::heads(G);
        // in the order of step -1: column c at position c + 1
        T v[RPT][W], nxt[RPT], l[RPT];
        int lab[RPT];                                          // the row each register row stands for
        #pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int i = gbase + tid + NT * q;
            lab[q] = i;
            const T* rowp = A + (r0 + (i < m ? i : 0)) * ld + c0;
            if (vec) {
                #pragma unroll
                for (int c = 0; c < W; c += VE) {
                    const vec_t x = *reinterpret_cast<const vec_t*>(rowp + c);
                    #pragma unroll
                    for (int e = 0; e < VE; ++e) v[q][(c + e + 1) % W] = x[e];
                }
            }
            else {
                #pragma unroll
                for (int c = 0; c < W; ++c) v[q][(c + 1) % W] = rowp[c < w ? c : 0];
            }
            #pragma unroll
            for (int c = 0; c < W; ++c) v[q][(c + 1) % W] = (i < m && c < w) ? v[q][(c + 1) % W] : T(0);
            nxt[q] = v[q][1];
            l[q] = T(0);
        }
        int pl = -1, pq = 0;                                   // the last pivot row's lane in this wave

        #pragma unroll 1
        for (int j = 0; j < w; ++j) {
            const uint32_t tag = tag0 + uint32_t(j);
            // (1) this wave's candidate: the largest entry of column j, the first of equals
            T babs = T(-1), bval = T(0), bfac = T(0), bnxt = T(0);
            uint32_t bidx = NONE;
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const T a = fabs(nxt[q]);
                const bool take = lab[q] >= j && lab[q] < m && (a > babs || (a == babs && uint32_t(lab[q]) < bidx));
                babs = take ? a : babs;
                bval = take ? nxt[q] : bval;
                bfac = take ? l[q] : bfac;
                bnxt = take ? v[q][2] : bnxt;
                bidx = take ? uint32_t(lab[q]) : bidx;
                if (lab[q] == j) s_cand[NW] = LeafHead<T>{nxt[q], l[q], v[q][2], uint32_t(j)};
            }
            const uint32_t key = argmax_key(babs);
            const uint32_t mk = wave_max_u32(key);
            const int wl = wave_argmax_lane(babs, bidx, key, mk);
            if (lane == wl) s_cand[wave] = LeafHead<T>{bval, bfac, bnxt, bidx};
            __syncthreads();
            // (2) the pivot row of column j - 1 goes out ...
            uint64_t* const rowb = rows + ((j + 1) & 1) * SL::REP * RW;
            if (pl >= 0) {
                #pragma unroll
                for (int q = 0; q < RPT; ++q)
                    if (q == pq && lane == pl) {
                        #pragma unroll
                        for (int c = 0; c < W; c += VE) {
                            vec_t x;
                            #pragma unroll
                            for (int e = 0; e < VE; ++e) x[e] = v[q][c + e];
                            *reinterpret_cast<vec_t*>(&s_row[wave][c]) = x;
                        }
                    }
                __builtin_amdgcn_wave_barrier();
                if (lane < (w - j + 1) * NWV && lane < RW) {
                    const uint32_t x = reinterpret_cast<const word_t*>(s_row[wave])[lane];
                    #pragma unroll
                    for (int r = 0; r < SL::REP; ++r) tw_store(rowb + r * RW + lane, x, tag - 1);
                }
            }
            // ... and comes in; finished columns are zero in it
            const int lim = w - j + 1;                         // positions lim .. of step j - 1 are finished
            uint32_t fv;
            if (pl < 0 && j > 0) {
                const int64_t off[1] = {lane < RW ? lane : 0};
                const bool val[1] = {lane < lim * NWV && lane >= NWV && lane < RW};
                uint32_t got[1];
                tw_gather<1>(rowb + (g & (SL::REP - 1)) * RW, off, val, tag - 1, got, error, 1);
                fv = got[0];
            }
            else {
                fv = reinterpret_cast<const word_t*>(s_row[wave])[lane < RW ? lane : 0];
            }
            const bool in = j > 0 && lane >= NWV && lane < lim * NWV && lane < RW;
            if (lane < RW) reinterpret_cast<word_t*>(s_row[wave])[lane] = in ? fv : 0u;
            // 0 * inf would reach finished rows and columns: what is not finite
            // is left out of the update and follows by itself
            constexpr uint32_t EXP = sizeof(T) == 8 ? 0x7FF00000u : 0x7F800000u;
            bool odd = in && lane % NWV == NWV - 1 && (fv & EXP) == EXP;
            T lz[RPT];
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const bool act = j > 0 && lab[q] >= j && lab[q] < m, fin = isfinite(l[q]);
                lz[q] = act && fin ? l[q] : T(0);
                odd = odd || (act && !fin);
            }
            const bool sel = __builtin_amdgcn_ballot_w64(odd) != 0;
            if (sel) {
                if (lane < W) {
                    const T x = s_row[wave][lane];
                    s_raw[wave][lane] = x;
                    if (!isfinite(x)) s_row[wave][lane] = T(0);
                }
            }
            __builtin_amdgcn_wave_barrier();
            // (3) update, and move down by one
            {
                T v0[RPT];
                #pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    v0[q] = v[q][0];
                    v[q][0] = nxt[q];
                }
                #pragma unroll
                for (int c = 0; c < W; c += VE) {
                    const vec_t x = *reinterpret_cast<const vec_t*>(&s_row[wave][c]);
                    #pragma unroll
                    for (int e = 0; e < VE; ++e)
                        if (c + e >= 2)
                            #pragma unroll
                            for (int q = 0; q < RPT; ++q) v[q][c + e - 1] = fma_of(-lz[q], x[e], v[q][c + e]);
                }
                #pragma unroll
                for (int q = 0; q < RPT; ++q) v[q][W - 1] = v0[q];
                if (sel) {
                    #pragma unroll
                    for (int c = 2; c < W; ++c) {
                        const T x = s_raw[wave][c];
                        #pragma unroll
                        for (int q = 0; q < RPT; ++q) {
                            const bool act = j > 0 && lab[q] >= j && lab[q] < m && c < lim;
                            if (act && (!isfinite(x) || !isfinite(l[q]))) v[q][c - 1] = fma_of(-l[q], x, v[q][c - 1]);
                        }
                    }
                }
                // before the barrier, not on the chain behind it
                #pragma unroll
                for (int q = 0; q < RPT; ++q)
                    #pragma unroll
                    for (int c = 0; c < W; ++c) asm volatile("" : "+v"(v[q][c]));
            }
            __syncthreads();
            // (4) interchange rows j and p, scale column j and finish column j + 1
            const LeafDec<T> d = s_dec;
            const int p = __builtin_amdgcn_readfirstlane(int(d.h.idx));
            const T pv = d.h.val;
            const T u1 = j > 0 ? fma_of(-d.h.fac, d.u2, d.h.nxt) : d.h.nxt;
            const bool zero = pv == T(0), tiny = fabs(pv) < safe_min;
            const T inv = T(1) / pv;
            pl = -1;
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int lb = lab[q];
                const uint64_t own = __builtin_amdgcn_ballot_w64(lb == p);
                if (own) { pl = __builtin_ctzll(own); pq = q; }
                lab[q] = lb == p ? j : (lb == j ? p : lb);
                const bool act = lab[q] > j && lab[q] < m;
                T t = v[q][0] * inv;
                if (zero || tiny) t = zero ? v[q][0] : v[q][0] / pv;
                l[q] = t;
                v[q][0] = act ? t : v[q][0];
                nxt[q] = (act && j + 1 < w) ? fma_of(-t, u1, v[q][1]) : v[q][1];
            }
        }

        // after w steps v[q][c] holds column (w - 1 + c) mod W
        #pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int i = lab[q];
            if (i < m) {
                T* rowp = A + (r0 + i) * ld + c0;
                if (vec) {
                    #pragma unroll
                    for (int c = 0; c < W; c += VE) {
                        vec_t x;
                        #pragma unroll
                        for (int e = 0; e < VE; ++e) x[e] = v[q][(c + e + 1) % W];
                        *reinterpret_cast<vec_t*>(rowp + c) = x;
                    }
                }
                else {
                    #pragma unroll
                    for (int c = 0; c < W; ++c) {
                        const int col = (w - 1 + c) & (W - 1);
                        if (col < w) rowp[col] = v[q][c];
                    }
                }
            }
        }
    }
    if (xpw > w) leaf_swap_others<T, W, NT + 64>(A, ld, r0, c0, w, xp0, xpw, s_pivs, G, g);
}

//------------------------------------------------------------------------------
// One-workgroup leaf (leaf_wg.hh) on a panel in memory.
template <class T, int W, int RPT, int VEC, int NT>
__global__ __launch_bounds__(NT)
void panel_leaf_wg_kernel(T* __restrict__ A, int64_t ld, int64_t r0, int64_t m_total, int64_t c0,
                          int w, int64_t* __restrict__ ipiv, int64_t* __restrict__ info, T threshold,
                          int64_t xp0, int64_t xpw)
{
    constexpr int VE = 16 / int(sizeof(T));
    typedef T vec_t __attribute__((ext_vector_type(VE)));
    const int tid = threadIdx.x;
    const int m = int(m_total - r0);
    __shared__ LeafWg<T, W, NT> s;

    T v[RPT][W];
    int lab[RPT];                                          // the row each register row stands for
    #pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int i = tid + NT * q;
        lab[q] = i;
        const T* rowp = A + (r0 + (i < m ? i : 0)) * ld + c0;
        if (VEC && w == W) {
            #pragma unroll
            for (int c = 0; c < W; c += VE) {
                const vec_t x = *reinterpret_cast<const vec_t*>(rowp + c);
                #pragma unroll
                for (int e = 0; e < VE; ++e) v[q][c + e] = x[e];
            }
        }
        else {
            #pragma unroll
            for (int c = 0; c < W; ++c) v[q][c] = rowp[c < w ? c : 0];
        }
        #pragma unroll
        for (int c = 0; c < W; ++c) v[q][c] = (i < m && c < w) ? v[q][c] : T(0);
    }
    leaf_wg_factor<T, W, RPT, NT>(s, v, lab, w, m, A, ld, r0, c0, info, threshold);

    // after w steps v[q][c] holds column (w + c) mod W
    #pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int i = lab[q];
        if (i < m) {
            T* rowp = A + (r0 + i) * ld + c0;
            if (VEC && w == W) {
                #pragma unroll
                for (int c = 0; c < W; c += VE) {
                    vec_t y;
                    #pragma unroll
                    for (int e = 0; e < VE; ++e) y[e] = v[q][c + e];
                    *reinterpret_cast<vec_t*>(rowp + c) = y;
                }
            }
            else {
                #pragma unroll
                for (int c = 0; c < W; ++c) {
                    const int col = (w + c) & (W - 1);
                    if (col < w) rowp[col] = v[q][c];
                }
            }
        }
    }
    if (tid < w) ipiv[c0 + tid] = r0 + s.pivs[tid];
    if (xpw > w) leaf_swap_others<T, W, NT, 64>(A, ld, r0, c0, w, xp0, xpw, s.pivs, 1, 0);
}

// Most rows of a one-workgroup leaf, one row per thread.  FP64, 32 columns:
// 500 rows 50 us in one workgroup, 63 us over two; 700 rows (two per thread)
// 64 and 62 us, 1000 rows 69 and 64 us.  FP32: 500 rows 42 and 52 us, 1000
// rows 53 and 54 us, 2000 rows 78 and 61 us.
static constexpr int64_t LEAF_WG_ROWS = 512;

template <class T, int W>
static void panel_leaf_w(T* A, int64_t ld, int64_t r0, int64_t m_total, int64_t c0, int w,
                         int64_t* ipiv, int64_t* info, double threshold, const PanelWork& pw,
                         uint32_t tag0, hipStream_t s, int64_t xp0, int64_t xpw);

template <class T>
void panel_leaf(T* A, int64_t ld, int64_t r0, int64_t m_total, int64_t c0, int w,
                int64_t* ipiv, int64_t* info, double threshold, const PanelWork& pw,
                uint32_t tag0, hipStream_t s, int64_t xp0, int64_t xpw)
{
    // FP64 leaves of at most 16 columns run the 16-wide register form (its
    // 2-row shape keeps two workgroups per CU on tall panels)
    if constexpr (sizeof(T) == 8) {
        if (w <= 16) {
            panel_leaf_w<T, 16>(A, ld, r0, m_total, c0, w, ipiv, info, threshold, pw, tag0, s, xp0, xpw);
            return;
        }
    }
    panel_leaf_w<T, LeafW<T>::W>(A, ld, r0, m_total, c0, w, ipiv, info, threshold, pw, tag0, s, xp0, xpw);
}

template <class T, int W>
static void panel_leaf_w(T* A, int64_t ld, int64_t r0, int64_t m_total, int64_t c0, int w,
                         int64_t* ipiv, int64_t* info, double threshold, const PanelWork& pw,
                         uint32_t tag0, hipStream_t s, int64_t xp0, int64_t xpw)
{
    const int64_t m = m_total - r0;
    SA_REQUIRE(w >= 1 && w <= W, -2, "panel_leaf: bad width");
    SA_REQUIRE(m >= w, -2, "panel_leaf: fewer rows than columns");
    SA_REQUIRE(m < int64_t(0xFFFFFFFFu), -2, "panel_leaf: panel too tall");
    const T thr = T(threshold);
    constexpr int VE = 16 / int(sizeof(T));
    const bool vec = (reinterpret_cast<uintptr_t>(A) % 16 == 0) && (ld % VE == 0) && (c0 % VE == 0);
    SA_REQUIRE(xpw == 0 || (r0 == c0 && xp0 <= c0 && c0 + w <= xp0 + xpw), -2,
               "panel_leaf: leaf outside the enclosing panel");
    if (m <= LEAF_WG_ROWS) {
#define SA_WG(NTV, V) hipLaunchKernelGGL((panel_leaf_wg_kernel<T, W, 1, V, NTV>), dim3(1), dim3(NTV), 0, s, \
                                          A, ld, r0, m_total, c0, w, ipiv, info, thr, xp0, xpw)
        if (m <= 256) { if (vec) SA_WG(256, 1); else SA_WG(256, 0); }
        else { if (vec) SA_WG(512, 1); else SA_WG(512, 0); }
#undef SA_WG
        SA_CHECK_LAUNCH();
        return;
    }
    uint64_t* slots = static_cast<uint64_t*>(pw.slots);
    const bool vec_rows = vec && w == W;
#define SA_LEAF(NTV, R, GM)                                                                       \
    do {                                                                                          \
        const int64_t G = ceildiv(m, int64_t(NTV) * (R));                                         \
        SA_REQUIRE(G <= (GM), -2, "panel_leaf: panel too tall");                                  \
        SA_REQUIRE((int64_t(sizeof(uint64_t)) * LeafSlots<T, W>::words(int(G)) <= pw.slots_bytes), -2, \
                   "panel_leaf: slot area too small");                                            \
        hipLaunchKernelGGL((panel_leaf_rot_kernel<T, W, R, NTV, GM>), dim3(G), dim3(NTV + 64), 0, s, A, ld, r0, \
                           m_total, c0, w, ipiv, info, thr, tag0, slots, pw.error, xp0, xpw, vec_rows); \
    } while (0)
    // Alone, more workgroups of one row per thread are fastest (FP64, 8192
    // rows: 256 x 1 2.34 us per column, 256 x 2 2.97).  Beside a trailing
    // update a leaf starts when enough CUs have retired a GEMM workgroup, and
    // 8 waves of at most 128 registers fit the place of one (256 registers on
    // each SIMD): with 256 x 1, 128 workgroups, a leaf of 32768 rows took 935
    // us beside the FP64 update and 89 alone, with 448 x 1, 74 workgroups, 379
    // (n = 32768: 660 and 490 ms).  Two rows of 128 bytes fit those registers,
    // two of 256 do not.  The heads of 32, 64 or 128 workgroups are 4, 8 or 16
    // loads per poll in FP64 (8192 rows: 2.34, 2.45, 2.72 us), half in FP32.
    if (m <= 32 * 256) SA_LEAF(256, 1, 32);
    else if (m <= 64 * 448) SA_LEAF(448, 1, 64);
    else if (W * sizeof(T) > 128 && m <= 128 * 448) SA_LEAF(448, 1, 128);
    else if (W * sizeof(T) <= 128 && m <= 64 * 896) SA_LEAF(448, 2, 64);
    else if (m <= 128 * 896) SA_LEAF(448, 2, 128);
    else SA_LEAF(512, 2, 128);
#undef SA_LEAF
    SA_CHECK_LAUNCH();
}

template void panel_leaf<double>(double*, int64_t, int64_t, int64_t, int64_t, int, int64_t*, int64_t*,
                                 double, const PanelWork&, uint32_t, hipStream_t, int64_t, int64_t);
template void panel_leaf<float>(float*, int64_t, int64_t, int64_t, int64_t, int, int64_t*, int64_t*,
                                double, const PanelWork&, uint32_t, hipStream_t, int64_t, int64_t);

//------------------------------------------------------------------------------
// Row interchanges.  The sequential LAPACK-style swap list (i, ipiv[i]),
// i = k1..k2-1, with ipiv[i] >= i (src/internal/internal_swap.cc:198-435 and
// the parallel-pivot map of :33-77), is turned into an explicit list of
// (dst row <- src row) moves: every touched row r receives the original row
// src(r) = t_k1(t_k1+1(...t_k2-1(r))), t_i the i-th transposition.  The apply
// kernel then gathers the sources of a column chunk into LDS and scatters
// them, which keeps every row access coalesced in the row-major layout.
static constexpr int PLAN_MAX = 2048;

// Rows are kept relative to k1 as 32-bit ints in LDS, padded to a multiple
// of 16 with identity transpositions, so both per-thread sweeps (the
// duplicate test and the backward walk of src_of) read sixteen entries per
// group of four broadcast LDS loads and do only register compares in between.
__global__ __launch_bounds__(1024)
void laswp_plan_kernel(int64_t k1, int64_t k2, int64_t nrows, const int64_t* __restrict__ ipiv,
                       int64_t* __restrict__ plan)
{
    __shared__ __attribute__((aligned(16))) int piv[PLAN_MAX];
    __shared__ int keep[PLAN_MAX];
    __shared__ int scan[PLAN_MAX];
    typedef int int4_t __attribute__((ext_vector_type(4)));
    const int tid = threadIdx.x, nt = blockDim.x;
    const int np = int(k2 - k1);
    const int np4 = (np + 15) & ~15;                     // padded to whole 16-entry groups
    for (int i = tid; i < np4; i += nt) {
        int v = i;                                          // padding / out-of-range: no swap
        if (i < np) {
            const int64_t p = ipiv[k1 + i];
            if (p >= k1 + i && p < nrows) v = int(p - k1);
        }
        piv[i] = v;
    }
    __syncthreads();
    for (int i = tid; i < np; i += nt) {
        const int p = piv[i];
        int k = p >= np;                                    // a row below the swapped block
        for (int i2 = 0; i2 < (i & ~15); i2 += 16) {
            int4_t q[4];
            #pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const int4_t*>(&piv[i2 + 4 * u]);
            #pragma unroll
            for (int u = 0; u < 4; ++u) k &= (q[u][0] != p) & (q[u][1] != p) & (q[u][2] != p) & (q[u][3] != p);
        }
        for (int i2 = i & ~15; i2 < i; ++i2) k &= (piv[i2] != p);
        keep[i] = k;
        scan[i] = k;
    }
    __syncthreads();
    // inclusive scan (Hillis-Steele)
    for (int off = 1; off < np; off <<= 1) {
        int vals[2];
        int cnt = 0;
        for (int i = tid; i < np; i += nt) vals[cnt++] = (i >= off) ? scan[i - off] : 0;
        __syncthreads();
        cnt = 0;
        for (int i = tid; i < np; i += nt) scan[i] += vals[cnt++];
        __syncthreads();
    }
    const int nkeep = np > 0 ? scan[np - 1] : 0;
    const int count = np + nkeep;
    // source of relative row x: t_0(t_1(...t_{np-1}(x))), t_i = (i piv[i])
    auto src_of = [&](int x) {
        for (int i = np4 - 16; i >= 0; i -= 16) {
            int4_t q[4];
            #pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const int4_t*>(&piv[i + 4 * u]);
            #pragma unroll
            for (int u = 15; u >= 0; --u) {
                const int a = i + u, b = q[u >> 2][u & 3];
                x = (x == a) ? b : ((x == b) ? a : x);
            }
        }
        return k1 + int64_t(x);
    };
    for (int e = tid; e < np; e += nt) {
        plan[1 + 2 * e] = k1 + e;
        plan[2 + 2 * e] = src_of(e);
    }
    for (int i = tid; i < np; i += nt)
        if (keep[i]) {
            const int e = np + scan[i] - 1;
            plan[1 + 2 * e] = k1 + int64_t(piv[i]);
            plan[2 + 2 * e] = src_of(piv[i]);
        }
    if (tid == 0) plan[0] = count;
}

template <class T>
__global__ __launch_bounds__(256)
void laswp_apply_kernel(T* __restrict__ A, int64_t ld, int64_t c0, int64_t c1, int ch,
                        const int64_t* __restrict__ plan)
{
    extern __shared__ unsigned char smem_raw[];
    T* buf = reinterpret_cast<T*>(smem_raw);
    const int count = int(plan[0]);
    const int64_t cb = c0 + int64_t(blockIdx.x) * ch;
    const int tid = threadIdx.x;
    const int c = tid % ch, e0 = tid / ch, es = 256 / ch;
    const bool ok = cb + c < c1;
    const int64_t cc = ok ? cb + c : c1 - 1;
    // Batches of 8 independent loads (clamped), so row fetches overlap.
    for (int e = e0; e < count; e += 8 * es) {
        T v[8];
        #pragma unroll
        for (int u = 0; u < 8; ++u) {
            int ee = e + u * es;
            int64_t src = plan[2 + 2 * (ee < count ? ee : count - 1)];
            v[u] = A[src * ld + cc];
        }
        #pragma unroll
        for (int u = 0; u < 8; ++u) {
            int ee = e + u * es;
            if (ee < count) buf[ee * ch + c] = ok ? v[u] : T(0);
        }
    }
    __syncthreads();
    for (int e = e0; e < count; e += es) {
        int64_t dst = plan[1 + 2 * e];
        if (ok) A[dst * ld + cb + c] = buf[e * ch + c];
    }
}

// Small interchange sequences (<= 64 pivots, the ones inside the recursive
// panel): every workgroup derives the (dst <- src) list itself in LDS and
// applies it to its column chunk, so no separate plan launch is needed.
// Entry e < np is row k1+e; entry np+i is pivot row ipiv[k1+i] when it lies
// at or beyond k2 and is its first occurrence, otherwise unused.
template <class T>
__global__ __launch_bounds__(256)
void laswp_small_kernel(T* __restrict__ A, int64_t ld, int64_t nrows, int64_t c0, int64_t c1, int ch,
                        int64_t k1, int np, const int64_t* __restrict__ ipiv)
{
    __shared__ int64_t piv[64];
    __shared__ int64_t dst[128], src[128];
    extern __shared__ unsigned char smem_raw[];
    T* buf = reinterpret_cast<T*>(smem_raw);
    const int tid = threadIdx.x;
    const int64_t k2 = k1 + np;
    if (tid < np) {
        int64_t p = ipiv[k1 + tid];
        piv[tid] = (p >= k1 + tid && p < nrows) ? p : k1 + tid;
    }
    __syncthreads();
    if (tid < 2 * np) {
        int64_t r = -1;
        if (tid < np) r = k1 + tid;
        else {
            int i = tid - np;
            int64_t p = piv[i];
            bool first = p >= k2;
            for (int i2 = 0; i2 < i; ++i2) first = first && (piv[i2] != p);
            if (first) r = p;
        }
        int64_t x = r;
        if (r >= 0)
            for (int i = np - 1; i >= 0; --i) {
                int64_t a = k1 + i, b = piv[i];
                if (x == a) x = b;
                else if (x == b) x = a;
            }
        dst[tid] = r;
        src[tid] = x;
    }
    __syncthreads();
    const int64_t cb = c0 + int64_t(blockIdx.x) * ch;
    const int c = tid % ch, e0 = tid / ch, es = 256 / ch;
    const bool ok = cb + c < c1;
    const int64_t cc = ok ? cb + c : c1 - 1;
    for (int e = e0; e < 2 * np; e += 8 * es) {
        T v[8];
        #pragma unroll
        for (int u = 0; u < 8; ++u) {
            int ee = e + u * es;
            int64_t sr = (ee < 2 * np && dst[ee] >= 0) ? src[ee] : k1;
            v[u] = A[sr * ld + cc];
        }
        #pragma unroll
        for (int u = 0; u < 8; ++u) {
            int ee = e + u * es;
            if (ee < 2 * np && dst[ee] >= 0) buf[ee * ch + c] = ok ? v[u] : T(0);
        }
    }
    __syncthreads();
    for (int e = e0; e < 2 * np; e += es)
        if (dst[e] >= 0 && ok) A[dst[e] * ld + cb + c] = buf[e * ch + c];
}

void laswp_plan(int64_t k1, int64_t k2, int64_t nrows, const int64_t* ipiv, int64_t* plan,
                hipStream_t s)
{
    SA_REQUIRE(k2 - k1 <= PLAN_MAX, -2, "laswp: too many pivots in one call");
    SA_REQUIRE(nrows - k1 < (int64_t(1) << 31), -2, "laswp: rows beyond 32-bit plan range");
    if (k2 <= k1) return;
    hipLaunchKernelGGL(laswp_plan_kernel, dim3(1), dim3(1024), 0, s, k1, k2, nrows, ipiv, plan);
    SA_CHECK_LAUNCH();
}

__global__ void laswp_invert_kernel(int64_t* plan, int64_t maxcount)
{
    const int64_t count = plan[0];
    for (int64_t e = threadIdx.x; e < count && e < maxcount; e += blockDim.x) {
        int64_t d = plan[1 + 2 * e];
        plan[1 + 2 * e] = plan[2 + 2 * e];
        plan[2 + 2 * e] = d;
    }
}

void laswp_invert_plan(int64_t* plan, int64_t npiv, hipStream_t s)
{
    if (npiv <= 0) return;
    hipLaunchKernelGGL(laswp_invert_kernel, dim3(1), dim3(1024), 0, s, plan, 2 * npiv);
    SA_CHECK_LAUNCH();
}

// Two-pass interchange: pass 0 copies source row plan[2+2e] (columns
// [c0, c1)) into tmp row e, pass 1 copies tmp row e into destination row
// plan[1+2e].  grid.y strides over entries, grid.x over 16-byte column groups.
template <class T, int PASS, int VEC>
__global__ __launch_bounds__(256)
void laswp_pass_kernel(T* __restrict__ A, int64_t ld, int64_t c0, int64_t ncol, T* __restrict__ tmp,
                       const int64_t* __restrict__ plan)
{
    constexpr int VE = VEC ? 16 / int(sizeof(T)) : 1;
    typedef T vec_t __attribute__((ext_vector_type(VE)));
    const int count = int(plan[0]);
    const int64_t col = (int64_t(blockIdx.x) * 256 + threadIdx.x) * VE;
    if (col >= ncol) return;
    for (int e = blockIdx.y; e < count; e += gridDim.y) {
        const int64_t row = plan[(PASS == 0 ? 2 : 1) + 2 * e];
        T* a = A + row * ld + c0 + col;
        T* t = tmp + int64_t(e) * ncol + col;
        if (VEC && col + VE <= ncol) {
            // each source element is read once: nontemporal loads
            if (PASS == 0) *reinterpret_cast<vec_t*>(t) = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(a));
            else *reinterpret_cast<vec_t*>(a) = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(t));
        }
        else {
            for (int q = 0; q < VE && col + q < ncol; ++q) {
                if (PASS == 0) t[q] = a[q];
                else a[q] = t[q];
            }
        }
    }
}

template <class T>
void laswp(T* A, int64_t ld, int64_t nrows, int64_t c0, int64_t c1, int64_t k1, int64_t k2,
           const int64_t* ipiv, int64_t* plan, hipStream_t s, bool plan_ready, T* tmp, int64_t tmp_elems)
{
    if (k2 <= k1) return;
    if (plan_ready && tmp && c1 > c0 && tmp_elems >= 2 * (k2 - k1) * (c1 - c0)) {
        constexpr int VE = 16 / int(sizeof(T));
        const int64_t ncol = c1 - c0;
        const bool vec = ld % VE == 0 && c0 % VE == 0 && ncol % VE == 0
                         && reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(tmp) % 16 == 0;
        const int64_t per = vec ? VE : 1;
        dim3 grid(unsigned(ceildiv(ncol, 256 * per)), unsigned(std::min<int64_t>(2 * (k2 - k1), 2048)));
        if (vec) {
            hipLaunchKernelGGL((laswp_pass_kernel<T, 0, 1>), grid, dim3(256), 0, s, A, ld, c0, ncol, tmp, plan);
            hipLaunchKernelGGL((laswp_pass_kernel<T, 1, 1>), grid, dim3(256), 0, s, A, ld, c0, ncol, tmp, plan);
        }
        else {
            hipLaunchKernelGGL((laswp_pass_kernel<T, 0, 0>), grid, dim3(256), 0, s, A, ld, c0, ncol, tmp, plan);
            hipLaunchKernelGGL((laswp_pass_kernel<T, 1, 0>), grid, dim3(256), 0, s, A, ld, c0, ncol, tmp, plan);
        }
        SA_CHECK_LAUNCH();
        return;
    }
    if (!plan_ready && k2 - k1 <= 64) {
        if (c1 <= c0) return;
        const int np = int(k2 - k1);
        int ch = 256;
        while (ch > 4 && int64_t(ch) * 2 * np * int64_t(sizeof(T)) > 65536) ch /= 2;
        while (ch > 4 && ch / 2 >= (c1 - c0)) ch /= 2;
        size_t lds = size_t(ch) * size_t(2 * np) * sizeof(T);
        int64_t nblk = ceildiv(c1 - c0, ch);
        hipLaunchKernelGGL(laswp_small_kernel<T>, dim3(unsigned(nblk)), dim3(256), lds, s,
                           A, ld, nrows, c0, c1, ch, k1, np, ipiv);
        SA_CHECK_LAUNCH();
        return;
    }
    if (!plan_ready) laswp_plan(k1, k2, nrows, ipiv, plan, s);
    if (c1 <= c0) return;
    const int64_t maxcount = 2 * (k2 - k1);
    // column chunk: power of two, LDS staging <= 64 KiB, 4..256 columns
    int ch = 256;
    while (ch > 4 && int64_t(ch) * maxcount * int64_t(sizeof(T)) > 65536) ch /= 2;
    while (ch > 4 && ch / 2 >= (c1 - c0)) ch /= 2;
    size_t lds = size_t(ch) * size_t(maxcount) * sizeof(T);
    SA_REQUIRE(lds <= 65536, -2, "laswp: LDS staging too large");
    int64_t nblk = ceildiv(c1 - c0, ch);
    hipLaunchKernelGGL(laswp_apply_kernel<T>, dim3(unsigned(nblk)), dim3(256), lds, s,
                       A, ld, c0, c1, ch, plan);
    SA_CHECK_LAUNCH();
}

template void laswp<double>(double*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                            const int64_t*, int64_t*, hipStream_t, bool, double*, int64_t);
template void laswp<float>(float*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                           const int64_t*, int64_t*, hipStream_t, bool, float*, int64_t);

} // namespace sa
