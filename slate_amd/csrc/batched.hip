// Batched factor-and-solve of many small systems of uneven size (gfx950).
//
// One persistent launch: each workgroup takes the next system from a work
// queue (an atomic ticket over a largest-first order), copies it into its
// own workspace in row-major order (interchanges then move contiguous rows),
// factors it with partial pivoting, solves, and refines in FP64 against the
// original matrix to SLATE's stopping rule (src/gesv_mixed.cc:190-259,
// internal_util.hh:121-138), with the FP64 factorization as the fallback when
// the refinement misses the tolerance.  The per-system steps mirror
// slate::gesv / gesv_mixed on a single tile column; the batching (one launch
// for thousands of systems of different n, no per-system launches or host
// round trips) is this library's own design.
//
// Per-system modes (BatchArgs::mode):
//   0 FP32 factor + FP64 IR, 1 FP64 factor, 2 BF16 factor (FP32 storage,
//   bf16-operand MFMA trailing updates with FP32 accumulation) + FP64 IR,
//   3 learned choice, 4/5/6 the learned path with its choice forced to
//   0/1/2 (labelling).
// The learned path factors in BF16 or FP32 first (the probe), solves once and
// forms the FP64 residual (iteration 0 of the refinement), and feeds the
// probe's normwise quantities to the selector network (the MLP of mlp.hip,
// run by one wave), which picks what runs: BF16 + IR (0), FP32 + IR (1) or
// FP64 (2) — keeping the probe factor when it has the chosen precision.
//
// Factorization: blocked right-looking LU.  A panel of NB columns is factored
// with its rows in registers (leaf_wg.hh: two barriers per column, rows that
// change labels instead of places) and stored to memory and to LDS (row pitch
// NB + 4 floats: fragment reads and row writes are conflict free).  Its
// interchanges are composed by one wave into at most 2 NB row moves
// (destination, source); one thread per column then applies them with all
// loads before any store (one memory round trip per panel instead of one per
// swap) and, right of the panel, solves U12 = L11^{-1} A12 on the rows it has
// just gathered.  A22 -= L21 U12 runs as 32 x 32 wave tiles of MFMA
// (v_mfma_f32_16x16x4f32, v_mfma_f32_16x16x32_bf16 or v_mfma_f64_16x16x4f64):
// a wave takes a strip of tiles, keeps the strip's U12 in registers, reads
// L21 from the LDS panel and streams C, the next tiles' loads in flight.
// Triangular solves: 64-row blocks, each diagonal block solved by one wave
// (no barriers), the rows below updated by the whole workgroup.
//
// Bounds: up to n of about 500 the panels' serial chain (about 1.3 us per
// column), above it the trailing matrix streamed once per NB columns.  With
// the panel in LDS (each thread reading and writing whole rows, the pivot
// row in registers by selects) a column took 4.5 - 5.4 us at any size, and
// 16-column panels streamed the trailing matrix twice as often.  4096 systems
// of 32 .. 1024 rows: 140 ms then, 62.7 ms now (n = 1000, all CUs busy: 25 and
// 10 ms per system, of which the updates take 4.5, the panels 1.4, the solves
// 1.1, the load 0.9).
//
// Systems of at most 64 rows (FP32 and FP64 factors) take one wave each, a
// workgroup's waves working on different ones: row i lives in lane i, the
// pivot row is broadcast by v_readlane, and no barrier is needed.
//
// The ticket counter and a count of finished workgroups live in `queue`; the
// last workgroup to finish zeroes both, so consecutive launches (and replays
// of a graph holding the launch) need no separate reset.
#include "common.hh"
#include "kernels.hh"
#include "leaf_wg.hh"

#include <cstring>
#include <limits>

namespace sa {

static constexpr int BMAXN = 1024;          // largest system
static constexpr int SEL_F = 24, SEL_H = 64, SEL_K = 8;   // selector network (mlp.hip layout)
static constexpr int SEL_CHOICES = 3;

// Panel width of storage type T for a configuration: NBF float columns (half
// as many in FP64, so both fit the same LDS and registers); with 512 threads
// the registers hold two such panels, which are factored as one.
template <class T, int NBF, int BT> struct Pan {
    static constexpr int NB = NBF * (BT == 512 ? 2 : 1) / (sizeof(T) == 8 ? 2 : 1);
    static constexpr int LD = NB + 16 / int(sizeof(T));    // LDS row pitch
    static constexpr int RPT = BMAXN / BT;                  // panel rows per thread
};
template <int NBF, int BT> constexpr int pan_lds_bytes()
{
    return BMAXN * Pan<float, NBF, BT>::LD * 4 > BMAXN * Pan<double, NBF, BT>::LD * 8
         ? BMAXN * Pan<float, NBF, BT>::LD * 4 : BMAXN * Pan<double, NBF, BT>::LD * 8;
}

__host__ __device__ inline int b_ldw(int n) { return (n + 3) & ~3; }

// W (row-major, ldw) = A (column-major n x n, FP64), cast to T.  Wave tiles of
// 64 rows x 32 columns: the column reads are coalesced, each lane then writes
// 32 consecutive elements of its row.
template <class T, int BT>
__device__ __forceinline__ void wg_load_rowmajor(const double* __restrict__ A, int n, T* __restrict__ W, int ldw)
{
    constexpr int NW = BT / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ti = (n + 63) >> 6, tj = (n + 31) >> 5;
    for (int t = wave; t < ti * tj; t += NW) {
        const int i = (t % ti) * 64 + lane, j0 = (t / ti) * 32;
        T v[32];
        #pragma unroll
        for (int c = 0; c < 32; ++c)
            v[c] = T(A[(i < n ? i : n - 1) + int64_t(j0 + c < n ? j0 + c : n - 1) * n]);
        #pragma unroll
        for (int c = 0; c < 32; ++c) v[c] = j0 + c < n ? v[c] : T(0);
        if (i < n) {
            // rows and column tiles start 16-byte aligned; the last vector may
            // run into the padding up to ldw
            constexpr int VE = 16 / int(sizeof(T));
            typedef T vec_t __attribute__((ext_vector_type(VE)));
            T* w = W + int64_t(i) * ldw + j0;
            #pragma unroll
            for (int c = 0; c < 32; c += VE)
                if (j0 + c < n) {
                    vec_t x;
                    #pragma unroll
                    for (int e = 0; e < VE; ++e) x[e] = v[c + e];
                    *reinterpret_cast<vec_t*>(w + c) = x;
                }
        }
    }
}

// C (nr x nr, row stride ldw) -= L (nr x NB, LDS, row stride LD) * U (NB x nr,
// row stride ldw) in 32-row wave tiles of VE 16-column blocks (VE elements =
// 16 bytes).  A lane's columns are consecutive (block b holds the columns
// VE c + b), so C moves in 16-byte vectors: with one element per access a
// tile took 32 loads and 32 stores, and two tiles in flight already exceeded
// the 63 a wave can have outstanding.  A wave takes a strip of tiles, keeps
// the strip's U (NB x 16 VE) in registers and has the next tile's loads
// (clamped, unguarded) in flight during the products.  Step s takes the
// products k = 4 s .. 4 s + 3, lane l the one of k = 4 s + l/16, so each sum
// runs in the order of k (rows of U grow with k: any other order has larger
// partial sums, 1.15 times the error of the FP32 factor of a uniform matrix);
// a row of L holds the columns 4 s + g at (NB/4) g + s (lds_column), so that a
// lane's are consecutive and L fragments are 16-byte reads.
// Row of accumulator register r: 4 r + l/16 (FP64), 4 (l/16) + r (FP32).
template <int NB> constexpr int lds_column(int p) { return 4 * (p % (NB / 4)) + p / (NB / 4); }

template <class T, int NB, int LD, int BT, bool BFU>
__device__ __forceinline__ void wg_update(T* __restrict__ C, const T* __restrict__ U, int ldw, const T* __restrict__ L,
                                          int nr)
{
    constexpr int NW = BT / 64, VE = 16 / int(sizeof(T));
    constexpr int KS = NB / 4;                          // k-steps of 4
    typedef T vec_t __attribute__((ext_vector_type(VE)));
    typedef T acc_t __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int tr = (nr + 31) >> 5, tc = (nr + 16 * VE - 1) / (16 * VE);
    const int parts = min(tr, (2 * NW + tc - 1) / tc);  // at least two items per wave where there are rows
    const int per = (tr + parts - 1) / parts;
    const int lastv = (nr - 1) & ~(VE - 1);             // the last vector of a row; it may run into the padding
    auto crow = [&](int a, int r) { return 16 * a + (sizeof(T) == 8 ? 4 * r + fg : 4 * fg + r); };
    for (int it = wave; it < tc * parts; it += NW) {
        const int t0 = (it / tc) * per, t1 = min(tr, t0 + per);
        const int jv = (it % tc) * 16 * VE + VE * fr, jc = min(jv, lastv);
        vec_t bv[KS];                                   // U rows k = 4 s + fg, element b for block b
        #pragma unroll
        for (int s = 0; s < KS; ++s) bv[s] = *reinterpret_cast<const vec_t*>(U + (4 * s + fg) * ldw + jc);
        vec_t cv[2][2][4];
        auto fetch = [&](int set, int t) {
            #pragma unroll
            for (int a = 0; a < 2; ++a)
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    cv[set][a][r] = *reinterpret_cast<const vec_t*>(C + min((t << 5) + crow(a, r), nr - 1) * ldw + jc);
        };
        auto tile = [&](int set, int t) {
            const int i0 = t << 5;
            acc_t acc[2][VE];
            #pragma unroll
            for (int a = 0; a < 2; ++a)
                #pragma unroll
                for (int b = 0; b < VE; ++b) acc[a][b] = acc_t{T(0), T(0), T(0), T(0)};
            T av[2][KS];
            #pragma unroll
            for (int a = 0; a < 2; ++a) {
                const T* lp = L + min(i0 + 16 * a + fr, nr - 1) * LD + KS * fg;
                #pragma unroll
                for (int s = 0; s < KS; s += VE) {
                    const vec_t x = *reinterpret_cast<const vec_t*>(lp + s);
                    #pragma unroll
                    for (int e = 0; e < VE; ++e) av[a][s + e] = x[e];
                }
            }
            if constexpr (sizeof(T) == 8) {
                #pragma unroll
                for (int s = 0; s < KS; ++s)
                    #pragma unroll
                    for (int a = 0; a < 2; ++a)
                        #pragma unroll
                        for (int b = 0; b < VE; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a][s], bv[s][b], acc[a][b], 0, 0, 0);
            }
            else if constexpr (BFU) {
                // one 32-deep product; a 16-column panel fills half of it
                v8bf a8[2], b8[VE];
                #pragma unroll
                for (int e = 0; e < 8; ++e) {
                    #pragma unroll
                    for (int a = 0; a < 2; ++a) a8[a][e] = __bf16(e < KS ? av[a][e < KS ? e : 0] : 0.f);
                    #pragma unroll
                    for (int b = 0; b < VE; ++b) b8[b][e] = __bf16(e < KS ? bv[e < KS ? e : 0][b] : 0.f);
                }
                #pragma unroll
                for (int a = 0; a < 2; ++a)
                    #pragma unroll
                    for (int b = 0; b < VE; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a8[a], b8[b], acc[a][b], 0, 0, 0);
            }
            else {
                #pragma unroll
                for (int s = 0; s < KS; ++s)
                    #pragma unroll
                    for (int a = 0; a < 2; ++a)
                        #pragma unroll
                        for (int b = 0; b < VE; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a][s], bv[s][b], acc[a][b], 0, 0, 0);
            }
            #pragma unroll
            for (int a = 0; a < 2; ++a)
                #pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = i0 + crow(a, r);
                    vec_t x = cv[set][a][r];
                    #pragma unroll
                    for (int b = 0; b < VE; ++b) x[b] -= acc[a][b][r];
                    if (i < nr && jv < nr) *reinterpret_cast<vec_t*>(C + i * ldw + jv) = x;
                }
        };
        if (t0 < t1) fetch(0, t0);
        for (int t = t0; t < t1; t += 2) {
            if (t + 1 < t1) fetch(1, t + 1);
            tile(0, t);
            if (t + 2 < t1) fetch(0, t + 2);
            if (t + 1 < t1) tile(1, t + 1);
        }
    }
}

// In-workgroup LU with partial pivoting of the row-major n x n matrix W
// (Tile_getrf.hh:197-366: largest magnitude, ties to the lower index, scaling
// by the reciprocal unless the pivot is below the safe minimum).
// perm[i] = original row now at position i (the interchanges composed).
// *s_info: first exactly-zero pivot.
// bf: bf16 operands in the trailing updates (T = float).
template <class T, int NBF, int BT>
__device__ __forceinline__ void wg_getrf(T* __restrict__ W, int n, int ldw, int* __restrict__ perm, int* s_info, bool bf,
                                         T* s_p, LeafWg<T, Pan<T, NBF, BT>::NB, BT>& s_leaf, int* s_dst, int* s_src)
{
    using P = Pan<T, NBF, BT>;
    constexpr int NB = P::NB, LD = P::LD, RPT = P::RPT, VE = 16 / int(sizeof(T));
    typedef T vec_t __attribute__((ext_vector_type(VE)));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < n; i += BT) perm[i] = i;
    for (int k0 = 0; k0 < n; k0 += NB) {
        const int kb = min(NB, n - k0);
        const int mr = n - k0;
        T* Wk = W + k0 * ldw + k0;
        {
            T v[RPT][NB];
            int lab[RPT];
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int i = tid + BT * q;
                lab[q] = i;
                const T* rowp = Wk + (i < mr ? i : 0) * ldw;
                #pragma unroll
                for (int c = 0; c < NB; c += VE) {
                    // whole vectors inside the row's padded length, which ends on one
                    const vec_t x = *reinterpret_cast<const vec_t*>(rowp + (c < kb ? c : 0));
                    #pragma unroll
                    for (int e = 0; e < VE; ++e) v[q][c + e] = (i < mr && c + e < kb) ? x[e] : T(0);
                }
            }
            leaf_wg_factor<T, NB, RPT, BT>(s_leaf, v, lab, kb, mr, W, ldw, k0, k0, s_info, T(1));
            // rows to their places, in memory and in LDS (L11 in the order of its
            // columns, L21 as wg_update reads it); v[q][c] holds column (kb + c) mod NB
            #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int i = lab[q];
                if (i >= mr) continue;
                T* rowp = Wk + i * ldw;
                T* sp = s_p + i * LD;
                if (kb == NB) {
                    #pragma unroll
                    for (int c = 0; c < NB; c += VE) {
                        vec_t x;
                        #pragma unroll
                        for (int e = 0; e < VE; ++e) x[e] = v[q][c + e];
                        *reinterpret_cast<vec_t*>(rowp + c) = x;
                        if (i < NB) *reinterpret_cast<vec_t*>(sp + c) = x;
                    }
                    if (i >= NB) {
                        #pragma unroll
                        for (int c = 0; c < NB; c += VE) {
                            vec_t x;
                            #pragma unroll
                            for (int e = 0; e < VE; ++e) x[e] = v[q][lds_column<NB>(c + e)];
                            *reinterpret_cast<vec_t*>(sp + c) = x;
                        }
                    }
                }
                else {
                    #pragma unroll
                    for (int c = 0; c < NB; ++c) {
                        const int col = (kb + c) & (NB - 1);
                        if (col < kb) rowp[col] = v[q][c];
                    }
                }
            }
        }
        // Net row moves of the panel's interchanges: lane t < kb follows row
        // k0 + t, lane kb + t the pivot row of column t; each lane tracks
        // which original row ends up in its row (lanes naming the same row
        // stay equal).  A row whose source is itself does not move.
        if (wave == 0) {
            const int cand = lane < kb ? k0 + lane : (lane < 2 * kb ? k0 + s_leaf.pivs[lane - kb] : -1);
            int src = cand;
            for (int j = 0; j < kb; ++j) {
                const int ra = k0 + j, rb = k0 + s_leaf.pivs[j];
                const int va = __shfl(src, j, 64), vb = __shfl(src, kb + j, 64);
                if (ra != rb) {
                    if (cand == ra) src = vb;
                    else if (cand == rb) src = va;
                }
            }
            s_dst[lane] = cand;
            s_src[lane] = src;
        }
        __syncthreads();
        // the moves on the columns left and right of the panel and on perm
        // (column n), one column per thread, every source loaded before any
        // row is written; right of the panel (which then has NB columns) the
        // rows k0 .. k0 + NB - 1 are solved against L11 before they are stored
        for (int c = tid; c <= n; c += BT) {
            if (c >= k0 && c < k0 + kb) continue;
            asm volatile("" ::: "memory");          // reread the move list per column (keeps registers free)
            if (c >= k0 + kb && c < n) {
                T x[NB], y[NB];
                #pragma unroll
                for (int t = 0; t < NB; ++t) {
                    x[t] = W[s_src[t] * ldw + c];
                    const int d = s_dst[NB + t], sr = s_src[NB + t];
                    y[t] = sr != d ? W[sr * ldw + c] : T(0);
                }
                asm volatile("" ::: "memory");      // reread the list below instead of keeping it live
                #pragma unroll
                for (int t = 0; t < NB; ++t) {
                    const int d = s_dst[NB + t], sr = s_src[NB + t];
                    if (sr != d) W[d * ldw + c] = y[t];
                }
                #pragma unroll
                for (int r = 1; r < NB; ++r) {
                    asm volatile("" ::: "memory");  // row r's L11 reads stay inside its step
                    T s = x[r];
                    #pragma unroll
                    for (int q = 0; q < r; q += VE) {
                        const vec_t l = *reinterpret_cast<const vec_t*>(s_p + r * LD + q);
                        #pragma unroll
                        for (int e = 0; e < VE; ++e) if (q + e < r) s -= l[e] * x[q + e];
                    }
                    x[r] = s;
                }
                #pragma unroll
                for (int r = 0; r < NB; ++r) W[(k0 + r) * ldw + c] = x[r];
            }
            else if (c < n) {
                T v[2 * NB];
                #pragma unroll
                for (int t = 0; t < 2 * NB; ++t) {
                    const int d = s_dst[t], sr = s_src[t];
                    v[t] = (d >= 0 && sr != d) ? W[sr * ldw + c] : T(0);
                }
                asm volatile("" ::: "memory");
                #pragma unroll
                for (int t = 0; t < 2 * NB; ++t) {
                    const int d = s_dst[t], sr = s_src[t];
                    if (d >= 0 && sr != d) W[d * ldw + c] = v[t];
                }
            }
            else {
                int v[2 * NB];
                #pragma unroll
                for (int t = 0; t < 2 * NB; ++t) {
                    const int d = s_dst[t], sr = s_src[t];
                    v[t] = (d >= 0 && sr != d) ? perm[sr] : 0;
                }
                asm volatile("" ::: "memory");
                #pragma unroll
                for (int t = 0; t < 2 * NB; ++t) {
                    const int d = s_dst[t], sr = s_src[t];
                    if (d >= 0 && sr != d) perm[d] = v[t];
                }
            }
        }
        __syncthreads();
        const int c1 = k0 + kb, nr = n - c1;
        if (nr <= 0) break;
        T* C = W + c1 * ldw + c1;
        const T* U = W + k0 * ldw + c1;
        if constexpr (sizeof(T) == 4) {
            if (bf) wg_update<T, NB, LD, BT, true>(C, U, ldw, s_p + kb * LD, nr);
            else wg_update<T, NB, LD, BT, false>(C, U, ldw, s_p + kb * LD, nr);
        }
        else {
            wg_update<T, NB, LD, BT, false>(C, U, ldw, s_p + kb * LD, nr);
        }
        __syncthreads();
    }
}

// x := op(LU)^{-1} x for the factors in W (row-major), x of length n in
// global memory (FP64).  Lower (unit) or upper, 64-row blocks: the diagonal
// block is staged in LDS (s_blk, 64 x 65 T) and solved by wave 0 with
// lane broadcasts, the solved piece is kept in LDS (s_x) and the rows below (above)
// are updated by the whole workgroup, one row per thread with eight
// independent partial sums.
template <class T, int BT>
__device__ __forceinline__ void wg_trsv(const T* __restrict__ W, int n, int ldw, double* __restrict__ x, bool lower,
                                        T* s_blk, double* s_x)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nblk = (n + 63) / 64;
    for (int bb = 0; bb < nblk; ++bb) {
        const int blk = lower ? bb : nblk - 1 - bb;
        const int b0 = blk * 64, bn = min(64, n - b0);
        for (int e = tid; e < 64 * 64; e += BT) {
            const int r = e >> 6, c = e & 63;
            s_blk[r * 65 + c] = (r < bn && c < bn) ? W[int64_t(b0 + r) * ldw + b0 + c] : T(0);
        }
        __syncthreads();
        if (wave == 0) {
            double y = lane < bn ? x[b0 + lane] : 0.0;
            const T* row = s_blk + lane * 65;
            if (lower) {
                #pragma unroll 8
                for (int j = 0; j < bn; ++j) {
                    const double yj = lane_val(y, j), l = double(row[j]);
                    y = lane > j ? y - l * yj : y;
                }
            }
            else {
                const double d = lane < bn ? double(row[lane]) : 1.0, dinv = 1.0 / d;
                if constexpr (sizeof(T) == 4) {
                    // a float factor's rows scaled by the diagonal, off the chain
                    y /= d;
                    #pragma unroll 8
                    for (int j = bn - 1; j >= 0; --j) {
                        const double yj = lane_val(y, j), u = double(row[j]) * dinv;
                        y = lane < j ? y - u * yj : y;
                    }
                }
                else {
                    // y stays the row's numerator; outside the quotients' range
                    // the block is solved again with divisions
                    const double y0 = y;
                    #pragma unroll 8
                    for (int j = bn - 1; j >= 0; --j) {
                        const double yj = lane_val(quot_by_inverse(y, d, dinv), j), u = double(row[j]);
                        y = lane < j ? y - u * yj : y;
                    }
                    double q = quot_by_inverse(y, d, dinv);
                    if (__ballot(!(quot_range(d) && quot_holds(y, q)))) {
                        y = y0;
                        #pragma unroll 1
                        for (int j = bn - 1; j >= 0; --j) {
                            const double yj = lane_val(y / d, j), u = double(row[j]);
                            y = lane < j ? y - u * yj : y;
                        }
                        q = y / d;
                    }
                    y = q;
                }
            }
            if (lane < bn) x[b0 + lane] = y;
            s_x[lane] = lane < bn ? y : 0.0;
        }
        __syncthreads();
        const int r0 = lower ? b0 + bn : 0, r1 = lower ? n : b0;
        for (int i = r0 + tid; i < r1; i += BT) {
            const T* wr = W + int64_t(i) * ldw + b0;
            double ps[8];
            #pragma unroll
            for (int u = 0; u < 8; ++u) ps[u] = 0.0;
            if (bn == 64) {
                #pragma unroll
                for (int j = 0; j < 64; j += 8)
                    #pragma unroll
                    for (int u = 0; u < 8; ++u) ps[u] += double(wr[j + u]) * s_x[j + u];
            }
            else {
                for (int j = 0; j < bn; ++j) ps[j & 7] += double(wr[j]) * s_x[j];
            }
            x[i] -= ((ps[0] + ps[1]) + (ps[2] + ps[3])) + ((ps[4] + ps[5]) + (ps[6] + ps[7]));
        }
        __syncthreads();
    }
}

struct BatchArgs {
    int count;
    int nbig;                       // order[0 .. nbig) take a workgroup each,
    int small_per;                  // the rest a wave each, small_per per workgroup
    const int* order;               // systems, each part largest first
    const int* n;                   // sizes
    const int* mode;                // per system, see the file comment
    const int64_t* offA;            // A_i at A + offA[i], column-major, ld n_i (FP64)
    const int64_t* offB;            // b_i / x_i at B + offB[i]
    const double* A;
    const double* B;
    double* X;
    int* iters;                     // refinement steps (>= 0), -(itermax+1) fallback, -3 singular factor
    int* info;                      // factorization info (FP64 path or fallback)
    double* berr;                   // ||b - A x||_inf / (||A||_inf ||x||_inf)
    int* choice;                    // what ran: 0 BF16 + IR, 1 FP32 + IR, 2 FP64
    float* feat;                    // learned path: SEL_F features per system (may be null)
    unsigned long long* ticks;      // wall-clock ticks per system (100 MHz; may be null)
    const float* sel;               // selector network parameters (learned path)
    int* queue;                     // [0] ticket, [1] finished workgroups; zero between launches
    char* work;                     // per-workgroup workspace
    int64_t work_stride;            // bytes per workgroup
    int itermax;
    double tol;                     // <= 0: eps * sqrt(n)
    int probe_bf16;                 // learned path: probe factor in BF16 (1) or FP32 (0)
};

// sum_j |A(i, j)| (ABS) or sum_j A(i, j) v_j over the n columns of the
// column-major A, with v read from LDS; eight independent partial sums keep
// eight loads in flight per thread.
template <bool ABS>
__device__ __forceinline__ double row_dot(const double* __restrict__ A, int n, int i, const double* s_v)
{
    double ps[8];
    #pragma unroll
    for (int u = 0; u < 8; ++u) ps[u] = 0.0;
    int j = 0;
    // 32 loads in flight per thread; column j + u still goes to partial sum
    // u mod 8 in column order, as in the 8-column loop below
    for (; j + 32 <= n; j += 32) {
        double av[32];
        #pragma unroll
        for (int u = 0; u < 32; ++u) av[u] = A[i + int64_t(j + u) * n];
        #pragma unroll
        for (int u = 0; u < 32; ++u) ps[u & 7] += ABS ? fabs(av[u]) : av[u] * s_v[j + u];
    }
    for (; j + 8 <= n; j += 8)
        #pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double a = A[i + int64_t(j + u) * n];
            ps[u] += ABS ? fabs(a) : a * s_v[j + u];
        }
    for (; j < n; ++j) {
        const double a = A[i + int64_t(j) * n];
        ps[j & 7] += ABS ? fabs(a) : a * s_v[j];
    }
    return ((ps[0] + ps[1]) + (ps[2] + ps[3])) + ((ps[4] + ps[5]) + (ps[6] + ps[7]));
}

// Norms keep NaN (fmax drops it): a factor or solution that overflowed has a
// norm that is not finite, and such a norm never meets the tolerance.
__device__ __forceinline__ double norm_max(double a, double b) { return (a > b || a != a) ? a : b; }
__device__ __forceinline__ bool b_converged(double rnorm, double xnorm, double anorm, double tol)
{
    const double lim = xnorm * anorm * tol;
    return isfinite(lim) && rnorm <= lim;
}
// ||b - A x|| / (||A|| ||x||), not finite where the solution is not.
__device__ __forceinline__ double b_backward_error(double rnorm, double xnorm, double anorm)
{
    const double den = anorm * xnorm;
    return den == 0 ? 0.0 : rnorm / den;
}

// r = b - A x (FP64, A column-major) and infinity norms: ||r|| in s_dred[0],
// ||x|| in s_dred[1].  s_v: n doubles of LDS for x.
template <int BT>
__device__ __forceinline__ void wg_residual(const double* __restrict__ A, int n, const double* __restrict__ b,
                            const double* __restrict__ x, double* __restrict__ r, double* s_dred, double* s_v)
{
    constexpr int NW = BT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < n; i += BT) s_v[i] = x[i];
    __syncthreads();
    double rmax = 0, xmax = 0;
    for (int i = tid; i < n; i += BT) {
        const double s = b[i] - row_dot<false>(A, n, i, s_v);
        r[i] = s;
        rmax = norm_max(rmax, fabs(s));
        xmax = norm_max(xmax, fabs(s_v[i]));
    }
    #pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        rmax = norm_max(rmax, __shfl_xor(rmax, o, 64));
        xmax = norm_max(xmax, __shfl_xor(xmax, o, 64));
    }
    __syncthreads();
    if (lane == 0) { s_dred[2 + wave] = rmax; s_dred[2 + NW + wave] = xmax; }
    __syncthreads();
    if (tid == 0) {
        double a = 0, c = 0;
        for (int w = 0; w < NW; ++w) { a = norm_max(a, s_dred[2 + w]); c = norm_max(c, s_dred[2 + NW + w]); }
        s_dred[0] = a;
        s_dred[1] = c;
    }
    __syncthreads();
}

// max over rows of the row sums of |A| (column-major) -> s_dred[0];
// max |v| of v (length n) -> s_dred[1].
template <int BT>
__device__ __forceinline__ void wg_norms(const double* __restrict__ A, int n, const double* __restrict__ v, double* s_dred)
{
    constexpr int NW = BT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double m = 0, vm = 0;
    for (int i = tid; i < n; i += BT) {
        m = norm_max(m, row_dot<true>(A, n, i, nullptr));
        vm = norm_max(vm, fabs(v[i]));
    }
    #pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        m = norm_max(m, __shfl_xor(m, o, 64));
        vm = norm_max(vm, __shfl_xor(vm, o, 64));
    }
    __syncthreads();
    if (lane == 0) { s_dred[2 + wave] = m; s_dred[2 + NW + wave] = vm; }
    __syncthreads();
    if (tid == 0) {
        double a = 0, c = 0;
        for (int w = 0; w < NW; ++w) { a = norm_max(a, s_dred[2 + w]); c = norm_max(c, s_dred[2 + NW + w]); }
        s_dred[0] = a;
        s_dred[1] = c;
    }
    __syncthreads();
}

// Selector network forward pass by wave 0 (h1 = relu(W1^T f + b1),
// h2 = relu(W2^T h1 + b2), z = W3^T h2 + b3; lane h holds hidden unit h);
// returns argmax over the first SEL_CHOICES outputs (lane 0 valid).
__device__ __forceinline__ int sel_choose(const float* __restrict__ P, const float* f)
{
    const int lane = threadIdx.x & 63;
    const float* W1 = P;
    const float* b1 = W1 + SEL_F * SEL_H;
    const float* W2 = b1 + SEL_H;
    const float* b2 = W2 + SEL_H * SEL_H;
    const float* W3 = b2 + SEL_H;
    const float* b3 = W3 + SEL_H * SEL_K;
    float h = b1[lane];
    for (int q = 0; q < SEL_F; ++q) h += f[q] * W1[q * SEL_H + lane];
    h = fmaxf(h, 0.f);
    float h2 = b2[lane];
    for (int g = 0; g < SEL_H; ++g) h2 += __shfl(h, g, 64) * W2[g * SEL_H + lane];
    h2 = fmaxf(h2, 0.f);
    const int k = lane & (SEL_K - 1);
    float z = b3[k];
    for (int g = 0; g < SEL_H; ++g) z += __shfl(h2, g, 64) * W3[g * SEL_K + k];
    int best = 0;
    float bz = __shfl(z, 0, 64);
    for (int c = 1; c < SEL_CHOICES; ++c) {
        const float zc = __shfl(z, c, 64);
        if (zc > bz) { bz = zc; best = c; }
    }
    return best;
}

//------------------------------------------------------------------------------
// Systems of at most 64 rows, one wave each.  Row i of the system is lane i;
// its row of the matrix sits in 64 registers while it is factored, the
// system's n columns in the last n column positions (k0 = 64 - n first ones
// unused), so that after the rotating factorization column position c is
// register c whatever n is.  n = 64 takes 106 us (51 of them the factor),
// n = 32 56 us, and the waves of a workgroup do not wait for each other; the
// workgroup path above takes 190 and 110 us per system of its CU (430 and
// 240 with the panel in LDS).
constexpr int BSMALL = 64;

// Steps [k, kend) (column positions) with C live registers (C >= 64 - k); as
// leaf_wg_steps: rows keep their lane, interchanges change labels.
template <class T, int C>
__device__ __forceinline__ void wave_factor_steps(T (&v)[64], int n, int& lab, int& pl, T& diag, int& info, int& k,
                                                  int kend)
{
    const int lane = threadIdx.x & 63, k0 = 64 - n;
    #pragma unroll 1
    for (; k < kend; ++k) {
        const int kk = k - k0, lim = 64 - k;
        const T a = fabs(v[0]);
        const T babs = (lab >= kk && lab < n && a >= T(0)) ? a : T(-1);
        const uint32_t key = argmax_key(babs), mk = wave_max_u32(key);
        const int wl = mk ? wave_argmax_lane(babs, uint32_t(lab), key, mk) : __builtin_ctzll(__ballot(lab == kk));
        const T pv = lane_val(v[0], wl);
        const int pos = __builtin_amdgcn_readlane(lab, wl);
        lab = lane == wl ? kk : lab == kk ? pos : lab;
        pl = lane == kk ? wl : pl;
        diag = lane == wl ? v[0] : diag;
        const bool act = lab > kk && lab < n;
        T l = v[0] * (T(1) / pv);
        if (pv == T(0) || fabs(pv) < std::numeric_limits<T>::min()) {
            if (pv == T(0) && info == 0) info = kk + 1;
            l = pv == T(0) ? v[0] : v[0] / pv;
        }
        const T t0 = act ? l : v[0];
        l = act ? l : T(0);
        #pragma unroll
        for (int c = 1; c < C; ++c) {
            const T xr = lane_val(v[c], wl);
            const T x = c > C - 16 ? (c < lim ? xr : T(0)) : xr;
            v[c - 1] = v[c] - l * x;
        }
        #pragma unroll
        for (int c = C; c < 64; ++c) v[c - 1] = v[c];
        v[63] = t0;
    }
}

// LU of A (column-major) cast to T, stored by column positions: column k at
// F[64 (64 - n + k) + lane].  lab: the row position this lane's row
// ends in; pl: lane k holds the lane of pivot row k; diag: this row's U(k, k).
// Returns the first exactly-zero pivot (1-based), else 0.
template <class T>
__device__ __forceinline__ int wave_factor(const double* __restrict__ A, int n, T* F, int& lab, int& pl, T& diag)
{
    const int lane = threadIdx.x & 63, i = min(lane, n - 1);
    T v[64];
    #pragma unroll
    for (int c = 0; c < 64; ++c) v[c] = T(A[i + min(c, n - 1) * n]);
    #pragma unroll
    for (int c = 0; c < 64; ++c) v[c] = (lane < n && c < n) ? v[c] : T(0);
    lab = lane;
    pl = 0;
    diag = T(1);
    int info = 0, k = 64 - n;
    wave_factor_steps<T, 64>(v, n, lab, pl, diag, info, k, 16);
    wave_factor_steps<T, 48>(v, n, lab, pl, diag, info, k, 32);
    wave_factor_steps<T, 32>(v, n, lab, pl, diag, info, k, 48);
    wave_factor_steps<T, 16>(v, n, lab, pl, diag, info, k, 64);
    // by column position: no address below F, whatever n is
    #pragma unroll
    for (int c = 0; c < 64; ++c) F[64 * c + lane] = v[c];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return info;
}

// (LU)^{-1} P rhs in FP64 from the factor as wave_factor stores it; rhs by
// original row, the result's entry k in lane k.
template <class T>
__device__ __forceinline__ double wave_lu_solve(const T* Fp, int n, int lab, int pl, T diag, double rhs)
{
    const int lane = threadIdx.x & 63;
    const T* F = Fp + 64 * (64 - n);
    double y = rhs, x = 0.0;
    #pragma unroll 8
    for (int k = 0; k < n; ++k) {
        const double yk = lane_val(y, __builtin_amdgcn_readlane(pl, k)), l = double(F[64 * k + lane]);
        y = lab > k ? y - l * yk : y;
    }
    const double d = double(diag), dinv = 1.0 / d;
    if constexpr (sizeof(T) == 4) {
        // a float factor's rows scaled by the diagonal, off the chain
        y /= d;
        #pragma unroll 8
        for (int k = n - 1; k >= 0; --k) {
            const double xk = lane_val(y, __builtin_amdgcn_readlane(pl, k)), u = double(F[64 * k + lane]) * dinv;
            y = lab < k ? y - u * xk : y;
            x = lane == k ? xk : x;
        }
    }
    else {
        // as in wg_trsv
        const double y0 = y;
        #pragma unroll 8
        for (int k = n - 1; k >= 0; --k) {
            const double xk = lane_val(quot_by_inverse(y, d, dinv), __builtin_amdgcn_readlane(pl, k));
            y = lab < k ? y - double(F[64 * k + lane]) * xk : y;
            x = lane == k ? xk : x;
        }
        if (__ballot(!(quot_range(d) && quot_holds(y, quot_by_inverse(y, d, dinv))))) {
            y = y0;
            #pragma unroll 1
            for (int k = n - 1; k >= 0; --k) {
                const double xk = lane_val(y / d, __builtin_amdgcn_readlane(pl, k));
                y = lab < k ? y - double(F[64 * k + lane]) * xk : y;
                x = lane == k ? xk : x;
            }
        }
    }
    return x;
}

// sum_j |A(i, j)| or sum_j A(i, j) x_j for this lane's row, summed as row_dot does.
template <bool ABS>
__device__ __forceinline__ double wave_row_dot(const double* __restrict__ A, int n, double x)
{
    const int i = min(int(threadIdx.x & 63), n - 1);
    asm volatile("" : "+s"(n));                         // bounds formed here, not ahead of the refinement loop
    double ps[8];
    #pragma unroll
    for (int u = 0; u < 8; ++u) ps[u] = 0.0;
    #pragma unroll
    for (int h = 0; h < 64; h += 32) {
        if (h >= n) break;
        double av[32];
        #pragma unroll
        for (int u = 0; u < 32; ++u) av[u] = A[i + min(h + u, n - 1) * n];
        #pragma unroll
        for (int u = 0; u < 32; ++u)
            if (h + u < n) ps[u & 7] += ABS ? fabs(av[u]) : av[u] * lane_val(x, h + u);
    }
    return ((ps[0] + ps[1]) + (ps[2] + ps[3])) + ((ps[4] + ps[5]) + (ps[6] + ps[7]));
}

__device__ __forceinline__ double wave_norm_max(double v)
{
    #pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = norm_max(v, __shfl_xor(v, o, 64));
    return v;
}

// The selector's features of a probe and its choice are the workgroup path's.
__device__ __forceinline__ void batch_features(float* f, int n, bool ok, double anorm, double bnorm, double xnorm, double rnorm,
                               double tol, bool probe_bf16)
{
    for (int q = 0; q < SEL_F; ++q) f[q] = 0.f;
    const double tiny = 1e-300;
    f[0] = 1.f;
    f[1] = float(log2(double(n)) / 10.0);
    if (ok) {
        f[2] = float(log10(fmax(anorm * xnorm / bnorm, tiny)) / 8.0);
        f[3] = float(log10(fmax(rnorm / (anorm * xnorm), tiny)) / 8.0);
        f[5] = float(log10(fmax(rnorm / bnorm, tiny)) / 8.0);
        f[6] = (rnorm <= xnorm * anorm * tol) ? 1.f : 0.f;
    }
    else {
        f[4] = 1.f;
    }
    f[7] = probe_bf16 ? 1.f : 0.f;
}

// One system (n <= 64; modes 0, 1 and, with an FP32 probe, 3 .. 6) by one
// wave, the steps of the workgroup path below.  s_feat: SEL_F floats of LDS;
// s_f: 64 x 64 floats of LDS for the float factor; F64: the same in doubles,
// in memory, for the FP64 one.
__device__ __forceinline__ void wave_system(const BatchArgs& a, const double* gA, const double* gB, double* gX, int sys,
                                            float* s_feat, float* s_f, double* F64)
{
    const unsigned long long t0 = wall_clock64();
    const int lane = threadIdx.x & 63;
    const int n = __builtin_amdgcn_readfirstlane(a.n[sys]), mode = __builtin_amdgcn_readfirstlane(a.mode[sys]);
    const double* A = gA + a.offA[sys];
    const double* b = gB + a.offB[sys];
    const double tol = a.tol > 0 ? a.tol : std::numeric_limits<double>::epsilon() * sqrt(double(n));
    const double bl = lane < n ? b[lane] : 0.0;
    double x = 0.0, r = 0.0, rnorm = 0.0, xnorm = 0.0;
    auto residual = [&] {
        const double s = bl - wave_row_dot<false>(A, n, x);
        r = lane < n ? s : 0.0;
        rnorm = wave_norm_max(fabs(r));
        xnorm = wave_norm_max(lane < n ? fabs(x) : 0.0);
    };
    const double anorm = wave_norm_max(lane < n ? wave_row_dot<true>(A, n, 0.0) : 0.0);
    const double bnorm = wave_norm_max(fabs(bl));

    int info = 0, iters = 0, ch = mode == 1 ? 2 : 1;
    bool need64 = mode == 1;
    if (mode != 1) {
        float diag;
        int lab, pl;
        const int pinfo = wave_factor<float>(A, n, s_f, lab, pl, diag);
        if (pinfo == 0) {
            x = wave_lu_solve<float>(s_f, n, lab, pl, diag, bl);
            residual();
        }
        bool keep = pinfo == 0;
        if (mode != 0) {
            const bool ok = pinfo == 0 && isfinite(rnorm) && isfinite(xnorm) && xnorm > 0 && bnorm > 0 && anorm > 0;
            if (lane == 0) batch_features(s_feat, n, ok, anorm, bnorm, xnorm, rnorm, tol, false);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (a.feat && lane < SEL_F) a.feat[int64_t(sys) * SEL_F + lane] = s_feat[lane];
            int c = mode - 4;
            if (mode == 3) c = __builtin_amdgcn_readfirstlane(sel_choose(a.sel, s_feat));
            if (c <= 1) c = ok ? 1 : 2;                 // choices 0 and 1 keep an FP32 probe that can be kept
            ch = c;
            keep = c == 1;
        }
        if (keep) {
            bool conv = false;
            for (int it = 0; it <= a.itermax; ++it) {
                if (it > 0) residual();
                conv = b_converged(rnorm, xnorm, anorm, tol);
                if (conv) { iters = it; break; }
                if (it == a.itermax) break;
                x += wave_lu_solve<float>(s_f, n, lab, pl, diag, r);
            }
            if (!conv) { need64 = true; iters = -a.itermax - 1; }
        }
        else {
            need64 = true;
            iters = mode == 0 ? -3 : 0;
        }
    }
    if (need64) {
        double diag;
        int lab, pl;
        info = wave_factor<double>(A, n, F64, lab, pl, diag);
        x = wave_lu_solve<double>(F64, n, lab, pl, diag, bl);
    }
    residual();
    if (lane < n) gX[a.offB[sys] + lane] = x;
    if (lane == 0) {
        a.iters[sys] = iters;
        a.info[sys] = info;
        a.berr[sys] = b_backward_error(rnorm, xnorm, anorm);
        if (a.choice) a.choice[sys] = ch;
        if (a.ticks) a.ticks[sys] = wall_clock64() - t0;
    }
}

template <int NBF, int BT>
__global__ __launch_bounds__(BT)
void batched_solve_kernel(BatchArgs a, char* gwork, const double* gA, const double* gB, double* gX)
{
    // The block's large arrays are arguments of their own, too: the compiler
    // knows those for global memory, while a pointer read from the block is
    // accessed by flat instructions, which wait on the LDS counter as well.
    constexpr int NW = BT / 64;
    __shared__ __attribute__((aligned(16))) char s_pan[pan_lds_bytes<NBF, BT>()];
    using LeafF = LeafWg<float, Pan<float, NBF, BT>::NB, BT>;
    using LeafD = LeafWg<double, Pan<double, NBF, BT>::NB, BT>;
    __shared__ __attribute__((aligned(16))) char s_leaf[sizeof(LeafF) > sizeof(LeafD) ? sizeof(LeafF) : sizeof(LeafD)];
    __shared__ float s_wfeat[NW][SEL_F];
    __shared__ int s_dst[64], s_src[64];
    __shared__ double s_dred[2 + 2 * NW];
    __shared__ float s_feat[SEL_F];
    __shared__ int s_sys, s_info, s_choice;
    const int tid = threadIdx.x;
    char* ws = gwork + int64_t(blockIdx.x) * a.work_stride;
    // workspace: W32 (1024^2 float) | W64 (1024^2 double) | perm (1024 int) | r, y (1024 double)
    float* W = reinterpret_cast<float*>(ws);
    double* W64 = reinterpret_cast<double*>(ws + int64_t(BMAXN) * BMAXN * sizeof(float));
    int* perm = reinterpret_cast<int*>(W64 + int64_t(BMAXN) * BMAXN);
    double* r = reinterpret_cast<double*>(perm + BMAXN);
    double* y = r + BMAXN;
    float* s_pf = reinterpret_cast<float*>(s_pan);
    double* s_pd = reinterpret_cast<double*>(s_pan);
    // outside the factorizations the panel LDS holds the solves' diagonal
    // block (64 x 65, up to FP64) and vectors: x for residuals, a solved piece
    static_assert(pan_lds_bytes<NBF, BT>() >= NW * 64 * 64 * 4, "panel LDS too small for the waves' factors");
    static_assert(pan_lds_bytes<NBF, BT>() >= 64 * 65 * 8 + BMAXN * 8 + 64 * 8, "panel LDS too small for the solves");
    double* s_v = reinterpret_cast<double*>(s_pan + 64 * 65 * 8);
    double* s_x = s_v + BMAXN;
    const double eps = std::numeric_limits<double>::epsilon();
    while (true) {
        if (tid == 0) {
            const int q = atomicAdd(&a.queue[0], 1);
            const int groups = a.small_per ? (a.count - a.nbig + a.small_per - 1) / a.small_per : 0;
            s_sys = q < a.nbig ? a.order[q] : q < a.nbig + groups ? -2 - (q - a.nbig) : -1;
            s_info = 0;
        }
        __syncthreads();
        const int sys = s_sys;
        if (sys == -1) break;                             // every wave leaves here
        if (sys < 0) {                                    // a group of small systems, one per wave
            const int w = __builtin_amdgcn_readfirstlane(tid >> 6), i = a.nbig + (-2 - sys) * a.small_per + w;
            if (w < a.small_per && i < a.count)
                wave_system(a, gA, gB, gX, __builtin_amdgcn_readfirstlane(a.order[i]), s_wfeat[w], s_pf + 64 * 64 * w,
                            W64 + 64 * 64 * w);
            __syncthreads();
            continue;
        }
        const unsigned long long t0 = wall_clock64();
        const int n = a.n[sys], ldw = b_ldw(n);
        const int mode = a.mode[sys];
        const double* A = gA + a.offA[sys];
        const double* b = gB + a.offB[sys];
        double* x = gX + a.offB[sys];
        const double tol = a.tol > 0 ? a.tol : eps * sqrt(double(n));

        // ||A||_inf and ||b||_inf
        wg_norms<BT>(A, n, b, s_dred);
        const double anorm = s_dred[0], bnorm = s_dred[1];
        __syncthreads();

        // One pass of the loop: factor (when asked to), solve, residual, and
        // what follows from it.  Every step is written once, so that it is
        // inlined: as separate functions the steps reach LDS and memory by
        // flat accesses (4096 systems 83 ms instead of 62.7).
        // kind: 0 FP32 factor, 1 BF16, 2 FP64.
        int kind = mode == 1 ? 2 : (mode == 2 || (mode >= 3 && a.probe_bf16)) ? 1 : 0;
        int ch = mode == 0 ? 1 : mode == 1 ? 2 : 0;
        int info = 0, iters = 0, it = 0;
        bool probing = mode >= 3, fresh = true;
        while (true) {
            bool singular = false;
            if (fresh) {
                if (tid == 0) s_info = 0;
                if (kind == 2) {
                    wg_load_rowmajor<double, BT>(A, n, W64, ldw);
                    __syncthreads();
                    wg_getrf<double, NBF, BT>(W64, n, ldw, perm, &s_info, false, s_pd, *reinterpret_cast<LeafD*>(s_leaf),
                                              s_dst, s_src);
                }
                else {
                    wg_load_rowmajor<float, BT>(A, n, W, ldw);
                    __syncthreads();
                    wg_getrf<float, NBF, BT>(W, n, ldw, perm, &s_info, kind == 1, s_pf, *reinterpret_cast<LeafF*>(s_leaf),
                                             s_dst, s_src);
                }
                __syncthreads();
                if (kind == 2) info = s_info;
                else singular = s_info != 0;
                it = 0;
                __syncthreads();                          // s_info read before it is reset
            }
            if (!singular) {
                // out = (LU)^{-1} P rhs
                const double* rhs = fresh ? b : r;
                double* out = fresh ? x : y;
                for (int i = tid; i < n; i += BT) out[i] = rhs[perm[i]];
                __syncthreads();
                for (int h = 0; h < 2; ++h) {
                    if (kind == 2) wg_trsv<double, BT>(W64, n, ldw, out, h == 0, s_pd, s_x);
                    else wg_trsv<float, BT>(W, n, ldw, out, h == 0, s_pf, s_x);
                }
                if (!fresh) {
                    for (int i = tid; i < n; i += BT) x[i] += y[i];
                    __syncthreads();
                }
                wg_residual<BT>(A, n, b, x, r, s_dred, s_v);
            }
            fresh = false;
            if (kind == 2) break;
            if (probing) {
                // learned path: the probe's normwise quantities pick what runs
                probing = false;
                const double rnorm = singular ? 0.0 : s_dred[0], xnorm = singular ? 0.0 : s_dred[1];
                const bool ok = !singular && isfinite(rnorm) && isfinite(xnorm) && xnorm > 0 && bnorm > 0 && anorm > 0;
                if (tid == 0) batch_features(s_feat, n, ok, anorm, bnorm, xnorm, rnorm, tol, a.probe_bf16 != 0);
                __syncthreads();
                if (a.feat && tid < SEL_F) a.feat[int64_t(sys) * SEL_F + tid] = s_feat[tid];
                int c = mode - 4;
                if (mode == 3) {
                    if (tid < 64) {
                        const int cc = sel_choose(a.sel, s_feat);
                        if (tid == 0) s_choice = cc;
                    }
                    __syncthreads();
                    c = s_choice;
                }
                // what runs: 0 BF16 + IR, 1 FP32 + IR, 2 FP64.  A singular or
                // non-finite probe cannot be kept (BF16 probe: FP32 instead; FP32
                // probe: FP64); with an FP32 probe choices 0 and 1 both keep it.
                bool keep;
                if (a.probe_bf16) {
                    if (c == 0 && !ok) c = 1;
                    keep = c == 0;
                }
                else {
                    if (c <= 1) c = ok ? 1 : 2;
                    keep = c == 1;
                }
                ch = c;
                if (!keep) {
                    kind = c == 1 ? 0 : 2;
                    fresh = true;
                    continue;
                }
            }
            else if (singular) {
                iters = -3;
                kind = 2;
                fresh = true;
                continue;
            }
            // refinement: the residual of x is in r, its norms in s_dred
            const bool conv = a.itermax >= 0 && b_converged(s_dred[0], s_dred[1], anorm, tol);
            __syncthreads();
            if (conv) { iters = it; break; }
            if (it >= a.itermax) {
                iters = -a.itermax - 1;
                kind = 2;
                fresh = true;
            }
            ++it;
        }
        // backward error from the last residual
        if (tid == 0) {
            a.iters[sys] = iters;
            a.info[sys] = info;
            a.berr[sys] = b_backward_error(s_dred[0], s_dred[1], anorm);
            if (a.choice) a.choice[sys] = ch;
            if (a.ticks) a.ticks[sys] = wall_clock64() - t0;
        }
        __syncthreads();
    }
    // the last workgroup to finish leaves the queue zeroed for the next launch
    if (tid == 0) {
        __threadfence();
        const int done = atomicAdd(&a.queue[1], 1);
        if (done == int(gridDim.x) - 1) {
            atomicExch(&a.queue[0], 0);
            atomicExch(&a.queue[1], 0);
        }
    }
}

int64_t batched_work_stride(int)
{
    int64_t b = int64_t(BMAXN) * BMAXN * (4 + 8) + int64_t(BMAXN) * (4 + 16) + 256;
    return (b + 255) & ~int64_t(255);
}

// Kernel of a tile configuration: float panel width nbf (16 or 32) and
// workgroup size bt (256; 512 with nbf 16 only: the 32-wide panel at 512
// threads spills most of its working registers).
static const void* batched_kernel_ptr(int nbf, int bt)
{
    if (nbf == 16) return bt == 512 ? (const void*)batched_solve_kernel<16, 512> : (const void*)batched_solve_kernel<16, 256>;
    return (const void*)batched_solve_kernel<32, 256>;
}

bool batched_config_valid(int nbf, int bt) { return (nbf == 16 && (bt == 256 || bt == 512)) || (nbf == 32 && bt == 256); }

int batched_max_wgs_per_cu(int nbf, int bt)
{
    SA_REQUIRE(batched_config_valid(nbf, bt), -2, "batched: bad tile configuration");
    int nb = 0;
    SA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, batched_kernel_ptr(nbf, bt), bt, 0));
    return nb;
}

void batched_fill_args(void* out, int count, int nbig, int small_per, const int* order, const int* n, const int* mode, const int64_t* offA,
                       const int64_t* offB, const double* A, const double* B, double* X, int* iters, int* info,
                       double* berr, int* choice, float* feat, unsigned long long* ticks, const float* sel,
                       int* queue, char* work, int itermax, double tol, int probe_bf16)
{
    BatchArgs a{count, nbig, small_per, order, n, mode, offA, offB, A, B, X, iters, info, berr, choice, feat, ticks, sel, queue,
                work, batched_work_stride(4), itermax, tol, probe_bf16};
    static_assert(sizeof(BatchArgs) <= BATCH_ARGS_BYTES, "BatchArgs size");
    std::memcpy(out, &a, sizeof(a));
}

void batched_launch(const void* args, int nbf, int bt, int grid, hipStream_t s)
{
    SA_REQUIRE(batched_config_valid(nbf, bt), -2, "batched: bad tile configuration");
    const BatchArgs& a = *static_cast<const BatchArgs*>(args);
    if (a.count <= 0) return;
    if (nbf == 16) {
        if (bt == 512) hipLaunchKernelGGL((batched_solve_kernel<16, 512>), dim3(unsigned(grid)), dim3(512), 0, s, a, a.work, a.A, a.B, a.X);
        else hipLaunchKernelGGL((batched_solve_kernel<16, 256>), dim3(unsigned(grid)), dim3(256), 0, s, a, a.work, a.A, a.B, a.X);
    }
    else {
        hipLaunchKernelGGL((batched_solve_kernel<32, 256>), dim3(unsigned(grid)), dim3(256), 0, s, a, a.work, a.A, a.B, a.X);
    }
    SA_CHECK_LAUNCH();
}

// A one-node graph holding the launch (the kernel resets its own queue, so
// replays need nothing else).  args must stay valid while the graph exists.
void batched_graph(void* args, int nbf, int bt, int grid, hipGraph_t* g, hipGraphExec_t* ge)
{
    SA_REQUIRE(batched_config_valid(nbf, bt), -2, "batched: bad tile configuration");
    SA_HIP(hipGraphCreate(g, 0));
    hipKernelNodeParams kp{};
    BatchArgs* a = static_cast<BatchArgs*>(args);
    void* kargs[5] = {args, &a->work, &a->A, &a->B, &a->X};
    kp.func = const_cast<void*>(batched_kernel_ptr(nbf, bt));
    kp.gridDim = dim3(unsigned(grid));
    kp.blockDim = dim3(unsigned(bt));
    kp.sharedMemBytes = 0;
    kp.kernelParams = kargs;
    kp.extra = nullptr;
    hipGraphNode_t node;
    SA_HIP(hipGraphAddKernelNode(&node, *g, nullptr, 0, &kp));
    SA_HIP(hipGraphInstantiate(ge, *g, nullptr, nullptr, 0));
}

int batched_max_n() { return BMAXN; }
int batched_small_n() { return BSMALL; }

} // namespace sa
