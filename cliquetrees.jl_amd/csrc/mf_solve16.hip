// mf_solve16.hip — gfx950 kernels of the supernodal triangular solves for more
// right-hand sides than go column by column (HostPlan::vcols), in blocks of
// sixteen on the matrix cores.
//
// The tasks, the tickets and the hand-off are those of mf_solve1.hip: an
// element that another workgroup waits for starts as a signalling NaN and is
// its own flag.  Blocks of sixteen columns are independent solves that share
// a launch: a ticket covers one unit of tasks for one block, the blocks of a
// unit side by side, so the chain of one block fills the waits of the others
// and the factor's tiles are read from a cache by all blocks but the first.
//
// Values in flight are kept row by row, sixteen columns (128 bytes in FP64)
// to a row: the solution (X forward, Z backward), the update vectors and the
// separator partials.  That is the layout the B operand of the 16x16x4
// matrix instructions loads in whole lines, straight from memory into
// registers, and gathered rows cost one line each.
//
// A wavefront takes a sixteen-wide slice of the product's inner dimension for
// all 64 rows (four row groups by four inner steps, 16 instructions a tile),
// so the operands of a chain step are the wavefront's own and there is no
// barrier in a chain; the wavefronts' sums meet in LDS once per task.
//
// Both directions with the permutations, 16 columns at a time inside one task
// and counters per front before -> this, us:
//   40 x 40 x 40 grid, n 64000, 75 columns    19170 -> 1530
//   56 x 60 x 52 grid, n 174720, 16 / 33      2840 -> 2070 / 29900 -> 2870
//   31 x 29 x 27 grid, n 24273, 16 / 33        830 ->  420 /  3760 ->  500
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "mf_kernels.h"
#include "mf_mfma.h"
#include "mf_vsolve.h"

namespace mf {

namespace {

constexpr int RB = 16;                         // columns of a block
constexpr int LR = RB + 1;                     // leading dimension of its rows in LDS
constexpr int VROWS = NB + NB * VT_ROWBLOCKS;  // rows of a one-task front

template <typename T>
using v4_t = typename Mfma<T>::v4;

// N values at once (settle): v holds earlier peeks, x the values (0 where off).
template <typename T, int N>
__device__ __forceinline__ void settle_n(bits_t<T> (&v)[N], const T* const (&p)[N], const bool (&on)[N], T (&x)[N],
                                         const Ctl& c) {
    auto missing = [&] {
        bool m = false;
#pragma unroll
        for (int i = 0; i < N; ++i) m |= on[i] && v[i] == unset<T>();
        return m;
    };
    if (__any(missing())) {
        Watch w;
        for (int spins = 1;; ++spins) {
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] = peek(p[i]);
            if (!__any(missing())) break;
            if ((spins & 255) == 0) {
                if (sync_ld(c.hang)) break;
                if (w.expired(0, c.ticket, c.stall)) {
                    if (missing()) give_up(c.hang, reinterpret_cast<const int32_t*>(p[0]), 1, 0, -1);
                    break;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = on[i] ? __builtin_bit_cast(T, v[i]) : (T)0;
}

// ---- operands -----------------------------------------------------------------
// Lane (li, lk).  Rows and columns outside a tile repeat its last ones: the
// other operand is 0 there or the sum unused.

// a[4 i + s] = base[16 i + li + (16 g + 4 s + lk) ld]
template <typename T>
__device__ __forceinline__ void load_a(const T* base, int64_t ld, int rows, int cols, int g, T (&a)[16]) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t c = (uint32_t)min(16 * g + 4 * s + lk, cols - 1) * (uint32_t)ld;
#pragma unroll
        for (int i = 0; i < 4; ++i) a[4 * i + s] = base[c + (uint32_t)min(16 * i + li, rows - 1)];
    }
}
// a[4 i + s] = base[(16 g + 4 lk + s) + (16 i + li) ld], row groups i with 16 i < cols (the transposed product)
template <typename T>
__device__ __forceinline__ void load_at(const T* base, int64_t ld, int rows, int cols, int g, T (&a)[16]) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (16 * i >= cols) break;
        const uint32_t c = (uint32_t)min(16 * i + li, cols - 1) * (uint32_t)ld;
        if (16 * g + 16 <= rows) {
            // four consecutive rows in one piece (aligned to an element only)
            __builtin_memcpy(&a[4 * i], base + 16 * g + (c + 4u * lk), 4 * sizeof(T));
            continue;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) a[4 * i + s] = base[c + (uint32_t)min(16 * g + 4 * lk + s, rows - 1)];
    }
}
// acc[i] += a[4 i + .] x over the four steps
template <typename T>
__device__ __forceinline__ void mma(const T (&a)[16], const T (&x)[4], v4_t<T> (&acc)[4], int groups) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= groups) break;
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[i] = Mfma<T>::op(a[4 * i + s], x[s], acc[i]);
    }
}
template <typename T>
__device__ __forceinline__ void zero(v4_t<T> (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = v4_t<T>{0, 0, 0, 0};
}
// Before anything but another matrix instruction touches the sums.  The
// number of row groups is a branch around matrix instructions; hipcc 7.2
// counts the 18 wait states such a result needs (FP64, 16 passes) along the
// longest way through the branches only, and on the short way (one group) the
// next instruction read the last register early: its low word was still 0.
// (tests/test_matrix_waits.py looks for such paths in the built library.)
template <typename T>
__device__ __forceinline__ void mma_done(v4_t<T> (&acc)[4]) {
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
}
// This wavefront's sums into its part of Red (4 x 64 rows).
template <typename T>
__device__ __forceinline__ void put(v4_t<T> (&acc)[4], T* Red, int g) {
    mma_done<T>(acc);
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) Red[(NB * g + 16 * i + Mfma<T>::row(lk, v)) * LR + li] = acc[i][v];
}
template <typename T>
__device__ __forceinline__ T sum4(const T* Red, int row, int col) {
    const int e = row * LR + col;
    return (Red[e] + Red[NB * LR + e]) + (Red[2 * NB * LR + e] + Red[3 * NB * LR + e]);
}

// ---- children -----------------------------------------------------------------
// CB children by RG groups of RP rows in flight, added into Y (rows rel - r0).
// RP = 16: a wavefront takes columns 4 g .. 4 g + 3 of every row (the four
// wavefronts share Y without meeting); RP = 4: all sixteen.
template <typename T, bool BLK, int RP, int CB, int RG>
__device__ __forceinline__ void gather_pass(const DevPlan& P, const DevBSolve<T>& V, int q, int qe, int blk, int r0, T* Y,
                                            int g, const Ctl& ctl) {
    const int lane = threadIdx.x & 63;
    const int ro = RP == 16 ? lane >> 2 : lane >> 4, col = RP == 16 ? 4 * g + (lane & 3) : lane & 15;
    int lo[CB], hi[CB], rel[CB], most = 0;
    const T* M[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        const VChild k = V.chd[min(q + c, qe - 1)];
        lo[c] = 0;
        hi[c] = uni(k.ma);
        if (BLK) {
            lo[c] = uni(P.sgstart[k.sg + blk]);
            hi[c] = uni(P.sgstart[k.sg + blk + 1]);
        }
        if (q + c >= qe) hi[c] = lo[c];
        rel[c] = uni(k.rel);
        M[c] = V.Mv + uni(k.mv) * RB;
        most = max(most, hi[c] - lo[c]);
    }
    for (int i0 = 0; i0 < most; i0 += RP * RG) {
        bits_t<T> v[CB * RG];
        const T* p[CB * RG];
        int yr[CB * RG];
        bool on[CB * RG];
        T x[CB * RG];
#pragma unroll
        for (int j = 0; j < CB * RG; ++j) {
            const int c = j / RG, at = lo[c] + i0 + RP * (j % RG);
            on[j] = at + ro < hi[c];
            p[j] = V.Mv;
            v[j] = 0;
            yr[j] = 0;
            if (at < hi[c]) {
                const int e = min(at + ro, hi[c] - 1);
                yr[j] = P.rel[rel[c] + e] - r0;
                p[j] = M[c] + (uint32_t)(e * RB + col);
                v[j] = peek(p[j]);
            }
        }
        settle_n<T, CB * RG>(v, p, on, x, ctl);
#pragma unroll
        for (int j = 0; j < CB * RG; ++j) {
            if (on[j]) Y[yr[j] * LR + col] += x[j];
            if (j % RG == RG - 1) wave_sync();
        }
    }
}
template <typename T, bool BLK, int RP>
__device__ __forceinline__ void gather(const DevPlan& P, const DevBSolve<T>& V, const Front& f, int blk, int r0, T* Y, int g,
                                       const Ctl& ctl) {
    if (f.chd1 - f.chd0 == 1) gather_pass<T, BLK, RP, 1, 8>(P, V, f.chd0, f.chd1, blk, r0, Y, g, ctl);
    else
        for (int q = f.chd0; q < f.chd1; q += 2) gather_pass<T, BLK, RP, 2, 4>(P, V, q, f.chd1, blk, r0, Y, g, ctl);
}

// ---- small fronts (nJ <= 64), one wavefront each ------------------------------
// Lane r keeps row r's sixteen values; the slab Y (64 rows) carries them to
// and from the row-by-row layout.

// What scale_panel returns, of a panel that it has scaled already (the
// diagonal keeps D).
template <typename T>
__device__ __forceinline__ void scaled_diagonal(int nn, int nj, const T* Ps, bool unit, T& d, T& rd, bool& exact) {
    const int rr = min((int)(threadIdx.x & 63), nn - 1);
    d = unit ? (T)1 : Ps[rr + rr * (nj | 1)];
    rd = (T)1 / d;
    exact = __any(abnormal(rd));
}

template <typename T>
__device__ __forceinline__ void store_rows(const T* Y, int r0, int rows, T* dst) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    for (int k = lk; k < rows; k += 4) publish(dst + (uint32_t)(k * RB + li), Y[(r0 + k) * LR + li]);
}

template <typename T>
__device__ void small_fwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, bool staged, T* Ps, T* Y,
                            const Ctl& ctl) {
    const int r = threadIdx.x & 63;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, ld = nj | 1;
    const bool unit = F.diag != 0;
    T y[RB];
    {
        const T* b = V.B + f.c0;
        const uint32_t rb = min(r, nn - 1);
#pragma unroll
        for (int c = 0; c < RB; ++c) y[c] = (b + (int64_t)min(c, V.ncol - 1) * V.ldb)[rb];
    }
#pragma unroll
    for (int c = 0; c < RB; ++c) {
        if (r >= nn || c >= V.ncol) y[c] = (T)0;
        Y[r * LR + c] = (T)0;
    }
    if (!staged) stage_panel(F.panel + f.poff, nj, nn, Ps);
    wave_sync();
    T d, rcp;
    bool exact;
    scale_panel(nj, nn, Ps, unit || staged, d, rcp, exact);
    if (staged) scaled_diagonal(nn, nj, Ps, unit, d, rcp, exact);
    gather<T, false, 4>(P, V, f, 0, 0, Y, 0, ctl);
    wave_sync();
#pragma unroll
    for (int c = 0; c < RB; ++c) y[c] += Y[r * LR + c];
    const int rr = min(r, nj - 1);
    for (int k = 0; k < nn; ++k) {
        const T l = -Ps[rr + k * ld];
        T yk[RB];
#pragma unroll
        for (int c = 0; c < RB; ++c) yk[c] = lane_of(y[c], k);
        if (r > k) {
#pragma unroll
            for (int c = 0; c < RB; ++c) y[c] = fma_(l, yk[c], y[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < RB; ++c) Y[r * LR + c] = (!unit && r < nn) ? quot(y[c], d, rcp, exact) : y[c];
    wave_sync();
    store_rows(Y, 0, nn, V.X + (int64_t)f.c0 * RB);
    store_rows(Y, nn, na, V.Mv + P.mvoff1[J] * RB);
}

template <typename T>
__device__ void small_bwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, bool staged, T* Ps, T* Y,
                            const Ctl& ctl) {
    const int r = threadIdx.x & 63, li = r & 15, lk = r >> 4;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, ld = nj | 1;
    const bool unit = F.diag != 0;
    const int32_t* rows = P.rows + f.rowoff + nn;
    // the right-hand side rows through the slab into lane r's registers
    const T* in = V.X + (int64_t)f.c0 * RB;
    T b[RB];
    const int rd = min(r, nn - 1);
#pragma unroll
    for (int c = 0; c < RB; ++c) b[c] = in[(uint32_t)(rd * RB + c)];
    const T dd = unit ? F.d[f.c0 + rd] : (T)1;
    if (!staged) stage_panel(F.panel + f.poff, nj, nn, Ps);
    wave_sync();
    T d, rcp;
    bool exact;
    scale_panel(nj, nn, Ps, unit || staged, d, rcp, exact);
    if (staged) scaled_diagonal(nn, nj, Ps, unit, d, rcp, exact);
    // separator part: -L21' x_sep, sixteen separator rows at a time
    v4_t<T> acc[4];
    zero<T>(acc);
    for (int q = 0; q < na; q += 16) {
        const T* p[4];
        bits_t<T> v[4];
        bool on[4];
        T x[4], a[16];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int e = q + 4 * s + lk;
            on[s] = e < na;
            p[s] = V.Z + ((int64_t)rows[min(e, na - 1)] * RB + li);
            v[s] = peek(p[s]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                a[4 * i + s] = 16 * i < nn ? -Ps[nn + min(q + 4 * s + lk, na - 1) + min(16 * i + li, nn - 1) * ld] : (T)0;
        settle_n<T, 4>(v, p, on, x, ctl);
        mma(a, x, acc, (nn + 15) >> 4);
    }
    put(acc, Y, 0);
    wave_sync();
    T y[RB];
#pragma unroll
    for (int c = 0; c < RB; ++c) {
        y[c] = unit ? b[c] / dd : quot(b[c], d, rcp, exact);
        y[c] += Y[r * LR + c];
    }
    for (int k = nn - 1; k > 0; --k) {
        const T l = -Ps[k + rd * ld];
        T xk[RB];
#pragma unroll
        for (int c = 0; c < RB; ++c) xk[c] = lane_of(y[c], k);
        if (r < k) {
#pragma unroll
            for (int c = 0; c < RB; ++c) y[c] = fma_(l, xk[c], y[c]);
        }
    }
    wave_sync();
#pragma unroll
    for (int c = 0; c < RB; ++c) Y[r * LR + c] = y[c];
    wave_sync();
    store_rows(Y, 0, nn, V.Z + (int64_t)f.c0 * RB);
    if (r < nn) {
        T* o = V.B + f.c0;
#pragma unroll
        for (int c = 0; c < RB; ++c)
            if (c < V.ncol) (o + (int64_t)c * V.ldb)[(uint32_t)r] = y[c];
    }
}

// ---- big fronts, one workgroup -----------------------------------------------

// Right-hand side rows [c0, c0 + rows) of this wavefront's row group g (the
// accumulator layout).
template <typename T>
__device__ __forceinline__ v4_t<T> rhs_group(const DevBSolve<T>& V, int c0, int rows, int g) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const T* b = V.B + (int64_t)min(li, V.ncol - 1) * V.ldb + c0;
    T w[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) w[v] = b[min(16 * g + Mfma<T>::row(lk, v), rows - 1)];
    v4_t<T> x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = (16 * g + Mfma<T>::row(lk, v) < rows && li < V.ncol) ? w[v] : (T)0;
    return x;
}
// acc[g] += x (g uniform, the array in registers)
template <typename T>
__device__ __forceinline__ void add_group(v4_t<T> (&acc)[4], const v4_t<T>& x, int g) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i == g) acc[i] += x;
}

// acc -= L(rows at base, blocks [0, nblk)) X, X read as the chain publishes it.
template <typename T>
__device__ __forceinline__ void left_sum(const T* base, int64_t nj, int rows, int nblk, int cols, const T* X, int g,
                                         v4_t<T> (&acc)[4], const Ctl& ctl) {
    if (nblk <= 0) return;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int groups = (rows + 15) >> 4;
    auto kb = [&](int ib) { return ib == nblk - 1 ? cols : NB; };
    auto at = [&](int ib, int s) {
        return X + (int64_t)ib * NB * RB + (uint32_t)(min(16 * g + 4 * s + lk, kb(ib) - 1) * RB + li);
    };
    T a0[16], a1[16];
    bits_t<T> x0[4], x1[4] = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) x0[s] = peek(at(0, s));
    load_a(base, nj, rows, kb(0), g, a0);
    auto step = [&](int ib, const T (&a)[16], bits_t<T> (&xv)[4], T (&an)[16], bits_t<T> (&xn)[4]) {
        if (ib + 1 < nblk) {
#pragma unroll
            for (int s = 0; s < 4; ++s) xn[s] = peek(at(ib + 1, s));
            load_a(base + (int64_t)(ib + 1) * NB * nj, nj, rows, kb(ib + 1), g, an);
        }
        const T* p[4];
        bool on[4];
        T x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            p[s] = at(ib, s);
            on[s] = 16 * g + 4 * s + lk < kb(ib);
        }
        settle_n<T, 4>(xv, p, on, x, ctl);
#pragma unroll
        for (int s = 0; s < 4; ++s) x[s] = -x[s];
        mma(a, x, acc, groups);
    };
    for (int ib = 0; ib < nblk; ib += 2) {
        step(ib, a0, x0, a1, x1);
        if (ib + 1 < nblk) step(ib + 1, a1, x1, a0, x0);
    }
}

// Sum over the wavefronts' parts of Red of this lane's four operand rows of
// slice g, rows 16 g + (4 s + lk, or 4 lk + s for the transposed order) < rows.
template <typename T, bool TR>
__device__ __forceinline__ void operand(const T* Red, int rows, int g, T (&x)[4]) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int row = 16 * g + (TR ? 4 * lk + s : 4 * s + lk);
        x[s] = row < rows ? sum4(Red, row, li) : (T)0;
    }
}

// The block's final rows (sum over the parts of Red), published row by row.
template <typename T>
__device__ __forceinline__ void publish_block(const T* Red, int rows, T* dst) {
    for (int e = threadIdx.x; e < rows * RB; e += 256) publish(dst + (uint32_t)e, sum4(Red, e >> 4, e & 15));
}

// Forward diagonal block [k0, k0 + kb) of a big front.
template <typename T>
__device__ void diag_fwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, int k0, int kb, T* Y,
                           T* Red, const Ctl& ctl) {
    const int g = uni((int)(threadIdx.x >> 6));
    const Front f = front_of(P, J);
    const int nj = f.nn + f.na;
    T wa[16];
    load_a(F.W + f.woff + k0, f.nn, kb, kb, g, wa);
    v4_t<T> acc[4];
    zero<T>(acc);
    add_group<T>(acc, rhs_group(V, f.c0 + k0, kb, g), g);
    for (int e = threadIdx.x; e < NB * LR; e += 256) Y[e] = (T)0;
    __syncthreads();
    gather<T, true, 16>(P, V, f, k0 / NB, k0, Y, g, ctl);
    left_sum(F.panel + f.poff + k0, nj, kb, k0 / NB, NB, V.X + (int64_t)f.c0 * RB, g, acc, ctl);
    put(acc, Red, g);
    __syncthreads();
    // the children's sums join one part
    for (int e = threadIdx.x; e < NB * RB; e += 256) Red[(e >> 4) * LR + (e & 15)] += Y[(e >> 4) * LR + (e & 15)];
    __syncthreads();
    T x[4];
    operand<T, false>(Red, kb, g, x);
    zero<T>(acc);
    mma(wa, x, acc, (kb + 15) >> 4);
    put(acc, Y, g);
    __syncthreads();
    publish_block(Y, kb, V.X + (int64_t)(f.c0 + k0) * RB);
}

// Forward update rows [r0, r1) (>= nn) of a big front.
template <typename T>
__device__ void rows_fwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, int r0, int r1, T* Y,
                           T* Red, const Ctl& ctl) {
    const int g = uni((int)(threadIdx.x >> 6));
    const Front f = front_of(P, J);
    const int nn = f.nn, nj = nn + f.na, m = r1 - r0, p = (nn + NB - 1) / NB;
    v4_t<T> acc[4];
    zero<T>(acc);
    for (int e = threadIdx.x; e < NB * LR; e += 256) Y[e] = (T)0;
    __syncthreads();
    gather<T, true, 16>(P, V, f, p + (r0 - nn) / NB, r0, Y, g, ctl);
    left_sum(F.panel + f.poff + r0, nj, m, p, nn - (p - 1) * NB, V.X + (int64_t)f.c0 * RB, g, acc, ctl);
    put(acc, Red, g);
    __syncthreads();
    T* dst = V.Mv + (P.mvoff1[J] + (r0 - nn)) * RB;
    for (int e = threadIdx.x; e < m * RB; e += 256)
        publish(dst + (uint32_t)e, sum4(Red, e >> 4, e & 15) + Y[(e >> 4) * LR + (e & 15)]);
}

// A whole big front of one diagonal block and at most VT_ROWBLOCKS row
// blocks, forward: wavefront g takes row block g.
template <typename T>
__device__ void front_fwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, T* Y, T* Red,
                            const Ctl& ctl) {
    const int lane = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6)), li = lane & 15, lk = lane >> 4;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, m = min(NB, na - NB * g), groups = (nn + 15) >> 4;
    T wa[16], la[16];
    load_a(F.W + f.woff, nn, nn, nn, g, wa);
    const T* Lg = F.panel + f.poff + nn + NB * min(g, max(na - 1, 0) / NB);
    if (m > 0) load_a(Lg, nj, m, nn, 0, la);
    const v4_t<T> b = rhs_group(V, f.c0, nn, g);
    for (int e = threadIdx.x; e < VROWS * LR; e += 256) Y[e] = (T)0;
    __syncthreads();
    gather<T, false, 16>(P, V, f, 0, 0, Y, g, ctl);
    __syncthreads();
    v4_t<T> acc[4];
    if (16 * g < nn) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = 16 * g + Mfma<T>::row(lk, v);
            if (row < nn) Y[row * LR + li] += b[v];
        }
        wave_sync();
        T x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int row = 16 * g + 4 * s + lk;
            x[s] = row < nn ? Y[row * LR + li] : (T)0;
        }
        zero<T>(acc);
        mma(wa, x, acc, groups);
        put(acc, Red, g);
    } else {
        for (int e = lane; e < NB * LR; e += 64) Red[NB * LR * g + e] = (T)0;
    }
    __syncthreads();
    publish_block(Red, nn, V.X + (int64_t)f.c0 * RB);
    if (m > 0) {
        zero<T>(acc);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * i + Mfma<T>::row(lk, v);
                acc[i][v] = row < m ? Y[(nn + NB * g + row) * LR + li] : (T)0;
            }
        for (int c = 0; 16 * c < nn; ++c) {
            if (c > 0) load_a(Lg, nj, m, nn, c, la);
            T x[4];
            operand<T, false>(Red, nn, c, x);
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = -x[s];
            mma(la, x, acc, (m + 15) >> 4);
        }
        mma_done<T>(acc);
        T* dst = V.Mv + (P.mvoff1[J] + NB * g) * RB;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * i + Mfma<T>::row(lk, v);
                if (row < m) publish(dst + (uint32_t)(row * RB + li), acc[i][v]);
            }
    }
}

// Transposed sums: acc -= L(rows, block k0)' x(rows) over row tiles of the
// panel, tile u covering panel rows [row0(u), min(row0(u) + 64, lim(u))); the
// wavefront takes rows 16 g .. 16 g + 15 of every tile.
template <typename T, typename R0, typename LIM>
__device__ __forceinline__ void sweep(const T* Pk, int64_t nj, int kb, const int32_t* rows, const T* Z, int g, int nu,
                                      R0 row0, LIM lim, v4_t<T> (&acc)[4], const Ctl& ctl) {
    if (nu <= 0) return;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int groups = (kb + 15) >> 4;
    auto ptrs = [&](int u, const T* (&p)[4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            p[s] = Z + ((int64_t)rows[min(row0(u) + 16 * g + 4 * lk + s, lim(u) - 1)] * RB + li);
    };
    auto tile = [&](int u, T (&a)[16]) { load_at(Pk + row0(u), nj, min(NB, lim(u) - row0(u)), kb, g, a); };
    T a0[16], a1[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) a0[j] = a1[j] = (T)0;
    const T *p0[4], *p1[4];
    bits_t<T> x0[4], x1[4] = {0, 0, 0, 0};
    ptrs(0, p0);
    ptrs(min(1, nu - 1), p1);
#pragma unroll
    for (int s = 0; s < 4; ++s) x0[s] = peek(p0[s]);
    tile(0, a0);
    auto step = [&](int u, const T (&a)[16], const T* (&p)[4], bits_t<T> (&xv)[4], T (&an)[16], const T* (&pn)[4],
                    bits_t<T> (&xn)[4]) {
        if (u + 1 < nu) {
#pragma unroll
            for (int s = 0; s < 4; ++s) xn[s] = peek(pn[s]);
            tile(u + 1, an);
        }
        bool on[4];
        T x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) on[s] = row0(u) + 16 * g + 4 * lk + s < lim(u);
        settle_n<T, 4>(xv, p, on, x, ctl);
        if (u + 2 < nu) ptrs(u + 2, p);
#pragma unroll
        for (int s = 0; s < 4; ++s) x[s] = -x[s];
        mma(a, x, acc, groups);
    };
    for (int u = 0; u < nu; u += 2) {
        step(u, a0, p0, x0, a1, p1, x1);
        if (u + 1 < nu) step(u + 1, a1, p1, x1, a0, p0, x0);
    }
}

// Backward separator product of diagonal block [k0, k0 + kb) over the
// separator tiles [t0, t1): the partial slot of the chunk.
template <typename T>
__device__ void sep_bwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, int k0, int t0, int t1,
                          T* Red, const Ctl& ctl) {
    const int g = uni((int)(threadIdx.x >> 6));
    const Front f = front_of(P, J);
    const int nn = f.nn, nj = nn + f.na, kb = min(NB, nn - k0);
    const int nsep = (f.na + NB - 1) / NB, nchk = (nsep + SEP_TILES - 1) / SEP_TILES;
    v4_t<T> acc[4];
    zero<T>(acc);
    sweep(F.panel + f.poff + (int64_t)k0 * nj, nj, kb, P.rows + f.rowoff, V.Z, g, t1 - t0,
          [&](int u) { return nn + NB * (t1 - 1 - u); }, [&](int) { return nj; }, acc, ctl);
    put(acc, Red, g);
    __syncthreads();
    publish_block(Red, kb, V.Mv + (P.sboff1[J] + (int64_t)((k0 / NB) * nchk + t0 / SEP_TILES) * NB) * RB);
}

// Backward diagonal block [k0, k0 + kb): y = C_k - L21' x_sep - sum_{ib > k}
// L_{ib,k}' X_ib (separator tiles first, farthest ancestors first, then the
// chain), X_k = W_k' y.
template <typename T>
__device__ void diag_bwd16(const DevPlan& P, const DevFactor<T>& F, const DevBSolve<T>& V, int J, int k0, int kb, T* Red,
                           T* Red2, const Ctl& ctl) {
    const int lane = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6)), li = lane & 15, lk = lane >> 4;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, p = (nn + NB - 1) / NB, kblk = k0 / NB, nch = p - 1 - kblk;
    const int nsep = (na + NB - 1) / NB, nchk = (nsep + SEP_TILES - 1) / SEP_TILES;
    const int64_t sb = P.sboff1[J];
    T wa[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) wa[j] = (T)0;
    load_at(F.W + f.woff + k0, f.nn, kb, kb, g, wa);
    v4_t<T> acc[4];
    zero<T>(acc);
    {
        // the right-hand side rows of row group g
        const T* in = V.X + (int64_t)(f.c0 + k0) * RB;
        v4_t<T> b;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = min(16 * g + Mfma<T>::row(lk, v), kb - 1);
            b[v] = in[(uint32_t)(row * RB + li)];
            if (F.diag != 0) b[v] /= F.d[f.c0 + k0 + row];
        }
        add_group<T>(acc, b, g);
    }
    const int ns = sb >= 0 ? 0 : nsep;
    sweep(F.panel + f.poff + (int64_t)k0 * nj, nj, kb, P.rows + f.rowoff, V.Z, g, ns + nch,
          [&](int u) { return u < ns ? nn + NB * (ns - 1 - u) : NB * (p - 1 - (u - ns)); },
          [&](int u) { return u < ns ? nj : nn; }, acc, ctl);
    mma_done<T>(acc);
    if (sb >= 0) {
        // the front's separator tasks: their partials, chunk c by wavefront c mod 4
        const T* slot = V.Mv + (sb + (int64_t)kblk * nchk * NB) * RB;
        for (int c = g; c < nchk; c += 4) {
            const T* sl = slot + (int64_t)c * NB * RB;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (16 * i >= kb) break;
                const T* q[4];
                bits_t<T> v[4];
                bool on[4];
                T x[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int row = 16 * i + Mfma<T>::row(lk, s);
                    on[s] = row < kb;
                    q[s] = sl + (uint32_t)(min(row, kb - 1) * RB + li);
                    v[s] = peek(q[s]);
                }
                settle_n<T, 4>(v, q, on, x, ctl);
#pragma unroll
                for (int s = 0; s < 4; ++s) acc[i][s] += x[s];
            }
        }
    }
    put(acc, Red, g);
    __syncthreads();
    T x[4];
    operand<T, true>(Red, kb, g, x);
    zero<T>(acc);
    mma(wa, x, acc, (kb + 15) >> 4);
    put(acc, Red2, g);
    __syncthreads();
    publish_block(Red2, kb, V.Z + (int64_t)(f.c0 + k0) * RB);
    if (lane < kb)
        for (int c = g; c < V.ncol; c += 4) (V.B + f.c0 + k0 + (int64_t)c * V.ldb)[(uint32_t)lane] = sum4(Red2, lane, c);
}

// LDS of a workgroup: small panels and the four slabs, or a one-task front's
// rows and the wavefronts' sums.
template <typename T>
union BLds {
    struct {
        T panel[VT_PANELS];
        T slab[4 * NB * LR];
    } s;
    struct {
        T Y[VROWS * LR];
        T Red[4 * NB * LR];
    } b;
};

// GROUP: a ticket covers V0.group blocks of a unit's tasks, one after the
// other (a small front's panel is staged and scaled for the first of them).
// One block a ticket / groups of up to four, us: 30000 systems of order 3, 33
// and 100 columns 616 / 475 and 1387 / 1036, 1500 of order 60 572 / 440 and
// 1306 / 1002, 2000 small grids, 33 and 75 columns 699 / 580 and 1148 / 974.
template <typename T, bool FWD, bool GROUP>
__global__ __launch_bounds__(256, 2) void k_bsolve16(DevPlan P, DevFactor<T> F, DevBSolve<T> V0) {
    static_assert(VROWS >= 4 * NB, "the second set of partial sums in Y");
    __shared__ BLds<T> S;
    __shared__ uint32_t s_tick;
    const int tid = threadIdx.x, g = uni(tid >> 6);
    const Ctl ctl{F.hang, V0.ticket, F.stall};
    const int nblk = (V0.nrhs + RB - 1) / RB, per = GROUP ? V0.group : 1;
    const uint32_t ngrp = (nblk + per - 1) / per, tickets = (uint32_t)V0.nunit * ngrp;
    for (;;) {
        if (tid == 0) s_tick = atomicAdd(V0.ticket, 1u);
        __syncthreads();
        const uint32_t tick = uni((int32_t)s_tick);
        if (tick >= tickets) break;
        const uint32_t u = tick / ngrp;
        const int blk0 = (int)(tick - u * ngrp) * per, blk1 = GROUP ? min(nblk, blk0 + per) : blk0 + 1;
        auto block = [&](int blk) {
            DevBSolve<T> V = V0;
            V.B += (int64_t)blk * RB * V.ldb;
            V.ncol = min(RB, V.nrhs - blk * RB);
            V.X += (int64_t)blk * RB * P.n;
            V.Z += (int64_t)blk * RB * P.n;
            V.Mv += (int64_t)blk * RB * V.mvs;
            return V;
        };
        const int t1 = V0.unit[u + 1];
        for (int t = V0.unit[u]; t < t1; ++t) {
            const unsigned long long t_begin = (V0.trace && tid == 0) ? wall_clock64() : 0;
            const VTask tk = V0.task[t];
            if (tk.kind == VT_SMALL) {
                const int J = uni(g == 0 ? tk.a : g == 1 ? tk.b : g == 2 ? tk.c : tk.d);
                const int o = uni(g == 0 ? 0 : g == 1 ? (tk.o12 & 0xffff) : g == 2 ? (int)((uint32_t)tk.o12 >> 16) : tk.o3);
                for (int blk = blk0; blk < blk1 && J >= 0; ++blk) {
                    const DevBSolve<T> V = block(blk);
                    if (FWD) small_fwd16(P, F, V, J, GROUP && blk > blk0, S.s.panel + o, S.s.slab + g * NB * LR, ctl);
                    else small_bwd16(P, F, V, J, GROUP && blk > blk0, S.s.panel + o, S.s.slab + g * NB * LR, ctl);
                }
            } else {
                for (int blk = blk0; blk < blk1; ++blk) {
                    const DevBSolve<T> V = block(blk);
                    if (GROUP && blk > blk0) __syncthreads();  // the LDS of the block before is free
                    if (FWD) {
                        if (tk.kind == VT_FRONT) front_fwd16(P, F, V, uni(tk.a), S.b.Y, S.b.Red, ctl);
                        else if (tk.kind == VT_DIAG) diag_fwd16(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.b.Y, S.b.Red, ctl);
                        else rows_fwd16(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.b.Y, S.b.Red, ctl);
                    } else {
                        if (tk.kind == VT_SEPB) sep_bwd16(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), uni(tk.d), S.b.Red, ctl);
                        else diag_bwd16(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.b.Red, S.b.Y, ctl);
                    }
                }
            }
            if (V0.trace && tid == 0) {  // (the last block's clocks stay)
                V0.trace[2 * tk.t0] = t_begin | ((unsigned long long)blockIdx.x << 48);
                V0.trace[2 * tk.t0 + 1] = wall_clock64();
            }
            __syncthreads();  // the LDS of this task is free; every thread has read s_tick
        }
    }
}

// The values that a solve's workgroups wait for, unset; both tickets 0.
template <typename T>
__global__ __launch_bounds__(256) void k_binit(bits_t<T>* XZ, int64_t n, bits_t<T>* Mv, int64_t m, uint32_t* ticket) {
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, st = (int64_t)gridDim.x * blockDim.x;
    if (i0 < 2) ticket[i0] = 0u;
    for (int64_t i = i0; i < n; i += st) XZ[i] = unset<T>();
    for (int64_t i = i0; i < m; i += st) Mv[i] = unset<T>();
}

}  // namespace

template <typename T>
void launch_solve16(const DevPlan& P, const DevFactor<T>& F, T* B, int64_t ldb, int nrhs, T* XZ, T* Mv, int64_t mvs,
                    const DevVPlan& D, unsigned long long* trace, int64_t ntrace_f, hipStream_t s) {
    if (D.nfu <= 0) return;
    const int64_t nblk = (nrhs + RB - 1) / RB, cols = nblk * RB, half = (int64_t)P.n * cols;
    const int64_t blocks = (std::max<int64_t>(mvs, 2 * (int64_t)P.n) * cols + 1023) / 1024;
    hipLaunchKernelGGL((k_binit<T>), dim3((unsigned)std::min<int64_t>(blocks, 4096)), dim3(256), 0, s, (bits_t<T>*)XZ, 2 * half,
                       (bits_t<T>*)Mv, mvs * cols, F.ticket);
    // blocks a ticket: several where the plan's tasks fill the chip by themselves
    // (HostPlan::vgroup) and many tickets are left all the same
    const int64_t group = D.group ? std::max<int64_t>(1, std::min<int64_t>({nblk, 4, nblk * D.nfu / 1024})) : 1;
    DevBSolve<T> V{B, XZ, XZ + half, Mv, ldb, mvs, nrhs, 0, (int32_t)group, D.ftask, D.funit, D.nfu, D.chd, F.ticket, trace};
    auto grid = [&](int64_t units) { return dim3((unsigned)std::min<int64_t>(units * ((nblk + group - 1) / group), 512)); };
    auto run = [&](auto fwd, int64_t units) {
        constexpr bool FWD = decltype(fwd)::value;
        if (group > 1) hipLaunchKernelGGL((k_bsolve16<T, FWD, true>), grid(units), dim3(256), 0, s, P, F, V);
        else hipLaunchKernelGGL((k_bsolve16<T, FWD, false>), grid(units), dim3(256), 0, s, P, F, V);
    };
    run(std::true_type(), D.nfu);
    V.task = D.btask;
    V.unit = D.bunit;
    V.nunit = D.nbu;
    V.ticket = F.ticket + 1;
    V.trace = trace ? trace + 2 * ntrace_f : nullptr;
    run(std::false_type(), D.nbu);
}

template void launch_solve16<double>(const DevPlan&, const DevFactor<double>&, double*, int64_t, int, double*, double*,
                                     int64_t, const DevVPlan&, unsigned long long*, int64_t, hipStream_t);
template void launch_solve16<float>(const DevPlan&, const DevFactor<float>&, float*, int64_t, int, float*, float*, int64_t,
                                    const DevVPlan&, unsigned long long*, int64_t, hipStream_t);

}  // namespace mf
