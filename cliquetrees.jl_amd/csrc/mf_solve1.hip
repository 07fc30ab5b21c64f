// mf_solve1.hip — gfx950 kernels of the supernodal triangular solves for few
// right-hand sides, column by column (mf_solve16.hip takes more than the plan
// says, HostPlan::vcols).
//
// Per-front recurrences of divide.jl:417-659, 864-1038, one persistent launch
// per direction.  With one column the solves are bound
// by latency: the chain of diagonal blocks up the root path and the hand-off
// between workgroups at each of its links.  Three things differ from the
// blocked kernels because of that:
//
//  * The data is its own flag.  Every element that another workgroup of the
//    launch waits for (the solution, the update vectors, the separator
//    partials) starts as a signalling NaN that no arithmetic returns, and the
//    consumer reads the element itself until it has changed.  Against a
//    counter published after the stores have drained and read before the data
//    is fetched, a hand-off takes one trip to memory in place of two
//    (0.54 us a link against 1.09, 200 links of 64 doubles).  There is no
//    counter per front and nothing to clear but the values.
//  * Products run on the vector units: one 64 x 64 tile times a vector is 16
//    fused multiply-adds a thread (about 150 cycles, the operand broadcast
//    inside 16 lanes by DPP, no LDS), where the matrix instructions spend
//    1024 cycles a wavefront on 16 columns of which one is wanted.
//  * Everything a task needs that does not come from another task of the
//    launch (factor tiles, inverses, index lists) is loaded before the task
//    waits.
//
// A ticket of the launch's counter costs 11.5 ns whatever runs (the counter
// is one address in memory), so tickets are a bound of their own when tasks
// are short: up to four small fronts share a task, a front of one diagonal
// block and at most four row blocks is one task, and in the middle of a long
// list one ticket covers up to four tasks.
//
// Several columns are independent solves that share the launch (the ticket
// order is unit by unit, the columns of a unit side by side).
//
// Both directions with the permutations, us, 1 / 3 / 4 / 6 / 8 columns, and
// mf_solve16.hip for up to 16 (its time hardly depends on the columns); with
// per-front counters and matrix instructions for one column before:
//   56 x 60 x 52 grid, n 174720   867 / 1350 / 1650 / 2290 / 2900   2030   (2237)
//   31 x 29 x 27 grid, n 24273    179 /  241 /  278 /  360 /  439    415   (670)
//   100 x 100 grid, n 10000       120 /  163 /  191 /  249 /  307    270   (390)
// The planner places the line between the two by the plan (solve_columns).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mf_kernels.h"
#include "mf_vsolve.h"

namespace mf {

namespace {

// s0 + s1 += sum over j < 16 of a[j] * (lane j of each row of sixteen lanes of x).
__device__ __forceinline__ void fma16(double& s0, double& s1, double x, const double (&a)[16]) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %2, %3 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %4 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %5 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %6 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %7 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %8 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %9 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %10 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %11 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %12 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %13 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %14 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %15 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %16 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %18 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "+v"(s0), "+v"(s1)
        : "v"(x), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
          "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]), "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15]));
}
__device__ __forceinline__ void fma16(float& s0, float& s1, float x, const float (&a)[16]) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %2, %3 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %4 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %5 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %6 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %7 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %8 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %9 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %10 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %11 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %12 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %13 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %14 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %15 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %16 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %2, %18 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "+v"(s0), "+v"(s1)
        : "v"(x), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
          "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]), "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15]));
}

// Children's update vectors added into Yw (this wavefront's own rows), the
// children q0, q0 + dq, ... of f, four in flight.  BLK: the entries landing
// in row block `blk` of the front, at Yw[rel - r0]; else entries [64 ch,
// 64 ch + 64) of every child, at Yw[rel].
template <typename T, bool BLK>
__device__ __forceinline__ void gather(const DevPlan& P, const DevVSolve<T>& V, const Front& f, int blk, int r0, int q0,
                                       int dq, int ch, T* Yw, const Ctl& ctl) {
    const int lane = threadIdx.x & 63;
    for (int q = f.chd0 + q0; q < f.chd1; q += 4 * dq) {
        const T* p[4];
        bits_t<T> v[4];
        int yr[4];
        bool on[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i > 0 && q + i * dq >= f.chd1) {
                p[i] = p[0];
                v[i] = 0;
                yr[i] = 0;
                on[i] = false;
                continue;
            }
            const VChild k = V.chd[q + i * dq];
            int lo = 64 * ch, hi = k.ma;
            if (BLK) {
                lo = P.sgstart[k.sg + blk];
                hi = P.sgstart[k.sg + blk + 1];
            }
            on[i] = lo + lane < hi;
            const int e = on[i] ? lo + lane : 0;
            yr[i] = P.rel[k.rel + e] - (BLK ? r0 : 0);
            p[i] = V.Mv + k.mv + e;
            v[i] = peek(p[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i > 0 && q + i * dq >= f.chd1) break;
            const T x = settle(v[i], p[i], on[i], ctl);
            if (on[i]) Yw[yr[i]] += x;
            wave_sync();
        }
    }
}

template <typename T>
__device__ void small_fwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, T* Ps, T* Yw,
                           const Ctl& ctl) {
    const int r = threadIdx.x & 63;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, ld = nj | 1;
    const bool unit = F.diag != 0;
    const T b = V.in[f.c0 + min(r, nn - 1)];
    Yw[r] = (T)0;
    stage_panel(F.panel + f.poff, nj, nn, Ps);
    wave_sync();
    T d, rcp;
    bool exact;
    scale_panel(nj, nn, Ps, unit, d, rcp, exact);
    gather<T, false>(P, V, f, 0, 0, 0, 1, 0, Yw, ctl);
    wave_sync();
    T y = Yw[r] + (r < nn ? b : (T)0);
    const int rr = min(r, nj - 1);
    for (int k = 0; k < nn; ++k) {
        const T l = Ps[rr + k * ld], yk = lane_of(y, k);
        if (r > k) y = fma_(-l, yk, y);
    }
    if (!unit && r < nn) y = quot(y, d, rcp, exact);
    if (r < nn) {
        publish(V.out + f.c0 + r, y);
        wipe(V.wipe + f.c0 + r);
    } else if (r < nj) {
        publish(V.Mv + P.mvoff1[J] + (r - nn), y);
    }
}

template <typename T>
__device__ void small_bwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, T* Ps, T* Yw,
                           const Ctl& ctl) {
    const int r = threadIdx.x & 63;
    const Front f = front_of(P, J);
    const int nn = f.nn, nj = nn + f.na, ld = nj | 1;
    const bool unit = F.diag != 0;
    const int rr = min(r, nj - 1), rd = min(r, nn - 1);
    const T* px = V.out + P.rows[f.rowoff + rr];
    bits_t<T> xv = peek(px);
    T y = V.in[f.c0 + rd];
    if (unit) y /= F.d[f.c0 + rd];
    stage_panel(F.panel + f.poff, nj, nn, Ps);
    wave_sync();
    T d, rcp;
    bool exact;
    scale_panel(nj, nn, Ps, unit, d, rcp, exact);
    if (!unit) y = quot(y, d, rcp, exact);
    // separator part: the sixteen values of a group from LDS, broadcast by DPP
    const T x = settle(xv, px, r >= nn && r < nj, ctl);
    Yw[r] = x;
    wave_sync();
    T s0 = (T)0, s1 = (T)0;
    // (without separator rows the stand-in row would be the last diagonal
    // entry's, and an infinite one times 0 is not 0)
    for (int q = nj > nn ? nn & ~15 : nj; q < nj; q += 16) {
        T a[16];
        const T xq = Yw[q + (r & 15)];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = q + j;
            a[j] = -Ps[min(max(i, nn), nj - 1) + rd * ld];
        }
        fma16(s0, s1, xq, a);
    }
    y += s0 + s1;
    for (int k = nn - 1; k > 0; --k) {
        const T l = Ps[k + rd * ld], xk = lane_of(y, k);
        if (r < k) y = fma_(-l, xk, y);
    }
    if (r < nn) publish(V.out + f.c0 + r, y);
}

// ---- big fronts, one workgroup -----------------------------------------------
// Thread (r, g): r = lane, g = wavefront.  A 64 x 64 tile A times a vector x
// is sum over g of A[r][16 g + j] x[16 g + j], j < 16, each wavefront taking
// its sixteen columns; the four partial sums meet in LDS (Red) at the end of
// a task's sums.

// The loaders take no sign and mask nothing: rows and columns outside the
// tile repeat its last ones, the products' x is 0 there or their sum unused.
// Column addresses are uniform (scalar registers, one lane offset).

// a[j] = base[r + (16 g + j) ld], r < rows, 16 g + j < cols
template <typename T>
__device__ __forceinline__ void load_cols(const T* base, int64_t ld, int rows, int cols, int g, T (&a)[16]) {
    const uint32_t r = min((int)(threadIdx.x & 63), rows - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = (base + (int64_t)min(16 * g + j, cols - 1) * ld)[r];
}
// a[j] = base[(16 g + j) + c ld], c = lane < cols, 16 g + j < rows (the transposed product)
template <typename T>
__device__ __forceinline__ void load_rows(const T* base, int64_t ld, int rows, int cols, int g, T (&a)[16]) {
    const uint32_t c = (uint32_t)min((int)(threadIdx.x & 63), cols - 1) * (uint32_t)ld;
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = (base + min(16 * g + j, rows - 1))[c];
}

constexpr int VROWS = NB + NB * VT_ROWBLOCKS;  // rows of a one-task front

// Sum over the four wavefronts' rows of Red (leading dimension VROWS).
template <typename T>
__device__ __forceinline__ T sum4(const T* Red, int i) {
    return (Red[i] + Red[VROWS + i]) + (Red[2 * VROWS + i] + Red[3 * VROWS + i]);
}

// s0 + s1 += -L(rows base.., blocks [0, nblk)) X, X read as the chain
// publishes it: the tile and the block of X of the next step load while this
// step's are awaited and multiplied.  cols: columns of the last block.
template <typename T>
__device__ __forceinline__ void left_sum(const T* base, int64_t nj, int rows, int nblk, int cols, const T* X, int g,
                                         T& s0, T& s1, const Ctl& ctl) {
    if (nblk <= 0) return;
    const int li = threadIdx.x & 15;
    auto kb = [&](int ib) { return ib == nblk - 1 ? cols : NB; };
    auto at = [&](int ib) { return X + ib * NB + min(16 * g + li, kb(ib) - 1); };
    T a0[16], a1[16];
    bits_t<T> x0 = peek(at(0)), x1 = 0;
    load_cols(base, nj, rows, kb(0), g, a0);
    auto step = [&](int ib, const T (&a)[16], bits_t<T> xv, T (&an)[16], bits_t<T>& xn) {
        if (ib + 1 < nblk) {
            xn = peek(at(ib + 1));
            load_cols(base + (int64_t)(ib + 1) * NB * nj, nj, rows, kb(ib + 1), g, an);
        }
        const T x = -settle(xv, at(ib), 16 * g + li < kb(ib), ctl);
        fma16(s0, s1, x, a);
    };
    for (int ib = 0; ib < nblk; ib += 2) {
        step(ib, a0, x0, a1, x1);
        if (ib + 1 < nblk) step(ib + 1, a1, x1, a0, x0);
    }
}

// Forward diagonal block [k0, k0 + kb) of a big front.
template <typename T>
__device__ void diag_fwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, int k0, int kb, T* Y,
                          T* Red, const Ctl& ctl) {
    const int r = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6)), li = r & 15;
    const Front f = front_of(P, J);
    const int nj = f.nn + f.na;
    const T* Pj = F.panel + f.poff;
    T wa[16];
    load_cols(F.W + f.woff + k0, f.nn, kb, kb, g, wa);
    const T b = g == 0 && r < kb ? V.in[f.c0 + k0 + r] : (T)0;
    T* Yw = Y + g * VROWS;
    Yw[r] = (T)0;
    wave_sync();
    gather<T, true>(P, V, f, k0 / NB, k0, g, 4, 0, Yw, ctl);
    wave_sync();
    T s0 = Yw[r] + b, s1 = (T)0;
    left_sum(Pj + k0, nj, kb, k0 / NB, NB, V.out + f.c0, g, s0, s1, ctl);
    Red[g * VROWS + r] = s0 + s1;
    __syncthreads();
    T t0 = (T)0, t1 = (T)0;
    fma16(t0, t1, 16 * g + li < kb ? sum4(Red, 16 * g + li) : (T)0, wa);
    Y[g * VROWS + r] = t0 + t1;
    __syncthreads();
    if (g == 0 && r < kb) {
        publish(V.out + f.c0 + k0 + r, sum4(Y, r));
        wipe(V.wipe + f.c0 + k0 + r);
    }
}

// Forward update rows [r0, r1) (>= nn) of a big front: M2 = gather - L21 X.
template <typename T>
__device__ void rows_fwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, int r0, int r1, T* Y,
                          T* Red, const Ctl& ctl) {
    const int r = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6));
    const Front f = front_of(P, J);
    const int nn = f.nn, nj = nn + f.na, m = r1 - r0, p = (nn + NB - 1) / NB;
    T* Yw = Y + g * VROWS;
    Yw[r] = (T)0;
    wave_sync();
    gather<T, true>(P, V, f, p + (r0 - nn) / NB, r0, g, 4, 0, Yw, ctl);
    wave_sync();
    T s0 = Yw[r], s1 = (T)0;
    left_sum(F.panel + f.poff + r0, nj, m, p, nn - (p - 1) * NB, V.out + f.c0, g, s0, s1, ctl);
    Red[g * VROWS + r] = s0 + s1;
    __syncthreads();
    if (g == 0 && r < m) publish(V.Mv + P.mvoff1[J] + (r0 - nn) + r, sum4(Red, r));
}

// A whole big front of one diagonal block and at most VT_ROWBLOCKS row
// blocks, forward: wavefront g takes row block g.
template <typename T>
__device__ void front_fwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, T* Y, T* Red,
                           const Ctl& ctl) {
    const int r = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6)), li = r & 15;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, m = min(NB, na - NB * g);
    T wa[16], la[2][16];
    load_cols(F.W + f.woff, nn, nn, nn, g, wa);
    const T* Lg = F.panel + f.poff + nn + NB * min(g, (na - 1) / NB);
    if (m > 0) {
        load_cols(Lg, nj, m, nn, 0, la[0]);
        if (nn > 16) load_cols(Lg, nj, m, nn, 1, la[1]);
    }
    const T b = V.in[f.c0 + min(16 * g + li, nn - 1)];
    T* Yw = Y + g * VROWS;
    for (int e = r; e < VROWS; e += 64) Yw[e] = (T)0;
    wave_sync();
    for (int ch = g; ch * 64 < nj; ch += 4) gather<T, false>(P, V, f, 0, 0, 0, 1, ch, Yw, ctl);
    __syncthreads();
    if (16 * g < nn) {
        T t0 = (T)0, t1 = (T)0;
        fma16(t0, t1, 16 * g + li < nn ? sum4(Y, 16 * g + li) + b : (T)0, wa);
        Red[g * VROWS + r] = t0 + t1;
    } else {
        Red[g * VROWS + r] = (T)0;
    }
    T acc = m > 0 ? sum4(Y, nn + NB * g + r) : (T)0;
    __syncthreads();
    if (g == 0 && r < nn) {
        publish(V.out + f.c0 + r, sum4(Red, r));
        wipe(V.wipe + f.c0 + r);
    }
    if (m > 0) {
        T s1 = (T)0;
        auto x = [&](int c) { return 16 * c + li < nn ? -sum4(Red, 16 * c + li) : (T)0; };
        fma16(acc, s1, x(0), la[0]);
        if (nn > 16) fma16(acc, s1, x(1), la[1]);
        for (int c = 2; 16 * c < nn; ++c) {
            load_cols(Lg, nj, m, nn, c, la[0]);
            fma16(acc, s1, x(c), la[0]);
        }
        if (r < m) publish(V.Mv + P.mvoff1[J] + NB * g + r, acc + s1);
    }
}

// Transposed sums: -L(rows, block k0)' x(rows) over row tiles of the panel,
// x in the tile's lanes, sixteen columns a wavefront, the loads coalesced
// along the rows and the lanes' partial sums kept apart until the end.  A
// block of kb <= 16 (32) columns is one (two) column groups; the wavefronts
// then split the tiles.  Tile u covers panel rows [row0(u), min(row0(u) + 64,
// lim(u))).
struct ColSplit {
    int ng, ci, sp, ns;  // column groups, this wavefront's group and split, splits
    __device__ __forceinline__ ColSplit(int kb, int g) {
        ng = kb <= 16 ? 1 : kb <= 32 ? 2 : 4;
        ns = 4 / ng;
        ci = g & (ng - 1);
        sp = g / ng;
    }
};
template <typename T, typename R0, typename LIM>
__device__ __forceinline__ void sweep(const T* Pk, int64_t nj, int kb, const int32_t* rows, const T* X, const ColSplit& cs,
                                      int nu, R0 row0, LIM lim, T (&acc)[16], const Ctl& ctl) {
    if (nu <= 0) return;
    const int lane = threadIdx.x & 63;
    const int c0 = 16 * cs.ci;
    auto idx = [&](int u) { return rows[min(row0(u) + lane, lim(u) - 1)]; };
    auto tile = [&](int u, T (&a)[16]) {
        const uint32_t r = min(row0(u) + lane, lim(u) - 1);
        const T* q = Pk + (int64_t)c0 * nj;
#pragma unroll
        for (int j4 = 0; j4 < 16; j4 += 4)
            if (c0 + j4 < kb) {
#pragma unroll
                for (int j = j4; j < j4 + 4; ++j) a[j] = (q + (int64_t)min(j, kb - 1 - c0) * nj)[r];
            }
    };
    T a0[16], a1[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) a0[j] = a1[j] = (T)0;
    int i1 = nu > 1 ? idx(1) : 0;
    const T *p0 = X + idx(0), *p1 = p0;
    bits_t<T> x0 = peek(p0), x1 = 0;
    tile(0, a0);
    auto step = [&](int u, const T (&a)[16], const T* p, bits_t<T> xv, T (&an)[16], const T*& pn, bits_t<T>& xn) {
        if (u + 1 < nu) {
            pn = X + i1;
            xn = peek(pn);
            tile(u + 1, an);
            if (u + 2 < nu) i1 = idx(u + 2);
        }
        const T x = -settle(xv, p, row0(u) + lane < lim(u), ctl);
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = fma_(a[j], x, acc[j]);
    };
    for (int u = 0; u < nu; u += 2) {
        step(u, a0, p0, x0, a1, p1, x1);
        if (u + 1 < nu) step(u + 1, a1, p1, x1, a0, p0, x0);
    }
}
// The lanes' partial sums of a sweep, transposed through R (64 x 65):
// thread (c, g) gets column c's sum over lanes [16 g, 16 g + 16).
template <typename T>
__device__ __forceinline__ T fold(const T (&acc)[16], const ColSplit& cs, int g, int kb, T* R) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < 16; ++j) R[(16 * g + j) * (NB + 1) + lane] = acc[j];
    __syncthreads();
    T s = (T)0;
    if (lane < kb)
        for (int sp = 0; sp < cs.ns; ++sp) {
            const T* q = R + (16 * (sp * cs.ng + (lane >> 4)) + (lane & 15)) * (NB + 1) + 16 * g;
#pragma unroll
            for (int i = 0; i < 16; ++i) s += q[i];
        }
    return s;
}

// Backward separator product of diagonal block [k0, k0 + kb) over the
// separator tiles [t0, t1): the partial slot of the chunk.
template <typename T>
__device__ void sep_bwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, int k0, int t0, int t1,
                         T* R, T* Red, const Ctl& ctl) {
    const int r = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6));
    const Front f = front_of(P, J);
    const int nn = f.nn, nj = nn + f.na, kb = min(NB, nn - k0);
    const int nsep = (f.na + NB - 1) / NB, nchk = (nsep + SEP_TILES - 1) / SEP_TILES;
    const ColSplit cs(kb, g);
    T acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = (T)0;
    const int last = t1 - 1 - cs.sp;  // descending: the nearest ancestors finish last
    sweep(F.panel + f.poff + (int64_t)k0 * nj, nj, kb, P.rows + f.rowoff, V.out, cs, last >= t0 ? (last - t0) / cs.ns + 1 : 0,
          [&](int u) { return nn + NB * (last - u * cs.ns); }, [&](int) { return nj; }, acc, ctl);
    Red[g * VROWS + r] = fold(acc, cs, g, kb, R);
    __syncthreads();
    if (g == 0 && r < kb) publish(V.Mv + P.sboff1[J] + (int64_t)((k0 / NB) * nchk + t0 / SEP_TILES) * NB + r, sum4(Red, r));
}

// Backward diagonal block [k0, k0 + kb): y = C_k - L21' x_sep - sum_{ib > k}
// L_{ib,k}' X_ib, X_k = W_k' y.  The last link of the chain (block k + 1) is
// the one the task waits for: its tile is loaded transposed, so that the
// product ends in the layout the W product starts from.
template <typename T>
__device__ void diag_bwd1(const DevPlan& P, const DevFactor<T>& F, const DevVSolve<T>& V, int J, int k0, int kb, T* R,
                          T* Red, T* Red2, const Ctl& ctl) {
    const int r = threadIdx.x & 63, g = uni((int)(threadIdx.x >> 6)), li = r & 15;
    const Front f = front_of(P, J);
    const int nn = f.nn, na = f.na, nj = nn + na, p = (nn + NB - 1) / NB, kblk = k0 / NB, nch = p - 1 - kblk;
    const int nsep = (na + NB - 1) / NB, nchk = (nsep + SEP_TILES - 1) / SEP_TILES;
    const T* Pj = F.panel + f.poff;
    const int64_t sb = P.sboff1[J];
    T wa[16];
    load_rows(F.W + f.woff + k0, f.nn, kb, kb, g, wa);
    T y = (T)0;
    if (g == 0 && r < kb) {
        y = V.in[f.c0 + k0 + r];
        if (F.diag != 0) y /= F.d[f.c0 + k0 + r];
    }
    const ColSplit cs(kb, g);
    const int last = sb >= 0 ? -1 : nsep - 1 - cs.sp;
    const int ns = last >= 0 ? last / cs.ns + 1 : 0, nc = max(nch - 1, 0);
    if (nc > 0 || (sb < 0 && nsep > 0)) {
        T acc[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = (T)0;
        // the separator tiles, farthest ancestors first, then blocks p - 1 .. k + 2
        sweep(Pj + (int64_t)k0 * nj, nj, kb, P.rows + f.rowoff, V.out, cs, ns + nc,
              [&](int u) { return u < ns ? nn + NB * (last - u * cs.ns) : NB * (p - 1 - (u - ns)); },
              [&](int u) { return u < ns ? nj : nn; }, acc, ctl);
        y += fold(acc, cs, g, kb, R);
    }
    if (sb >= 0) {
        // the front's separator tasks: their partials, chunk c by wavefront c mod 4
        const T* slot = V.Mv + sb + (int64_t)kblk * nchk * NB + min(r, kb - 1);
        for (int c = g; c < nchk; c += 4) y += settle(peek(slot + c * NB), slot + c * NB, r < kb, ctl);
    }
    T s1 = (T)0;
    if (nch > 0) {
        const int row = k0 + NB, rows = min(NB, nn - row);
        const T* px = V.out + f.c0 + row + min(16 * g + li, rows - 1);
        T la[16];
        load_rows(Pj + row + (int64_t)k0 * nj, nj, rows, kb, g, la);
        const T x = -settle(peek(px), px, 16 * g + li < rows, ctl);
        fma16(y, s1, x, la);
    }
    Red[g * VROWS + r] = y + s1;
    __syncthreads();
    T t0 = (T)0, t1 = (T)0;
    fma16(t0, t1, 16 * g + li < kb ? sum4(Red, 16 * g + li) : (T)0, wa);
    Red2[g * VROWS + r] = t0 + t1;
    __syncthreads();
    if (g == 0 && r < kb) publish(V.out + f.c0 + k0 + r, sum4(Red2, r));
}

// LDS of a workgroup: small panels (or the transposed partial sums), the
// wavefronts' gathered rows, their partial sums.
template <typename T>
struct VLds {
    T panel[VT_PANELS];
    T Y[4 * VROWS];
    T Red[4 * VROWS];
    uint32_t unit;
};

template <typename T, bool FWD>
__global__ __launch_bounds__(256, 3) void k_vsolve(DevPlan P, DevFactor<T> F, DevVSolve<T> V0) {
    static_assert(VT_PANELS >= NB * (NB + 1), "the transposed partial sums and a 64 x 64 small front");
    __shared__ VLds<T> S;
    const int tid = threadIdx.x, g = uni(tid >> 6);
    const Ctl ctl{F.hang, V0.ticket, F.stall};
    const uint32_t nc = V0.cols, tickets = (uint32_t)V0.nunit * nc;
    for (;;) {
        if (tid == 0) S.unit = atomicAdd(V0.ticket, 1u);
        __syncthreads();
        const uint32_t tick = uni((int32_t)S.unit);
        if (tick >= tickets) break;
        // the columns are independent; the same unit's tickets are neighbours,
        // so that the factor's tiles come out of a cache for all but the first
        const uint32_t u = tick / nc;
        const int64_t col = tick - u * nc;
        DevVSolve<T> V = V0;
        V.in += col * V.ldin;
        V.wipe += col * V.ldin;
        V.out += col * V.ldout;
        V.Mv += col * V.mvs;
        const int t1 = V.unit[u + 1];
        for (int t = V.unit[u]; t < t1; ++t) {
            const unsigned long long t_begin = (V.trace && tid == 0) ? wall_clock64() : 0;
            const VTask tk = V.task[t];
            if (tk.kind == VT_SMALL) {
                const int J = uni(g == 0 ? tk.a : g == 1 ? tk.b : g == 2 ? tk.c : tk.d);
                const int o = uni(g == 0 ? 0 : g == 1 ? (tk.o12 & 0xffff) : g == 2 ? (int)((uint32_t)tk.o12 >> 16) : tk.o3);
                if (J >= 0) {
                    if (FWD) small_fwd1(P, F, V, J, S.panel + o, S.Y + g * VROWS, ctl);
                    else small_bwd1(P, F, V, J, S.panel + o, S.Y + g * VROWS, ctl);
                }
            } else if (FWD) {
                if (tk.kind == VT_FRONT) front_fwd1(P, F, V, uni(tk.a), S.Y, S.Red, ctl);
                else if (tk.kind == VT_DIAG) diag_fwd1(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.Y, S.Red, ctl);
                else rows_fwd1(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.Y, S.Red, ctl);
            } else {
                if (tk.kind == VT_SEPB) sep_bwd1(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), uni(tk.d), S.panel, S.Red, ctl);
                else diag_bwd1(P, F, V, uni(tk.a), uni(tk.b), uni(tk.c), S.panel, S.Red, S.Y, ctl);
            }
            if (V.trace && tid == 0) {  // (the last column's clocks stay)
                V.trace[2 * tk.t0] = t_begin | ((unsigned long long)blockIdx.x << 48);
                V.trace[2 * tk.t0 + 1] = wall_clock64();
            }
            __syncthreads();  // the LDS of this task is free; every thread has read S.unit
        }
    }
}

// The values that a solve's workgroups wait for, unset; both tickets 0.
template <typename T>
__global__ __launch_bounds__(256) void k_vinit(bits_t<T>* X, int64_t n, bits_t<T>* Mv, int64_t m, uint32_t* ticket) {
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, st = (int64_t)gridDim.x * blockDim.x;
    if (i0 < 2) ticket[i0] = 0u;
    for (int64_t i = i0; i < n; i += st) X[i] = unset<T>();
    for (int64_t i = i0; i < m; i += st) Mv[i] = unset<T>();
}

}  // namespace

template <typename T>
void launch_solve1(const DevPlan& P, const DevFactor<T>& F, T* B, int64_t ldb, int cols, T* X, T* Mv, int64_t mvs,
                   const DevVPlan& D, int n, unsigned long long* trace, int64_t ntrace_f, hipStream_t s) {
    if (D.nfu <= 0) return;
    const int64_t blocks = ((mvs > n ? mvs : n) * cols + 1023) / 1024;
    hipLaunchKernelGGL((k_vinit<T>), dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, s, (bits_t<T>*)X,
                       (int64_t)n * cols, (bits_t<T>*)Mv, mvs * cols, F.ticket);
    auto grid = [&](int64_t units) { return dim3((unsigned)(units * cols < 1024 ? units * cols : 1024)); };
    // forward: B -> X, leaving B unset; backward: X -> B
    DevVSolve<T> V{B, X, Mv, B, ldb, n, mvs, D.ftask, D.funit, D.nfu, cols, D.chd, F.ticket, trace};
    hipLaunchKernelGGL((k_vsolve<T, true>), grid(D.nfu), dim3(256), 0, s, P, F, V);
    V = DevVSolve<T>{X, B, Mv, X, n, ldb, mvs, D.btask, D.bunit, D.nbu, cols, D.chd, F.ticket + 1,
                     trace ? trace + 2 * ntrace_f : nullptr};
    hipLaunchKernelGGL((k_vsolve<T, false>), grid(D.nbu), dim3(256), 0, s, P, F, V);
}

template void launch_solve1<double>(const DevPlan&, const DevFactor<double>&, double*, int64_t, int, double*, double*,
                                    int64_t, const DevVPlan&, int, unsigned long long*, int64_t, hipStream_t);
template void launch_solve1<float>(const DevPlan&, const DevFactor<float>&, float*, int64_t, int, float*, float*,
                                   int64_t, const DevVPlan&, int, unsigned long long*, int64_t, hipStream_t);

}  // namespace mf
