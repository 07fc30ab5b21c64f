// mf_factor.hip — gfx950 kernels of the multifrontal numeric factorization.
//
//   k_small     fused front kernel for internal fronts with nJ <= 64: the
//               front lives in LDS; extend-add of the children's update
//               matrices, assembly, partial factorization and the write-out
//               of the panel and of U in one workgroup.  Persistent mode
//               hands out fronts by ticket in postorder levels and waits on
//               the children's completion flags (bounded wait).
//               Reference: chol_loop_snd!/nod! cholesky.jl:434-692,
//               chol_send! cholesky.jl:950-983, potrf2! blas/potrf.jl:3-41.
//   k_dag       persistent tile-DAG over all big fronts: extend-add
//               tiles (F11/F21 += F, cholesky.jl:520-521; M22 <- F22,
//               cholesky.jl:542), small fronts above the small region,
//               diagonal-tile factor + inverse (potrf2!), panel solve tiles
//               (trsm!, blas/trsx.jl:156-159, as a product with the inverted
//               diagonal tile), trailing-update tiles and update-matrix tiles
//               M22 -= L21 [D] L21' (syrk!, blas/syrk.jl:137-159).
//   k_diag      diagonal-tile inverse alone (solves of a factor given in the
//               reference layout).
//   k_copyout   internal panels -> the reference's Dval/Lval/d layout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "mf_kernels.h"
#include "mf_mfma.h"
#include "mf_pivots.h"
#include "mf_sync.h"

namespace mf {

namespace {

template <typename T>
__device__ __forceinline__ double sign_of(const DevFactor<T>& F, int gcol) {
    if (F.signs) return F.signs[gcol];
    return F.diag == 0 ? 1.0 : 0.0;
}

// regularize(R, S, Djj, j): no_regularization.jl:27-33 and
// dynamic_regularization.jl:75-90.  0 signals a failed pivot.
template <typename T>
__device__ __forceinline__ double regularize(const DevFactor<T>& F, double s, double Djj) {
    if (F.reg_kind == 1) return (s * Djj < F.eps) ? F.delta * s : Djj;
    if (s != 0.0 && !(s * Djj > 0.0)) return 0.0;
    return Djj;
}

// Julia's max of floats: NaN when either argument is NaN.
__device__ __forceinline__ double jmax(double a, double b) {
    if (a != a || b != b) return a + b;
    return a > b ? a : b;
}

// GMW81 regularize (gmw81.jl:109-155): s * max(|Djj|, amax^2 / beta, delta),
// amax the largest magnitude below the pivot in its front column as the
// column stands after the previous pivots (GMW81 never fails a pivot).
template <typename T>
__device__ __forceinline__ double regularize_gmw(const DevFactor<T>& F, double s, double Djj, double amax) {
    return s * jmax(jmax(fabs(Djj), amax * amax / F.gmw[2]), F.delta);
}

// Largest value over the wavefront (NaN-propagating), in every lane; over
// each half of it with LANES = 32.
template <int LANES = 64>
__device__ __forceinline__ double wave_max(double v) {
    for (int o = LANES / 2; o > 0; o >>= 1) v = jmax(v, __shfl_xor(v, o));
    return v;
}

// Waits until this wave's global stores (and loads) have completed.  Task
// outputs are device-coherent stores, so once every wave has drained before
// the closing barrier, the counter update that thread 0 makes afterwards
// follows all of the task's data.
__device__ __forceinline__ void drain_stores() { __builtin_amdgcn_s_waitcnt(0); }

__device__ __forceinline__ int ld_rel(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Update matrices of small fronts are written and read with device-coherent
// (sc1) accesses: a small front then publishes with its stores drained and a
// flag, and its parent reads U without a cache-wide invalidate.
template <typename T>
__device__ __forceinline__ T ldc(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void stc(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr int LDS = SMALL_NJ + 1;  // leading dimension of LDS fronts and tiles
constexpr int LDT = 64 + 4;        // leading dimension of the 64-wide tile's LDS operand
constexpr int GEMM_LDS = 4 * 16 * 128;  // two stages of two operands of a long product

// A plan record that every lane of the workgroup has loaded from the same
// place, into scalar registers: sizes, strides and offsets then cost no vector
// registers or vector arithmetic.
template <typename S>
__device__ __forceinline__ S uniform(const S& v) {
    static_assert(sizeof(S) % 4 == 0, "whole words");
    struct Words {
        int w[sizeof(S) / 4];
    };
    Words x = __builtin_bit_cast(Words, v);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(S) / 4); ++i) x.w[i] = __builtin_amdgcn_readfirstlane(x.w[i]);
    return __builtin_bit_cast(S, x);
}

// Computes v here, before the stores that follow.  A store under a per-lane
// predicate is a branch; arithmetic left to that branch waits there for its
// operands' loads, and on this hardware that wait covers the stores already
// issued, so a run of predicated stores would take one memory round trip each
// (660 cycles per store in the extend-add, 16 stores per tile).
template <typename T, int N>
__device__ __forceinline__ void pin(T (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}

// 1 / sqrt(d) and 1 / d to full double precision: the hardware estimate
// (about 24 bits) and one step of third order, a chain of five and three
// operations.
__device__ __forceinline__ double rsqrt_full(double d) {
    const double y = __builtin_amdgcn_rsq(d);
    const double e = __builtin_fma(-(d * y), y, 1.0);
    return __builtin_fma(y, e * __builtin_fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ double rcp_full(double d) {
    const double y = __builtin_amdgcn_rcp(d);
    const double e = __builtin_fma(-d, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}
// Lane k of v, to every lane (k is uniform).
__device__ __forceinline__ double lane_of(double v, int k) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, k), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), k);
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}
__device__ __forceinline__ float lane_of(float v, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, v), k));
}

// The children of a front final: one lane a child, by a whole wavefront.
template <typename T>
__device__ __forceinline__ void wait_children(const DevPlan& P, const DevFactor<T>& F, int q0, int q1, int lane) {
    for (int b = q0; b < q1; b += 64) {
        const bool on = b + lane < q1;
        const int32_t* w = F.flags + P.vchd[min(b + lane, q1 - 1)].front;
        Watch watch;
        for (int spins = 1;; ++spins) {
            const bool ok = !on || ld_rel(w) >= 1;
            if (__all(ok)) break;
            if ((spins & 255) == 0) {
                // once any wait has given up, every other wait returns at once
                if (ld_rel(F.hang)) return;
                if (watch.expired((int32_t)__popcll(__ballot(ok)), F.ticket, F.stall)) {
                    if (!ok) give_up(F.hang, w, 1, 0, -1);
                    return;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
}

// The pivot of column k from its diagonal entry and (GMW81) the magnitudes
// below it: the pivot (0: failed), its scale (1 / sqrt or 1 /) and, for
// Cholesky, its root.  sgn: the signs of the front's columns, one a lane (read
// where there are any).  The estimates of rsqrt_full and rcp_full hold where the
// pivot and its reciprocal are normal numbers (exponents 1 to 2044); any other
// takes the square root and the division, so that an infinite diagonal entry
// (a pinned unknown) scales its column to zero and a subnormal one is as
// accurate as the rest.
// LANES: rows that differ (32: the wavefront's halves hold the same ones).
template <int LANES, typename T>
__device__ __forceinline__ double small_pivot(const DevFactor<T>& F, double sgn, int k, double akk, double below, double* scale,
                                              double* root) {
    const double sg = F.signs ? lane_of(sgn, k) : F.diag == 0 ? 1.0 : 0.0;
    const double piv = F.reg_kind == 2 ? regularize_gmw(F, sg, akk, wave_max<LANES>(below)) : regularize(F, sg, akk);
    *scale = F.diag == 0 ? rsqrt_full(piv) : rcp_full(piv);
    *root = piv * *scale;
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(__builtin_bit_cast(unsigned long long, piv) >> 32));
    if (__builtin_expect(((hi >> 20) & 0x7ff) - 1 >= 2044, 0)) {
        *root = sqrt(piv);
        *scale = 1.0 / (F.diag == 0 ? *root : piv);
    }
    return piv;
}

// One small front (nJ <= 64) by a workgroup: the panel's A entries and the
// children's update matrices meet in LDS (M), then wavefront g keeps columns
// c = g mod 4, row r in lane r, in registers for the partial factorization:
// the wavefront that owns column k scales it and leaves it in LDS, and after
// one barrier every wavefront subtracts it from its later columns.  The
// owned columns shift down by one register every four columns, so the pivot
// is always in the first.  Both small-front kernels on a 100 x 100 grid: 199
// -> 156 us of the small region.  WAIT: the children are waited for here, after the
// loads that do not depend on them.  Returns after a failed pivot (recorded
// in F.info).
// Bound: the chain of pivots (square root, LDS, barrier and the update) and
// the loads' round trips.  A front of the DAG took 28 us with the columns in
// LDS, one thread's square root and division and three barriers a pivot, and
// the children's records read one by one.
template <typename T, bool WAIT>
__device__ __forceinline__ void small_front(const DevPlan& P, const DevFactor<T>& F, int J, T* M, T* s_piv, int* s_fail,
                                            const int tid) {
    const Front f = uniform(P.fronts[J]);
    const int nn = f.nn, na = f.na, nj = nn + na;
    const int r = tid & 63, g = __builtin_amdgcn_readfirstlane(tid >> 6);
    T* Pj = F.panel + f.poff;
    T a[NB / 4];
    for (int c0 = 0; c0 < nj; c0 += 32) {
        T v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Pj[min(r, nj - 1) + (int64_t)min(c0 + 4 * i + g, nn - 1) * nj];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int c = c0 + 4 * i + g;
            if (c < nj) M[r + c * LDS] = (c < nn && c <= r && r < nj) ? v[i] : (T)0;
        }
    }
    if (WAIT && g == 0) wait_children(P, F, f.chd0, f.chd1, r);
    __syncthreads();
    for (int qb = f.chd0; qb < f.chd1; qb += 64) {
        const int ns = min(64, f.chd1 - qb);
        const VChild x = P.vchd[qb + min(r, ns - 1)];  // one child a lane
        auto get = [&](int32_t v, int q) { return __builtin_amdgcn_readlane(v, q); };
        // wavefront g: columns c = g mod 4 of the child, row in the lane, all in flight
        auto load = [&](int q, T (&v)[NB / 4], int& rr) {
            const int ma = get(x.ma, q);
            const uint64_t uo = (uint32_t)get((int32_t)(uint64_t)x.u, q) |
                                (uint64_t)(uint32_t)get((int32_t)((uint64_t)x.u >> 32), q) << 32;
            const uint32_t row = min(r, ma - 1);
            rr = (P.rel + get(x.rel, q))[row];
            const T* u = F.U + uo;
#pragma unroll
            for (int h = 0; h < NB / 4; h += 4) {
                if (4 * h >= ma) break;  // uniform
#pragma unroll
                for (int i = h; i < h + 4; ++i) v[i] = ldc(u + (int64_t)min(4 * i + g, ma - 1) * ma + row);
            }
        };
        auto add = [&](int q, const T (&v)[NB / 4], int rr) {
            const int ma = get(x.ma, q);
#pragma unroll
            for (int h = 0; h < NB / 4; h += 4) {
                if (4 * h >= ma) break;  // uniform
#pragma unroll
                for (int i = h; i < h + 4; ++i) {
                    const int c = 4 * i + g;
                    const int cc = get(rr, min(c, ma - 1));
                    if (c <= r && r < ma) M[rr + cc * LDS] += v[i];
                }
            }
        };
        T v0[NB / 4], v1[NB / 4];
        int r0 = 0, r1 = 0;
        load(0, v0, r0);
        for (int q = 0; q < ns; q += 2) {
            if (q + 1 < ns) load(q + 1, v1, r1);
            add(q, v0, r0);
            __syncthreads();
            if (q + 1 >= ns) break;
            if (q + 2 < ns) load(q + 2, v0, r0);
            add(q + 1, v1, r1);
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) a[i] = 4 * i + g < nj && r < nj ? M[r + (4 * i + g) * LDS] : (T)0;
    __syncthreads();
    const bool chol = F.diag == 0;
    int k4 = 0;  // first column of the wavefronts' first registers
    const double sgn = F.signs ? F.signs[f.c0 + min(r, nn - 1)] : 0.0;
    struct Fail {
        int* p;
        bool writer;  // one lane of the owner
        __device__ __forceinline__ void set(int v) const {
            if (writer) *p = v;
        }
        __device__ __forceinline__ int get() const { return *p; }
    };
    // column k, held in the owner's first register
    auto own = [&](int k) {
        double sc, rt;
        const double piv = small_pivot<64>(F, sgn, k, (double)lane_of(a[0], k),
                                       (r > k && r < nj) ? fabs((double)a[0]) : 0.0, &sc, &rt);
        if (piv == 0.0) {
            if (r == 0) atomicMin(F.info, (unsigned long long)(f.c0 + k + 1));
            return false;
        }
        if (r == 0) {
            *s_piv = chol ? (T)1 : (T)piv;
            if (!chol) stc(F.d + f.c0 + k, (T)piv);
        }
        M[r + k * LDS] = r > k ? a[0] * (T)sc : (r == k && chol) ? (T)rt : a[0];
        return true;
    };
    auto update = [&](int k) {
        const int o = k & 3;
        const T lr = -M[r + k * LDS] * *s_piv;
#pragma unroll
        for (int h = 0; h < NB / 4; h += 4) {
            if (k4 + 4 * h >= nj) break;  // uniform
#pragma unroll
            for (int i = h; i < h + 4; ++i)
                if (i > 0 || g > o) a[i] += lr * M[min(k4 + 4 * i + g, NB - 1) + k * LDS];
        }
        if (o == 3) {
            k4 += 4;
#pragma unroll
            for (int i = 0; i + 1 < NB / 4; ++i) a[i] = a[i + 1];
        }
    };
    // (closed for LDLt: s_piv is one column's)
    if (!pivot_columns(nn, g, !chol, own, Fail{s_fail, r == 0}, [] { __syncthreads(); }, update)) return;
    // the update matrix's columns (c >= nn) and the panel
    pin(a);
    if (na > 0) {
        T* Uj = F.U + f.uoff;
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) {
            const int c = k4 + 4 * i + g;
            if (c >= nn && c < nj && r >= c && r < nj) stc(Uj + (r - nn) + (int64_t)(c - nn) * na, a[i]);
        }
    }
    for (int c = g; c < nn; c += 4)
        if (r >= c && r < nj) stc(Pj + r + (int64_t)c * nj, M[r + c * LDS]);
}

constexpr int LDT1 = TINY_NJ + 1;     // leading dimension of a wavefront's LDS front
static_assert(TINY_NJ == 32, "both halves of a wavefront hold the rows of a tiny front");

// One tiny front (nJ <= TINY_NJ) by one wavefront: as small_front, with the
// whole front in the wavefront's registers (row in the lane, one register a
// column, four columns to a step of the loop) and its own LDS slab Mw for
// the sums and the finished columns.  A wavefront's LDS operations complete
// in order, so no barrier is needed.  Children are added two at a time, even
// columns by lanes 0..31 and odd ones by lanes 32..63.
template <typename T>
__device__ __forceinline__ void wave_front(const DevPlan& P, const DevFactor<T>& F, int J, T* Mw, const int lane) {
    const Front f = uniform(P.fronts[J]);
    const int nn = f.nn, na = f.na, nj = nn + na;
    const int r = lane & (TINY_NJ - 1), half = lane >> 5;
    T* Pj = F.panel + f.poff;
    auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int c0 = 0; c0 < TINY_NJ; c0 += 16) {
        if (c0 >= nj) break;  // uniform
        T v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Pj[min(r, nj - 1) + (int64_t)min(c0 + 2 * i + half, nn - 1) * nj];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int c = c0 + 2 * i + half;
            Mw[r + c * LDT1] = (c < nn && c <= r && r < nj) ? v[i] : (T)0;
        }
    }
    const double sgn = F.signs ? F.signs[f.c0 + min(r, nn - 1)] : 0.0;
    wait_children(P, F, f.chd0, f.chd1, lane);
    sync();
    for (int qb = f.chd0; qb < f.chd1; qb += 64) {
        const int ns = min(64, f.chd1 - qb);
        const VChild x = P.vchd[qb + min(lane, ns - 1)];
        auto get = [&](int32_t v, int q) { return __builtin_amdgcn_readlane(v, q); };
        auto load = [&](int q, T (&v)[TINY_NJ / 2], int& rr) {
            const int ma = get(x.ma, q);
            const uint64_t uo = (uint32_t)get((int32_t)(uint64_t)x.u, q) |
                                (uint64_t)(uint32_t)get((int32_t)((uint64_t)x.u >> 32), q) << 32;
            const uint32_t row = min(r, ma - 1);
            rr = (P.rel + get(x.rel, q))[row];
            const T* u = F.U + uo;
#pragma unroll
            for (int h = 0; h < TINY_NJ / 2; h += 4) {
                if (2 * h >= ma) break;  // uniform
#pragma unroll
                for (int i = h; i < h + 4; ++i) v[i] = ldc(u + (row + (uint32_t)(min(2 * i + half, ma - 1) * ma)));
            }
        };
        auto add = [&](int q, const T (&v)[TINY_NJ / 2], int rr) {
            const int ma = get(x.ma, q);
#pragma unroll
            for (int h = 0; h < TINY_NJ / 2; h += 4) {
                if (2 * h >= ma) break;  // uniform
#pragma unroll
                for (int i = h; i < h + 4; ++i) {
                    const int c = 2 * i + half;
                    const int c0 = get(rr, min(2 * i, ma - 1)), c1 = get(rr, min(2 * i + 1, ma - 1));
                    if (c <= r && r < ma) Mw[rr + (half ? c1 : c0) * LDT1] += v[i];
                }
            }
            sync();
        };
        T v0[TINY_NJ / 2], v1[TINY_NJ / 2];
        int r0 = 0, r1 = 0;
        for (int q = 0; q < ns; q += 2) {
            load(q, v0, r0);
            if (q + 1 < ns) load(q + 1, v1, r1);
            add(q, v0, r0);
            if (q + 1 < ns) add(q + 1, v1, r1);
        }
    }
    T a[TINY_NJ];
#pragma unroll
    for (int c = 0; c < TINY_NJ; ++c) a[c] = (c & ~3) < nj ? Mw[r + c * LDT1] : (T)0;
    const bool chol = F.diag == 0;
    int k4 = 0;
    bool failed = false;
    // column k = k4 + O, held in register O
    auto pivot = [&](auto O) {
        constexpr int o = decltype(O)::value;
        const int k = k4 + o;
        if (k >= nn || failed) return;  // uniform
        double sc, rt;
        const double piv = small_pivot<TINY_NJ>(F, sgn, k, (double)lane_of(a[o], k), (r > k && r < nj) ? fabs((double)a[o]) : 0.0, &sc, &rt);
        if (piv == 0.0) {
            if (lane == 0) atomicMin(F.info, (unsigned long long)(f.c0 + k + 1));
            failed = true;
            return;
        }
        if (!chol && lane == 0) stc(F.d + f.c0 + k, (T)piv);
        const T l = r > k ? a[o] * (T)sc : (r == k && chol) ? (T)rt : a[o];
        Mw[r + k * LDT1] = l;
        const T lr = chol ? -l : -l * (T)piv;
        // (out of the loop at the first group past the front: a test of every
        // group is an execution mask each, 10 us a front of nine columns on a
        // path of 50000 unknowns against 8.7)
#pragma unroll
        for (int h = 0; h < TINY_NJ; h += 4) {
            if (k4 + h >= nj) break;
#pragma unroll
            for (int i = h; i < h + 4; ++i)
                if (i > o) a[i] += lr * lane_of(l, min(k4 + i, TINY_NJ - 1));
        }
    };
    for (;;) {
        pivot(std::integral_constant<int, 0>());
        pivot(std::integral_constant<int, 1>());
        pivot(std::integral_constant<int, 2>());
        pivot(std::integral_constant<int, 3>());
        if (failed) return;  // the front stays unfinished; info reports the column
        if (k4 + 4 > nn) break;
        k4 += 4;
#pragma unroll
        for (int i = 0; i + 4 < TINY_NJ; ++i) a[i] = a[i + 4];
    }
    pin(a);
    sync();
    // the update matrix's columns, odd and even in the two halves' lanes
    if (na > 0) {
        T* Uj = F.U + f.uoff;
#pragma unroll
        for (int i = 0; i < TINY_NJ; ++i) {
            const int c = k4 + i;
            if ((i & 1) == half && c >= nn && c < nj && r >= c && r < nj) stc(Uj + (r - nn) + (c - nn) * na, a[i]);
        }
    }
    for (int c = half; c < nn; c += 2)
        if (r >= c && r < nj) stc(Pj + r + (int64_t)c * nj, Mw[r + c * LDT1]);
}

// Persistent walk of the small region.  Tickets are units of the planner's
// children-first order: one front of nJ > TINY_NJ (the whole workgroup), or
// up to four consecutive tiny fronts (one per wavefront, each waiting for
// its own children; a child in the same unit belongs to another wavefront,
// which progresses on its own).  Update matrices go through device-coherent
// accesses, so a front is published by draining its stores and setting its
// flag; no cache-wide write-back or invalidate.  (Several units a ticket, as
// the solves take their tasks, were slower: 600 systems 655 -> 706 us.)
template <typename T>
__global__ __launch_bounds__(256, 4) void k_small(DevPlan P, DevFactor<T> F, int tickets) {
    constexpr int MS = SMALL_NJ * LDS > 4 * TINY_NJ * LDT1 ? SMALL_NJ * LDS : 4 * TINY_NJ * LDT1;
    __shared__ T M[MS];
    __shared__ T s_piv;
    __shared__ int s_fail, s_t;
    for (;;) {
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        if (tid == 0) s_t = (int)atomicAdd(F.ticket, 1u);
        __syncthreads();
        const int t = s_t;
        __syncthreads();
        if (t >= tickets) break;
        const int u = P.small_units[t], start = u >> 3, cnt = u & 7;
        if (cnt == 0) {  // one front, the whole workgroup
            const int J = P.small_order[start];
            if (tid == 0) s_fail = 0;
            small_front<T, true>(P, F, J, M, &s_piv, &s_fail, tid);
            drain_stores();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(F.flags + J, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
            if (wave < cnt) {
                const int J = P.small_order[start + wave];
                wave_front<T>(P, F, J, M + wave * TINY_NJ * LDT1, lane);
                drain_stores();
                __builtin_amdgcn_wave_barrier();
                if (lane == 0) __hip_atomic_store(F.flags + J, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        // closes the ticket before the back-edge: every thread reaches the
        // next ticket together
        __syncthreads();
    }
}

constexpr int EA_LDS = 17 * LDS;  // LDS elements of a wavefront's extend-add columns

// Extend-add of one 64 x 64 tile (F11/F21 += F, cholesky.jl:520-521, or
// M22 <- F22, cholesky.jl:542).  Wavefront w takes the tile's columns
// [16w, 16w + 16) in an LDS accumulator of its own (acc, 16 columns of LDS),
// so no barrier is needed.  Per child (in the reference's reverse order) lane
// l is the child's row ra + l, which lands in one row of the tile; the
// child's columns landing in the wavefront's (at most sixteen) are all in
// flight at once, the next child's while this one's are added, eight
// independent read-add-writes in LDS at a time (a wavefront's LDS operations
// complete in order, so children add up in their order).  The finished columns are added to the panel or written to
// U row-contiguously.  Bound: the load round trips (source record and rel
// map, then U); one tile takes 5.2 us of a workgroup on an idle chip (about 22
// us per 4,096 elements when each wavefront took one parent column at a time
// through a 1,024-row window).
template <typename T>
__device__ __forceinline__ void ea_tile(const DevPlan& P, const DevFactor<T>& F, const EaTask e, T* lds, const int tid) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = 16 * wave;
    const Front f = uniform(P.fronts[e.front]);
    const int p = (f.nn + NB - 1) / NB, nj = f.nn + f.na;
    const int r0 = e.I < p ? e.I * NB : f.nn + (e.I - p) * NB, c0 = e.J < p ? e.J * NB : f.nn + (e.J - p) * NB;
    const int m = min(NB, (e.I < p ? f.nn : nj) - r0), n = min(NB, (e.J < p ? f.nn : nj) - c0);
    if (cw >= n) return;
    const bool to_u = e.J >= p;
    const int64_t ld = to_u ? f.na : nj;
    T* dst = to_u ? F.U + f.uoff + (r0 - f.nn) + (int64_t)(c0 - f.nn) * ld : F.panel + f.poff + r0 + (int64_t)c0 * ld;
    T* acc = lds + wave * EA_LDS;  // sixteen columns and a spare one
    const bool diag = e.I == e.J;
    T pre[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        // the assembled A entries (an earlier launch wrote them)
        pre[j] = to_u ? (T)0 : dst[min(lane, m - 1) + (int64_t)min(cw + j, n - 1) * ld];
        acc[lane + j * LDS] = (T)0;
    }
    // One source in flight: its rel maps, then its part of U (up to sixteen
    // columns of the tile's)
    struct Src {
        int rr, rc, i, rb, t0, t1, ta;
        T v[16];
    };
    // Thin sources (the planner's choice: many, and few of them more than
    // sixteen rows high in the tile), eight at a time: lane (i, j) =
    // (l mod 16, l / 16) is row i of columns j, j + 4, ... of the source's in
    // this wavefront's strip, so a source is a load and an LDS addition per
    // four columns, and eight sources' round trips are one.  20000 children of
    // 20 rows in a front of 500: 20.7 -> 7.3 ms a factorization, of 60 rows in
    // 4000: 57.5 -> 15.0.  A group with a higher source goes one by one.
    for (int sb = e.src0; e.thin && sb < e.src1; sb += 64) {
        const int ns = min(64, e.src1 - sb);
        const EaSrc x = P.ea_src[sb + min(lane, ns - 1)];
        const unsigned long long high = __ballot(x.rb - x.ra > 16);
        auto get = [&](int32_t v, int q) { return __builtin_amdgcn_readlane(v, q); };
        const int li = lane & 15, lj = lane >> 4;
        // the source's columns in the strip: the first, their number, this lane's column's place
        struct Cols {
            int t0, nt, rc;
        };
        auto cols = [&](int q, int rc, bool valid) {
            const bool has = valid && lane < get(x.tb, q) - get(x.ta, q);
            const int t0 = (int)__popcll(__ballot(has && rc < cw));
            return Cols{t0, (int)__popcll(__ballot(has && rc < cw + 16)) - t0, rc};
        };
        // columns j + 4 h, row `row` (at place pr of the tile): value and place (a spare one if there is none)
        auto fetch = [&](int q, const Cols& c, int h, int row, int pr, T& v, int& at) {
            const int ta = get(x.ta, q), rb = get(x.rb, q);
            const uint64_t uo = (uint32_t)get((int32_t)(uint64_t)x.u_off, q) |
                                (uint64_t)(uint32_t)get((int32_t)((uint64_t)x.u_off >> 32), q) << 32;
            const int j = lj + 4 * h, t = min(c.t0 + j, get(x.tb, q) - ta - 1);
            const bool on = j < c.nt && row < rb && (!diag || row >= ta + t);
            const int col = __shfl(c.rc, t) - cw;  // (by every lane)
            at = on ? col * LDS + pr : 16 * LDS + lane;
            const T u = ldc(F.U + uo + min(row, rb - 1) + (int64_t)(ta + t) * get(x.ma, q));
            v = on ? u : (T)0;
        };
        constexpr int G = 8;
        for (int q0 = 0; q0 < ns; q0 += G) {
            if (((high >> q0) & ((1u << G) - 1)) != 0) {
#pragma unroll 1
                for (int q = q0; q < min(q0 + G, ns); ++q) {
                    const int32_t* rel = P.rel + get(x.rel_off, q);
                    const Cols c = cols(q, rel[min(get(x.ta, q) + lane, get(x.tb, q) - 1)] - c0, true);
                    for (int row = get(x.ra, q) + li, r1 = get(x.rb, q), g = 0; 16 * g < r1 - get(x.ra, q); ++g, row += 16) {
                        const int pr = rel[min(row, r1 - 1)] - r0;
                        for (int h = 0; 4 * h < c.nt; ++h) {
                            T v;
                            int at;
                            fetch(q, c, h, row, pr, v, at);
                            acc[at] += v;
                        }
                    }
                }
                continue;
            }
            int pr[G], most = 0;
            Cols c[G];
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int q = min(q0 + i, ns - 1);
                const int32_t* rel = P.rel + get(x.rel_off, q);
                pr[i] = rel[min(get(x.ra, q) + li, get(x.rb, q) - 1)];
                c[i].rc = rel[min(get(x.ta, q) + lane, get(x.tb, q) - 1)];
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                pr[i] -= r0;
                c[i] = cols(min(q0 + i, ns - 1), c[i].rc - c0, q0 + i < ns);
                most = max(most, c[i].nt);
            }
            T v[4][G];
            int at[4][G];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                if (4 * h >= most) break;  // uniform
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const int q = min(q0 + i, ns - 1);
                    fetch(q, c[i], h, get(x.ra, q) + li, pr[i], v[h][i], at[h][i]);
                }
            }
#pragma unroll
            for (int i = 0; i < G; ++i)
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (4 * h < c[i].nt) acc[at[h][i]] += v[h][i];
        }
    }
    for (int sb = e.src0; !e.thin && sb < e.src1; sb += 64) {
        const int ns = min(64, e.src1 - sb);
        // the source records, one per lane
        const EaSrc x = P.ea_src[sb + min(lane, ns - 1)];
        auto get = [&](int32_t v, int q) { return __builtin_amdgcn_readlane(v, q); };
        auto rels = [&](int q, Src& s) {
            const int32_t* rel = P.rel + get(x.rel_off, q);
            const int ra = get(x.ra, q), tb = get(x.tb, q);
            s.ta = get(x.ta, q);
            s.rb = get(x.rb, q);
            s.i = ra + lane;
            s.rr = rel[min(s.i, s.rb - 1)] - r0;            // this lane's row of the tile
            s.rc = rel[min(s.ta + lane, tb - 1)] - c0;      // column of the tile of child column ta + lane
            s.t1 = tb;
        };
        auto cols = [&](int q, Src& s) {
            const bool has = lane < s.t1 - s.ta;
            s.t0 = s.ta + (int)__popcll(__ballot(has && s.rc < cw));
            s.t1 = s.ta + (int)__popcll(__ballot(has && s.rc < cw + 16));
            const uint64_t uo = (uint32_t)get((int32_t)(uint64_t)x.u_off, q) |
                                (uint64_t)(uint32_t)get((int32_t)((uint64_t)x.u_off >> 32), q) << 32;
            const int ma = get(x.ma, q);
            const T* u = F.U + uo + min(s.i, s.rb - 1);
#pragma unroll
            for (int h = 0; h < 16; h += 8) {
                if (s.t0 + h >= s.t1) break;  // uniform
#pragma unroll
                for (int j = h; j < h + 8; ++j) s.v[j] = ldc(u + (int64_t)min(s.t0 + j, s.t1 - 1) * ma);
            }
        };
        // columns past the child's last go to the spare column
        auto add = [&](const Src& s) {
            if (s.i >= s.rb) return;
#pragma unroll
            for (int h = 0; h < 16; h += 8) {
                if (s.t0 + h >= s.t1) break;  // uniform
                T o[8];
                int pc[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int t = s.t0 + h + j;
                    const int c = t < s.t1 ? get(s.rc, t - s.ta) - cw : 16;
                    pc[j] = c * LDS + s.rr;
                    o[j] = acc[pc[j]];
                }
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    acc[pc[j]] = o[j] + (!diag || s.i >= s.t0 + h + j ? s.v[h + j] : (T)0);
            }
        };
        Src s0, s1;
        rels(0, s0);
        if (ns > 1) rels(1, s1);
        cols(0, s0);
        for (int q = 0; q < ns; q += 2) {
            if (q + 1 < ns) cols(q + 1, s1);
            add(s0);
            if (q + 2 < ns) rels(q + 2, s0);
            if (q + 1 < ns) add(s1);
            if (q + 3 < ns) rels(q + 3, s1);
            if (q + 2 < ns) cols(q + 2, s0);
        }
    }
    // all LDS reads first, then the stores
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const T a = acc[lane + j * LDS];
        pre[j] = to_u ? a : pre[j] + a;
    }
    pin(pre);
#pragma unroll
    for (int j = 0; j < 16; ++j)
        if (lane < m && cw + j < n && (!diag || lane >= cw + j)) stc(dst + lane + (int64_t)(cw + j) * ld, pre[j]);
}

constexpr int PB = 16;            // block size inside the diagonal tile
constexpr int LDP = PB + 1;       // leading dimension of the tile's inverse diagonal blocks
constexpr int PTILE = NB * LDS + (NB / PB) * PB * LDP + 3 * NB;  // LDS elements of potrf_blocked

// Column operations with the multiplier broadcast inside each row of sixteen
// lanes (DPP row_newbcast): a(q) += (lane L0 + q of s) * m for q < N.  One
// instruction per element, where a readlane pair and a multiply-add take
// 20 cycles against 9.5 (FP64, one wavefront).  The leading s_nop covers the
// two wait states between a vector write of s and its first DPP read.
template <int L0>
__device__ __forceinline__ void dpp_fma1(double& a0, double s, double m) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(a0) : "v"(s), "v"(m), "n"(L0));
}
template <int L0>
__device__ __forceinline__ void dpp_fma4(double& a0, double& a1, double& a2, double& a3, double s, double m) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(s), "v"(m), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
}
template <int L0>
__device__ __forceinline__ void dpp_fma1(float& a0, float s, float m) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(a0) : "v"(s), "v"(m), "n"(L0));
}
template <int L0>
__device__ __forceinline__ void dpp_fma4(float& a0, float& a1, float& a2, float& a3, float s, float m) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(s), "v"(m), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
}
// a[j] += (lane j of s) * m for K < j < 16
template <int K, typename T>
__device__ __forceinline__ void dpp_cols(T (&a)[PB], T s, T m) {
    constexpr int G = (K + 4) / 4 * 4;  // first whole group of four columns
    if constexpr (K + 1 < G) dpp_fma1<K + 1>(a[K + 1], s, m);
    if constexpr (K + 2 < G) dpp_fma1<K + 2>(a[K + 2], s, m);
    if constexpr (K + 3 < G) dpp_fma1<K + 3>(a[K + 3], s, m);
    if constexpr (G <= 4) dpp_fma4<4>(a[4], a[5], a[6], a[7], s, m);
    if constexpr (G <= 8) dpp_fma4<8>(a[8], a[9], a[10], a[11], s, m);
    if constexpr (G <= 12) dpp_fma4<12>(a[12], a[13], a[14], a[15], s, m);
}
// Lane K of every row of sixteen lanes, to all its lanes.
template <int K>
__device__ __forceinline__ double dpp_bcast(double s) {
    double v;
    asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(v) : "v"(s), "n"(K));
    return v;
}
template <int K>
__device__ __forceinline__ float dpp_bcast(float s) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x150 + K, 0xf, 0xf, true));
}


// Pivot rules of the diagonal tile.  PR_RULE: signs and regularization, one
// call of regularize per pivot; PR_CHOL / PR_LDLT: the default signs (fails
// unless the pivot is positive / on a zero pivot only); PR_INV / PR_INV_UNIT:
// the block is factored already (Cholesky / LDLt) and only carries the other
// rows along.
enum { PR_RULE = 0, PR_CHOL = 1, PR_LDLT = 2, PR_INV = 3, PR_INV_UNIT = 4 };

// Columns K..15 of a 16-column block by one wavefront.  x: row (lane & 15) of
// the diagonal block, repeated in each row of sixteen lanes (so that DPP can
// broadcast its column); y: one other row per lane.  Per pivot k with s =
// 1 / l_kk (Cholesky) or 1 / d_k (LDLt): l = x_k s, and every later column
// takes x_j -= l_jk m, y_j -= l_jk m_y, with m, m_y the finished x_k, y_k:
// l for Cholesky, the unscaled column a_ik for LDLt (the caller multiplies
// by s where it needs l).  The rows below the block (a panel solve) and rows
// of the identity (which become rows of L^-T) are the same operation.
// Finished columns go to LDS at once (xw, yw: this lane's rows, column
// strides LDS and ys; what lands above the diagonal is not read).  pv / sc
// (LDS): the pivots and s for LDLt.  fails: bit k for a failed pivot.
template <typename T, int RULE, int K>
__device__ __forceinline__ void pivot_cols(T (&x)[PB], T (&y)[PB], const DevFactor<T>& F, const int gcol0,
                                           const int nk, const bool chol, T* pv, T* sc, T* xw, T* yw,
                                           const int ys, unsigned& fails, const int lane) {
    if constexpr (K < PB) {
        T l, m, my;
        if constexpr (RULE == PR_INV_UNIT) {
            l = x[K];
            my = y[K];
        } else if constexpr (RULE == PR_INV) {
            l = x[K];
            my = y[K] * ((T)1 / dpp_bcast<K>(x[K]));  // (a factor from elsewhere: any number)
        } else {
            double piv = (double)dpp_bcast<K>(x[K]);
            const bool ch = RULE == PR_CHOL || (RULE == PR_RULE && chol);
            bool bad = false;
            if constexpr (RULE == PR_RULE) {
                // padding columns (K >= nk) keep their pivot 1: no sign is read
                if (K < nk) piv = regularize(F, sign_of(F, gcol0 + K), piv);
                bad = piv == 0.0;
            } else {
                bad = RULE == PR_CHOL ? !(piv > 0.0) : piv == 0.0;
            }
            fails |= bad ? 1u << K : 0u;
            if constexpr (RULE == PR_RULE) {
                if (bad) piv = 1.0;
            }
            const double s = ch ? rsqrt_full(piv) : rcp_full(piv);
            l = x[K] * (T)s;
            if constexpr (RULE == PR_RULE) {
                // the (possibly replaced) pivot on the diagonal
                if ((lane & (PB - 1)) == K && ch) l = (T)(piv * s);
            }
            m = ch ? l : x[K];
            my = ch ? y[K] * (T)s : y[K];
            if (!ch && lane == 0) {
                pv[K] = (T)piv;
                sc[K] = (T)s;
            }
            dpp_cols<K>(x, l, -m);
            if (lane < PB) xw[K * LDS] = m;
        }
        dpp_cols<K>(y, l, -my);
        yw[K * ys] = my;
        pivot_cols<T, RULE, K + 1>(x, y, F, gcol0, nk, chol, pv, sc, xw, yw, ys, fails, lane);
    }
}

// Diagonal tile, blocked by 16 columns: the 64 x 64 tile A lives in LDS.  The
// factor and its inverse come out of one pass over [A; I]: the column
// operations that turn A into L turn the identity into L^-T.  Rows of A use
// the tile's lower blocks and rows of the identity its upper blocks, which A
// does not use; the identity's diagonal blocks have a place of their own
// (WD).  So "row block w" is rows [16w, 16w + 16) of A for w > b and of the
// identity for w <= b, 64 rows beside the diagonal block in every block step
// b.  A block step:
// (1) wavefront 0 takes the diagonal block and all 64 other rows through the
//     block's 16 pivots in registers (pivot_cols), while the other
//     wavefronts finish the previous step's update;
// (2) the rank-16 update X_wc -= X_wb (s L_cb)' on the matrix cores, first
//     the next block column (wavefront w its row block), then, beside the
//     next step's pivots, the later ones (c <= w for rows of A).
// Bound: wavefront 0's instruction issue in the chain of 64 pivots (FP64
// operations issue every 8 cycles on one wavefront).  A full tile on an idle
// CU, load to last store: FP64 13.6 us, FP32 12.4 us (19.0 and
// 16.0 us with the pivot row broadcast by readlane, one wavefront per row
// block; 40 us with the rows below and the inverse in passes of their own).
// W = L^-1 (ld = nn, zeros above the diagonal) goes to the W pool; L stays in
// LDS for store_diag.  invert_only: the tile already holds L and only W is
// formed.  resident: the tile is in LDS already (chain_step left it there).
// LDS: PTILE elements.
template <typename T>
__device__ __forceinline__ void potrf_blocked(const DevFactor<T>& F, const Front f, int k0, bool invert_only,
                              bool resident, T* lds, const int tid) {
    typedef typename Mfma<T>::v4 v4;
    constexpr int NBLK = NB / PB;
    T* A = lds;                          // 64 x LDS, column-major
    T* WD = lds + NB * LDS;              // diagonal blocks of L^-T, PB x LDP each
    T* sc = WD + NBLK * PB * LDP;        // 1 (Cholesky) or the reciprocal pivots (LDLt)
    T* pv = sc + NB;                     // the pivots (LDLt)
    const int nj = f.nn + f.na, kb = min(NB, f.nn - k0), gc0 = f.c0 + k0;
    T* blk = F.panel + f.poff + k0 + (int64_t)k0 * nj;
    const int r = tid & 63, cg = tid >> 6, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const bool chol = F.diag == 0;
    // the identity's diagonal blocks: block = wave, four elements per thread
#pragma unroll
    for (int q = 0; q < 4; ++q) WD[wave * PB * LDP + li + (lk + 4 * q) * LDP] = li == lk + 4 * q ? (T)1 : (T)0;
    if (tid < NB) sc[tid] = (T)1;
    if (!resident) {
        // all sixteen loads in flight (outside the tile: the tile's first
        // element stands in), then the LDS writes
        T tv[NB / 4];
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) {
            const int c = cg + 4 * i;
            tv[i] = ldc(blk + ((r < kb && c < kb && c <= r) ? r + (int64_t)c * nj : 0));
        }
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) {
            const int c = cg + 4 * i;
            A[r + c * LDS] = (r < kb && c < kb && c <= r) ? tv[i] : (r == c ? (T)1 : (T)0);
        }
    }
    __syncthreads();
    // X_wc -= X_wb (s L_cb)' for row block w of block step b
    auto update = [&](int w, int b, int c) {
        const T* xa = w == b ? WD + b * PB * LDP : A + PB * w + PB * b * LDS;
        const int xs = w == b ? LDP : LDS;
        T av[4], bv[4], xv[4];
        v4 acc = v4{0, 0, 0, 0};
        T* xc = A + PB * w + (PB * c + li) * LDS;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            av[s] = xa[li + (4 * s + lk) * xs];
            bv[s] = A[(PB * c + li) + (PB * b + 4 * s + lk) * LDS] * sc[PB * b + 4 * s + lk];
            xv[s] = xc[Mfma<T>::row(lk, s)];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = Mfma<T>::op(av[s], bv[s], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) xc[Mfma<T>::row(lk, v)] = xv[v] - acc[v];
    };
#pragma unroll 1
    for (int b = 0; b < NBLK; ++b) {
        const int c0 = b * PB;
        if (c0 >= kb) break;  // uniform
        if (wave == 0) {
            T x[PB], y[PB];
            T* xw = A + (c0 + li) + c0 * LDS;
            T* yw = lk == b ? WD + b * PB * LDP + li : A + lane + c0 * LDS;  // this lane's other row
            const int ys = lk == b ? LDP : LDS;
#pragma unroll
            for (int j = 0; j < PB; ++j) x[j] = xw[j * LDS];
#pragma unroll
            for (int j = 0; j < PB; ++j) y[j] = yw[j * ys];
            const int nk = min(PB, kb - c0), g0 = gc0 + c0;
            T *pb = pv + c0, *sb = sc + c0;
            unsigned fails = 0;
            if (invert_only) {
                // rows of A below the block are final: their results go to a spare place
                if (lk > b) yw = pv + NB + lane;
                const int yi = lk > b ? 0 : ys;
                if (chol) pivot_cols<T, PR_INV, 0>(x, y, F, g0, nk, true, pb, sb, xw, yw, yi, fails, lane);
                else pivot_cols<T, PR_INV_UNIT, 0>(x, y, F, g0, nk, false, pb, sb, xw, yw, yi, fails, lane);
            } else if (F.signs != nullptr || F.reg_kind != 0) {
                // signs or a regularization take the general form
                pivot_cols<T, PR_RULE, 0>(x, y, F, g0, nk, chol, pb, sb, xw, yw, ys, fails, lane);
            } else if (chol) {
                pivot_cols<T, PR_CHOL, 0>(x, y, F, g0, nk, true, pb, sb, xw, yw, ys, fails, lane);
            } else {
                pivot_cols<T, PR_LDLT, 0>(x, y, F, g0, nk, false, pb, sb, xw, yw, ys, fails, lane);
            }
            if (fails != 0 && lane == 0)
                atomicMin(F.info, (unsigned long long)(g0 + __builtin_ctz(fails) + 1));
        } else if (b > 0) {
            // the later block columns of the previous step, beside the pivots
            int q = 0;
            for (int w = 0; w < NBLK; ++w)
                for (int c = b + 1; c <= (w > b - 1 ? w : NBLK - 1); ++c, ++q)
                    if (q % 3 == wave - 1 && !(invert_only && w > b - 1)) update(w, b - 1, c);
        }
        __syncthreads();
        // the next block column
        if (b + 1 < NBLK && c0 + PB < kb && !(invert_only && wave > b)) update(wave, b, b + 1);
        __syncthreads();
    }
    // W(r, c) = L^-T(c, r): the panel solves wait for it.  All of a thread's
    // LDS reads first, then its stores.
    T* W = F.W + f.woff + k0;
    T v[NB / 4];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int c = cg + 4 * i, bc = i / 4, br = r / PB;
        const T* src = bc == br ? WD + bc * PB * LDP + (c & (PB - 1)) + (r & (PB - 1)) * LDP : A + c + r * LDS;
        v[i] = (c <= r) ? *src : (T)0;
    }
    pin(v);
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int c = cg + 4 * i;
        if (r < kb && c < kb) stc(W + r + (int64_t)c * f.nn, v[i]);
    }
    if (!invert_only && !chol && tid < kb) stc(F.d + gc0 + tid, pv[tid]);
}

// The factored tile, from LDS (as potrf_blocked leaves it) to the panel.
template <typename T>
__device__ __forceinline__ void store_diag(const DevFactor<T>& F, const Front f, int k0, const T* lds, const int tid) {
    const T* sc = lds + NB * LDS + (NB / PB) * PB * LDP;
    const int nj = f.nn + f.na, kb = min(NB, f.nn - k0), r = tid & 63, cg = tid >> 6;
    T* blk = F.panel + f.poff + k0 + (int64_t)k0 * nj;
    T v[NB / 4];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int c = cg + 4 * i;
        v[i] = lds[r + c * LDS] * (r > c ? sc[c] : (T)1);
    }
    pin(v);
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int c = cg + 4 * i;
        if (r < kb && c <= r) stc(blk + r + (int64_t)c * nj, v[i]);
    }
}

// A 64 x 64 tile of C in the row-contiguous layout of memory: thread (r, g)
// holds C(r, g + 4i).  The matrix cores' output registers hold 16 columns by
// 4 rows per instruction, 32-byte pieces of 16 cache lines; read and written
// like that a tile cost 2 us in loads and 3 us in stores, in this layout
// about 1 us each.  Products therefore leave through LDS (Cs, leading
// dimension LDS, complete on entry).
template <typename T>
__device__ __forceinline__ void fetch_c(const T* C, int64_t ldc_, int m, int n, T (&c)[NB / 4], const int tid) {
    const int r = min(tid & 63, m - 1), g = tid >> 6;
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) c[i] = ldc(C + r + min(g + 4 * i, n - 1) * ldc_);
}
// C = c - Cs (sub) or Cs
template <typename T, bool SUB>
__device__ __forceinline__ void write_c(T* C, int64_t ldc_, int m, int n, bool lower, const T (&c)[NB / 4],
                                        const T* Cs, const int tid) {
    const int r = tid & 63, g = tid >> 6;
    T x[NB / 4];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const T y = Cs[r + (g + 4 * i) * LDS];
        x[i] = SUB ? c[i] - y : y;
    }
    pin(x);
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int col = g + 4 * i;
        if (r < m && col < n && (!lower || r >= col)) stc(C + r + col * ldc_, x[i]);
    }
}

// The two products that follow a diagonal tile on the critical chain, by the
// workgroup that factored it (potrf_blocked has just returned: lds still
// holds L, W' = L^-T and the pivots): the panel solve of the tile below,
// L1 = A1 W' (/ D), and the update of the next diagonal tile,
// C -= L1 (D) L1'.  t: the panel solve's product, u: the update's.  W' is
// read from LDS (its zero blocks skipped), A1 goes straight from memory into
// the matrix cores' operand registers, and L1 takes the diagonal tile's place
// in LDS for the update.  The diagonal tile's own L leaves here, behind the
// loads, since no task waits for it.  The caller has seen A1 and C final
// through the previous block column.  keep: the next diagonal tile stays in
// LDS, where potrf_blocked's tile goes, instead of going to memory.  LDS:
// PTILE + NB * LDS elements.
template <typename T>
__device__ __forceinline__ void chain_step(const DevFactor<T>& F, const Front f, int k0, const GemmTask t,
                                           const GemmTask u, bool keep, T* lds, const int tid) {
    typedef typename Mfma<T>::v4 v4;
    constexpr int NBLK = NB / PB;
    T* A = lds;
    const T* WD = lds + NB * LDS;
    const T* pv = WD + NBLK * PB * LDP + NB;
    T* Cs = lds + PTILE;
    const int lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
    const bool chol = F.diag == 0;
    const int m = t.m, nj = t.lda;
    T* A1 = F.panel + t.a_off;
    T* C = F.panel + u.c_off;
    // rows 16 wave + li of A1 (t.k = 64 columns)
    T a[NB / 4], c[NB / 4];
    {
        const int row = min(PB * wave + li, m - 1);
#pragma unroll
        for (int s = 0; s < NB / 4; ++s) a[s] = ldc(A1 + row + (int64_t)(4 * s + lk) * nj);
    }
    fetch_c(C, nj, m, m, c, tid);
    store_diag<T>(F, f, k0, lds, tid);
    v4 acc[NBLK];
#pragma unroll
    for (int j = 0; j < NBLK; ++j) acc[j] = v4{0, 0, 0, 0};
#pragma unroll
    for (int kb = 0; kb < NBLK; ++kb)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = 4 * s + lk;
#pragma unroll
            for (int j = kb; j < NBLK; ++j) {
                const T b = j == kb ? WD[j * PB * LDP + k + li * LDP] : A[(PB * kb + k) + (PB * j + li) * LDS];
                acc[j] = Mfma<T>::op(a[4 * kb + s], b, acc[j]);
            }
        }
    if (!chol)
#pragma unroll
        for (int j = 0; j < NBLK; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[j][v] /= pv[PB * j + li];
    __syncthreads();  // every wavefront has read L and W'
    // L1 (rows past m are zero) takes the tile's place
#pragma unroll
    for (int j = 0; j < NBLK; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = PB * wave + Mfma<T>::row(lk, v);
            A[row + (PB * j + li) * LDS] = row < m ? acc[j][v] : (T)0;
        }
    __syncthreads();
    write_c<T, false>(A1, nj, m, NB, false, c, A, tid);
    // the ten 16 x 16 blocks (br, bc) of C's lower triangle: block q to
    // wavefront q % 4 (blocks past the tenth repeat block 0 and are dropped)
    const T *pa[3], *pb[3];
    int dst[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int e = wave + 4 * q;
        int br = e < 1 ? 0 : e < 3 ? 1 : e < 6 ? 2 : 3;
        int bc = e - br * (br + 1) / 2;
        if (e >= 10) br = bc = 0;
        pa[q] = A + PB * br + li + lk * LDS;
        pb[q] = A + PB * bc + li + lk * LDS;
        dst[q] = PB * br + (PB * bc + li) * LDS;
        acc[q] = v4{0, 0, 0, 0};
    }
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
        const T sc = chol ? (T)1 : pv[4 * s + lk];
#pragma unroll
        for (int q = 0; q < 3; ++q) acc[q] = Mfma<T>::op(pa[q][4 * s * LDS] * sc, pb[q][4 * s * LDS], acc[q]);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
        if (wave + 4 * q < 10)  // uniform
#pragma unroll
            for (int v = 0; v < 4; ++v) Cs[dst[q] + Mfma<T>::row(lk, v)] = acc[q][v];
    __syncthreads();
    if (!keep) {
        write_c<T, true>(C, nj, m, m, true, c, Cs, tid);
        return;
    }
    const int r = tid & 63, g = tid >> 6;
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int col = g + 4 * i;
        const T x = c[i] - Cs[r + col * LDS];
        A[r + col * LDS] = (r < m && col < m && col <= r) ? x : (r == col ? (T)1 : (T)0);
    }
}

// Diagonal tile under GMW81 (chol_factor! GMW81 specialization,
// cholesky.jl:739-875): every pivot takes the largest magnitude below it in
// the whole front column, so the task waits for its whole block column (each
// tile final through the previous block column) and reads the rows below the
// tile.  In the tile, right-looking column by column in LDS.  Below it,
// column j as it stands after the tile's pivots 0..j-1 is
//   a_ij - sum_{q<j} a_iq w_q,  w_q = sum_{p=q}^{j-1} l_jp W_pq,
// with a the block column's values (the panel solve has not run yet), l row j
// of the tile's L (unit for LDLt) and W = L^-1, built row by row alongside:
// W_jq = -w_q / l_jj (l_jj = 1 for LDLt), W_jj = 1 / l_jj.  L goes to the
// panel and W to the W pool, as the blocked path writes them.  LDS:
// 2 NB LDS + NB elements and 6 doubles.  Only the GMW81 instance of the
// persistent kernel holds it.
template <typename T>
__device__ __forceinline__ void potrf_gmw(const DevFactor<T>& F, const Front& f, int k0, T* lds,
                                          const int tid) {
    T* A = lds;                // the tile, 64 x LDS, lower triangle
    T* Wt = lds + NB * LDS;    // W = L^-1 of the tile, row by row
    T* w = Wt + NB * LDS;      // w of the current pivot
    double* s_red = (double*)(w + NB);  // per-wave maxima, then the pivot's l and 1 / l
    double& s_l = s_red[4];
    double& s_inv = s_red[5];
    const int nj = f.nn + f.na, kb = min(NB, f.nn - k0), gc0 = f.c0 + k0, nbelow = nj - k0;
    T* blk = F.panel + f.poff + k0 + (int64_t)k0 * nj;
    const int r = tid & 63, cg = tid >> 6, lane = tid & 63, wave = tid >> 6;
    const bool chol = F.diag == 0;
    for (int c = cg; c < NB; c += 4) {
        A[r + c * LDS] = (r < kb && c < kb && c <= r) ? ldc(blk + r + (int64_t)c * nj) : (r == c ? (T)1 : (T)0);
        Wt[r + c * LDS] = (T)0;
    }
    __syncthreads();
    for (int j = 0; j < kb; ++j) {
        // (1) w_q = sum_{p=q}^{j-1} l_jp W_pq, one thread per q < j
        if (tid < j) {
            T acc = (T)0;
            for (int p = tid; p < j; ++p) acc += A[j + p * LDS] * Wt[p + tid * LDS];
            w[tid] = acc;
        }
        __syncthreads();
        // (2) the largest magnitude below the pivot: tile rows from LDS, rows
        // below the tile from the block column
        double m = (r > j && r < kb && cg == 0) ? fabs((double)A[r + j * LDS]) : 0.0;
        // RB rows per thread and QB columns per step, as many independent loads
        // in flight (the rows are device-coherent loads from far memory, a
        // round trip a step: with 4 x 4 for every height a column of a band of
        // 100 took 6.7 us, 5.0 now); out-of-range rows and columns read row kb /
        // column 0 and are dropped
        auto below = [&](int i0, auto rows, auto cols) {
            constexpr int RB = decltype(rows)::value, QB = decltype(cols)::value;
            T acc[RB];
            int64_t ro[RB];
#pragma unroll
            for (int u = 0; u < RB; ++u) {
                const int i = i0 + tid + 256 * u;
                ro[u] = i < nbelow ? i : kb;
                acc[u] = ldc(blk + ro[u] + (int64_t)j * nj);
            }
            for (int q0 = 0; q0 < j; q0 += QB) {
                T a[QB][RB], wq[QB];
#pragma unroll
                for (int qq = 0; qq < QB; ++qq) {
                    const int q = q0 + qq < j ? q0 + qq : 0;
                    wq[qq] = q0 + qq < j ? w[q] : (T)0;
#pragma unroll
                    for (int u = 0; u < RB; ++u) a[qq][u] = ldc(blk + ro[u] + (int64_t)q * nj);
                }
#pragma unroll
                for (int qq = 0; qq < QB; ++qq)
#pragma unroll
                    for (int u = 0; u < RB; ++u) acc[u] -= a[qq][u] * wq[qq];
            }
#pragma unroll
            for (int u = 0; u < RB; ++u)
                if (i0 + tid + 256 * u < nbelow) m = jmax(m, fabs((double)acc[u]));
        };
        for (int i0 = kb; i0 < nbelow; i0 += 1024) {
            if (nbelow - i0 > 512) below(i0, std::integral_constant<int, 4>(), std::integral_constant<int, 4>());
            else if (nbelow - i0 > 256) below(i0, std::integral_constant<int, 2>(), std::integral_constant<int, 8>());
            else below(i0, std::integral_constant<int, 1>(), std::integral_constant<int, 16>());
        }
        m = wave_max(m);
        if (lane == 0) s_red[wave] = m;
        __syncthreads();
        if (tid == 0) {
            const double amax = jmax(jmax(s_red[0], s_red[1]), jmax(s_red[2], s_red[3]));
            const double piv = regularize_gmw(F, sign_of(F, gc0 + j), (double)A[j + j * LDS], amax);
            if (chol) {
                const double l = sqrt(piv);
                s_l = l;
                s_inv = 1.0 / l;
            } else {
                stc(F.d + gc0 + j, (T)piv);
                s_l = piv;
                s_inv = 1.0 / piv;
            }
        }
        __syncthreads();
        // (3) column j of L (the LDLt diagonal keeps the unregularized value)
        // and row j of W
        const T inv = (T)s_inv, pj = (T)s_l;
        if (cg == 0) {
            if (r > j && r < kb) A[r + j * LDS] *= inv;
            if (r == j && chol) A[j + j * LDS] = pj;
        } else if (cg == 1 && r <= j) {
            Wt[j + r * LDS] = r == j ? (chol ? inv : (T)1) : -w[r] * (chol ? inv : (T)1);
        }
        __syncthreads();
        // (4) rank-1 update of the trailing tile: a_rc -= l_rj (d_j) l_cj
        if (r > j && r < kb) {
            const T lr = A[r + j * LDS] * (chol ? (T)1 : pj);
            for (int c = j + 1 + cg; c <= r; c += 4) A[r + c * LDS] -= lr * A[c + j * LDS];
        }
        __syncthreads();
    }
    for (int c = cg; c < kb; c += 4)
        if (r < kb && c <= r) stc(blk + r + (int64_t)c * nj, A[r + c * LDS]);
    T* W = F.W + f.woff + k0;
    for (int c = cg; c < kb; c += 4)
        if (r < kb) stc(W + r + (int64_t)c * f.nn, (c <= r) ? Wt[r + c * LDS] : (T)0);
}

template <typename T>
__global__ __launch_bounds__(256) void k_diag(DevPlan P, DevFactor<T> F, int t0) {
    __shared__ T lds[PTILE];
    const DiagTask dt = P.diag[t0 + blockIdx.x];
    potrf_blocked<T>(F, P.fronts[dt.front], dt.k0, true, false, lds, (int)threadIdx.x);
}

template <typename T>
__device__ __forceinline__ T* arr_base(const DevFactor<T>& F, int a) {
    return a == ARR_PANEL ? F.panel : (a == ARR_U ? F.U : F.W);
}

// Sixteen bytes per lane from memory straight into LDS (lds: the wavefront's
// first lane's place, the lanes follow contiguously), device-coherent like
// ldc.  Only the global address's dword alignment is needed, so any row
// offset and leading dimension will do.
__device__ __forceinline__ void load_lds16(const void* g, void* lds) {
    typedef __attribute__((address_space(1))) const void gptr;
    typedef __attribute__((address_space(3))) void lptr;
    constexpr int SC1 = 16;  // device scope
    __builtin_amdgcn_global_load_lds((gptr*)g, (lptr*)lds, 16, 0, SC1);
}

// E x E output tile C -= A diag(s) B' (lower part only on the diagonal): the
// update-matrix tiles (E = 128 for long k) and the multi-step trailing
// updates (E = 64).  Wave w owns the (E/2) x (E/2) quarter (w & 1, w >> 1) as
// MFMA blocks (v_mfma_*_16x16x4: lane l holds A[l%16][l/16] and
// B[l/16][l%16]; the row of output register v is Mfma<T>::row); the strictly
// upper quarter of a diagonal tile does no MFMA work.  The k-loop runs on two
// LDS stages of KW columns of A and B (leading dimension E, no padding: every
// load instruction writes whole 128-byte lines): while the waves multiply out
// of one stage, the next chunk goes from memory straight into the other
// (load_lds16), one barrier per chunk.  Rows past the tile are loaded too
// (the panel pool has 2 NB elements of slack behind its end) and only reach
// rows and columns of C that are not stored.  C leaves through LDS in rounds
// (fetch_c's reason).  Bound: the matrix cores, which reach 75 TFLOP/s from
// LDS alone; FP64, 1,176 tiles of 128 x 128 x 512 on 512 workgroups in step:
// 43.9 TFLOP/s (52.7 before pin() ordered the stores of C, which left the
// DAG's task times as they were; 34.9 with the chunks staged through
// registers), 4,656 tiles of 64 x 64 x 512: 45.8 (39.4).
template <typename T, int E>
__device__ __forceinline__ void gemm_tile(const DevFactor<T>& F, const GemmTask g, T* S, const int tid) {
    typedef typename Mfma<T>::v4 v4;
    constexpr int KW = E == 128 ? 16 : 32;           // columns per stage
    constexpr int EPL = 16 / (int)sizeof(T);         // elements per lane and load
    constexpr int LPC = E / EPL, CPI = 64 / LPC;     // lanes per column, columns per load
    constexpr int ST = KW * E, M = E / 32, Q = E / 2;
    static_assert(4 * ST <= GEMM_LDS, "stages");
    const T* A = arr_base(F, g.arrA) + g.a_off;
    const T* B = arr_base(F, g.arrB) + g.b_off;
    T* C = arr_base(F, g.arrC) + g.c_off;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = (wave & 1) * Q, wc = (wave >> 1) * Q;
    const int li = lane & 15, lk = lane >> 4;
    const bool idle = g.lower && wc > wr;  // strictly above the diagonal
    const T* s = (F.diag != 0 && g.s_col >= 0) ? F.d + g.s_col : nullptr;
    v4 acc[M][M];
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) acc[i][j] = v4{0, 0, 0, 0};
    T sv[KW / 4];  // the LDLt pivots of the chunk in flight
    auto load = [&](int k0, T* st) {
        if (k0 + KW <= g.k) {
            const T* a = A + EPL * (lane % LPC) + (int64_t)(k0 + lane / LPC) * g.lda;
            const T* b = B + EPL * (lane % LPC) + (int64_t)(k0 + lane / LPC) * g.ldb;
#pragma unroll
            for (int i = 0; i < KW / CPI / 4; ++i) {
                const int k = (wave + 4 * i) * CPI;
                load_lds16(a + (int64_t)k * g.lda, st + k * E);
                load_lds16(b + (int64_t)k * g.ldb, st + ST + k * E);
            }
        } else {
            // the last, shorter chunk: its missing columns are zero
            for (int e = tid; e < ST; e += 256) {
                const int r = e % E, k = k0 + e / E;
                const T x = ldc(A + min(r, g.m - 1) + (int64_t)min(k, g.k - 1) * g.lda);
                const T y = ldc(B + min(r, g.n - 1) + (int64_t)min(k, g.k - 1) * g.ldb);
                st[e] = k < g.k ? x : (T)0;
                st[ST + e] = k < g.k ? y : (T)0;
            }
        }
        if (s)
#pragma unroll
            for (int i = 0; i < KW / 4; ++i) sv[i] = ldc(s + min(k0 + 4 * i + lk, g.k - 1));
    };
    load(0, S);
    int buf = 0;
    for (int k0 = 0; k0 < g.k; k0 += KW, buf ^= 1) {
        // the chunk has arrived (each wave waits for its own loads, then the
        // barrier) and the other stage is no longer read
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        T cs[KW / 4];
        if (s)
#pragma unroll
            for (int i = 0; i < KW / 4; ++i) cs[i] = sv[i];
        if (k0 + KW < g.k) load(k0 + KW, S + (buf ^ 1) * 2 * ST);
        if (!idle) {
            const T* a0 = S + buf * 2 * ST;
            const T* b0 = a0 + ST;
#pragma unroll
            for (int kk = 0; kk < KW; kk += 4) {
                T a[M], b[M];
#pragma unroll
                for (int i = 0; i < M; ++i) {
                    a[i] = a0[(kk + lk) * E + wr + 16 * i + li];
                    b[i] = b0[(kk + lk) * E + wc + 16 * i + li];
                }
                if (s)
#pragma unroll
                    for (int i = 0; i < M; ++i) a[i] *= cs[kk / 4];
#pragma unroll
                for (int i = 0; i < M; ++i)
#pragma unroll
                    for (int j = 0; j < M; ++j) acc[i][j] = Mfma<T>::op(a[i], b[j], acc[i][j]);
            }
        }
    }
    __syncthreads();  // every wave is done with the stages
    // C in rounds of NC columns: the wavefronts that own them put their
    // products in LDS (Cs: E x NC, over the stages), then every thread updates
    // row-contiguous pieces; the next round's C is fetched meanwhile
    constexpr int NC = 32, LDC = E + 1, CPER = E * NC / 256, CS = 256 / E;
    T* Cs = S;
    const int r = tid % E, kq = tid / E;
    T cv[CPER];
    auto fetch_round = [&](int q) {
#pragma unroll
        for (int i = 0; i < CPER; ++i)
            cv[i] = ldc(C + min(r, g.m - 1) + (int64_t)min(NC * q + kq + CS * i, g.n - 1) * g.ldc);
    };
    fetch_round(0);
#pragma unroll
    for (int q = 0; q < E / NC; ++q) {
        if (NC * q >= g.n) break;  // uniform
        if (NC * q / Q == wave >> 1 && !idle) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < M; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        Cs[(wr + 16 * i + Mfma<T>::row(lk, v)) + (16 * j + li) * LDC] = acc[i][(2 * q + j) % M][v];
        }
        __syncthreads();
        T x[CPER];
#pragma unroll
        for (int i = 0; i < CPER; ++i) x[i] = cv[i] - Cs[r + (kq + CS * i) * LDC];
        pin(x);
        if (q + 1 < E / NC) fetch_round(q + 1);
#pragma unroll
        for (int i = 0; i < CPER; ++i) {
            const int col = NC * q + kq + CS * i;
            if (r < g.m && col < g.n && (!g.lower || r >= col)) stc(C + r + (int64_t)col * g.ldc, x[i]);
        }
        __syncthreads();
    }
}

// 64 x 64 output tile with k <= 64 (every panel solve and the single-step
// trailing updates of the critical chain).  Wave w owns the rows
// [16w, 16w + 16): its A operand goes from memory straight into the matrix
// cores' operand registers, B is staged whole in LDS (Bs: 64 x LDT), so the
// tile costs one load round trip and one barrier.  The product is summed on
// its own and subtracted from C once (FP32 accuracy).  All loads are unconditional from clamped addresses.
// TRSM: B = W = L^-1 is lower triangular, the zero blocks are skipped.  Bound:
// the load round trip from the other XCDs' writes plus 40 (panel solve) or 64
// matrix-core operations of 64 cycles per wavefront; a full panel-solve tile
// on an idle chip takes 5.3 us (10.4 in two 32-wide chunks), a
// single-step update 6.2 us (7.4).
template <typename T, bool TRSM>
__device__ __forceinline__ void gemm_tile64(const DevFactor<T>& F, const GemmTask g, T* Bs, T* Cs, const int tid) {
    typedef typename Mfma<T>::v4 v4;
    constexpr int NBLK = NB / PB;
    const T* A = arr_base(F, g.arrA) + g.a_off;
    const T* B = arr_base(F, g.arrB) + g.b_off;
    T* C = arr_base(F, g.arrC) + g.c_off;
    const int wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const T* s = (!TRSM && F.diag != 0 && g.s_col >= 0) ? F.d + g.s_col : nullptr;
    T b[NB / 4], a[NB / 4], cv[NB / 4];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i)
        b[i] = ldc(B + min(lane, g.n - 1) + (int64_t)min(wave + 4 * i, g.k - 1) * g.ldb);
    const int row = PB * wave + li;
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) a[i] = ldc(A + min(row, g.m - 1) + (int64_t)min(4 * i + lk, g.k - 1) * g.lda);
    if constexpr (!TRSM) fetch_c(C, g.ldc, g.m, g.n, cv, tid);
    if (s) {
#pragma unroll
        for (int i = 0; i < NB / 4; ++i) a[i] *= ldc(s + min(4 * i + lk, g.k - 1));
    }
    // the LDLt pivots of this thread's columns
    T dcol[NBLK];
    if (TRSM && F.diag != 0)
#pragma unroll
        for (int j = 0; j < NBLK; ++j) dcol[j] = ldc(F.d + g.s_col + min(PB * j + li, g.n - 1));
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int k = wave + 4 * i;
        Bs[k * LDT + lane] = (k < g.k && lane < g.n) ? b[i] : (T)0;
        a[i] = 4 * i + lk < g.k ? a[i] : (T)0;
    }
    v4 acc[NBLK];
#pragma unroll
    for (int j = 0; j < NBLK; ++j) acc[j] = v4{0, 0, 0, 0};
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB / 4; ++i)
#pragma unroll
        for (int j = TRSM ? i / 4 : 0; j < NBLK; ++j)
            acc[j] = Mfma<T>::op(a[i], Bs[(4 * i + lk) * LDT + PB * j + li], acc[j]);
#pragma unroll
    for (int j = 0; j < NBLK; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            T x = acc[j][v];
            if (TRSM && F.diag != 0) x /= dcol[j];
            Cs[(PB * wave + Mfma<T>::row(lk, v)) + (PB * j + li) * LDS] = x;
        }
    __syncthreads();
    write_c<T, !TRSM>(C, g.ldc, g.m, g.n, g.lower != 0, cv, Cs, tid);
}

// Dependency q of DAG task d: the counter w that must reach target.  Returns
// false when d has no dependency q; *nw is the number of dependencies.
template <typename T, bool GMW>
__device__ __forceinline__ bool dag_dep(const DevPlan& P, const DevFactor<T>& F, const DevDag& D, const DagTask& d,
                        int q, int32_t** w, int* target, int* nw) {
    const int J = d.front;
    const DagFront g = D.df[J];
    int32_t* cnt = D.cnt + g.toff;
    switch (d.kind) {
        case DT_EA:
        case DT_SMALL: {  // children complete, earlier users of the U slot consumed
            const int g0 = D.gate_ptr[J];
            *nw = D.gate_ptr[J + 1] - g0;
            if (q >= *nw) return false;
            const int c = D.gate[g0 + q];
            *w = c < 0 ? F.flags + ~c : D.eacnt + c;
            *target = c < 0 ? D.df[~c].n_done : D.df[c].n_ea;
            return true;
        }
        case DT_POTRF:
            // the diagonal tile (the fused products wait for their own tiles
            // inside the task, after the factorization); under GMW81 every
            // tile of the block column, updated through the previous column
            *nw = GMW ? g.R - d.a : 1;
            if (q >= *nw) return false;
            *w = cnt + d.a * g.R + d.a + q;
            *target = d.a + 1;
            return true;
        case DT_TRSM:
            *nw = 2;
            if (q >= *nw) return false;
            *w = cnt + d.c * g.R + (q == 0 ? d.c : d.b);
            *target = q == 0 ? d.c + 2 : d.c + 1;
            return true;
        case DT_UPD: {  // columns [K0, K1): rows I, Jc final through K1 - 1
            const int K0 = d.d & 0xffff, K1 = d.d >> 16;
            *nw = 3;
            if (q >= *nw) return false;
            *w = q == 2 ? cnt + d.c * g.R + d.b : cnt + (K1 - 1) * g.R + (q == 0 ? d.b : d.c);
            *target = q == 2 ? K0 + 1 : K1 + 1;
            return true;
        }
        default: {  // DT_SYRK: the tile's row blocks of the panel are final, and
                    // every extend-add of the front (the update-matrix columns) is done
            *nw = 3 + (d.d & 1) + ((d.d >> 1) & 1);
            if (q >= *nw) return false;
            if (q == *nw - 1) {
                *w = D.eacnt + J;
                *target = g.n_ea;
                return true;
            }
            const int blk = q == 0 ? d.b : q == 1 ? d.c : (q == 2 && (d.d & 1)) ? d.b + 1 : d.c + 1;
            *w = cnt + (g.p - 1) * g.R + blk;
            *target = g.p + 1;
            return true;
        }
    }
}

// Tickets a workgroup holds at once, and lanes of wave 0 per held ticket
// (one dependency each).  Holding more than one ticket lets a workgroup run a
// later ready ticket first, but every held ticket then waits for its holder:
// measured on the 64^3 7-point Laplacian the launch took 36.4 ms with one
// ticket, 39.2 ms with two, 41.5 ms with four and 44.3 ms with eight.
constexpr int WIN = 1;
constexpr int WDEP = 64;
constexpr unsigned long long WMASK = WDEP == 64 ? ~0ull : (1ull << (WDEP & 63)) - 1;

// Thread 0's clocks of a finished task.
__device__ __forceinline__ void dag_clock(const DevDag& D, int kind, int t, unsigned long long& mark,
                                          unsigned long long begin) {
    const unsigned long long now = wall_clock64();
    if (D.trace) {
        D.trace[2 * t] = begin | ((unsigned long long)blockIdx.x << 48);
        D.trace[2 * t + 1] = now;
    }
    atomicAdd(D.prof + 3 * kind, begin - mark);
    atomicAdd(D.prof + 3 * kind + 1, now - begin);
    atomicAdd(D.prof + 3 * kind + 2, 1ull);
    mark = now;
}

// Persistent tile-DAG factorization of the big region.  Tickets are handed
// out in the planner's order (a list schedule, critical path first); a task
// depends only on tasks with smaller tickets.  Each workgroup holds WIN
// tickets and runs whichever of them is ready (the oldest first), so it
// blocks only when none of its tickets is ready.  The smallest unfinished
// ticket always belongs to some workgroup and is ready (its dependencies all
// have smaller tickets), so the launch is deadlock-free on any number of
// resident workgroups.  Counters:
//   F.flags[J]   finished update-matrix tiles of front J (1 for a small front)
//   D.eacnt[J]   finished extend-add tasks of J (1 for a small front)
//   D.cnt[toff_J + K*R_J + I]  tile (I, K) of the panel: 0 until its
//                extend-add is done (1 at the start where no child reaches the
//                tile), 1 + the panel columns applied, K+2 once it is final
// Synchronization per task: lanes of wave 0 poll the dependencies of the
// held tickets with relaxed loads (WDEP lanes per ticket).  Every value a
// task reads that another task of this launch wrote is loaded with a
// device-coherent (sc1) load, and every task output is stored with a
// device-coherent store, so no L2 write-back or invalidate is needed: at the
// end every wave drains its stores, the workgroup meets at a barrier, and
// thread 0 publishes with relaxed counter updates.  (Whole-L2 write-backs per
// task cost 3 ms of the 35 ms launch on the 64^3 Laplacian.)
// GMW: the GMW81 instance (diagonal tiles by potrf_gmw, block-column waits);
// the other regularizations run the instance without it.
template <typename T, bool GMW>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 2) void k_dag(DevPlan P, DevFactor<T> F, DevDag D) {
    constexpr int S1 = PTILE + NB * LDS, S2 = NB * LDT + NB * LDS, S3 = GEMM_LDS;
    constexpr int SMEM = S1 > S2 ? (S1 > S3 ? S1 : S3) : (S2 > S3 ? S2 : S3);
    static_assert(SMALL_NJ * LDS <= SMEM && 4 * EA_LDS <= SMEM && 32 * 129 <= SMEM, "LDS");
    static_assert(SMEM >= 2 * NB * LDS + NB + 6 * (int)(sizeof(double) / sizeof(T)), "potrf_gmw LDS");
    __shared__ __align__(16) T smem[SMEM];
    __shared__ T s_piv;
    __shared__ int s_fail, s_sel, s_drop;
    __shared__ int s_win[WIN];
    if (threadIdx.x == 0) s_drop = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < WIN; ++i) {
            const int t = (int)atomicAdd(F.ticket, 1u);
            s_win[i] = t < D.ntask ? t : -1;
        }
    __syncthreads();
    // wave 0, lane (slot, q): dependency q of the ticket held in slot
    int my_t = -3, my_tgt = 0, my_extra = 0, my_drop = 0;
    bool my_has = false;
    int32_t* my_w = nullptr;
    unsigned long long t_mark = 0;
    if (D.prof && threadIdx.x == 0) t_mark = wall_clock64();
    for (;;) {
        // an opaque copy of the thread index: values derived from it are
        // recomputed per task instead of being held (and spilled) across the
        // whole persistent loop
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        if (tid < 64) {
            const int slot = tid / WDEP, q = tid & (WDEP - 1);
            int sel = -1;
            Watch watch;
            for (int spins = 0;; ++spins) {
                const int t = s_win[slot];
                if (t != my_t) {  // a new ticket in this slot
                    my_t = t;
                    my_has = false;
                    my_extra = 0;
                    if (t >= 0) {
                        const DagTask dd = D.task[t];
                        int nw = 0;
                        my_has = dag_dep<T, GMW>(P, F, D, dd, q, &my_w, &my_tgt, &nw);
                        my_drop = dd.kind == DT_POTRF ? dd.a + 2 : 0;
                        if (q == 0 && nw > WDEP) my_extra = nw;
                    }
                }
                const int seen = my_has ? ld_rel(my_w) : my_tgt;
                bool ok = seen >= my_tgt;
                if (my_extra) {  // more dependencies than lanes (many children): checked here
                    const DagTask dd = D.task[my_t];
                    for (int k = WDEP; k < my_extra && ok; ++k) {
                        int32_t* w2;
                        int tg2, nw2;
                        if (dag_dep<T, GMW>(P, F, D, dd, k, &w2, &tg2, &nw2)) ok = ld_rel(w2) >= tg2;
                    }
                }
                const unsigned long long okm = __ballot(ok);
                if (tid == 0) {
                    int best = -1, bt = 0x7fffffff;
                    bool any = false;
                    for (int i = 0; i < WIN; ++i) {
                        const int ti = s_win[i];
                        if (ti < 0) continue;
                        any = true;
                        if (((okm >> (WDEP * i)) & WMASK) == WMASK && ti < bt) {
                            bt = ti;
                            best = i;
                        }
                    }
                    sel = any ? best : -2;
                    // the watchdog of mf_sync.h: progress is a satisfied
                    // dependency more or a ticket taken anywhere in the launch
                    if (sel == -1 && (spins & 255) == 255) {
                        if (ld_rel(F.hang)) {
                            sel = -2;
                        } else if (watch.expired(__popcll(okm), F.ticket, F.stall)) {
                            give_up(F.hang, my_w, my_tgt, my_w ? ld_rel(my_w) : 0, my_t);
                            sel = -2;
                        }
                    }
                }
                // a diagonal tile that the workgroup before it in the chain has
                // factored already: drop the ticket
                if (!GMW && tid == 0) s_drop = sel >= 0 && my_drop > 0 && seen >= my_drop;
                sel = __shfl(sel, 0);
                if (sel != -1) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (tid == 0) {
                s_sel = sel;
                s_fail = 0;
                const unsigned long long a0 = D.prof ? wall_clock64() : 0;
                // no acquire: every read of data this launch wrote is a
                // device-coherent load (ldc), so no cache needs an invalidate
                if (D.prof) atomicAdd(D.prof + 3 * DT_KINDS + 1, wall_clock64() - a0);
            }
        }
        __syncthreads();
        const int sel = s_sel;
        if (sel < 0) break;
        if (s_drop) {
            __syncthreads();
            if (tid == 0) {
                const int nt = (int)atomicAdd(F.ticket, 1u);
                s_win[sel] = nt < D.ntask ? nt : -1;
            }
            __syncthreads();
            continue;
        }
        int t = __builtin_amdgcn_readfirstlane(s_win[sel]);
        DagTask d = uniform(D.task[t]);
        const int J = d.front;
        const DagFront g = uniform(D.df[J]);
        int32_t* cnt = D.cnt + g.toff;
        unsigned long long t_begin = 0;
        if (D.prof && tid == 0) t_begin = wall_clock64();
        // critical-chain tasks may issue ahead of the co-resident workgroup's
        // matrix-core waves (wave priority; uniform branch)
        const bool raise = ((D.prio >> d.kind) & 1) ||
                           (((D.prio >> DT_KINDS) & 1) && d.kind == DT_UPD && d.c == (d.d >> 16));
        if (raise) __builtin_amdgcn_s_setprio(3);
        switch (d.kind) {
            case DT_EA: {
                for (int e = d.a; e < d.b; ++e) ea_tile<T>(P, F, uniform(P.ea[e]), smem, tid);
                break;
            }
            case DT_SMALL:
                small_front<T, false>(P, F, J, smem, &s_piv, &s_fail, tid);
                break;
            case DT_POTRF:
                for (bool resident = false;;) {
                    int tid = (int)threadIdx.x;  // opaque again: nothing derived is kept across steps
                    asm volatile("" : "+v"(tid));
                    if constexpr (GMW) potrf_gmw<T>(F, uniform(P.fronts[J]), d.a * NB, smem, tid);
                    else potrf_blocked<T>(F, uniform(P.fronts[J]), d.a * NB, false, resident, smem, tid);
                    if (d.b < 0) {
                        if constexpr (!GMW) store_diag<T>(F, uniform(P.fronts[J]), d.a * NB, smem, tid);
                        break;
                    }
                    // publish the diagonal tile (the other panel solves of column a
                    // need only it), then the fused panel solve of tile (a+1, a) and
                    // the update of the next diagonal tile, once both tiles are
                    // updated through column a - 1: set by tasks with smaller tickets
                    // (the planner checks), so the waits end.
                    // The next diagonal tile is then final through column a, and if
                    // its ticket d.d has been handed out, this workgroup factors it
                    // as well, from LDS: its holder waits for nothing else, finds
                    // the tile already final and drops the ticket.  (Every ticket
                    // before d.d has a holder then, so the fused step's waits end.)
                    // Otherwise the tile goes to memory for whoever takes it.
                    drain_stores();
                    __syncthreads();
                    if (tid == 0) {
                        __builtin_amdgcn_s_waitcnt(0);
                        __hip_atomic_store(cnt + d.a * g.R + d.a, d.a + 2, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                        const uint32_t taken = sync_ld(F.ticket);
                        (void)bounded_wait(cnt + d.a * g.R + d.a + 1, d.a + 1, F.hang, F.ticket, F.stall, 1);
                        (void)bounded_wait(cnt + (d.a + 1) * g.R + d.a + 1, d.a + 1, F.hang, F.ticket, F.stall, 1);
                        s_sel = (!GMW && taken > (uint32_t)d.d) ? 1 : 0;
                    }
                    __syncthreads();
                    const bool keep = __builtin_amdgcn_readfirstlane(s_sel) != 0;
                    if constexpr (GMW) {
                        gemm_tile64<T, true>(F, uniform(P.gemm[d.b]), smem, smem + NB * LDT, tid);
                        // the update reads the panel solve's tile back from memory
                        drain_stores();
                        __syncthreads();
                        gemm_tile64<T, false>(F, uniform(P.gemm[d.c]), smem, smem + NB * LDT, tid);
                    } else {
                        chain_step<T>(F, uniform(P.fronts[J]), d.a * NB, uniform(P.gemm[d.b]),
                                      uniform(P.gemm[d.c]), keep, smem, tid);
                    }
                    if (!keep) break;
                    drain_stores();
                    __syncthreads();
                    if (tid == 0) {
                        __hip_atomic_store(cnt + d.a * g.R + d.a + 1, d.a + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (D.prof) dag_clock(D, d.kind, t, t_mark, t_begin);
                        if (D.prof) t_begin = t_mark;
                    }
                    t = d.d;
                    d = uniform(D.task[t]);
                    resident = true;
                }
                break;
            default: {
                const GemmTask gt = uniform(P.gemm[d.a]);
                if (gt.wide) gemm_tile<T, 128>(F, gt, smem, tid);
                else if (gt.mode == G_TRSM) gemm_tile64<T, true>(F, gt, smem, smem + NB * LDT, tid);
                else if (gt.k <= NB) gemm_tile64<T, false>(F, gt, smem, smem + NB * LDT, tid);
                else gemm_tile<T, 64>(F, gt, smem, tid);
                break;
            }
        }
        if (raise) __builtin_amdgcn_s_setprio(0);
        drain_stores();
        __syncthreads();
        if (tid == 0) {
            if (D.prof) dag_clock(D, d.kind, t, t_mark, t_begin);
            const unsigned long long r0 = D.prof ? wall_clock64() : 0;
            // every task output is written through (device-coherent stores), and
            // every wave drained its stores before the barrier: no L2 write-back
            __builtin_amdgcn_s_waitcnt(0);
            constexpr int R = __ATOMIC_RELAXED, S = __HIP_MEMORY_SCOPE_AGENT;
            switch (d.kind) {
                case DT_EA:
                    for (int e = d.a; d.c && e < d.b; ++e)
                        __hip_atomic_store(cnt + P.ea[e].J * g.R + P.ea[e].I, 1, R, S);
                    __hip_atomic_fetch_add(D.eacnt + J, 1, R, S);
                    break;
                case DT_SMALL:
                    __hip_atomic_store(D.eacnt + J, 1, R, S);
                    __hip_atomic_store(F.flags + J, 1, R, S);
                    break;
                case DT_POTRF:
                    __hip_atomic_store(cnt + d.a * g.R + d.a, d.a + 2, R, S);
                    if (d.b >= 0) __hip_atomic_store(cnt + d.a * g.R + d.a + 1, d.a + 2, R, S);
                    if (d.c >= 0) __hip_atomic_store(cnt + (d.a + 1) * g.R + d.a + 1, d.a + 2, R, S);
                    break;
                case DT_TRSM: __hip_atomic_store(cnt + d.c * g.R + d.b, d.c + 2, R, S); break;
                case DT_UPD: __hip_atomic_store(cnt + d.c * g.R + d.b, (d.d >> 16) + 1, R, S); break;
                default: __hip_atomic_fetch_add(F.flags + J, 1, R, S); break;
            }
            const unsigned long long r1 = D.prof ? wall_clock64() : 0;
            const int nt = (int)atomicAdd(F.ticket, 1u);
            s_win[sel] = nt < D.ntask ? nt : -1;
            if (D.prof) {
                atomicAdd(D.prof + 3 * DT_KINDS, r1 - r0);
                atomicAdd(D.prof + 3 * DT_KINDS + 2, wall_clock64() - r1);
            }
        }
        // closes the thread-0 block before the back-edge
        __syncthreads();
    }
}

__global__ void k_copy_i32(const int32_t* src, int32_t* dst, int64_t count) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) dst[i] = src[i];
}

template <typename T>
__global__ void k_fill(T* p, int64_t count, T value) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) p[i] = value;
}

// Reference-layout Dval/Lval (assembled A, or a factor) -> internal panels
// (zeroed before); one workgroup per global column.  uplo 0 (:L): the
// diagonal block is nn x nn lower and the off-diagonal block na x nn;
// uplo 1 (:U): both transposed, the block above being nn x na
// (chordal_triangular.jl:852-926, 1015-1055).  adiag[g] receives the
// diagonal entry of column g.
template <typename T>
__global__ __launch_bounds__(256) void k_assemble_ref(DevPlan P, DevFactor<T> F,
                                                      const double* Dval, const double* Lval,
                                                      int uplo, double* adiag) {
    const int g = blockIdx.x;
    const OutFront o = P.out[P.col2ref[g]];
    const Front f = P.fronts[o.J];
    const int nj = f.nn + f.na, c = g - o.r0, cl = o.r0 - f.c0;
    T* col = F.panel + f.poff + (int64_t)(cl + c) * nj;
    if (uplo == 0) {
        for (int r = c + threadIdx.x; r < o.nn; r += blockDim.x)
            col[cl + r] = (T)Dval[o.Dp + r + (int64_t)c * o.nn];
        for (int i = threadIdx.x; i < o.na; i += blockDim.x)
            col[P.septpos[o.sepoff + i]] = (T)Lval[o.Lp + i + (int64_t)c * o.na];
    } else {
        for (int r = c + threadIdx.x; r < o.nn; r += blockDim.x)
            col[cl + r] = (T)Dval[o.Dp + c + (int64_t)r * o.nn];
        for (int i = threadIdx.x; i < o.na; i += blockDim.x)
            col[P.septpos[o.sepoff + i]] = (T)Lval[o.Lp + c + (int64_t)i * o.nn];
    }
    if (threadIdx.x == 0) adiag[g] = Dval[o.Dp + c + (int64_t)c * o.nn];
}

// setflatindex! for every nonzero into the panels (tp: panel slot or -1);
// td: the permuted column of a diagonal entry or -1 (adiag keeps the
// assembled diagonal for the LDLt copy-out of nn = 1 fronts).
template <typename T>
__global__ void k_refresh(DevFactor<T> F, const int64_t* tp, const int64_t* td, const double* x,
                          int64_t nnz, double* adiag) {
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnz) return;
    const double v = x[k];
    const int64_t p = tp[k];
    if (p >= 0) F.panel[p] = (T)v;
    const int64_t q = td[k];
    if (q >= 0) adiag[q] = v;
}

// Internal panels -> the reference's Dval/Lval/d; one workgroup per global
// column.  Every entry of the column's blocks is written (zeros outside the
// stored triangle), so the arrays need no clearing before.  uplo as for
// k_assemble_ref.
template <typename T>
__global__ __launch_bounds__(256) void k_copyout(DevPlan P, DevFactor<T> F, double* Dval,
                                                 double* Lval, double* dout, int uplo,
                                                 const double* adiag) {
    const int g = blockIdx.x;
    const OutFront o = P.out[P.col2ref[g]];
    const Front f = P.fronts[o.J];
    const int nj = f.nn + f.na, c = g - o.r0, cl = o.r0 - f.c0;
    const T* col = F.panel + f.poff + (int64_t)(cl + c) * nj;
    const bool keep_diag = (F.diag != 0 && o.nn == 1);  // chol_loop_nod!: Dval keeps A's entry
    if (Dval) {
        for (int r = threadIdx.x; r < o.nn; r += blockDim.x) {
            double v = r >= c ? (double)col[cl + r] : 0.0;
            if (r == c && keep_diag) v = adiag[g];
            if (uplo == 0) Dval[o.Dp + r + (int64_t)c * o.nn] = v;
            else Dval[o.Dp + c + (int64_t)r * o.nn] = v;
        }
    }
    if (Lval) {
        for (int i = threadIdx.x; i < o.na; i += blockDim.x) {
            const double v = (double)col[P.septpos[o.sepoff + i]];
            if (uplo == 0) Lval[o.Lp + i + (int64_t)c * o.na] = v;
            else Lval[o.Lp + c + (int64_t)i * o.nn] = v;
        }
    }
    if (dout && F.diag != 0 && threadIdx.x == 0) dout[g] = (double)F.d[g];
}

// dst[i] = (double)src[i]: the FP64 copy of an FP32 factor's panels that
// the FP64-arithmetic solves read.
__global__ void k_widen(const float* src, double* dst, int64_t count) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) dst[i] = (double)src[i];
}

inline int grid_for(int64_t count, int block) {
    int64_t g = (count + block - 1) / block;
    if (g > 65536) g = 65536;
    return (int)(g < 1 ? 1 : g);
}

}  // namespace

template <typename T>
void launch_fill(T* p, int64_t count, T value, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_fill<T>, dim3(grid_for(count, 256)), dim3(256), 0, s, p, count, value);
}

void launch_copy_i32(const int32_t* src, int32_t* dst, int64_t count, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_copy_i32, dim3(grid_for(count, 256)), dim3(256), 0, s, src, dst, count);
}

template <typename T>
void launch_assemble_ref(const DevPlan& P, const DevFactor<T>& F, const double* Dval,
                         const double* Lval, int uplo, double* adiag, hipStream_t s) {
    if (P.n <= 0) return;
    hipLaunchKernelGGL(k_assemble_ref<T>, dim3(P.n), dim3(256), 0, s, P, F, Dval, Lval, uplo,
                       adiag);
}

template <typename T>
void launch_refresh(const DevFactor<T>& F, const int64_t* tp, const int64_t* td,
                    const double* nzval, int64_t nnz, double* adiag, hipStream_t s) {
    if (nnz <= 0) return;
    hipLaunchKernelGGL(k_refresh<T>, dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, s, F, tp,
                       td, nzval, nnz, adiag);
}

template <typename T>
void launch_small(const DevPlan& P, const DevFactor<T>& F, int tickets, hipStream_t s) {
    if (tickets <= 0) return;
    const int grid = tickets < 2048 ? tickets : 2048;
    hipLaunchKernelGGL(k_small<T>, dim3(grid), dim3(256), 0, s, P, F, tickets);
}

template <typename T>
void launch_diag(const DevPlan& P, const DevFactor<T>& F, int t0, int t1, hipStream_t s) {
    if (t1 <= t0) return;
    hipLaunchKernelGGL(k_diag<T>, dim3(t1 - t0), dim3(256), 0, s, P, F, t0);
}

template <typename T>
void launch_dag(const DevPlan& P, const DevFactor<T>& F, const DevDag& D, hipStream_t s) {
    if (D.ntask <= 0) return;
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const bool gmw = F.reg_kind == 2;
    if (gmw) (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_dag<T, true>, 256, 0);
    else (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_dag<T, false>, 256, 0);
    if (D.wg_per_cu > 0 && D.wg_per_cu < per) per = D.wg_per_cu;
    int grid = std::max(1, cus) * std::max(1, per);
    if (grid > D.ntask) grid = D.ntask;
    if (gmw) hipLaunchKernelGGL((k_dag<T, true>), dim3(grid), dim3(256), 0, s, P, F, D);
    else hipLaunchKernelGGL((k_dag<T, false>), dim3(grid), dim3(256), 0, s, P, F, D);
}

// gmw81_beta (gmw81.jl:74-101): the largest diagonal and off-diagonal
// magnitudes of the assembled matrix (the panels hold A before the
// factorization), one workgroup per internal front, combined with atomicMax
// on the bit patterns (non-negative doubles order as their bits; a NaN
// orders above every number and propagates).
template <typename T>
__global__ __launch_bounds__(256) void k_gmw_reduce(DevPlan P, DevFactor<T> F, unsigned long long* acc) {
    const Front f = P.fronts[blockIdx.x];
    const int nj = f.nn + f.na;
    const T* pn = F.panel + f.poff;
    double g = 0.0, x = 0.0;
    const int64_t total = (int64_t)nj * f.nn;
    for (int64_t e = threadIdx.x; e < total; e += 256) {
        const int c = (int)(e / nj), r = (int)(e - (int64_t)c * nj);
        if (r < c) continue;
        const double v = fabs((double)pn[e]);
        if (r == c) g = jmax(g, v);
        else x = jmax(x, v);
    }
    g = wave_max(g);
    x = wave_max(x);
    if ((threadIdx.x & 63) == 0) {
        atomicMax(acc, (unsigned long long)__builtin_bit_cast(unsigned long long, g));
        atomicMax(acc + 1, (unsigned long long)__builtin_bit_cast(unsigned long long, x));
    }
}

// beta = max(gamma, xi / sqrt(n^2 - 1), eps(T)), rounded to T
__global__ void k_gmw_final(double* gmw, double n, double eps_t, int f32) {
    const unsigned long long* acc = (const unsigned long long*)gmw;
    const double gamma = __builtin_bit_cast(double, acc[0]), xi = __builtin_bit_cast(double, acc[1]);
    const double b = jmax(jmax(gamma, xi / sqrt(n * n - 1.0)), eps_t);
    gmw[2] = f32 ? (double)(float)b : b;
}

template <typename T>
void launch_gmw_beta(const DevPlan& P, const DevFactor<T>& F, double* gmw, int64_t n, hipStream_t s) {
    launch_fill<unsigned long long>((unsigned long long*)gmw, 2, 0ull, s);
    if (P.nJ > 0)
        hipLaunchKernelGGL(k_gmw_reduce<T>, dim3(P.nJ), dim3(256), 0, s, P, F, (unsigned long long*)gmw);
    const double eps_t = sizeof(T) == 4 ? 1.1920928955078125e-07 : 2.220446049250313e-16;
    hipLaunchKernelGGL(k_gmw_final, dim3(1), dim3(1), 0, s, gmw, (double)n, eps_t, sizeof(T) == 4 ? 1 : 0);
}

void launch_widen(const float* src, double* dst, int64_t count, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_widen, dim3(grid_for(count, 256)), dim3(256), 0, s, src, dst, count);
}

template <typename T>
void launch_copyout(const DevPlan& P, const DevFactor<T>& F, double* Dval, double* Lval,
                    double* dout, int uplo, const double* adiag, hipStream_t s) {
    if (P.n <= 0) return;
    hipLaunchKernelGGL(k_copyout<T>, dim3(P.n), dim3(256), 0, s, P, F, Dval, Lval, dout, uplo,
                       adiag);
}

#define MF_INST(T)                                                                              \
    template void launch_fill<T>(T*, int64_t, T, hipStream_t);                                  \
    template void launch_assemble_ref<T>(const DevPlan&, const DevFactor<T>&, const double*,    \
                                         const double*, int, double*, hipStream_t);             \
    template void launch_refresh<T>(const DevFactor<T>&, const int64_t*, const int64_t*,        \
                                    const double*, int64_t, double*, hipStream_t);              \
    template void launch_small<T>(const DevPlan&, const DevFactor<T>&, int, hipStream_t);                            \
    template void launch_copyout<T>(const DevPlan&, const DevFactor<T>&, double*, double*,      \
                                    double*, int, const double*, hipStream_t);                  \
    template void launch_dag<T>(const DevPlan&, const DevFactor<T>&, const DevDag&, hipStream_t); \
    template void launch_gmw_beta<T>(const DevPlan&, const DevFactor<T>&, double*, int64_t, hipStream_t);
MF_INST(double)
MF_INST(float)
template void launch_diag<double>(const DevPlan&, const DevFactor<double>&, int, int, hipStream_t);
template void launch_fill<int32_t>(int32_t*, int64_t, int32_t, hipStream_t);
template void launch_fill<uint32_t>(uint32_t*, int64_t, uint32_t, hipStream_t);
template void launch_fill<unsigned long long>(unsigned long long*, int64_t, unsigned long long,
                                              hipStream_t);

}  // namespace mf
