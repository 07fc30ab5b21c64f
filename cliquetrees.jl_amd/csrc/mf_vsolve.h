// mf_vsolve.h — what the triangular-solve kernels share (device code only):
// values that are their own flags, uniform records, small panels in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mf_kernels.h"
#include "mf_sync.h"

namespace mf {

namespace {

template <typename T>
using bits_t = typename std::conditional<sizeof(T) == 8, unsigned long long, uint32_t>::type;
// Signalling NaNs: every arithmetic instruction returns a quiet one.
template <typename T>
__device__ __forceinline__ constexpr bits_t<T> unset() {
    if constexpr (sizeof(T) == 8) return 0x7FF4A5A5DEADBEE1ull;
    else return 0x7FA5A5A5u;
}
template <typename T>
__device__ __forceinline__ constexpr bits_t<T> quiet() {
    if constexpr (sizeof(T) == 8) return 0x7FF8000000000000ull;
    else return 0x7FC00000u;
}

template <typename T>
__device__ __forceinline__ bits_t<T> peek(const T* p) {
    return __hip_atomic_load(reinterpret_cast<const bits_t<T>*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void publish(T* p, T v) {
    bits_t<T> b = __builtin_bit_cast(bits_t<T>, v);
    if (b == unset<T>()) b = quiet<T>();
    __hip_atomic_store(reinterpret_cast<bits_t<T>*>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A right-hand side entry that has been read (its owner is its only reader)
// becomes the unset solution entry of the backward launch.
template <typename T>
__device__ __forceinline__ void wipe(T* p) {
    *reinterpret_cast<bits_t<T>*>(p) = unset<T>();
}

// What a wait needs: the watchdog's record and the counter that shows progress.
struct Ctl {
    int32_t* hang;
    const uint32_t* ticket;
    unsigned long long stall;
};

// The value at p once it is set; v is an earlier peek at it.  Whole
// wavefronts: lanes that want nothing pass on = false (with a valid p) and
// get 0.
template <typename T>
__device__ __forceinline__ T settle(bits_t<T> v, const T* p, bool on, const Ctl& c) {
    if (__any(on && v == unset<T>())) {
        Watch w;
        for (int spins = 1;; ++spins) {
            v = peek(p);
            if (!__any(on && v == unset<T>())) break;
            if ((spins & 255) == 0) {
                // once any wait has given up, every other wait returns at once
                if (sync_ld(c.hang)) break;
                if (w.expired(0, c.ticket, c.stall)) {
                    if (on && v == unset<T>()) give_up(c.hang, reinterpret_cast<const int32_t*>(p), 1, 0, -1);
                    break;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    return on ? __builtin_bit_cast(T, v) : (T)0;
}

// LDS traffic inside one wavefront completes in order; this keeps the
// compiler from reordering it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
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
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// A front's record in scalar registers (the front is uniform).
__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (int64_t)((unsigned long long)lo | ((unsigned long long)hi << 32));
}
__device__ __forceinline__ Front front_of(const DevPlan& P, int J) {
    Front f = P.fronts[J];
    f.poff = uni(f.poff);
    f.woff = uni(f.woff);
    f.c0 = uni(f.c0);
    f.nn = uni(f.nn);
    f.na = uni(f.na);
    f.rowoff = uni(f.rowoff);
    f.chd0 = uni(f.chd0);
    f.chd1 = uni(f.chd1);
    return f;
}

// y / d: the reciprocal of d is taken once, ahead of the substitution chain,
// and one correction step gives the quotient its last bits (q + r (y - q d)).
// `exact` (uniform): some reciprocal is not a normal number, divide instead.
template <typename T>
__device__ __forceinline__ T quot(T y, T d, T rd, bool exact) {
    if (exact) return y / d;
    const T q = y * rd, c = fma_(fma_(-q, d, y), rd, q);
    return __builtin_isfinite(q) ? c : q;
}
template <typename T>
__device__ __forceinline__ bool abnormal(T v) {
    return !__builtin_isnormal(v);
}

// ---- small fronts (nJ <= 64), one wavefront each ------------------------------

// The front's panel (contiguous, leading dimension nj) into Ps with leading
// dimension nj | 1 (odd: rows and columns are both read without conflicts).
template <typename T>
__device__ __forceinline__ void stage_panel(const T* Pj, int nj, int nn, T* Ps) {
    const int lane = threadIdx.x & 63, tot = nj * nn, ld = nj | 1;
    // e / nj for e < 4096, nj <= 64: (e * ceil(2^20 / nj)) >> 20 (nj >= 2; nj = 1 has e = 0)
    const uint32_t mul = nj > 1 ? ((1u << 20) / (uint32_t)nj + 1) : 0;
    for (int e0 = 0; e0 < tot; e0 += 64 * 8) {
        T v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Pj[min(e0 + 64 * i + lane, tot - 1)];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = e0 + 64 * i + lane;
            const int c = (int)(((uint32_t)e * mul) >> 20);
            if (e < tot) Ps[e - c * nj + c * ld] = v[i];
        }
    }
}

// The staged panel with every column divided by its diagonal entry (L = L' D,
// L' unit lower): the substitution chains then hold no division, and the
// divisions by D run in all rows at once, before (backward) or after
// (forward) the chain.  Rows r = lane; the diagonal keeps D; `d`, `rd`,
// `exact`: D, its reciprocal and the flag of quot for this lane's column.
template <typename T>
__device__ __forceinline__ void scale_panel(int nj, int nn, T* Ps, bool unit, T& d, T& rd, bool& exact) {
    const int r = threadIdx.x & 63, ld = nj | 1, rr = min(r, nn - 1);
    d = unit ? (T)1 : Ps[rr + rr * ld];
    rd = (T)1 / d;
    exact = __any(abnormal(rd));
    if (unit) return;
    for (int c = 0; c < nn; ++c) {
        const T dc = lane_of(d, c), rc = lane_of(rd, c);
        if (r > c && r < nj) Ps[r + c * ld] = quot(Ps[r + c * ld], dc, rc, exact);
    }
    wave_sync();
}

}  // namespace

}  // namespace mf
