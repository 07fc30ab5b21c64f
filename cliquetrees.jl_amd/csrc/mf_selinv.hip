// mf_selinv.hip — gfx950 kernel of the selected inversion of a Cholesky
// factor (selinv!, src/Multifrontal.jl/src/selinv.jl:38-424).
//
//   k_selinv   persistent: workgroups take tickets of the schedule built by
//              mf_selinv_plan.cpp (root first) and run one task each:
//              ST_XDIAG   X(K, K) = W_K, a diagonal tile of L11^-1 from the
//                         factor's inverted 64 x 64 tiles
//              ST_GEMM    one tile of at most 64 x 64, C = sum of up to two products
//                         sgn A B' (operands plain or transposed), on MFMA:
//                         the recursion of X = L11^-1, Lt = L21 X,
//                         Sigma21 = -M Lt, Sigma11 = X' X - Lt' Sigma21
//              ST_GATHER  a tile of M = Sigma(sep, sep) from the parent's
//                         frontal matrix and its mirror image (selinv_send!,
//                         copygathertri!, utils.jl:529-553)
//              ST_SMALL   a whole front with nJ <= 64 in LDS
//              (selinv_loop_snd!/nod!, selinv.jl:122-379).
// Synchronization is the tile-DAG factorization's: a task waits (bounded,
// mf_sync.h) on counters advanced only by tasks with smaller tickets; every
// value a task reads that this launch wrote is a device-coherent load and
// every output a device-coherent store; a task publishes once all its waves
// drained their stores and met at a barrier.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mf_kernels.h"
#include "mf_mfma.h"
#include "mf_sync.h"
#include "mf_vsolve.h"

namespace mf {

namespace {

template <typename T>
__device__ __forceinline__ T ldc(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void stc(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void drain_stores() { __builtin_amdgcn_s_waitcnt(0); }

constexpr int FLD = 64 + 1;  // leading dimension of LDS fronts and tiles

// One output tile of at most E x E: acc = sum over the task's products of
// sgn A B', then C = acc (lower triangle only for a diagonal tile).  Wave w
// owns the quarter (w & 1, w >> 1), E/32 x E/32 MFMA blocks.  Each chunk of
// KC inner columns of A and B goes through LDS; the next chunk is fetched
// into registers while the current one is multiplied.  A plain operand is
// fetched down its columns (lane = row), a transposed one along its rows
// (lane = k), so both are coalesced; the loads are unconditional (clamped)
// and the predicates applied when they go to LDS.
//
// E = 64, KC = 32 and E = 32, KC = 128 hold the same 2048 and 4096 values an
// operand; both spend 32 matrix instructions a wavefront (0.9 us in FP64) on
// a chunk, so a 32-wide tile runs its inner dimension four times as fast.
// The tiles of one front's phase rarely fill the chip and the phases down the
// tree are a chain, so phases of few tiles take the small one (28 x 30 x 26
// grid, with the gathers a task per tile: 2553 -> 1192 us).
template <typename T, int E, int KC>
__device__ __forceinline__ void sel_tile(const DevSel<T>& S, const SelTask& t, const SelPart* parts, T* As, T* Bs,
                                         const int tid) {
    typedef typename Mfma<T>::v4 v4;
    constexpr int PER = KC * E / 256, LD = E + 1, Q = E / 32, RS = 256 / KC, KS = 256 / E;
    const int wave = tid >> 6, lane = tid & 63;
    const int wr = (wave & 1) * (E / 2), wc = (wave >> 1) * (E / 2);
    const int li = lane & 15, lk = lane >> 4;
    v4 acc[Q][Q];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int j = 0; j < Q; ++j) acc[i][j] = v4{0, 0, 0, 0};
    // element i of this thread in a chunk: plain (row tid % E, k tid / E + KS i),
    // transposed (row tid / KC + RS i, k tid % KC)
    // (A, lda uniform: one base in scalar registers and a lane offset a load)
    auto fetch = [&](const T* A, int lda, bool tr, int rows, int k0, int k1, T (&v)[PER]) {
        const T* q = A + (tr ? (int64_t)k0 : (int64_t)k0 * lda);
        const int kn = k1 - k0;
        if (tr) {
            const uint32_t k = min(tid % KC, kn - 1);
#pragma unroll
            for (int i = 0; i < PER; ++i) v[i] = ldc(q + (k + (uint32_t)min(tid / KC + RS * i, rows - 1) * (uint32_t)lda));
        } else {
            const uint32_t r = min(tid % E, rows - 1);
#pragma unroll
            for (int i = 0; i < PER; ++i) v[i] = ldc(q + (r + (uint32_t)min(tid / E + KS * i, kn - 1) * (uint32_t)lda));
        }
    };
    auto put = [&](const T (&v)[PER], bool tr, int rows, int k0, int k1, T sg, T* X) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int r = tr ? tid / KC + RS * i : tid % E, k = tr ? tid % KC : tid / E + KS * i;
            X[k * LD + r] = (r < rows && k0 + k < k1) ? sg * v[i] : (T)0;
        }
    };
    for (int q = 0; q < t.np; ++q) {
        SelPart p = parts[q];
        p.a_off = uni(p.a_off);
        p.b_off = uni(p.b_off);
        p.lda = uni(p.lda);
        p.ldb = uni(p.ldb);
        p.k = uni(p.k);
        p.ta = (int8_t)uni((int32_t)p.ta);
        p.tb = (int8_t)uni((int32_t)p.tb);
        p.arrA = (int8_t)uni((int32_t)p.arrA);
        p.arrB = (int8_t)uni((int32_t)p.arrB);
        const T* A = S.base[p.arrA] + p.a_off;
        const T* B = S.base[p.arrB] + p.b_off;
        T ra[PER], rb[PER];
        fetch(A, p.lda, p.ta, t.m, 0, p.k, ra);
        fetch(B, p.ldb, p.tb, t.n, 0, p.k, rb);
        for (int k0 = 0; k0 < p.k; k0 += KC) {
            put(ra, p.ta, t.m, k0, p.k, (T)p.sgn, As);
            put(rb, p.tb, t.n, k0, p.k, (T)1, Bs);
            __syncthreads();
            if (k0 + KC < p.k) {
                fetch(A, p.lda, p.ta, t.m, k0 + KC, p.k, ra);
                fetch(B, p.ldb, p.tb, t.n, k0 + KC, p.k, rb);
            }
            const int ke = min(KC, (p.k - k0 + 3) & ~3);
#pragma unroll 8
            for (int kk = 0; kk < ke; kk += 4) {
                T a[Q], b[Q];
#pragma unroll
                for (int i = 0; i < Q; ++i) a[i] = As[(kk + lk) * LD + wr + 16 * i + li];
#pragma unroll
                for (int j = 0; j < Q; ++j) b[j] = Bs[(kk + lk) * LD + wc + 16 * j + li];
#pragma unroll
                for (int i = 0; i < Q; ++i)
#pragma unroll
                    for (int j = 0; j < Q; ++j) acc[i][j] = Mfma<T>::op(a[i], b[j], acc[i][j]);
            }
            __syncthreads();
        }
    }
    T* C = S.base[t.arrC] + t.c_off;
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int j = 0; j < Q; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = wr + i * 16 + Mfma<T>::row(lk, v), col = wc + j * 16 + li;
                if (row < t.m && col < t.n && (!t.lower || row >= col))
                    stc(C + row + (int64_t)col * t.ldc, acc[i][j][v]);
            }
}

// X(K, K) = W_K (kb x kb, zeros above the diagonal included).
template <typename T>
__device__ void sel_xdiag(const DevPlan& P, const DevSel<T>& S, int J, int K, const int tid) {
    const Front f = P.fronts[J];
    const int kb = min(NB, f.nn - NB * K);
    const T* W = S.base[SP_W] + f.woff + (int64_t)NB * K;
    T* X = S.base[SP_X] + S.xoff[J] + (int64_t)NB * K + (int64_t)NB * K * f.nn;
    const int r = tid & 63;
    for (int c = tid >> 6; c < kb; c += 4)
        if (r < kb) stc(X + r + (int64_t)c * f.nn, ldc(W + r + (int64_t)c * f.nn));
}

// Address of an element of the parent's frontal matrix [Sigma11, .; Sigma21, M]
// (lower triangle, p >= q, positions in the parent's row list).
template <typename T>
__device__ __forceinline__ const T* parent_addr(const T* sig, const T* M, int nn, int na, int p, int q) {
    return q < nn ? sig + p + (int64_t)q * (nn + na) : M + (p - nn) + (int64_t)(q - nn) * na;
}

// Tile (ib, jb), ib >= jb, of M and its mirror image above the diagonal:
// M(a, b) = F_parent(rel[max(a, b)], rel[min(a, b)]).  All of a thread's
// sixteen elements load at once (one at a time, with a store after each, a
// tile took sixteen trips to memory).
template <typename T>
__device__ void sel_gather(const DevPlan& P, const DevSel<T>& S, int J, int jb, int ib, T* Ts, const int tid) {
    const Front f = P.fronts[J];
    const Front pf = P.fronts[f.parent];
    const int32_t* rel = P.rel + f.reloff;
    T* M = S.base[SP_M] + S.moff[J];
    const T* sig = S.base[SP_SIG] + pf.poff;
    const T* pM = S.base[SP_M] + S.moff[f.parent];
    const int na = f.na, b0 = NB * jb, cb = min(NB, na - b0), a0 = NB * ib, rb = min(NB, na - a0);
    const int r = tid & 63, g = tid >> 6;
    const int ra = rel[min(a0 + r, na - 1)];
    T v[NB / 4];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int rc = rel[min(b0 + g + 4 * i, na - 1)];  // rel is increasing
        v[i] = ldc(parent_addr(sig, pM, pf.nn, pf.na, max(ra, rc), min(ra, rc)));
    }
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int c = g + 4 * i;
        if (r < rb && c < cb) stc(M + (a0 + r) + (int64_t)(b0 + c) * na, v[i]);
        Ts[r + c * FLD] = v[i];
    }
    if (ib == jb) return;
    __syncthreads();
    // the mirrored tile, written down its columns
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) v[i] = Ts[(g + 4 * i) + r * FLD];
#pragma unroll
    for (int i = 0; i < NB / 4; ++i)
        if (r < cb && g + 4 * i < rb) stc(M + (b0 + r) + (int64_t)(a0 + g + 4 * i) * na, v[i]);
}

// A whole front with nJ <= 64 in LDS: L = [L11; L21] in Lf (ld FLD), M in
// Mf; Lt = L21 L11^-1 and X = L11^-1 in place, Sigma21 = -M Lt into Mf,
// Sigma11 = X' X - Lt' Sigma21 straight to the output panel.  Up to eight
// columns a wavefront load at once, in pairs that stop at the front's last (a
// chain of fronts of nine columns, 8.3 us a front; 9.3 with all eight always).
template <typename T>
__device__ void sel_small(const DevPlan& P, const DevSel<T>& S, int J, T* Lf, T* Mf, const int tid) {
    const Front f = P.fronts[J];
    const int nn = f.nn, na = f.na, nJ = nn + na;
    const T* Lp = S.base[SP_PANEL] + f.poff;
    const int r = tid & 63, g = uni(tid >> 6);
    for (int c0 = g; c0 < nn; c0 += 32) {
        T v[8];
#pragma unroll
        for (int h = 0; h < 8; h += 2) {
            if (c0 + 4 * h >= nn) break;  // uniform
#pragma unroll
            for (int i = h; i < h + 2; ++i) v[i] = Lp[min(r, nJ - 1) + (int64_t)min(c0 + 4 * i, nn - 1) * nJ];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (r < nJ && c0 + 4 * i < nn) Lf[r + (c0 + 4 * i) * FLD] = v[i];
    }
    if (na > 0) {
        const Front pf = P.fronts[f.parent];
        const T* sig = S.base[SP_SIG] + pf.poff;
        const T* pM = S.base[SP_M] + S.moff[f.parent];
        const int32_t* rel = P.rel + f.reloff;
        T* Mo = S.base[SP_M] + S.moff[J];
        const bool keep = f.chd1 > f.chd0;  // the children gather from it
        const int ra = rel[min(r, na - 1)];
        for (int c0 = g; c0 < na; c0 += 32) {
            T v[8];
#pragma unroll
            for (int h = 0; h < 8; h += 2) {
                if (c0 + 4 * h >= na) break;  // uniform
#pragma unroll
                for (int i = h; i < h + 2; ++i) {
                    const int rc = rel[min(c0 + 4 * i, na - 1)];
                    v[i] = ldc(parent_addr(sig, pM, pf.nn, pf.na, max(ra, rc), min(ra, rc)));
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int c = c0 + 4 * i;
                if (r < na && c < na) {
                    Mf[r + c * FLD] = v[i];
                    if (keep) stc(Mo + r + (int64_t)c * na, v[i]);
                }
            }
        }
    }
    __syncthreads();
    // Lt = L21 L11^-1, last column first: Lt(:, c) = L21'(:, c) / L(c, c), then
    // L21'(:, j) -= Lt(:, c) L(c, j) for j < c
    for (int c = nn - 1; c >= 0 && na > 0; --c) {
        const T inv = (T)1 / Lf[c + c * FLD];
        if (tid < na) Lf[nn + tid + c * FLD] *= inv;
        __syncthreads();
        if (r < na)
            for (int j = g; j < c; j += 4) Lf[nn + r + j * FLD] -= Lf[nn + r + c * FLD] * Lf[c + j * FLD];
        __syncthreads();
    }
    // X = L11^-1 in place, last column first: X(i, j) = -X(j, j) sum_{k=j+1}^{i} X(i, k) L(k, j)
    for (int j = nn - 1; j >= 0; --j) {
        const T xjj = (T)1 / Lf[j + j * FLD];
        T v = (T)0;
        const int i = j + 1 + tid;
        if (i < nn) {
            T s = (T)0;
            for (int k = j + 1; k <= i; ++k) s += Lf[i + k * FLD] * Lf[k + j * FLD];
            v = -xjj * s;
        }
        __syncthreads();
        if (i < nn) Lf[i + j * FLD] = v;
        if (tid == 0) Lf[j + j * FLD] = xjj;
        __syncthreads();
    }
    // Sigma21 = -M Lt (na x nn, at most 4 entries per thread), then into Mf
    T s21[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = tid + 256 * q;
        T s = (T)0;
        if (e < na * nn) {
            const int r = e % na, c = e / na;
            for (int k = 0; k < na; ++k) s += Mf[r + k * FLD] * Lf[nn + k + c * FLD];
        }
        s21[q] = -s;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = tid + 256 * q;
        if (e < na * nn) Mf[e % na + (e / na) * FLD] = s21[q];
    }
    __syncthreads();
    T* Sg = S.base[SP_SIG] + f.poff;
    for (int e = tid; e < nJ * nn; e += 256) {
        const int r = e % nJ, c = e / nJ;
        T v = (T)0;
        if (r >= nn) {
            v = Mf[(r - nn) + c * FLD];
        } else if (r >= c) {
            for (int k = r; k < nn; ++k) v += Lf[k + r * FLD] * Lf[k + c * FLD];
            T s = (T)0;
            for (int k = 0; k < na; ++k) s += Lf[nn + k + r * FLD] * Mf[k + c * FLD];
            v -= s;
        }
        stc(Sg + r + (int64_t)c * nJ, v);
    }
}

template <typename T>
__global__ __launch_bounds__(256, 2) void k_selinv(DevPlan P, DevSel<T> S) {
    constexpr int SM1 = 2 * 64 * FLD, SM2 = 2 * 128 * 33;
    __shared__ T smem[SM1 > SM2 ? SM1 : SM2];
    __shared__ int s_t;
    for (;;) {
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        if (tid == 0) s_t = (int)atomicAdd(S.ticket, 1u);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(s_t);
        __syncthreads();
        if (t >= S.ntask) break;
        const SelTask tk = S.task[t];
        if (tid == 0)
            for (int w = 0; w < 2; ++w)
                if (tk.wait[w] >= 0) (void)bounded_wait(S.cnt + tk.wait[w], tk.target[w], S.hang, S.ticket, S.stall, 1);
        __syncthreads();
        switch (tk.kind) {
            case ST_XDIAG: sel_xdiag<T>(P, S, tk.front, tk.a, tid); break;
            case ST_GEMM:
                if (tk.m <= 32 && tk.n <= 32) sel_tile<T, 32, 128>(S, tk, S.task[t].p, smem, smem + 128 * 33, tid);
                else sel_tile<T, 64, 32>(S, tk, S.task[t].p, smem, smem + 32 * 65, tid);
                break;
            case ST_GATHER: sel_gather<T>(P, S, tk.front, tk.a, tk.b, smem, tid); break;
            default: sel_small<T>(P, S, tk.front, smem, smem + 64 * FLD, tid); break;
        }
        drain_stores();
        __syncthreads();
        if (tid == 0) {
            __builtin_amdgcn_s_waitcnt(0);
            __hip_atomic_fetch_add(S.cnt + tk.front, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // closes the thread-0 block before the back-edge
        __syncthreads();
    }
}

}  // namespace

template <typename T>
void launch_selinv(const DevPlan& P, const DevSel<T>& S, hipStream_t s) {
    if (S.ntask <= 0) return;
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_selinv<T>, 256, 0);
    int grid = std::max(1, cus) * std::max(1, per);
    if (grid > S.ntask) grid = S.ntask;
    hipLaunchKernelGGL(k_selinv<T>, dim3(grid), dim3(256), 0, s, P, S);
}

template void launch_selinv<double>(const DevPlan&, const DevSel<double>&, hipStream_t);
template void launch_selinv<float>(const DevPlan&, const DevSel<float>&, hipStream_t);

}  // namespace mf
