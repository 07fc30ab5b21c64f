// mf_solve.hip — the permutations around the triangular solves.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mf_kernels.h"

namespace mf {

namespace {

// dst[i] = src[perm[i]] (P*B, multiply.jl:277-280) or dst[perm[i]] = src[i].
template <typename TB>
__global__ void k_permute(const double* src, int64_t lds, TB* dst, int64_t ldd, const int64_t* perm,
                          int n, int nrhs, int inverse) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n * nrhs) return;
    int r = (int)(i % n), c = (int)(i / n);
    int64_t p = perm[r] - 1;
    if (!inverse) dst[r + c * ldd] = (TB)src[p + c * lds];
    else dst[p + c * ldd] = (TB)src[r + c * lds];
}

template <typename TS>
__global__ void k_permute_back(const TS* src, int64_t lds, double* dst, int64_t ldd,
                               const int64_t* perm, int n, int nrhs) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n * nrhs) return;
    int r = (int)(i % n), c = (int)(i / n);
    dst[(perm[r] - 1) + c * ldd] = (double)src[r + c * lds];
}

inline unsigned blocks_for(int64_t tot) { return (unsigned)((tot + 255) / 256); }

}  // namespace

template <typename TB>
void launch_permute(const double* src, int64_t lds, TB* dst, int64_t ldd, const int64_t* perm,
                    int n, int nrhs, bool inverse, hipStream_t s) {
    int64_t tot = (int64_t)n * nrhs;
    if (tot <= 0) return;
    hipLaunchKernelGGL(k_permute<TB>, dim3(blocks_for(tot)), dim3(256), 0, s, src, lds, dst, ldd,
                       perm, n, nrhs, inverse ? 1 : 0);
}

void launch_permute_back(const void* src, int64_t lds, bool src_f32, double* dst, int64_t ldd,
                         const int64_t* perm, int n, int nrhs, hipStream_t s) {
    int64_t tot = (int64_t)n * nrhs;
    if (tot <= 0) return;
    if (src_f32)
        hipLaunchKernelGGL(k_permute_back<float>, dim3(blocks_for(tot)), dim3(256), 0, s,
                           (const float*)src, lds, dst, ldd, perm, n, nrhs);
    else
        hipLaunchKernelGGL(k_permute_back<double>, dim3(blocks_for(tot)), dim3(256), 0, s,
                           (const double*)src, lds, dst, ldd, perm, n, nrhs);
}

template void launch_permute<double>(const double*, int64_t, double*, int64_t, const int64_t*, int, int, bool,
                                     hipStream_t);
template void launch_permute<float>(const double*, int64_t, float*, int64_t, const int64_t*, int, int, bool, hipStream_t);

}  // namespace mf
