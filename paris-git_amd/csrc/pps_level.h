// pps_level.h -- a multigrid level as the kernels see it, and the small
// device helpers that the sweeps, the coarse tail and the outer kernels share.
#pragma once

#include "pps_internal.h"

namespace pps {

// ---------------------------------------------------------------------
// kernel-side level view
// ---------------------------------------------------------------------
template <class T> struct LevelK {
    int nx, ny, nz;
    const T *cx, *cy, *cz, *dg;
};

// a compile-time index as an argument
template <int I> struct Ic { static constexpr int value = I; };

// sum over the 64 lanes of a wavefront (result in lane 0)
__device__ __forceinline__ double wsum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

__device__ __forceinline__ int wrap_m(int i, int n) { return i == 0 ? n - 1 : i - 1; }
__device__ __forceinline__ int wrap_p(int i, int n) { return i == n - 1 ? 0 : i + 1; }

// Diagonal of a row whose excess A7 - sum(couplings) is zero (every row
// of a singular system): the sum of its six couplings, in one fixed order
// shared by every kernel of the V-cycle.
template <class T>
__device__ __forceinline__ T diag_sum(T cxm, T cx, T cym, T cy, T czm, T cz) {
    return ((cxm + cx) + (cym + cy)) + (czm + cz);
}

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Writes the block sum of v to part[block linear id].  Any block of at most
// 1024 threads whose x extent is a multiple of 64 (each wavefront is 64
// consecutive linear thread ids); wavefront sums are added in a fixed order.
__device__ __forceinline__ void block_partial(double v, double *part) {
    __shared__ double sm[16];
    const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int b = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int nw = (blockDim.x * blockDim.y * blockDim.z) >> 6;
    v = wsum(v);
    if ((t & 63) == 0) sm[t >> 6] = v;
    __syncthreads();
    if (t == 0) {
        double a = 0.0;
        for (int w = 0; w < nw; ++w) a += sm[w];
        part[b] = a;
    }
    __syncthreads();
}

// Coarsening from a level to the next.
struct Coarsening {
    int fx, fy, fz;      // 1 or 2 per axis
    int cnx, cny, cnz;   // coarse sizes, ceil(n / f)
};

}  // namespace pps
