// pps_scal.h -- the outer iteration's scalars: block partials to sums, the
// stopping test and the host's mailbox.  The sums are formed by a kernel of
// one workgroup (3 to 7 us a launch and its gap), or, where there are few
// partials, by every block of the kernel that needs them.
#pragma once

#include "pps_level.h"

namespace pps {

// ---------------------------------------------------------------------
// Scalars of the FP64 outer iteration, on the device
// ---------------------------------------------------------------------
// (S_RZ, S_RZ + 1: rho of the iterations of even and odd number)
enum { S_RZ = 0, S_ZMEAN = 2, S_BETA, S_DQ, S_ALPHA, S_RR, S_BB, S_STOP, S_N };
// alpha of the direction in ring slot j: S[S_AH + j] (j < kRingSlots;
// the scalars take 64 doubles)
constexpr int kRingSlots = 9;   // directions held for deferred x updates
constexpr int S_AH = S_N;
static_assert(S_AH + kRingSlots <= 64, "ring alphas fit the scalars");

// fixed-order sum of nb partials, the same value in every thread (any
// block of at most 1024 threads whose x extent is a multiple of 64)
template <int LOADS = 1>   // of a thread in flight
__device__ __forceinline__ double sum_partials(const double *part, int nb) {
    __shared__ double sm[16];
    const int nt = blockDim.x * blockDim.y * blockDim.z;
    const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int nw = nt >> 6;
    double v = 0.0;
#pragma unroll LOADS
    for (int b = tid; b < nb; b += nt) v += part[b];
    v = wsum(v);
    if ((tid & 63) == 0) sm[tid >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < nw; ++w) t += sm[w];
    __syncthreads();
    return t;
}

// three such sums at once (slots 0, 1, 2 of the partials)
__device__ __forceinline__ void sum_partials3(const double *part, int nb, double out[3]) {
    __shared__ double sm[3][16];
    const int nt = blockDim.x * blockDim.y * blockDim.z;
    const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int nw = nt >> 6;
    double v[3] = {0.0, 0.0, 0.0};
    for (int b = tid; b < nb; b += nt)
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] += part[c * kRedBlocks + b];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v[c] = wsum(v[c]);
        if ((tid & 63) == 0) sm[c][tid >> 6] = v[c];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        out[c] = 0.0;
        for (int w = 0; w < nw; ++w) out[c] += sm[c][w];
    }
    __syncthreads();
}

// a value that every lane holds, in scalar registers
__device__ __forceinline__ double uniform(double v) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_readfirstlane(u.i[0]);
    u.i[1] = __builtin_amdgcn_readfirstlane(u.i[1]);
    return u.d;
}

// Most partials that a consuming kernel's blocks sum themselves.  Of beta's
// (three sums, in k_dq_tiled): the 32^3 solve has 64 and saves the launch; at
// 64^3 FP64 (144) k_dq_tiled would grow from 7.4 to 12.5 us, as much as the
// kernel (4.1 us) and its gap take, and from 700 blocks on, two rounds on the
// card, it would pay twice.
constexpr int kFoldParts = 128;
// Of alpha's (k_update) and r.r's (the next cycle's first leg), one sum: up to
// 1024, a load for each thread of a leg and four for one of k_update.  128^3:
// k_update 12.9 -> 13.3 us without k_scal_alpha's 4.2, k_march PRE 23.3 ->
// 23.5 (means that take in a solve's last one, which returns at once) without
// k_scal_rr's 4.6; solves at 128^3 1576 -> 1555 us, 64^3 FP64 873
// -> 860, 49x64x40 FP64 1088 -> 1060.
constexpr int kFoldWide = 1024;

// beta from the nb partials of (r, z), sum z, sum r: zmean, rho = r.(z - zmean),
// beta = rho / rho_old, 0 in the first iteration.  rd, wr: the places of
// rho_old and rho in S.
struct BetaK {
    int nb, singular, first, rd, wr;
    long long n;
};
__device__ __forceinline__ void beta_of(const BetaK &k, const double sums[3], double rho_old, double *beta,
                                        double *zm, double *rho) {
    *zm = k.singular ? sums[1] / (double)k.n : 0.0;
    *rho = sums[0] - *zm * sums[2];
    *beta = k.first ? 0.0 : *rho / rho_old;
}

// alpha = rho / d.q (nb 0: it is in S; rz: the place of rho; slot: the
// direction's)
struct AlphaK {
    int nb, rz, slot;
};

// r.r likewise, with the stopping test sqrt(r.r / N) < tol, both written to
// the host's mailbox by the first block.  skip (nb 0): the test's outcome,
// put there by a kernel of its own.
struct StopK {
    const double *skip;
    const double *part;
    int nb;
    double N, tol;
    double *S;
    Mailbox *mb;
    unsigned long long seq;
};
// the values, then seq with a system-scope release: a host that reads seq
// (acquire) sees them
__device__ __forceinline__ void post(Mailbox *mb, unsigned long long seq, double rr, double bb, double flags,
                                     double stop) {
    mb->rr = rr;
    mb->bb = bb;
    mb->flags = flags;
    mb->pad = stop;
    __hip_atomic_store(&mb->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ bool stopped(const StopK &k) {
    if (!k.nb) return k.skip && *k.skip != 0.0;
    const double rr = sum_partials(k.part, k.nb);
    const bool stop = sqrt(rr / k.N) < k.tol;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        k.S[S_RR] = rr;
        post(k.mb, k.seq, rr, 0.0, 0.0, stop ? 1.0 : 0.0);
    }
    return stop;
}

}  // namespace pps
