// pps_march.h -- one smoothing leg of a large level in one pass over memory.
//
// A leg of the default cycle is two red-black sweeps: before them the
// iterate is zero, and after them the residual is restricted (PRE); or the
// coarse correction is added before them (POST).  Sweep by sweep the level's
// couplings, right-hand side and iterate stream from HBM two or three times.
// Here a block marches the planes of a region of 64 x 32 cells (FP64 32 x 32)
// once, its four colour passes (and the residual) trailing each other by one plane:
//   step s:  plane s    rows and right-hand side, first values of colour 0
//            plane s-1  colour 1
//            plane s-2  colour 0
//            plane s-3  colour 1
//            plane s-4  colour 0 (POST) or its residual (PRE); output
// Each pass is right one cell further inside than the one before, so the
// inner 56 x 24 cells (FP64 24 x 24) are those of the sweeps on the whole
// level; cells are computed 1.5 times over (FP64 1.8) and the halo read again
// from the L2, where neighbouring tiles (numbered XCD by XCD) find each
// other's lines if they march at one pace.  So a block fills a CU: of two
// 512-thread blocks (32 x 32 in FP32 too) one was served first and ran up to
// 30 planes ahead, and its lines had gone when the other came: 389 and 534 MB
// fetched at 256^3 (PRE, POST; least 268 and 310) instead of 337 and 423.
//
// Planes are loaded straight into LDS (buffer loads with an LDS target, two
// planes ahead: no registers are held by loads in flight, and a load's
// latency spans two steps).  Rows of one parity issue them at the start of a
// step and the others at its end, so that half of the wavefronts compute
// while the other half waits for the load unit (PRE + POST at 128^3 26.0 + 24.5
// us, 27.4 + 26.7 with all at the start; FP64 36.5 + 30.5 against 38.9 + 35.2,
// 256^3 FP64 178 + 206 against 181 + 209; 256^3 FP32 105 + 121 either way, 512^3
// 785 + 882 against 777 + 872).  A thread owns the column of one x-pair (2m,
// 2m+1) of one row: the rows of its last planes and all vertical neighbours
// are in its registers, neighbours along x in the next lanes'; those along y
// come from LDS, where each stage leaves the value it formed for the stage
// behind it, one step later.  A
// stage reads only what earlier steps wrote: one barrier a step.
// j + k has one parity over a wavefront, so the position in the pair that
// all stages of a step update is the same and uniform; the steps are
// unrolled by six (positions alternate, three planes in flight) for each
// parity, and every register index is a constant.
//
// Between PRE and POST only colour 0 of the iterate is needed (POST's first
// pass overwrites colour 1 unread), so PRE stores that colour alone, one
// value a pair.  After PRE's last pass the residual of colour 1 is zero (its
// equations were just solved), so only colour 0's is formed.
//
// What lies beyond a wall (cells, planes) and the missing second cell of an
// odd row are inert: no couplings, reciprocal diagonal 0, value 0.  Cells
// inside reach them through couplings of 0 only, but zero times a value is
// zero only if that is finite, and the row of the nearest cell in their place
// can have a diagonal of 0 (its one open face the one towards the cells
// inside).  No output depends on the edge of the region.  A periodic axis
// wraps.  Singular systems only (every diagonal is the coupling sum).
#pragma once

#include "pps_leg.h"
#include "pps_scal.h"
#include "pps_tail.h"
#include "pps_xcd.h"

namespace pps {

constexpr int kMarchHalo = 4;
constexpr int kMarchOut = 24;                                       // output rows of a tile
template <class T> constexpr int kMarchPairs = sizeof(T) == 4 ? 32 : 16;   // pairs of a row of a region
template <class T> constexpr int kMarchOutX = 2 * kMarchPairs<T> - 2 * kMarchHalo;   // output cells of it
template <class T> constexpr int kMarchThreads = 32 * kMarchPairs<T>;

struct MarchK {
    int px, py, pz;      // periodic axes
    int tx, ty;          // tiles
    int zc;              // output planes of a block (even)
};

// A buffer resource over an array of n elements (less than 4 GiB): loads
// take a uniform base o (the plane) and an offset c of the lane, both in
// elements.
template <class T> struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Buf(const T *p, long long n)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), 0, (int)(n * (long long)sizeof(T)), 0x00020000)) {}
    __device__ __forceinline__ Pair2<T> at2(unsigned o, unsigned c) const {   // elements c, c + 1
        if constexpr (sizeof(T) == 4)
            return __builtin_bit_cast(Pair2<T>, __builtin_amdgcn_raw_buffer_load_b64(r, c * 4u, o * 4u, 0));
        else
            return __builtin_bit_cast(Pair2<T>, __builtin_amdgcn_raw_buffer_load_b128(r, c * 8u, o * 8u, 0));
    }
    // BYTES a lane to consecutive places in LDS (lds uniform); byte: the
    // lane's byte offset
    template <int BYTES> __device__ __forceinline__ void to_lds(void *lds, unsigned o, unsigned byte) const {
        // (the low half of a generic pointer to LDS is its LDS address)
        auto *to = (__attribute__((address_space(3))) void *)(unsigned)reinterpret_cast<unsigned long long>(lds);
        static_assert(BYTES == 4 || BYTES == 16, "sizes of an LDS load");
        if constexpr (BYTES == 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, byte, o * (unsigned)sizeof(T), 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 16, byte, o * (unsigned)sizeof(T), 0, 0);
    }
};

// Until at most N of the wavefront's loads and stores are outstanding (they
// are counted in the order of their issue).
template <int N> __device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// v of the lane above (UP) or below: within rows of 16 lanes (R 16) or within
// the wavefront; 0 beyond the end.
template <bool UP, int R> __device__ __forceinline__ int beside(int v) {
    constexpr int ctrl = R == 16 ? (UP ? 0x101 : 0x111) : (UP ? 0x130 : 0x138);   // row / wave shl, shr
    return __builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, true);
}
template <bool UP, int R> __device__ __forceinline__ float beside(float v) {
    return __builtin_bit_cast(float, beside<UP, R>(__builtin_bit_cast(int, v)));
}
template <bool UP, int R> __device__ __forceinline__ double beside(double v) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = beside<UP, R>(u.i[0]);
    u.i[1] = beside<UP, R>(u.i[1]);
    return u.d;
}

// Workgroup barrier over LDS reads and writes.  lds_barrier's fence would
// also wait for every load on its way into LDS; those are waited for by
// count (wait_vm) before the barrier that publishes them.
__device__ __forceinline__ void march_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// One plane in LDS: 16 x 32 pairs, rows of one parity next to each other
// (even rows, then odd); PRE also the column left of the region and the row
// below it, POST the colour-0 iterate (one a pair) and the correction of it.
template <class T> struct alignas(2 * sizeof(T)) LdsPair { T a, b; };   // one LDS access
template <class T, bool PRE> struct alignas(16) MarchPlane {
    static constexpr int N = kMarchThreads<T>;
    LdsPair<T> cx[N], cy[N], cz[N], b[N];
    T e0[PRE ? 32 : N], e1[PRE ? 2 * kMarchPairs<T> : N];
};

// V16: rows are multiples of 16 bytes, and planes are loaded 16 bytes a lane
// (a wavefront half an array); otherwise 4 bytes a lane, any row length.
template <class T, bool PRE, bool DOT, bool V16>
__global__ void __launch_bounds__(kMarchThreads<T>, sizeof(T) == 4 ? 4 : 2)
k_march(LevelK<T> L, MarchK g, Coarsening cg, const T *__restrict__ b, const T *__restrict__ xc,
        const T *__restrict__ ec, T *__restrict__ xo, T *__restrict__ bc, double *__restrict__ part,
        StopK stop) {
    if (PRE && stopped(stop)) return;
    using Pl = MarchPlane<T, PRE>;
    // three planes, distinct arrays (so that the compiler can tell a read of
    // one from the loads into another)
    __shared__ Pl A0, A1, A2;
    // what each stage formed in the last two steps, one a pair, and PRE's
    // residuals
    constexpr int kW = kMarchThreads<T>, kR = kMarchPairs<T>, kC = 2 * kR;   // pairs, pairs and cells of a row
    __shared__ T Wm[4 * 2 * kW];
    __shared__ T Rz[PRE ? 2 * kW : 1];
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = xcd_order(blockIdx.x, gridDim.x);
    const int ox = t % g.tx * kMarchOutX<T>, oy = t / g.tx % g.ty * kMarchOut;
    const int k0 = t / (g.tx * g.ty) * g.zc, k1 = min(k0 + g.zc, (nz + 1) & ~1);
    auto place = [](int i, int n, int per) {   // wrapped, or moved to the nearest cell
        if (i >= 0 && i < n) return i;
        if (!per) return i < 0 ? 0 : n - 1;
        i %= n;
        return i < 0 ? i + n : i;
    };
    // the row of the region that lies at place r of a plane in LDS
    auto row_at = [](int r) { return 2 * (r & 15) + (r >> 4); };

    // the thread's pair: the pairs of 64 / kR rows of one parity jl a wavefront
    const int m = tid & (kR - 1), jl = wv & 1, jh = lane / kR + (wv >> 1) * (64 / kR), j = 2 * jh + jl;
    const int own = m + kR * jh + kW / 2 * jl;
    const int rs = own + (jl ? -kW / 2 : kW / 2 - kR), rn = own + (jl ? kR - kW / 2 : kW / 2);   // rows below, above
    const int ui = ox - kMarchHalo + 2 * m, uj = oy - kMarchHalo + j;
    const int gi = place(ui, nx, g.px) & ~1, gj = place(uj, ny, g.py);
    const bool two = V16 || gi + 1 < nx;     // the pair's second cell exists
    // the pair's first cell lies in the level
    const bool real = (g.px || (ui >= 0 && ui < nx)) && (g.py || (uj >= 0 && uj < ny));
    const bool mine = m >= 2 && m < kR - 2 && j >= 4 && j < 28 && ui < nx && uj < ny;
    const bool wallw = ui == 0 && !g.px, walls = uj == 0 && !g.py;   // no coupling to the left, below
    const long long sz = (long long)nx * ny, n = sz * nz;
    const unsigned np = (nx + 1) >> 1, pcol = (gi >> 1) + np * gj;
    const long long psz = (long long)np * ny;

    // loads of a plane's four arrays, NC a wavefront (V16: of its own array
    // wv / (kR / 8), else of each), and the lane's byte offsets in a plane
    constexpr int DW = sizeof(T) / 4, NC = 2 * DW;
    unsigned off[NC], pof[DW], eof[DW], off_w = 0, off_s = 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        // cell of the plane in LDS; V16: the first of the lane's 4 / DW cells,
        // all inside the row or all outside
        const int e = V16 ? (((wv & (kR / 8 - 1)) * NC + c) * 64 + lane) * (4 / DW) : ((wv * NC + c) * 64 + lane) / DW;
        int i = place(ox - kMarchHalo + (e & (kC - 1)), nx, g.px);
        if (V16) i &= ~(4 / DW - 1);
        off[c] = (i + (unsigned)nx * place(oy - kMarchHalo + row_at(e / kC), ny, g.py)) * (unsigned)sizeof(T) +
                 (V16 ? 0u : (lane % DW) * 4u);
    }
    if (PRE) {
        const int e = lane / DW;   // 32 rows, kC cells
        off_w = (place(ox - kMarchHalo - 1, nx, g.px) +
                 (unsigned)nx * place(oy - kMarchHalo + row_at(e & 31), ny, g.py)) * (unsigned)sizeof(T) + (lane % DW) * 4u;
        off_s = (place(ox - kMarchHalo + (e & (kC - 1)), nx, g.px) +
                 (unsigned)nx * place(oy - kMarchHalo - 1, ny, g.py)) * (unsigned)sizeof(T) + (lane % DW) * 4u;
    } else {
        // the wavefront's own 64 pairs; the second cell's parent
        // where cells and not pairs are children (fx 1) is the next element
#pragma unroll
        for (int c = 0; c < DW; ++c) {
            const int e = (c * 64 + lane) / DW, em = e & (kR - 1), ej = 2 * (e / kR + (wv >> 1) * (64 / kR)) + jl;
            const int i = place(ox - kMarchHalo + 2 * em, nx, g.px) & ~1, jj = place(oy - kMarchHalo + ej, ny, g.py);
            pof[c] = ((i >> 1) + np * jj) * (unsigned)sizeof(T) + (lane % DW) * 4u;
            eof[c] = ((i >> (cg.fx - 1)) + (unsigned)cg.cnx * (jj >> (cg.fy - 1))) * (unsigned)sizeof(T) + (lane % DW) * 4u;
        }
    }
    const Buf<T> Bx(L.cx, n), By(L.cy, n), Bz(L.cz, n), Bb(b, n);
    const Buf<T> Bm(wv < kR / 8 ? L.cx : wv < kR / 4 ? L.cy : wv < 3 * kR / 8 ? L.cz : b, n);   // V16: this wavefront's array
    const Buf<T> Bc(PRE ? b : xc, PRE ? n : psz * nz);
    const Buf<T> Be(PRE ? b : ec, PRE ? n : (long long)cg.cnx * cg.cny * cg.cnz);
    auto plane_of = [&](int k) {   // wrapped; -1 beyond a wall (uniform)
        if (k >= 0 && k < nz) return k;
        if (!g.pz) return -1;
        k %= nz;
        return k < 0 ? k + nz : k;
    };
    const int s0 = k0 - kMarchHalo, s1 = k1 - 1 + kMarchHalo;
    // start loading plane s (if the march gets to it) into A; e: the position
    // of colour 0 in this wavefront's rows of it
    auto request = [&](Pl &A, int s, int e) -> bool {
        const int k = s > s1 ? -1 : plane_of(s);
        if (k < 0) return false;
        const unsigned o = (unsigned)sz * k;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (V16) {   // the four arrays follow each other in A
                Bm.template to_lds<16>((char *)&A + (wv * NC + c) * 1024, o, off[c]);
            } else {
                const int d = (wv * NC + c) * 256;
                Bx.template to_lds<4>((char *)A.cx + d, o, off[c]);
                By.template to_lds<4>((char *)A.cy + d, o, off[c]);
                Bz.template to_lds<4>((char *)A.cz + d, o, off[c]);
                Bb.template to_lds<4>((char *)A.b + d, o, off[c]);
            }
        }
        if (PRE) {
            if (wv == 0 && lane < 32 * DW) Bx.template to_lds<4>(A.e0, o, off_w);
            if (wv == 1 && lane < kC * DW) By.template to_lds<4>(A.e1, o, off_s);
        } else {
            const unsigned ko = (unsigned)(cg.cnx * cg.cny) * (k >> (cg.fz - 1)) + (cg.fx == 1 ? e : 0);
#pragma unroll
            for (int c = 0; c < DW; ++c) {
                const int d = 64 * (wv >> 1) + kW / 2 * jl + c * 64 / DW;
                Bc.template to_lds<4>(A.e0 + d, (unsigned)psz * k, pof[c]);
                Be.template to_lds<4>(A.e1 + d, ko, eof[c]);
            }
        }
        return true;
    };
    // A plane's loads at least (the count of every wavefront).  A step waits
    // until nothing older than what it and the step before issued since is
    // outstanding: its loads for plane s + 2 and both steps' stores, which
    // stay in flight (to wait for one of those loads costs a memory latency a
    // step: 256^3 FP32 PRE 111 us, POST 127; counted 105 and 121).  A count too
    // low is safe; one that takes in a store older than the loads waited for
    // is not, so a wavefront that requests at the start of a step must issue
    // those loads before the step's stores, which touch other memory: the
    // empty asm there keeps the order.
    constexpr int kLoads = (V16 ? 1 : 4) * NC + (PRE ? 0 : 2 * DW);

    // rows of the last planes by position, and the values of both colours in
    // them; everything zero before the first plane
    T co[6], cx[6][2], cs[6][2], cn[6][2], cu[6][2], bb[6][2], rd[6][2];
    T xr[6], xk[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        co[q] = xr[q] = xk[q] = (T)0;
#pragma unroll
        for (int e = 0; e < 2; ++e) cx[q][e] = cs[q][e] = cn[q][e] = cu[q][e] = bb[q][e] = rd[q][e] = (T)0;
    }
    for (int e = tid; e < 4 * 2 * kW; e += kW) Wm[e] = (T)0;
    double sbx = 0.0, sx = 0.0, sb = 0.0;
    // whether the wavefront stores (a value a step), and how often in two
    // steps it stores a restricted one (PRE)
    const bool storing = __any(mine);
    const int bstores = !PRE || (cg.fy == 2 && jl) ? 0 : cg.fz == 2 ? 1 : 2;

    // restriction of plane k, whose residuals were formed in the step before
    // (rlast, and the next row's in LDS); e: position of colour 0 in this
    // row of plane k, 1 - e in the next row.  Rows pair up when fy is 2 (the
    // lower row's thread sums both), planes when fz is 2 (rsum holds the
    // lower plane's).
    T rlast = 0, rsum[2] = {0, 0};
    auto finish = [&](int k, int e) {
        if (cg.fy == 2 && jl) return;   // uniform
        const T r2 = cg.fy == 2 ? Rz[(k & 1) * kW + own + kW / 2] : (T)0;
        T va = e ? r2 : rlast, vb = e ? rlast : r2;
        if (cg.fz == 2 && !(k & 1)) {
            rsum[0] = va;
            rsum[1] = vb;
            return;
        }
        if (cg.fz == 2) { va += rsum[0]; vb += rsum[1]; }
        const T scale = (T)1 / (T)(cg.fx * cg.fy * cg.fz);
        const int K = k >> (cg.fz - 1), J = gj >> (cg.fy - 1);
        if (!mine || K >= cg.cnz) return;
        T *o = bc + ((long long)cg.cnx * cg.cny * K + (long long)cg.cnx * J);
        if (cg.fx == 2) {
            o[gi >> 1] = (va + vb) * scale;
        } else {
            o[gi] = va * scale;
            if (two) o[gi + 1] = vb * scale;
        }
    };

    // step s at place P0 of the register rings, LATE: requests last, the active position E, the
    // plane in A, and An the LDS to load plane s + 2 into
    auto step = [&](auto LC, auto PC, auto EC, Pl &A, Pl &An, int s) {
        constexpr bool LATE = decltype(LC)::value;
        constexpr int P0 = decltype(PC)::value, E = decltype(EC)::value, H = P0 & 1;
        constexpr int P1 = (P0 + 5) % 6, P2 = (P0 + 4) % 6, P3 = (P0 + 3) % 6, P4 = (P0 + 2) % 6;
        // a stage's output of this step, and of the step before
        auto W = [&](int st, int i) -> T & { return Wm[(st * 2 + H) * kW + i]; };
        auto V = [&](int st, int i) -> T { return Wm[(st * 2 + 1 - H) * kW + i]; };
        // b + sum of the couplings of the cell at position E of plane slot q,
        // the neighbours of stage st; xp its pair's other cell, xd / xu the
        // cells below and above, cd the coupling to the one below (the +z
        // one of the plane below)
        auto sum = [&](auto QC, int st, T xp, T cd, T xd, T xu) {
            constexpr int q = decltype(QC)::value;
            T v = bb[q][E] + co[q] * xp;
            v += cx[q][E] * beside<E == 1, kR>(xp);   // the same stage's value of the next pair
            v += cs[q][E] * V(st, rs);
            v += cn[q][E] * V(st, rn);
            v += cd * xd;
            v += cu[q][E] * xu;
            return v;
        };
        bool ahead = false;
        if (!LATE) {
            ahead = request(An, s + 2, E);
            asm volatile("" ::: "memory");   // before this step's stores (see kLoads)
        }
        if (PRE && s - 5 >= k0) finish(s - 5, 1 - E);
        // plane s
        if (plane_of(s) >= 0 && real) {
            const LdsPair<T> vx = A.cx[own], vn = A.cy[own], vs = A.cy[rs], vu = A.cz[own], vb = A.b[own];
            T left = beside<false, kR>(vx.b);
            if (PRE) left = m == 0 ? A.e0[jh + 16 * jl] : left;
            co[P0] = vx.a;
            cx[P0][0] = wallw ? (T)0 : left;
            cx[P0][1] = vx.b;
            cs[P0][0] = walls ? (T)0 : vs.a; cs[P0][1] = walls ? (T)0 : vs.b;
            if (PRE && j == 0) { cs[P0][0] = A.e1[2 * m]; cs[P0][1] = A.e1[2 * m + 1]; }
            cn[P0][0] = vn.a; cn[P0][1] = vn.b;
            cu[P0][0] = vu.a; cu[P0][1] = vu.b;
            bb[P0][0] = vb.a; bb[P0][1] = vb.b;
            rd[P0][0] = (T)1 / diag_sum(cx[P0][0], co[P0], cs[P0][0], cn[P0][0], cu[P1][0], cu[P0][0]);
            rd[P0][1] = two ? (T)1 / diag_sum(co[P0], cx[P0][1], cs[P0][1], cn[P0][1], cu[P1][1], cu[P0][1]) : (T)0;
            xr[P0] = PRE ? bb[P0][E] * rd[P0][E] : E == 1 && !two ? (T)0 : A.e0[own] + A.e1[own];
        } else {
            co[P0] = xr[P0] = (T)0;
#pragma unroll
            for (int e = 0; e < 2; ++e) cx[P0][e] = cs[P0][e] = cn[P0][e] = cu[P0][e] = bb[P0][e] = rd[P0][e] = (T)0;
        }
        W(0, own) = xr[P0];
        const T cu5 = cu[(P0 + 1) % 6][E], xk5 = xk[(P0 + 1) % 6];   // plane s-5
        xk[P1] = sum(Ic<P1>(), 0, xr[P1], cu[P2][E], xr[P2], xr[P0]) * rd[P1][E];
        W(1, own) = xk[P1];
        xr[P2] = sum(Ic<P2>(), 1, xk[P2], cu[P3][E], xk[P3], xk[P1]) * rd[P2][E];
        W(2, own) = xr[P2];
        xk[P3] = sum(Ic<P3>(), 2, xr[P3], cu[P4][E], xr[P4], xr[P2]) * rd[P3][E];
        W(3, own) = xk[P3];
        const int k = s - 4;
        if constexpr (PRE) {
            const T d = diag_sum(E ? co[P4] : cx[P4][0], E ? cx[P4][1] : co[P4], cs[P4][E], cn[P4][E], cu5, cu[P4][E]);
            T r = sum(Ic<P4>(), 3, xk[P4], cu5, xk5, xk[P3]) - d * xr[P4];
            if (uj >= ny || (E == 1 && !two)) r = (T)0;   // not of the level
            if (mine && k >= k0 && k < k1 && k < nz) xo[psz * k + pcol] = xr[P4];
            rlast = r;
            Rz[H * kW + own] = r;
        } else {
            xr[P4] = sum(Ic<P4>(), 3, xk[P4], cu5, xk5, xk[P3]) * rd[P4][E];
            if (mine && k >= k0 && k < k1 && k < nz) {
                const T va = E ? xk[P4] : xr[P4], vb = E ? xr[P4] : xk[P4];
                T *o = xo + sz * k + (gi + (long long)nx * gj);
                if (two) *reinterpret_cast<Pair2<T> *>(o) = Pair2<T>{va, vb};
                else o[0] = va;
                if (DOT) {
                    sbx += (double)bb[P4][0] * (double)va;
                    sx += (double)va;
                    sb += (double)bb[P4][0];
                    if (two) {
                        sbx += (double)bb[P4][1] * (double)vb;
                        sx += (double)vb;
                        sb += (double)bb[P4][1];
                    }
                }
            }
        }
        if (LATE) ahead = request(An, s + 2, E);
        // plane s + 1 (requested a step ago) has landed
        if (!ahead) wait_vm<0>();
        else if (!(storing && k - (PRE ? 2 : 1) >= k0 && k < nz)) wait_vm<kLoads>();
        else if (LATE) wait_vm<kLoads + 1>();
        else if (bstores == 0) wait_vm<kLoads + 2>();
        else if (bstores == 1) wait_vm<kLoads + 3>();
        else wait_vm<kLoads + 4>();
        march_barrier();
        __builtin_amdgcn_sched_barrier(0);   // nothing of the next step moves up (registers)
    };
    {   // the first plane's -z couplings (its diagonals need them)
        const int k = plane_of(s0 - 1);
        if (k >= 0) {
            const unsigned sh = two ? 0 : 1;   // an odd row's last cell is loaded as the second of two
            const Pair2<T> v = Bz.at2((unsigned)sz * k, gi + (unsigned)nx * gj - sh);
            cu[5][0] = sh ? v.b : v.a;
            cu[5][1] = v.b;
        }
    }
    // every wavefront runs the same number of steps (and barriers), in the
    // loop of its rows' parity: s0 is even, so colour 0 of the first plane is
    // at position jl, and the number of steps is even
    request(A0, s0, jl);
    if (request(A1, s0 + 1, 1 - jl)) wait_vm<kLoads>();
    else wait_vm<0>();
    march_barrier();
    auto run = [&](auto EC) {
        constexpr int E = decltype(EC)::value;
        for (int s = s0;; s += 6) {
            step(EC, Ic<0>(), Ic<E>(), A0, A2, s);
            step(EC, Ic<1>(), Ic<1 - E>(), A1, A0, s + 1);
            if (s + 2 > s1) break;
            step(EC, Ic<2>(), Ic<E>(), A2, A1, s + 2);
            step(EC, Ic<3>(), Ic<1 - E>(), A0, A2, s + 3);
            if (s + 4 > s1) break;
            step(EC, Ic<4>(), Ic<E>(), A1, A0, s + 4);
            step(EC, Ic<5>(), Ic<1 - E>(), A2, A1, s + 5);
            if (s + 6 > s1) break;
        }
    };
    if (jl) run(Ic<1>());
    else run(Ic<0>());
    if (PRE) finish(k1 - 1, (jl ^ (k1 - 1)) & 1);
    if (DOT) {
        block_partial(sbx, part);
        block_partial(sx, part + kRedBlocks);
        block_partial(sb, part + 2 * kRedBlocks);
    }
}

}  // namespace pps
