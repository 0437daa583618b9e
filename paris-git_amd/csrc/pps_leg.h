// pps_leg.h -- one smoothing leg of a level in one launch.
//
// A leg of the default cycle is two red-black sweeps: before them the
// iterate is zero, and after them the residual is restricted (k_leg_pre); or
// the coarse correction is added before them (k_leg_post).  Launched sweep
// by sweep, a level of some 10^4 to 10^5 cells spends its time in launches
// of a few microseconds that are bound by latency, not by bytes.  Here a
// block computes its 8 x 8 x OZ output cells from a region four cells larger
// on every side: each of the four colour passes (and the residual) is right
// one cell further inside than the one before, so the outputs are those of
// the sweeps on the whole level, and the halo cells computed several times
// over cost less than the launches saved.
//
// A thread holds P x-pairs of cells (2m, 2m+1) of one (m, row), their rows
// and right-hand sides in registers; the iterate lies in LDS as two arrays by
// position in the pair, so that all addresses are unit-stride across a
// wavefront and constants apart.  j + k has one parity over a wavefront,
// which makes the position that a colour pass updates uniform.  The -y and
// -z couplings are the +y and +z ones of the pairs below and come through
// LDS, so every coupling is loaded once.  Cells at the region's edge are
// updated like the others, from whatever lies next to them in LDS: finite,
// and never read by a cell that an output depends on.
// Any size and coarsening: a periodic axis wraps, a cell beyond a wall is
// inert (no couplings, right-hand side 0, diagonal 1), as is the missing
// second cell of an odd row's last pair.
#pragma once

#include "pps_scal.h"
#include "pps_tail.h"
#include "pps_xcd.h"

namespace pps {

constexpr int kLegHalo = 4;              // colour passes of a leg
constexpr int kLegOut = 8;               // output cells along x and y
constexpr int kLegRow = 8;               // pairs along x of the region
constexpr int kLegPlane = kLegRow * 16;  // pairs of one of its planes (16 rows)
constexpr int kLegThreads = 1024;
constexpr int kLegStep = kLegThreads / kLegPlane;   // planes between a thread's pairs

struct LegK {
    int px, py, pz;      // periodic axes
    int tx, ty, tz;      // tiles
};

// element i of a plane, 32-bit byte offsets (levels of at most 2^28 cells)
template <class T> __device__ __forceinline__ T at(const T *p, unsigned i) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (unsigned)sizeof(T));
}
// elements i, i + 1 in one load (any alignment of a T)
template <class T> struct __attribute__((packed, aligned(sizeof(T)))) Pair2 { T a, b; };
template <class T> __device__ __forceinline__ Pair2<T> at2(const T *p, unsigned i) {
    return *reinterpret_cast<const Pair2<T> *>(reinterpret_cast<const char *>(p) + i * (unsigned)sizeof(T));
}

// the value of the lane below within 16 lanes (junk for the first of them)
__device__ __forceinline__ float lane_below(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_below(double v) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], 0x111, 0xf, 0xf, true);
    u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], 0x111, 0xf, 0xf, true);
    return u.d;
}

// LDS of a leg: X[position] of every pair of the region, with a plane and a
// pair of padding at both ends for the edge cells' reads, and the +y and +z
// couplings by position.
template <class T, int EZ> struct LegLds {
    static constexpr int kPairs = kLegPlane * EZ;
    static constexpr int kPad = kLegPlane;
    T X[2][kPairs + 2 * kPad];
    T cy[2][kPairs], cz[2][kPairs];
};

template <class T, bool DGI, int EZ> struct Leg {
    static constexpr int P = EZ / kLegStep;
    static constexpr int kPairs = kLegPlane * EZ;
    static constexpr int kOz = EZ - 2 * kLegHalo;
    static constexpr int kOutPairs = kLegOut / 2 * kLegOut * kOz;
    using Lds = LegLds<T, EZ>;
    static_assert(EZ % kLegStep == 0 && kLegStep % 2 == 0, "whole pairs a thread, one parity a wavefront");
    Lds &S;
    // rows by position: co couples the pair's cells, cxo the outer x faces
    T co[P], cxo[P][2], cs[P][2], cn[P][2], cd[P][2], cu[P][2], rd[P][2];
    T b[P][2], x[P][2];
    int c[P];            // cell of the pair's first cell in the level, -1 outside
    int gk[P];
    int m, j, k0, own0, ds, dn, gi, gj;
    bool two;            // the pair's second cell exists
    bool odd;            // j + k odd (uniform over a wavefront): colour 0 is the second cell

    __device__ __forceinline__ explicit Leg(Lds &lds) : S(lds) {}
    static __device__ __forceinline__ int wrap(int i, int n, int per) {
        if (i >= 0 && i < n) return i;
        if (!per) return -1;   // outside
        i %= n;
        return i < 0 ? i + n : i;
    }
    __device__ __forceinline__ int own(int p) const { return own0 + p * kLegThreads; }
    __device__ __forceinline__ int plane(int p) const { return k0 + p * kLegStep; }
    __device__ __forceinline__ T &X(int pos, int i) const { return S.X[pos][Lds::kPad + i]; }

    // rows and right-hand side; (ox, oy, oz): the block's first output cell
    __device__ __forceinline__ void load(const LevelK<T> &L, const LegK &g, const T *__restrict__ rhs, int ox,
                                         int oy, int oz) {
        // lanes: 8 pairs x every other row; the row's parity by wavefront.
        // Rows of one parity lie next to each other in LDS (own0 = tid), so
        // the rows above and below are 64 or 56 pairs away
        const int tid = threadIdx.x, jl = __builtin_amdgcn_readfirstlane((tid >> 6) & 1);
        m = tid & (kLegRow - 1);
        j = 2 * ((tid >> 3) & 7) + jl;
        k0 = __builtin_amdgcn_readfirstlane(tid >> 7);
        own0 = tid;
        odd = (jl ^ k0) & 1;
        ds = jl ? -64 : 56;
        dn = jl ? -56 : 64;
        gi = wrap(ox - kLegHalo + 2 * m, L.nx, g.px);
        gj = wrap(oy - kLegHalo + j, L.ny, g.py);
        two = gi >= 0 && gi + 1 < L.nx;
        const unsigned sy = L.nx, sz = (unsigned)L.nx * L.ny;
        T ga[P], gb[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            gk[p] = wrap(oz - kLegHalo + plane(p), L.nz, g.pz);
            const bool in = gi >= 0 && gj >= 0 && gk[p] >= 0;
            c[p] = in ? (int)(gi + sy * gj + sz * gk[p]) : -1;
            co[p] = (T)0;
#pragma unroll
            for (int q = 0; q < 2; ++q) cxo[p][q] = cn[p][q] = cu[p][q] = b[p][q] = (T)0;
            ga[p] = gb[p] = (T)1;
            if (in && two) {
                const Pair2<T> vx = at2(L.cx, c[p]), vy = at2(L.cy, c[p]), vz = at2(L.cz, c[p]), vb = at2(rhs, c[p]);
                co[p] = vx.a; cxo[p][1] = vx.b;
                cn[p][0] = vy.a; cn[p][1] = vy.b;
                cu[p][0] = vz.a; cu[p][1] = vz.b;
                b[p][0] = vb.a; b[p][1] = vb.b;
                if (!DGI) { const Pair2<T> vd = at2(L.dg, c[p]); ga[p] = vd.a; gb[p] = vd.b; }
            } else if (in) {
                co[p] = at(L.cx, c[p]);
                cn[p][0] = at(L.cy, c[p]);
                cu[p][0] = at(L.cz, c[p]);
                b[p][0] = at(rhs, c[p]);
                if (!DGI) ga[p] = at(L.dg, c[p]);
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                S.cy[q][own(p)] = cn[p][q];
                S.cz[q][own(p)] = cu[p][q];
            }
        }
        // the padding of X
        if (tid < 2 * Lds::kPad)
            for (int q = 0; q < 2; ++q) S.X[q][tid < Lds::kPad ? tid : kPairs + tid] = (T)0;
        // the couplings that reach out of the region
        const bool w0 = m == 0, s0 = j == 0;
        T xw[P], se[P][2], de[2] = {(T)0, (T)0};
#pragma unroll
        for (int p = 0; p < P; ++p) {
            xw[p] = se[p][0] = se[p][1] = (T)0;
            if (c[p] < 0) continue;
            if (w0) xw[p] = at(L.cx, gi == 0 ? c[p] + (sy - 1) : c[p] - 1);
            if (s0) {
                const unsigned cc = gj == 0 ? c[p] + sz - sy : c[p] - sy;
                se[p][0] = at(L.cy, cc);
                if (two) se[p][1] = at(L.cy, cc + 1);
            }
            if (p == 0 && k0 == 0) {
                const unsigned cc = gk[0] == 0 ? c[0] + sz * (L.nz - 1) : c[0] - sz;
                de[0] = at(L.cz, cc);
                if (two) de[1] = at(L.cz, cc + 1);
            }
        }
        lds_barrier();
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const T xl = lane_below(cxo[p][1]);
            cxo[p][0] = w0 ? xw[p] : xl;
            if (c[p] < 0) cxo[p][0] = (T)0;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                cs[p][q] = s0 ? se[p][q] : S.cy[q][own(p) + ds];
                cd[p][q] = p == 0 && k0 == 0 ? de[q] : S.cz[q][own(p) - kLegPlane];
                if (c[p] < 0 || (q && !two)) cs[p][q] = cd[p][q] = (T)0;
            }
            if (DGI && c[p] >= 0) {
                ga[p] = diag<0>(p);
                if (two) gb[p] = diag<1>(p);
            }
            rd[p][0] = (T)1 / ga[p];
            rd[p][1] = (T)1 / gb[p];
        }
    }
    // the coupling sum of a cell
    template <int POS> __device__ __forceinline__ T diag(int p) const {
        return POS ? diag_sum(co[p], cxo[p][1], cs[p][1], cn[p][1], cd[p][1], cu[p][1])
                   : diag_sum(cxo[p][0], co[p], cs[p][0], cn[p][0], cd[p][0], cu[p][0]);
    }
    // b + sum coupling * neighbour
    template <int POS> __device__ __forceinline__ T sum(int p) const {
        const int o = own(p);
        T v = b[p][POS] + co[p] * x[p][1 - POS];
        v += cxo[p][POS] * X(1 - POS, o + (POS ? 1 : -1));
        v += cs[p][POS] * X(POS, o + ds);
        v += cn[p][POS] * X(POS, o + dn);
        v += cd[p][POS] * X(POS, o - kLegPlane);
        v += cu[p][POS] * X(POS, o + kLegPlane);
        return v;
    }
    template <int POS> __device__ __forceinline__ void update() {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            x[p][POS] = sum<POS>(p) * rd[p][POS];
            X(POS, own(p)) = x[p][POS];
        }
    }
    // one colour pass
    template <int Q> __device__ __forceinline__ void pass() {
        if (odd != (Q != 0)) update<1>();
        else update<0>();
        lds_barrier();
    }
    __device__ __forceinline__ bool out(int p) const {
        return m >= kLegHalo / 2 && m < (kLegHalo + kLegOut) / 2 && j >= kLegHalo && j < kLegHalo + kLegOut &&
               plane(p) >= kLegHalo && plane(p) < EZ - kLegHalo;
    }
    // whether the pair's cells are the block's to store (a tile past the end
    // of a short periodic axis holds copies)
    __device__ __forceinline__ bool stores(int p, const LevelK<T> &L, int ox, int oy, int oz) const {
        return out(p) && c[p] >= 0 && ox - kLegHalo + 2 * m < L.nx && oy - kLegHalo + j < L.ny &&
               oz - kLegHalo + plane(p) < L.nz;
    }
    __device__ __forceinline__ void store(int p, T *__restrict__ xo) const {
        xo[c[p]] = x[p][0];
        if (two) xo[c[p] + 1] = x[p][1];
    }
};

__device__ __forceinline__ void leg_tile(const LegK &g, int oz_cells, int &ox, int &oy, int &oz) {
    const int t = xcd_order(blockIdx.x, gridDim.x);
    ox = t % g.tx * kLegOut;
    oy = t / g.tx % g.ty * kLegOut;
    oz = t / (g.tx * g.ty) * oz_cells;
}

// xo = two sweeps (colour 0 first) from zero for the right-hand side b, and
// bc = the restricted residual.  Nothing once the outer iteration has stopped.
template <class T, bool DGI, int EZ>
__global__ void __launch_bounds__(kLegThreads)
k_leg_pre(LevelK<T> L, LegK g, Coarsening cg, const T *__restrict__ b, T *__restrict__ xo, T *__restrict__ bc,
          StopK stop) {
    if (stopped(stop)) return;
    using Lg = Leg<T, DGI, EZ>;
    __shared__ typename Lg::Lds lds;
    int ox, oy, oz;
    leg_tile(g, Lg::kOz, ox, oy, oz);
    Lg S(lds);
    S.load(L, g, b, ox, oy, oz);
    // the first pass needs no neighbours; the other colour starts at zero
#pragma unroll
    for (int p = 0; p < Lg::P; ++p) {
        S.x[p][0] = S.odd ? (T)0 : S.b[p][0] * S.rd[p][0];
        S.x[p][1] = S.odd ? S.b[p][1] * S.rd[p][1] : (T)0;
        S.X(0, S.own(p)) = S.x[p][0];
        S.X(1, S.own(p)) = S.x[p][1];
    }
    lds_barrier();
    S.template pass<1>();
    S.template pass<0>();
    S.template pass<1>();
    // residuals by position over the output cells, in the LDS of the couplings
    T *R = &lds.cy[0][0];
#pragma unroll
    for (int p = 0; p < Lg::P; ++p) {
        if (!S.out(p)) continue;
        T d0 = 0, d1 = 0;
        if (DGI) {
            d0 = S.template diag<0>(p);
            d1 = S.template diag<1>(p);
        } else if (S.c[p] >= 0) {
            d0 = at(L.dg, S.c[p]);
            if (S.two) d1 = at(L.dg, S.c[p] + 1);
        }
        const int r = S.m - kLegHalo / 2 + kLegOut / 2 * (S.j - kLegHalo + kLegOut * (S.plane(p) - kLegHalo));
        R[r] = S.template sum<0>(p) - d0 * S.x[p][0];
        R[Lg::kOutPairs + r] = S.template sum<1>(p) - d1 * S.x[p][1];
        if (S.stores(p, L, ox, oy, oz)) S.store(p, xo);
    }
    lds_barrier();
    const int cx = kLegOut / cg.fx, cy = kLegOut / cg.fy, cz = Lg::kOz / cg.fz;
    for (int e = threadIdx.x; e < cx * cy * cz; e += kLegThreads) {
        int I, J, K;
        split3(e, cx, cy, I, J, K);
        const int gI = ox / cg.fx + I, gJ = oy / cg.fy + J, gK = oz / cg.fz + K;
        if (gI >= cg.cnx || gJ >= cg.cny || gK >= cg.cnz) continue;
        T acc = 0;
        for (int k = cg.fz * K; k < cg.fz * (K + 1); ++k)
            for (int j = cg.fy * J; j < cg.fy * (J + 1); ++j) {
                const T *r = R + kLegOut / 2 * (j + kLegOut * k);
                acc += cg.fx == 2 ? r[I] + r[Lg::kOutPairs + I] : r[((I & 1) ? Lg::kOutPairs : 0) + (I >> 1)];
            }
        bc[gI + (long long)cg.cnx * (gJ + (long long)cg.cny * gK)] =
            acc * ((T)1 / (T)(cg.fx * cg.fy * cg.fz));
    }
}

// xo = two sweeps (colour 1 first) from x + P ec, ec the coarse level's
// iterate (only the colour-0 values of x + P ec are read: the first pass
// overwrites the others).  DOT: block sums of b xo, xo and b over the output
// cells, laid out as k_rb_sweep's.
template <class T, bool DGI, int EZ, bool DOT>
__global__ void __launch_bounds__(kLegThreads)
k_leg_post(LevelK<T> L, LegK g, Coarsening cg, const T *__restrict__ b, const T *__restrict__ x,
           const T *__restrict__ ec, T *__restrict__ xo, double *__restrict__ part) {
    using Lg = Leg<T, DGI, EZ>;
    __shared__ typename Lg::Lds lds;
    int ox, oy, oz;
    leg_tile(g, Lg::kOz, ox, oy, oz);
    Lg S(lds);
    S.load(L, g, b, ox, oy, oz);
    const int o = S.odd ? 1 : 0;   // the colour-0 cell of the pair
#pragma unroll
    for (int p = 0; p < Lg::P; ++p) {
        T v = 0;
        if (S.c[p] >= 0 && (!o || S.two))
            v = at(x, S.c[p] + o) + at(ec, ((S.gi + o) >> (cg.fx - 1)) +
                                               cg.cnx * ((S.gj >> (cg.fy - 1)) + cg.cny * (S.gk[p] >> (cg.fz - 1))));
        S.x[p][0] = o ? (T)0 : v;
        S.x[p][1] = o ? v : (T)0;
        S.X(0, S.own(p)) = S.x[p][0];
        S.X(1, S.own(p)) = S.x[p][1];
    }
    lds_barrier();
    S.template pass<1>();
    S.template pass<0>();
    S.template pass<1>();
    S.template pass<0>();
    double sbx = 0.0, sx = 0.0, sb = 0.0;
#pragma unroll
    for (int p = 0; p < Lg::P; ++p) {
        if (!S.stores(p, L, ox, oy, oz)) continue;
        S.store(p, xo);
        if (DOT) {
            sbx += (double)S.b[p][0] * (double)S.x[p][0] + (double)S.b[p][1] * (double)S.x[p][1];
            sx += (double)S.x[p][0] + (double)S.x[p][1];
            sb += (double)S.b[p][0] + (double)S.b[p][1];
        }
    }
    if (DOT) {
        block_partial(sbx, part);
        block_partial(sx, part + kRedBlocks);
        block_partial(sb, part + 2 * kRedBlocks);
    }
}

}  // namespace pps
