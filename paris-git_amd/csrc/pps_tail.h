// pps_tail.h -- x-pairs ordered by colour, and the coarse end of a V-cycle
// in one workgroup.
//
// Along x the cells go in pairs (2m, 2m+1); in every row a pair holds one
// cell of each colour ((i+j+k)&1), and on a wall axis of odd size the last
// pair's second cell is missing (no couplings, diagonal 1, value 0).  The
// iterate of a level lies in LDS as two arrays, X[q][pair] the colour-q cell
// of a pair: of a cell's six neighbours one is its pair's other cell (in a
// register), and the other five have unit-stride addresses across a
// wavefront, where cells in their own order would be two apart.
#pragma once

#include "pps_level.h"

namespace pps {

// The rows of a pair's two cells, by colour: co the coupling of the pair's
// cells, cxo the x coupling to the neighbouring pair, cs / cn, cd / cu the
// -y / +y, -z / +z couplings, rd the reciprocal of the diagonal (a division
// in each update, ten dependent instructions, would be most of a pass).
template <class T> struct PairRow {
    T co, cxo[2], cs[2], cn[2], cd[2], cu[2], rd[2];
};
constexpr int kPairFields = 13;   // values of a PairRow

// LDS pair indices of the neighbours: o[q] the pair across the outer x face
// of the colour-q cell.
struct PairNb {
    int own, s, n, d, u, o[2];
};

// What the rows of pair m of row j, plane k are formed from: loaded first for
// all of a thread's pairs, so that one latency covers them.
template <class T, bool DGI> struct PairLoad {
    T xw, xa, xb, sa, sb, na, nb, da, db, ua, ub, ga, gb;
    __device__ __forceinline__ void load(const LevelK<T> &L, int m, int j, int k) {
        const int sy = L.nx, sz = L.nx * L.ny, i = 2 * m;
        const long long c = i + (long long)sy * j + (long long)sz * k;
        const int o = i + 1 < L.nx ? 1 : 0;
        const long long cw = m == 0 ? c + (L.nx - 1) : c - 1;
        const long long cs = c + (long long)(wrap_m(j, L.ny) - j) * sy;
        const long long cd = c + (long long)(wrap_m(k, L.nz) - k) * sz;
        xw = L.cx[cw], xa = L.cx[c], xb = L.cx[c + o];
        sa = L.cy[cs], sb = L.cy[cs + o], na = L.cy[c], nb = L.cy[c + o];
        da = L.cz[cd], db = L.cz[cd + o], ua = L.cz[c], ub = L.cz[c + o];
        if (!DGI) { ga = L.dg[c]; gb = L.dg[c + o]; }
    }
    // o: the pair's second cell exists; e: colour 0 is that cell (j + k odd)
    __device__ __forceinline__ void form(bool o, bool e, PairRow<T> &P) {
        if (DGI) {
            ga = diag_sum(xw, xa, sa, na, da, ua);
            gb = diag_sum(xa, xb, sb, nb, db, ub);
        }
        if (!o) { xb = sb = nb = db = ub = (T)0; gb = (T)1; }
        P.co = xa;
        P.cxo[0] = e ? xb : xw; P.cxo[1] = e ? xw : xb;
        P.cs[0] = e ? sb : sa; P.cs[1] = e ? sa : sb;
        P.cn[0] = e ? nb : na; P.cn[1] = e ? na : nb;
        P.cd[0] = e ? db : da; P.cd[1] = e ? da : db;
        P.cu[0] = e ? ub : ua; P.cu[1] = e ? ua : ub;
        P.rd[0] = (T)1 / (e ? gb : ga); P.rd[1] = (T)1 / (e ? ga : gb);
    }
};

// b + sum coupling * neighbour of the pair's colour-Q cell: xo the pair's
// other cell, O the other colour's LDS array
template <int Q, class T>
__device__ __forceinline__ T pair_sum(const PairRow<T> &P, const PairNb &N, T b, T xo, const T *O) {
    T v = b;
    v += P.co * xo + P.cxo[Q] * O[N.o[Q]];
    v += P.cs[Q] * O[N.s] + P.cn[Q] * O[N.n];
    v += P.cd[Q] * O[N.d] + P.cu[Q] * O[N.u];
    return v;
}

// Diagonal of the colour-Q cell of pair (m, j, k): the coupling sum, or
// stored (DGI false; any finite value does for a missing second cell).
template <int Q, bool DGI, class T>
__device__ __forceinline__ T pair_diag(const PairRow<T> &P, const LevelK<T> &L, int m, int j, int k) {
    if (DGI) return diag_sum(P.co, P.cxo[Q], P.cs[Q], P.cn[Q], P.cd[Q], P.cu[Q]);
    const int i = min(2 * m + (Q ^ ((j + k) & 1)), L.nx - 1);
    return L.dg[i + (long long)L.nx * (j + (long long)L.ny * k)];
}

// ---------------------------------------------------------------------
// Levels 0 .. nl-1 of the tail (level nl-1 is the coarsest, solved with its
// dense inverse) run in one workgroup: smoothing, restriction, the bottom
// solve and prolongation on LDS with workgroup barriers in between, one
// launch instead of several per level.  It is bound by the latency of its
// passes, so each pass is kept short: level 0's rows and right-hand side
// stay in registers for the whole launch (up to P pairs a thread), the rows
// of the levels below are staged in LDS by pair and held in registers
// while a level is smoothed, addresses are formed once per level, and every
// global load is issued before the first pass.  Any level of the plan
// qualifies (odd sizes, semi-coarsening); the smoothing is the colour
// passes of k_rb (pre: colour 0 first, post: colour 1 first).
// From 16^3, FP32: 15.5 us a launch (27.5 with every operand in LDS, 64-bit
// addresses formed again for each cell and a division an update; 16.5 with
// the inverse and the middle levels loaded after level 0 was formed).  FP64
// from 16^3: 25.8 us, some registers spilled, against 12 us from 8^3 and 27 us
// for the 16^3 level's own launches.
// ---------------------------------------------------------------------
constexpr int kTailMax = 8;
constexpr int kTailThreads = 1024;
template <class T> struct TailK {
    int nl, nb, nu_pre, nu_post;
    LevelK<T> L[kTailMax];   // operators in global memory
    Coarsening g[kTailMax];  // to the next level
    const T *b0;             // right-hand side of level 0 (global)
    T *x0;                   // iterate of level 0 (global, written at the end)
    const T *minv;
    // LDS offsets in elements of T: X of levels 1 .. nl-1 (two arrays of its
    // pairs; level 0's lies at 0, P kTailThreads apart), rows and right-hand side of levels 1 .. nl-2 (kPairFields + 2
    // arrays of their pairs), residual of the level being left (two arrays
    // of level 0's pairs), right-hand side and inverse of the coarsest
    int off_x[kTailMax], off_op[kTailMax];
    int off_r, off_b, off_minv;
};

__host__ __device__ inline int pairs_of(int nx, int ny, int nz) { return ((nx + 1) >> 1) * ny * nz; }

// (a, b, c) of linear index e in an na x nb x nc box: shifts and masks when
// na and nb are powers of two, divisions otherwise
__device__ __forceinline__ void split3(int e, int na, int nb, int &a, int &b, int &c) {
    if (((na & (na - 1)) | (nb & (nb - 1))) == 0) {
        const int la = __builtin_ctz(na), lb = __builtin_ctz(nb);
        a = e & (na - 1);
        b = (e >> la) & (nb - 1);
        c = e >> (la + lb);
    } else {
        a = e % na;
        b = (e / na) % nb;
        c = e / (na * nb);
    }
}

// neighbours of pair p = (m, j, k) of a whole level (wrapped: the coupling
// through a wall is 0)
__device__ __forceinline__ PairNb pair_nb(int p, int m, int j, int k, int np, int ny, int nz) {
    PairNb N;
    N.own = p;
    N.s = p + (wrap_m(j, ny) - j) * np;
    N.n = p + (wrap_p(j, ny) - j) * np;
    N.d = p + (wrap_m(k, nz) - k) * np * ny;
    N.u = p + (wrap_p(k, nz) - k) * np * ny;
    const int w = p + wrap_m(m, np) - m, e = p + wrap_p(m, np) - m;
    const bool odd = (j + k) & 1;
    N.o[0] = odd ? e : w;   // colour 0 is the first cell where j + k is even
    N.o[1] = odd ? w : e;
    return N;
}

// P pairs a thread of one level in registers.  st: pairs between the two
// colours' LDS arrays (a constant for level 0, so that it folds into the
// offsets of the LDS instructions).
template <class T, bool DGI, int P> struct PairSet {
    PairRow<T> row[P];
    PairNb nb[P];
    T b[P][2], x[P][2];
    bool on[P];

    template <int Q, bool FIRST> __device__ __forceinline__ void pass(T *X, int st) {
        T *Xq = X + Q * st;
        const T *O = X + (1 - Q) * st;
#pragma unroll
        for (int p = 0; p < P; ++p)
            if (on[p]) {
                const T v = FIRST ? b[p][Q] : pair_sum<Q>(row[p], nb[p], b[p][Q], x[p][1 - Q], O);
                x[p][Q] = v * row[p].rd[Q];
                Xq[nb[p].own] = x[p][Q];
            }
        lds_barrier();
    }
    __device__ __forceinline__ void pre(T *X, int st, int nu) {
        pass<0, true>(X, st);
        pass<1, false>(X, st);
        for (int q = 1; q < nu; ++q) {
            pass<0, false>(X, st);
            pass<1, false>(X, st);
        }
    }
    __device__ __forceinline__ void post(T *X, int st, int nu) {
        for (int q = 0; q < nu; ++q) {
            pass<1, false>(X, st);
            pass<0, false>(X, st);
        }
    }
    // residual of pair p at (m, j, k) into the arrays R (tot pairs each)
    __device__ __forceinline__ void resid(int p, const LevelK<T> &L, int m, int j, int k, const T *X, int st,
                                          T *R, int tot) {
        const T d0 = pair_diag<0, DGI>(row[p], L, m, j, k), d1 = pair_diag<1, DGI>(row[p], L, m, j, k);
        R[nb[p].own] = pair_sum<0>(row[p], nb[p], b[p][0], x[p][1], X + st) - d0 * x[p][0];
        R[tot + nb[p].own] = pair_sum<1>(row[p], nb[p], b[p][1], x[p][0], X) - d1 * x[p][1];
    }
};

// restriction: the children's residuals of coarse cell (I, J, K), divided by
// the nominal number of children; R the two colour arrays of the fine level
template <class T>
__device__ __forceinline__ T gather_resid(const T *R, const LevelK<T> &F, const Coarsening &g, int I, int J,
                                          int K) {
    const int np = (F.nx + 1) >> 1, tot = np * F.ny * F.nz;
    const int j1 = min(g.fy * J + g.fy, F.ny), k1 = min(g.fz * K + g.fz, F.nz);
    T acc = 0;
    for (int k = g.fz * K; k < k1; ++k)
        for (int j = g.fy * J; j < j1; ++j) {
            const T *r = R + np * (j + F.ny * k);
            // two x children are a pair (a missing second cell has residual 0)
            acc += g.fx == 2 ? r[I] + r[tot + I] : r[(((I + j + k) & 1) ? tot : 0) + (I >> 1)];
        }
    return acc * ((T)1 / (T)(g.fx * g.fy * g.fz));
}

// value of cell (i, j, k) of a level whose iterate is X (st pairs between
// the colours)
template <class T>
__device__ __forceinline__ T pair_value(const T *X, int st, int nx, int ny, int i, int j, int k) {
    const int np = (nx + 1) >> 1;
    return X[(((i + j + k) & 1) ? st : 0) + (i >> 1) + np * (j + ny * k)];
}

template <class T, bool DGI, int P>
__global__ void __launch_bounds__(kTailThreads)
k_tail(TailK<T> K) {
    extern __shared__ unsigned char smem_raw[];
    T *sm = reinterpret_cast<T *>(smem_raw);
    const int tid = threadIdx.x, NT = blockDim.x;
    const int nl = K.nl, nb = K.nb;
    const LevelK<T> &L0 = K.L[0];
    const int np0 = (L0.nx + 1) >> 1, tot0 = np0 * L0.ny * L0.nz;

    // Loads: level 0's couplings and right-hand side, those of a pair of the
    // middle levels (all their pairs in turn, pair tid here) and four values
    // of the inverse
    PairSet<T, DGI, P> S;
    PairLoad<T, DGI> W[P], Wm;
    T ba[P], bb[P], mv[4];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int e = tid + p * NT;
        S.on[p] = e < tot0;
        int m, j, k;
        split3(S.on[p] ? e : 0, np0, L0.ny, m, j, k);
        W[p].load(L0, m, j, k);
        const int c = 2 * m + L0.nx * (j + L0.ny * k);
        ba[p] = K.b0[c];
        bb[p] = K.b0[c + (2 * m + 1 < L0.nx ? 1 : 0)];
    }
    int at_m = 0, tm = 0, base = 0;   // Wm: its place in LDS, pairs of its level (0: none)
    bool om = false, em = false;
    for (int l = 1; l < nl - 1; ++l) {
        const LevelK<T> &L = K.L[l];
        const int tot = pairs_of(L.nx, L.ny, L.nz);
        if (tid >= base && tid < base + tot) {
            at_m = K.off_op[l] + tid - base;
            tm = tot;
            int m, j, k;
            split3(tid - base, (L.nx + 1) >> 1, L.ny, m, j, k);
            om = 2 * m + 1 < L.nx;
            em = (j + k) & 1;
            Wm.load(L, m, j, k);
        }
        base += tot;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (tid + c * NT < nb * nb) mv[c] = K.minv[tid + c * NT];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int e = S.on[p] ? tid + p * NT : 0;
        int m, j, k;
        split3(e, np0, L0.ny, m, j, k);
        const bool two = 2 * m + 1 < L0.nx, odd = (j + k) & 1;
        W[p].form(two, odd, S.row[p]);
        S.nb[p] = pair_nb(e, m, j, k, np0, L0.ny, L0.nz);
        if (!two) bb[p] = (T)0;
        S.b[p][0] = odd ? bb[p] : ba[p];
        S.b[p][1] = odd ? ba[p] : bb[p];
    }
    // the middle levels' rows and the inverse into LDS
    auto rows_to_lds = [&](int at, int tot, const PairRow<T> &row) {
        T *o = sm + at;
        o[0] = row.co;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            o[(1 + q) * tot] = row.cxo[q];
            o[(3 + q) * tot] = row.cs[q];
            o[(5 + q) * tot] = row.cn[q];
            o[(7 + q) * tot] = row.cd[q];
            o[(9 + q) * tot] = row.cu[q];
            o[(11 + q) * tot] = row.rd[q];
        }
    };
    if (tm) {
        PairRow<T> row;
        Wm.form(om, em, row);
        rows_to_lds(at_m, tm, row);
    }
    for (int e = tid + NT; e < base; e += NT) {
        int l = 1, p = e, tot;
        for (; p >= (tot = pairs_of(K.L[l].nx, K.L[l].ny, K.L[l].nz)); ++l) p -= tot;
        const LevelK<T> &L = K.L[l];
        int m, j, k;
        split3(p, (L.nx + 1) >> 1, L.ny, m, j, k);
        PairRow<T> row;
        Wm.load(L, m, j, k);
        Wm.form(2 * m + 1 < L.nx, (j + k) & 1, row);
        rows_to_lds(K.off_op[l] + p, tot, row);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (tid + c * NT < nb * nb) sm[K.off_minv + tid + c * NT] = mv[c];
    for (int e = tid + 4 * NT; e < nb * nb; e += NT) sm[K.off_minv + e] = K.minv[e];
    auto rows_from_lds = [&](int l, int p, int tot, PairRow<T> &row) {
        const T *o = sm + K.off_op[l] + p;
        row.co = o[0];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            row.cxo[q] = o[(1 + q) * tot];
            row.cs[q] = o[(3 + q) * tot];
            row.cn[q] = o[(5 + q) * tot];
            row.cd[q] = o[(7 + q) * tot];
            row.cu[q] = o[(9 + q) * tot];
            row.rd[q] = o[(11 + q) * tot];
        }
    };
    T *R = sm + K.off_r;
    T *X0 = sm;
    constexpr int ST0 = P * kTailThreads;
    S.pre(X0, ST0, K.nu_pre);   // its first barrier publishes the staged rows
#pragma unroll
    for (int p = 0; p < P; ++p)
        if (S.on[p]) {
            int m, j, k;
            split3(S.nb[p].own, np0, L0.ny, m, j, k);
            S.resid(p, L0, m, j, k, X0, ST0, R, tot0);
        }
    lds_barrier();

    // down the middle levels: one pair a thread
    for (int l = 1; l < nl - 1; ++l) {
        const LevelK<T> &L = K.L[l];
        const int np = (L.nx + 1) >> 1, tot = np * L.ny * L.nz;
        PairSet<T, DGI, 1> M;
        M.on[0] = tid < tot;
        int m, j, k;
        split3(M.on[0] ? tid : 0, np, L.ny, m, j, k);
        M.nb[0] = pair_nb(M.on[0] ? tid : 0, m, j, k, np, L.ny, L.nz);
        if (M.on[0]) {
            rows_from_lds(l, tid, tot, M.row[0]);
            const T ba = gather_resid(R, K.L[l - 1], K.g[l - 1], 2 * m, j, k);
            const T bb = 2 * m + 1 < L.nx ? gather_resid(R, K.L[l - 1], K.g[l - 1], 2 * m + 1, j, k) : (T)0;
            const bool o = (j + k) & 1;
            M.b[0][0] = o ? bb : ba;
            M.b[0][1] = o ? ba : bb;
            T *bs = sm + K.off_op[l] + kPairFields * tot + tid;
            bs[0] = M.b[0][0];
            bs[tot] = M.b[0][1];
        }
        T *X = sm + K.off_x[l];
        M.pre(X, tot, K.nu_pre);
        if (M.on[0]) M.resid(0, L, m, j, k, X, tot, R, tot);
        lds_barrier();
    }
    // the coarsest level: 16 lanes a row of the inverse
    {
        const LevelK<T> &L = K.L[nl - 1];
        T *sb = sm + K.off_b, *X = sm + K.off_x[nl - 1];
        for (int c = tid; c < nb; c += NT) {
            int i, j, k;
            split3(c, L.nx, L.ny, i, j, k);
            sb[c] = gather_resid(R, K.L[nl - 2], K.g[nl - 2], i, j, k);
        }
        lds_barrier();
        const T *mi = sm + K.off_minv;
        const int np = (L.nx + 1) >> 1, tot = np * L.ny * L.nz;
        for (int r = tid >> 4; r < ((nb + 3) & ~3); r += NT >> 4) {   // whole wavefronts
            T acc = 0;
            if (r < nb)
                for (int e = tid & 15; e < nb; e += 16) acc += mi[r * nb + e] * sb[e];
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 16);
            if (r < nb && (tid & 15) == 0) {
                int i, j, k;
                split3(r, L.nx, L.ny, i, j, k);
                X[(((i + j + k) & 1) ? tot : 0) + (i >> 1) + np * (j + L.ny * k)] = acc;
            }
        }
        lds_barrier();
    }
    // x += the parent's value, both cells of a pair; published for the passes
    auto correct = [&](int l, int p, int m, int j, int k, T *x, T *X, int tot) {
        const Coarsening &g = K.g[l];
        const T *Xc = sm + K.off_x[l + 1];
        const int st = pairs_of(g.cnx, g.cny, g.cnz);
        const int J = g.fy == 2 ? j >> 1 : j, Kz = g.fz == 2 ? k >> 1 : k;
        const T ea = pair_value(Xc, st, g.cnx, g.cny, g.fx == 2 ? m : 2 * m, J, Kz);
        const T eb = g.fx == 2 ? ea
                               : (2 * m + 1 < K.L[l].nx ? pair_value(Xc, st, g.cnx, g.cny, 2 * m + 1, J, Kz) : (T)0);
        const bool o = (j + k) & 1;
        x[0] += o ? eb : ea;
        x[1] += o ? ea : eb;
        X[p] = x[0];
        X[tot + p] = x[1];
    };
    for (int l = nl - 2; l >= 1; --l) {
        const LevelK<T> &L = K.L[l];
        const int np = (L.nx + 1) >> 1, tot = np * L.ny * L.nz;
        PairSet<T, DGI, 1> M;
        M.on[0] = tid < tot;
        int m, j, k;
        split3(M.on[0] ? tid : 0, np, L.ny, m, j, k);
        M.nb[0] = pair_nb(M.on[0] ? tid : 0, m, j, k, np, L.ny, L.nz);
        T *X = sm + K.off_x[l];
        if (M.on[0]) {
            rows_from_lds(l, tid, tot, M.row[0]);
            const T *bs = sm + K.off_op[l] + kPairFields * tot + tid;
            M.b[0][0] = bs[0];
            M.b[0][1] = bs[tot];
            M.x[0][0] = X[tid];
            M.x[0][1] = X[tot + tid];
            correct(l, tid, m, j, k, M.x[0], X, tot);
        }
        lds_barrier();
        M.post(X, tot, K.nu_post);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
        if (S.on[p]) {
            int m, j, k;
            split3(tid + p * NT, np0, L0.ny, m, j, k);
            correct(0, S.nb[p].own, m, j, k, S.x[p], X0, ST0);
        }
    lds_barrier();
    S.post(X0, ST0, K.nu_post);
#pragma unroll
    for (int p = 0; p < P; ++p)
        if (S.on[p]) {
            int m, j, k;
            split3(tid + p * NT, np0, L0.ny, m, j, k);
            const int c = 2 * m + L0.nx * (j + L0.ny * k);
            const bool odd = (j + k) & 1;
            K.x0[c] = odd ? S.x[p][1] : S.x[p][0];
            if (2 * m + 1 < L0.nx) K.x0[c + 1] = odd ? S.x[p][0] : S.x[p][1];
        }
}

}  // namespace pps
