// One-sided block Jacobi SVD on Gram tiles (FP64 and FP32).
//
// The matrix J (rows x ncols, column-major) is orthogonalised column-wise: J V = Z with V
// orthogonal and the columns of Z mutually orthogonal; sigma_j = |z_j|.  Columns are grouped in
// blocks of GJ_B = 8; a tile is a pair of blocks (16 columns) and belongs to one wave, or to NS
// waves that share its rows:
//   1. G = Y^T Y, the tile's 16 x 16 Gram matrix, on the matrix cores (K = rows), so that every
//      dot product of the tile comes out of one pass over its columns without a wave reduction;
//   2. one pass of rotations over the tile's column pairs on G alone (two-sided, J^T G J), the
//      rotations accumulated in a 16 x 16 V.  Lane (p, q) of the 8 x 8 lane grid holds the 2 x 2
//      blocks of pairs p and q of G, and two rows of V; a round computes the 8 rotations in the
//      diagonal lanes, passes them along the grid's rows and columns, and moves the second column of
//      every pair to the next lane;
//   3. Y <- Y V on the matrix cores.
// A round is thus about a dozen lane exchanges and one rotation's arithmetic, whatever the number of
// rows; the rows cost 8 matrix-core steps per 16 rows and visit.  (The form before it kept the
// tile's rows in registers and reduced the 24 dot products of each round across the wave: 8 wave
// reductions per visit, 0.26-0.37 ms per sweep of a 65-99-column core.)
// A step visits disjoint block pairs in the circle (round-robin) ordering: step 0 of every
// sweep rotates all pairs of the tile's columns, later steps only the pairs across its blocks.
//
// G is formed afresh from the columns at every visit, so errors of the two-sided updates do not
// accumulate; within a visit they are relative to the columns' norms (the scaled Gram matrix of a
// QR-preconditioned core is well conditioned), and the measured singular values and vectors are as
// accurate as with dot products taken before every rotation.
//
// Convergence test: |z_p . z_q| <= sqrt(rows) * eps * |z_p| |z_q| (relative, as LAPACK's
// one-sided Jacobi), pairs involving a column whose norm is below eps * ||J||_F are not rotated
// (those columns carry rounding-level singular values).  A sweep ends the iteration when every pair
// it visited had a cosine of at most JacobiStopCos on arrival: Jacobi converges quadratically, so the
// cosines it leaves are of the order of that bound's square, and the sweeps that would only shrink
// them further are skipped.  The plain, one-update-at-a-time form stops at 0.1 sqrt(eps), which
// leaves U orthonormal to rounding as LAPACK's SVD does; the batched form stops at 1e-5 in FP64
// (cosines left of order 1e-10, U orthonormal to about 1e-10, singular values exact to rounding),
// one sweep fewer.  The test is on the cosine and not on the rotation's angle: two columns of
// nearly equal norm take a large rotation even when nearly orthogonal.
#pragma once

#include "device_common.hpp"

namespace hcamd {

// Bits a tile's visit returns: it was rotated, and some pair was far from orthogonal on arrival (the
// sweep has not converged).
enum : int { JROT_APPLIED = 1, JROT_LARGE = 2 };

template <typename T>
struct JacobiStopCos;
template <>
struct JacobiStopCos<double> {
    static constexpr double tight = 1.4901161193847656e-09;  // 0.1 * sqrt(2^-52)
    static constexpr double loose = 1e-5;
};
template <>
struct JacobiStopCos<float> {
    static constexpr float tight = 3.4526698e-05f;  // 0.1 * sqrt(2^-23)
    static constexpr float loose = 3.4526698e-05f;
};

constexpr int GJ_B = 8;               // columns per block; a tile is two blocks
constexpr int GJ_TW = 2 * GJ_B;
constexpr int GJ_LD = GJ_TW + 1;      // odd, so that a row or a column of a tile matrix spans the LDS banks
constexpr int GJ_SC = GJ_TW * GJ_LD;  // LDS elements of one wave's tile matrix

// Tolerances of one Jacobi.  Gram entries are scaled by a power of two so that ||J||_F^2 is about 1
// (FP64) or 2^60 (FP32): products of two entries, and the squares of the smallest that can still ask
// for a rotation, then neither overflow nor underflow (columns below eps ||J||_F do not take part).
// Cosines are compared by their squares, in full precision.
template <typename T>
struct GramTol {
    T tol2, stop2, floor2, scale;  // squares of the two bounds on a cosine, of the smallest norm that takes part
    __device__ __forceinline__ GramTol(T fro2, int rows, T stop) {
        int ex = 0;
        constexpr int top = sizeof(T) == 8 ? 0 : 60, lim = sizeof(T) == 8 ? 1000 : 120;
        if (fro2 > T(0) && fro2 < T(INFINITY)) ex = top - ilogb(fro2);
        ex = ex < -lim ? -lim : (ex > lim ? lim : ex);
        scale = scalbn(T(1), ex);
        tol2 = T(rows) * (Eps<T>::value * Eps<T>::value);
        stop2 = stop * stop;
        floor2 = Eps<T>::value * Eps<T>::value * (fro2 * scale);
    }
};

// 1 / sqrt(x) to rounding for x in the normal range: the hardware's estimate (relative error e of
// about 2^-24 in FP64, 2^-22 in FP32) and one third-order step, y (1 + e' / 2 + 3 e'^2 / 8) with
// e' = 1 - x y^2.
__device__ __forceinline__ double rsqrt_full(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ float rsqrt_full(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float e = fmaf(-(x * y), y, 1.0f);
    return fmaf(y * e, fmaf(e, 0.375f, 0.5f), y);
}

// Rotation (c, s) that annihilates apq for the Gram entries (app, aqq, apq) of a column pair, or
// (1, 0) when the pair is already orthogonal to tolerance or involves a numerically zero column.
// With d = aqq - app and e = 2 apq, the smaller rotation has cos 2t = |d| / h, sin 2t = sign(d) e / h for
// h = hypot(d, e); c = sqrt((1 + cos 2t) / 2), s = sin 2t / (2 c): two reciprocal square roots in
// turn and no division.
template <typename T>
__device__ __forceinline__ void jacobi_rotation(T app, T aqq, T apq, const GramTol<T> &g, T &c, T &s) {
    const bool act = app > g.floor2 && aqq > g.floor2 && apq * apq > g.tol2 * (app * aqq);
    const T d = aqq - app, e = T(2) * apq;
    const T r = rsqrt_full(d * d + e * e);
    const T c2 = fma(T(0.5) * fabs(d), r, T(0.5));
    const T ic = rsqrt_full(c2);
    c = act ? c2 * ic : T(1);
    s = act ? (d >= T(0) ? e : -e) * (T(0.5) * r) * ic : T(0);
}

// The rotations of one visit, on the tile's scaled Gram matrix in `sc` (wave-private LDS, row i at
// i * GJ_LD); V is left in `sc`.  A stage pairs the first h columns of each group of 2 h with its
// last h: pair p is (a, b) with a = 2 h (p / h) + p % h and b = a + h at first; after each of the
// stage's h rounds b moves on to the next pair of the group, so every a meets every b and the
// columns are back in place.  A cross tile is the stage h = 8; a full tile adds h = 4, 2, 1, which
// together visit every pair of the 16 columns once.
template <typename T>
__device__ __forceinline__ void gram_rotate(T *sc, bool full, const GramTol<T> &g) {
    const int l = lane_id(), p = l >> 3, q = l & 7;
    T v0a = T(0), v0b = T(0), v1a = T(0), v1b = T(0);  // rows p and p + 8 of V, columns a_q and b_q
#pragma unroll 1
    for (int h = GJ_B; h > 0; h = full ? h >> 1 : 0) {
        const int ap = ((p & ~(h - 1)) << 1) | (p & (h - 1)), aq = ((q & ~(h - 1)) << 1) | (q & (h - 1));
        const int bp = ap + h, bq = aq + h;
        T gaa = sc[ap * GJ_LD + aq], gab = sc[ap * GJ_LD + bq], gba = sc[bp * GJ_LD + aq], gbb = sc[bp * GJ_LD + bq];
        if (h == GJ_B) {
            v0a = T(p == aq);
            v1b = T(p + GJ_B == bq);
        } else {
            // V's columns in the order of this stage (the previous stage's went through sc below)
            wave_fence();
            const int h2 = 2 * h;
            const int oq = ((q & ~(h2 - 1)) << 1) | (q & (h2 - 1));
            sc[p * GJ_LD + oq] = v0a;
            sc[p * GJ_LD + oq + h2] = v0b;
            sc[(p + GJ_B) * GJ_LD + oq] = v1a;
            sc[(p + GJ_B) * GJ_LD + oq + h2] = v1b;
            wave_fence();
            v0a = sc[p * GJ_LD + aq];
            v0b = sc[p * GJ_LD + bq];
            v1a = sc[(p + GJ_B) * GJ_LD + aq];
            v1b = sc[(p + GJ_B) * GJ_LD + bq];
        }
        // lanes the second columns come from: the next pair of the group along either axis
        const int qs = (q & ~(h - 1)) | ((q + 1) & (h - 1)), ps = (p & ~(h - 1)) | ((p + 1) & (h - 1));
        const int from_q = 8 * p + qs, from_p = 8 * ps + q, from_pq = 8 * ps + qs;
#pragma unroll 1
        for (int rd = 0; rd < h; ++rd) {
            T c, s;
            jacobi_rotation(gaa, gbb, gab, g, c, s);  // pair p's in lane (p, p)
            const T cq = lane_fetch(c, 9 * q), sq = lane_fetch(s, 9 * q);
            const T cp = lane_fetch(c, 9 * p), sp = lane_fetch(s, 9 * p);
            const T raa = cp * gaa - sp * gba, rba = sp * gaa + cp * gba;
            const T rab = cp * gab - sp * gbb, rbb = sp * gab + cp * gbb;
            gaa = cq * raa - sq * rab;
            gab = lane_fetch(sq * raa + cq * rab, from_q);
            gba = lane_fetch(cq * rba - sq * rbb, from_p);
            gbb = lane_fetch(sq * rba + cq * rbb, from_pq);
            const T w0 = v0a, w1 = v1a;
            v0a = cq * w0 - sq * v0b;
            v1a = cq * w1 - sq * v1b;
            v0b = lane_fetch(sq * w0 + cq * v0b, from_q);
            v1b = lane_fetch(sq * w1 + cq * v1b, from_q);
        }
        wave_fence();
        if (full && h > 1) {
            sc[ap * GJ_LD + aq] = gaa;
            sc[ap * GJ_LD + bq] = gab;
            sc[bp * GJ_LD + aq] = gba;
            sc[bp * GJ_LD + bq] = gbb;
        } else {
            sc[p * GJ_LD + aq] = v0a;
            sc[p * GJ_LD + bq] = v0b;
            sc[(p + GJ_B) * GJ_LD + aq] = v1a;
            sc[(p + GJ_B) * GJ_LD + bq] = v1b;
        }
        wave_fence();
    }
}

// One visit's rotations from the tile's Gram matrix, in the accumulator layout in gv: leaves V in `sc`
// (wave-private LDS) and returns the JROT flags; 0, and no V, when no pair the visit covers needs a
// rotation.
template <typename T>
__device__ __forceinline__ int gram_solve(const T (&gv)[4], T *sc, bool full, const GramTol<T> &g) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4;
    wave_fence();
#pragma unroll
    for (int v = 0; v < 4; ++v) sc[MF::row(v, k4) * GJ_LD + i16] = gv[v] * g.scale;
    wave_fence();
    bool any = false, large = false;
    const T dj = sc[i16 * (GJ_LD + 1)];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = MF::row(v, k4);
        const T di = sc[i * (GJ_LD + 1)];
        const bool pair = full ? i < i16 : (i < GJ_B && i16 >= GJ_B);
        if (pair && di > g.floor2 && dj > g.floor2) {
            const T x = gv[v] * g.scale, c2 = x * x, d2 = di * dj;
            any = any || c2 > g.tol2 * d2;
            large = large || c2 > g.stop2 * d2;
        }
    }
    if (__ballot(any) == 0) return 0;
    const int flags = JROT_APPLIED | (__ballot(large) ? JROT_LARGE : 0);
    wave_fence();
    gram_rotate(sc, full, g);
    return flags;
}

// Y <- Y V for 16 columns of M (rows x ncols, ld ldm): columns [cI, cI + 8) and [cJ, cJ + 8), V^T's
// operand values in va (va[s] = V[4 s + k4][i16]).  The product is formed transposed, V^T Y^T, so
// that 16 lanes read and write 16 consecutive rows of a column.  Waves sub of NS take every NS-th
// group of 16 rows.  Columns past ncols are zero in Y and not written.
template <typename T, int NS>
__device__ __forceinline__ void gram_apply(const T (&va)[4], T *M, int64_t ldm, int rows, int ncols, int cI, int cJ,
                                           int sub) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4;
    auto colp = [&](int k) -> T * {  // null past the last column
        const int c = k < GJ_B ? cI + k : cJ + k - GJ_B;
        return c < ncols ? M + (int64_t) c * ldm : nullptr;
    };
    const T *src[4];
    T *dst[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        src[s] = colp(4 * s + k4);
        dst[s] = colp(MF::row(s, k4));
    }
    constexpr int GR = 4;  // groups in flight
    for (int r0 = 16 * sub; r0 < rows; r0 += 16 * NS * GR) {
        T y[GR][4];
#pragma unroll
        for (int gi = 0; gi < GR; ++gi) {
            const int r = r0 + 16 * NS * gi + i16;
#pragma unroll
            for (int s = 0; s < 4; ++s) y[gi][s] = (src[s] && r < rows) ? src[s][r] : T(0);
        }
#pragma unroll
        for (int gi = 0; gi < GR; ++gi) {
            if (r0 + 16 * NS * gi >= rows) break;
            typename MF::acc a = MF::zero();
#pragma unroll
            for (int s = 0; s < 4; ++s) a = MF::mma(va[s], y[gi][s], a);
            const int r = r0 + 16 * NS * gi + i16;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (dst[v] && r < rows) dst[v][r] = a[v];
        }
    }
}

// One visit of the tile with columns [cI, cI + 8) and [cJ, cJ + 8) of J (rows x ncols, ld ldj), by NS
// waves (sub = this wave's number among them); columns past ncols count as zero.  `sc`: this wave's
// GJ_SC elements of LDS, the NS waves' one after another.  With NS > 1 every wave of the workgroup
// must call it (it synchronises twice), with act = false where it has no tile, and the caller
// synchronises before the next visit.  V (vrows x ncols, ld ldv) is rotated too when given.  Returns
// the JROT flags, the same in all NS waves.
template <typename T, int NS>
__device__ __forceinline__ int gram_tile(bool act, T *J, int64_t ldj, int rows, int ncols, int cI, int cJ, bool full,
                                         const GramTol<T> &g, T *sc, int sub, T *V = nullptr, int64_t ldv = 0,
                                         int vrows = 0) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4;
    const int gc = i16 < GJ_B ? cI + i16 : cJ + i16 - GJ_B;
    const bool cok = act && gc < ncols;
    const T *col = J + (int64_t) (cok ? gc : 0) * ldj;
    typename MF::acc acc0 = MF::zero(), acc1 = MF::zero();
    if (act) {
        // lane (i16, k4) supplies rows r0 + 4 k4 .. + 3 of column i16 (the sum may take the rows in any
        // order): both operands of Y^T Y hold the same values
        int r0 = 16 * sub;
        for (; r0 + 16 * NS * 3 + 16 <= rows; r0 += 16 * NS * 4) {
            T a[4][4];
#pragma unroll
            for (int gi = 0; gi < 4; ++gi)
#pragma unroll
                for (int s = 0; s < 4; ++s) a[gi][s] = cok ? col[r0 + 16 * NS * gi + 4 * k4 + s] : T(0);
#pragma unroll
            for (int gi = 0; gi < 4; gi += 2)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    acc0 = MF::mma(a[gi][s], a[gi][s], acc0);
                    acc1 = MF::mma(a[gi + 1][s], a[gi + 1][s], acc1);
                }
        }
        for (; r0 < rows; r0 += 16 * NS) {
            T a[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int r = r0 + 4 * k4 + s;
                a[s] = (cok && r < rows) ? col[r] : T(0);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) acc0 = MF::mma(a[s], a[s], acc0);
        }
    }
    T gv[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) gv[v] = acc0[v] + acc1[v];
    int flags = 0;
    T *first = sc;
    if constexpr (NS > 1) {
        // partial sums of the waves that share the tile; the first of them adds up and rotates
        first = sc - sub * GJ_SC;
#pragma unroll
        for (int v = 0; v < 4; ++v) sc[MF::row(v, k4) * GJ_LD + i16] = gv[v];
        __syncthreads();
        if (act && sub == 0) {
#pragma unroll
            for (int w = 1; w < NS; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) gv[v] += first[w * GJ_SC + MF::row(v, k4) * GJ_LD + i16];
            flags = gram_solve<T>(gv, sc, full, g);
            if (l == 0) sc[GJ_TW] = T(flags);  // the padding element of row 0
        }
        __syncthreads();
        if (!act) return 0;
        flags = (int) first[GJ_TW];
    } else {
        if (!act) return 0;
        flags = gram_solve<T>(gv, sc, full, g);
    }
    if (!flags) return 0;
    T va[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) va[s] = first[(4 * s + k4) * GJ_LD + i16];
    if constexpr (NS == 1) wave_fence();
    gram_apply<T, NS>(va, J, ldj, rows, ncols, cI, cJ, sub);
    if (V) gram_apply<T, NS>(va, V, ldv, vrows, ncols, cI, cJ, sub);
    return flags;
}

// Block pair bp of round-robin step `step` over nbp blocks of B columns: its first columns (cI,
// cJ) and whether it exists (the padding block of an odd block count pairs with nothing).
__device__ __forceinline__ bool jacobi_pair_cols(int bp, int step, int nbp, int B, int ncols, int &cI, int &cJ) {
    int bI, bJ;
    if (bp == 0) {
        bI = nbp - 1;
        bJ = step;
    } else {
        bI = (step + bp) % (nbp - 1);
        bJ = (step - bp + nbp - 1) % (nbp - 1);
    }
    if (bI > bJ) {
        const int t = bI;
        bI = bJ;
        bJ = t;
    }
    cI = bI * B;
    cJ = bJ * B;
    return cI < ncols;
}

// LDS elements of the whole-workgroup Jacobis below ahead of any staged columns: a reduction slot per
// wave and the sweep's flag, then one tile matrix per wave.
template <typename T>
__host__ __device__ constexpr int gram_jacobi_lds(int nwaves) {
    return 16 + nwaves * GJ_SC;
}

// Whole-workgroup Jacobi over `nw` waves, a wave per tile: J (rows x ncols, ld ldj) in LDS or global
// memory, V (vrows x ncols, ld ldv) rotated along when given.  `lds`: gram_jacobi_lds<T>(nw)
// elements.  Returns the sweeps used (max_sweeps when it did not converge).
template <typename T>
__device__ __forceinline__ int wg_gram_jacobi(T *J, int64_t ldj, int rows, int ncols, T *V, int64_t ldv, int vrows,
                                              T fro2, T stop, int max_sweeps, int nw, T *lds) {
    if (ncols <= 1) return 0;
    int &s_rot = *reinterpret_cast<int *>(lds + 8);
    T *sc = lds + 16 + wave_id() * GJ_SC;
    const GramTol<T> g(fro2, rows, stop);
    const int nblk = (ncols + GJ_B - 1) / GJ_B;
    const int nbp = nblk + (nblk & 1);
    int sweep = 0;
    for (; sweep < max_sweeps; ++sweep) {
        if (threadIdx.x == 0) s_rot = 0;
        __syncthreads();
        int any = 0;
        for (int step = 0; step < nbp - 1; ++step) {
            for (int bp = wave_id(); bp < nbp / 2; bp += nw) {
                int cI, cJ;
                if (!jacobi_pair_cols(bp, step, nbp, GJ_B, ncols, cI, cJ)) continue;
                if (step > 0 && cJ >= ncols) continue;
                any |= gram_tile<T, 1>(true, J, ldj, rows, ncols, cI, cJ, step == 0, g, sc, 0, V, ldv, vrows);
            }
            __syncthreads();
        }
        if ((any & JROT_LARGE) && lane_id() == 0) atomicOr(&s_rot, 1);
        __syncthreads();
        const int rot = s_rot;
        __syncthreads();
        if (!rot) break;
    }
    return sweep;
}

// Jacobi without V for a core too large for LDS, staged through it by super-blocks, by one workgroup
// of NWAVES waves, NS of them per tile.  The columns form super-blocks of W = GJ_B * NWAVES / NS
// columns and each sweep visits the super-block pairs (I, J > I) row by row: SI stays in local columns [0, W) of the
// LDS buffer Jl (ld rows | 1) while SJ after SJ passes through [W, 2 W), the next one on its way into
// registers as the waves rotate the block pairs of this one, round by round.  (One workgroup does them one
// after the other, so nothing asks for the disjoint pairs of a round-robin, which copied both super-blocks in and
// out per pair.  At 128 to 160 columns, two workgroups per CU: 647 us per sweep and 5.8 sweeps then, 617 and
// 5.1 now, since later pairs meet columns that earlier ones have turned; beyond, 1195 and 5.6, 1130 and 5.2.)
// The pairs (0, 1), (2, 3), ... run the round-robin over all their 2 W / GJ_B local blocks (in whose first round
// each block appears once, as a full tile: its internal column pairs), the others only the block pairs across SI and
// SJ, W / GJ_B rounds.  So every column pair is visited once per sweep, as in wg_gram_jacobi.  Columns past
// ncols are zero, so they never rotate.  A thread moves the same elements of a super-block wherever it goes,
// so the copies need no barrier among themselves.
// J: rows x ncols (ld rows), rows <= 64 RC; lds: gram_jacobi_lds<T>(NWAVES) elements of LDS, Jl: 2 W (rows | 1).
// Returns the sweeps used.
template <typename T, int NS, int RC>
__device__ __forceinline__ int wg_staged_jacobi(T *J, int rows, int ncols, T *Jl, T stop, int max_sweeps, T *lds) {
    constexpr int A = NWAVES / NS, W = GJ_B * A, LC = 2 * W, CW = W / NWAVES;
    T *s_red = lds;
    int &s_rot = *reinterpret_cast<int *>(lds + 8);
    T *sc = lds + 16 + wave_id() * GJ_SC;
    const int sub = wave_id() % NS, grp = wave_id() / NS;
    const int64_t ne = (int64_t) rows * ncols;
    T part = T(0);
    for (int64_t e = threadIdx.x; e < ne; e += NT) {
        const T a = J[e];
        part += a * a;
    }
    const GramTol<T> g(wg_sum(part, s_red), rows, stop);
    if (ncols <= 1) return 0;
    const int ld = rows | 1;
    const int ns = (ncols + W - 1) / W;
    // super-block S between memory (ld rows), registers and local columns [c0, c0 + W): a wave takes every
    // NWAVES-th column, a lane every 64th row
    T next[RC][CW];
    auto each = [&](int S, int c0, auto &&f) {
#pragma unroll
        for (int t = 0; t < RC; ++t)
#pragma unroll
            for (int u = 0; u < CW; ++u) {
                const int r = lane_id() + WAVE * t, c = wave_id() + u * NWAVES;
                f(t, u, J + r + (int64_t) (S * W + c) * rows, Jl + r + (c0 + c) * ld, r < rows, S * W + c < ncols);
            }
    };
    auto fetch = [&](int S) {
        each(S, 0, [&](int t, int u, const T *m, T *, bool row, bool col) { next[t][u] = row && col ? *m : T(0); });
    };
    auto put = [&](int c0) {
        each(0, c0, [&](int t, int u, T *, T *q, bool row, bool) {
            if (row) *q = next[t][u];
        });
    };
    auto save = [&](int S, int c0) {
        each(S, c0, [&](int, int, T *m, const T *q, bool row, bool col) {
            if (row && col) *m = *q;
        });
    };
    int sweep = 0;
    for (; sweep < max_sweeps; ++sweep) {
        if (threadIdx.x == 0) s_rot = 0;
        __syncthreads();
        int any = 0;
        for (int I = 0; I < ns; ++I) {
            // the last super-block has no partner: alone, only if no pair has visited its inside
            const bool solo = I == ns - 1;
            if (solo && (I & 1)) break;
            fetch(I);
            put(0);
            fetch(I + 1);  // zeros past the end
            const int nI = (ncols - I * W) < W ? (ncols - I * W) : W;
            for (int S = I + 1; S < ns || (solo && S == ns); ++S) {
                put(W);
                __syncthreads();
                if (S + 1 < ns) fetch(S + 1);
                const int left = ncols - S * W, nJ = left < 0 ? 0 : (left < W ? left : W);
                // a tile is skipped when no pair of it can rotate (a cross tile with an empty block, a
                // full tile with two)
                auto real = [&](int lc) { return lc < W ? lc < nI : lc - W < nJ; };
                int rot = 0;
                auto visit = [&](int lI, int lJ, bool full) {
                    const bool act = full ? (real(lI) || real(lJ)) : (real(lI) && real(lJ));
                    if (NS > 1 || act) rot |= gram_tile<T, NS>(act, Jl, ld, rows, LC, lI, lJ, full, g, sc, sub);
                };
                // the round-robin over the local blocks, all 2 A of them, or those across
                const bool inside = S == I + 1 && !(I & 1);
                const int rounds = inside ? 2 * A - 1 : A;
                for (int t = 0; t < rounds; ++t) {
                    int lI = grp * GJ_B, lJ = W + (grp + t < A ? grp + t : grp + t - A) * GJ_B;
                    if (inside) jacobi_pair_cols(grp, t, 2 * A, GJ_B, LC, lI, lJ);
                    visit(lI, lJ, inside && t == 0);
                    __syncthreads();
                }
                any |= rot;
                if (S < ns) save(S, W);
            }
            save(I, 0);
        }
        if ((any & JROT_LARGE) && lane_id() == 0) atomicOr(&s_rot, 1);
        __syncthreads();
        const int rot = s_rot;
        __syncthreads();
        if (!rot) break;
    }
    __syncthreads();
    return sweep;
}

// ---------------------------------------------------------------------------
// Multi-workgroup Jacobi (plain form, wide cores): one launch per round-robin step over the blocks.
// Workgroup (bp, 0) rotates block pair bp, its eight waves sharing the rows (each row is read once, kept
// in registers and written back), and records the tile's 16 x 16 V; workgroups (bp, 1 + k) of the next
// launch apply that record to rows [128 k, 128 k + 128) of V meanwhile, off the critical path.  One
// tile per workgroup and eight waves: a step is bound by the latency of its parts (launch, one pass over
// the tile from another XCD's writes, the 8 rounds) and by one CU's matrix cores, so wider super-blocks
// (32 columns per workgroup, half the steps) measured no faster per sweep.
// ---------------------------------------------------------------------------
constexpr int MW_WAVES = 8;
constexpr int MW_VROWS = 16 * MW_WAVES;     // rows of V per workgroup
constexpr int MW_REC = GJ_TW * GJ_TW;       // elements of one record
constexpr int MW_LDS = MW_WAVES * 2 * GJ_SC;

// The rotations of one tile (columns [cI, cI + 8) and [cJ, cJ + 8) of J, ld rows, rows <= 16 MW_WAVES
// GROUPS); `rec` receives V, `used` whether there is one; lds: MW_LDS elements.  `live` false: nothing
// is rotated (tested after the loads are under way).  Returns the JROT flags.
template <typename T, int GROUPS>
__device__ __forceinline__ int mw_rotate_tile(T *J, int rows, int ncols, int cI, int cJ, bool full, bool live,
                                              const GramTol<T> &g, T *rec, int32_t *used, T *lds) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4, w = wave_id();
    auto colp = [&](int k) -> T * {
        const int c = k < GJ_B ? cI + k : cJ + k - GJ_B;
        return c < ncols ? J + (int64_t) c * rows : nullptr;
    };
    // 16-row groups w, w + 8, ...: y[t][s] is row i16 of column 4 s + k4, the apply's operand
    T y[GROUPS][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const T *c = colp(4 * s + k4);
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) {
            const int r = 16 * (w + MW_WAVES * t) + i16;
            y[t][s] = (c && r < rows) ? c[r] : T(0);
        }
    }
    if (!live) return 0;
    // Gram matrix: a group's transpose goes through the wave's LDS, two groups at a time
    T *sc = lds + w * 2 * GJ_SC;
    typename MF::acc acc[2] = {MF::zero(), MF::zero()};
#pragma unroll
    for (int t0 = 0; t0 < GROUPS; t0 += 2) {
        wave_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (t0 + u < GROUPS)
#pragma unroll
                for (int s = 0; s < 4; ++s) sc[u * GJ_SC + (4 * s + k4) * GJ_LD + i16] = y[t0 + u][s];
        wave_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (t0 + u < GROUPS)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const T a = sc[u * GJ_SC + i16 * GJ_LD + 4 * k4 + s];
                    acc[u] = MF::mma(a, a, acc[u]);
                }
    }
    wave_fence();
    T gv[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        gv[v] = acc[0][v] + acc[1][v];
        sc[MF::row(v, k4) * GJ_LD + i16] = gv[v];
    }
    __syncthreads();
    int flags = 0;
    if (w == 0) {
#pragma unroll
        for (int ww = 1; ww < MW_WAVES; ++ww)
#pragma unroll
            for (int v = 0; v < 4; ++v) gv[v] += lds[ww * 2 * GJ_SC + MF::row(v, k4) * GJ_LD + i16];
        flags = gram_solve<T>(gv, lds, full, g);
        if (l == 0) {
            lds[GJ_TW] = T(flags);  // the padding element of row 0
            *used = flags & JROT_APPLIED;
        }
    }
    __syncthreads();
    flags = (int) lds[GJ_TW];
    if (!flags) return 0;
    T va[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) va[s] = lds[(4 * s + k4) * GJ_LD + i16];
    if (w == 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s) rec[(4 * s + k4) * GJ_TW + i16] = va[s];
    }
    T *dst[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) dst[v] = colp(MF::row(v, k4));
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        typename MF::acc a = MF::zero();
#pragma unroll
        for (int s = 0; s < 4; ++s) a = MF::mma(va[s], y[t][s], a);
        const int r = 16 * (w + MW_WAVES * t) + i16;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (dst[v] && r < rows) dst[v][r] = a[v];
    }
    return flags;
}

// Applies a tile's record to rows [r0, r0 + MW_VROWS) of V (nv x ncols, ld nv).
template <typename T>
__device__ __forceinline__ void mw_apply_v(T *V, int nv, int ncols, int cI, int cJ, const T *rec, int r0) {
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4;
    T va[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) va[s] = rec[(4 * s + k4) * GJ_TW + i16];
    const int nr = nv - r0 < MW_VROWS ? nv - r0 : MW_VROWS;
    gram_apply<T, MW_WAVES>(va, V + r0, nv, nr, ncols, cI, cJ, wave_id());
}

}  // namespace hcamd
