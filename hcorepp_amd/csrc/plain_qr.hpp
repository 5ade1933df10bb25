// Householder QR and Q application of the plain (one update at a time) form, where a single update has
// the GPU to itself: 16-column panels, one launch per panel and one per trailing update, and register
// blocks shared by 8 or 16 waves.
//
// Layout of a 16-column block in registers: rows are taken in groups of 16, group G by wave G % WAVES; lane
// (i16, k4) holds rows 16 G + 4 k4 .. + 3 of column i16.  That is both operands' layout for a product
// over the rows (P^T B) and, with the output rows of the second product permuted (prow), the layout B -= P W
// comes out in, so a block is read once and written once per use.
//
// The QR of Y (pivoted) moves no columns: piv[position] names the column of Y at each position, the
// selection permutes piv, reflectors stay in the column they were formed in, and R goes to the core
// J = P R_Y^T, whose row is the column's own number, as it is formed.  (Moving the chosen and the
// displaced columns took 6-13 us per panel, and building J from R another 50-590 us.)
#pragma once

#include "recompress.hpp"

namespace hcamd {

constexpr int PQ_NB = 16;                 // panel width
constexpr int PQ_MAX_COLS = JACOBI_ROWS_MAX;  // columns of a pivoted QR

// One QR of the plain form: A (m x ncols, ld m).  pivot: the QR of Y, with piv, the trailing columns'
// squared norms by position in cn, and the core J (ld ncols) that receives R^T.
template <typename T>
struct PlainQr {
    T *A, *tau, *tsave, *J, *cn;
    int32_t *piv;
    int64_t *hdr;
    int m, ncols, pivot;
};

// Within each row of 16 lanes: the first lane's value in all of them, and every lane's value one lane down
// (lane i takes lane i + 1's, the last the first's).
constexpr int DPP_ROW_BCAST0 = 0x150, DPP_ROW_DOWN1 = 0x12F;
template <int CTRL>
__device__ __forceinline__ double row_move(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float row_move(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Sum over the four lanes that hold a column (lane bits 4 and 5), in all of them.
template <typename T>
__device__ __forceinline__ T col_sum(T v) {
    T a = v, b = v;
    permlane_swap<32>(a, b);
    v = a + b;
    a = v;
    b = v;
    permlane_swap<16>(a, b);
    return a + b;
}

// Largest value of the wave, in every lane.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
    auto step = [&](unsigned o) { v = o > v ? o : v; };
    auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = r[0];
    step(r[1]);
    r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = r[0];
    step(r[1]);
    step(__builtin_amdgcn_mov_dpp((int) v, DPP_ROW_MIRROR, 0xF, 0xF, true));
    step(__builtin_amdgcn_mov_dpp((int) v, DPP_ROW_HALF_MIRROR, 0xF, 0xF, true));
    step(__builtin_amdgcn_mov_dpp((int) v, DPP_QUAD_XOR2, 0xF, 0xF, true));
    step(__builtin_amdgcn_mov_dpp((int) v, DPP_QUAD_XOR1, 0xF, 0xF, true));
    return v;
}

// Four consecutive elements at q: two or one wide accesses where `wide` says that q is aligned to 16 bytes.
__device__ __forceinline__ void load4(const double *q, bool wide, double (&v)[4]) {
    if (wide) {
        const double2 a = *reinterpret_cast<const double2 *>(q), b = *reinterpret_cast<const double2 *>(q + 2);
        v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y;
    } else {
        v[0] = q[0], v[1] = q[1], v[2] = q[2], v[3] = q[3];
    }
}
__device__ __forceinline__ void load4(const float *q, bool wide, float (&v)[4]) {
    if (wide) {
        const float4 a = *reinterpret_cast<const float4 *>(q);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    } else {
        v[0] = q[0], v[1] = q[1], v[2] = q[2], v[3] = q[3];
    }
}
__device__ __forceinline__ void store4(double *q, bool wide, const double (&v)[4]) {
    if (wide) {
        *reinterpret_cast<double2 *>(q) = double2{v[0], v[1]};
        *reinterpret_cast<double2 *>(q + 2) = double2{v[2], v[3]};
    } else {
        q[0] = v[0], q[1] = v[1], q[2] = v[2], q[3] = v[3];
    }
}
__device__ __forceinline__ void store4(float *q, bool wide, const float (&v)[4]) {
    if (wide) *reinterpret_cast<float4 *>(q) = float4{v[0], v[1], v[2], v[3]};
    else q[0] = v[0], q[1] = v[1], q[2] = v[2], q[3] = v[3];
}
// Rows r .. r + 3 of a column of `rows` rows, zero (not written) past its end.  Blocks of more than eight groups make every
// load, at the column's last row where its own is past the end (load_any), and clear what was not asked for afterwards: with
// branches around them the branches' state took the registers.  (The kernels of 1025 to 2048 rows had 310 to 750 bytes of scratch
// per lane; below about 270 each launch is 60 us shorter, an update of rank 1 in a 2048 x 2048 tile 260 -> 170 us, of rank 128
// 6.66 -> 3.28 ms.)
template <typename T>
__device__ __forceinline__ void load_any(const T *col, int r, int rows, T (&v)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = col[r + s < rows ? r + s : rows - 1];
}
template <typename T>
__device__ __forceinline__ void clear_rows(int r, int rows, bool ok, T (&v)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = (ok && r + s < rows) ? v[s] : T(0);
}
template <int GROUPS, typename T>
__device__ __forceinline__ void load_rows(const T *col, int r, int rows, bool ok, bool wide, T (&v)[4]) {
    if constexpr (GROUPS > 8) {
        load_any(col, r, rows, v);
        clear_rows(r, rows, ok, v);
    } else if (ok && r + 3 < rows) {
        load4(col + r, wide, v);
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) v[s] = (ok && r + s < rows) ? col[r + s] : T(0);
    }
}
template <int GROUPS, typename T>
__device__ __forceinline__ void store_rows(T *col, int r, int rows, bool ok, bool wide, const T (&v)[4]) {
    if (GROUPS <= 8 && ok && r + 3 < rows) {
        store4(col + r, wide, v);
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (ok && r + s < rows) col[r + s] = v[s];
    }
}
// Whether every column of a matrix of `ld` rows that starts on 16 bytes does too.
template <typename T>
__device__ __forceinline__ bool wide_columns(const T *A, int64_t ld) {
    return (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (ld * (int64_t) sizeof(T)) % 16 == 0;
}

// Blocks of more than eight groups leave no registers for the next groups' addresses and operands, nor for row numbers
// kept from the loads to the stores: group_end keeps a group's instructions together, own_rows gives row numbers that are
// computed anew.
template <int GROUPS>
__device__ __forceinline__ void group_end() {
    if constexpr (GROUPS > 8) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int GROUPS>
__device__ __forceinline__ int own_rows(int r) {
    if constexpr (GROUPS > 8) asm volatile("" : "+v"(r));
    return r;
}

// A wave's rows of a column (groups wave, wave + WAVES, ..).  Past eight groups all loads are made before the first value is
// looked at: cleared group by group, each group waited for its own (a panel of one column of 2048 rows 26.6 us, 22.0 now).
template <int WAVES, int GROUPS, typename T>
__device__ __forceinline__ void load_block(const T *col, int rows, bool ok, bool wide, T (&b)[GROUPS][4]) {
    const int r0 = 16 * wave_id() + 4 * (lane_id() >> 4);
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        const int r = own_rows<GROUPS>(r0 + 16 * WAVES * t);
        if constexpr (GROUPS > 8) load_any(col, r, rows, b[t]);
        else load_rows<GROUPS>(col, r, rows, ok, wide, b[t]);
        group_end<GROUPS>();
    }
    if constexpr (GROUPS > 8) {
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) {
            clear_rows(own_rows<GROUPS>(r0 + 16 * WAVES * t), rows, ok, b[t]);
            group_end<GROUPS>();
        }
    }
}

__device__ __forceinline__ double rcp_full(double d) {
    const double y = __builtin_amdgcn_rcp(d), e = fma(-d, y, 1.0);
    return fma(y * e, 1.0 + e, y);
}
__device__ __forceinline__ float rcp_full(float d) {
    const float y = __builtin_amdgcn_rcpf(d), e = fmaf(-d, y, 1.0f);
    return fmaf(y * e, 1.0f + e, y);
}

// The reflector of (alpha, x) with |x|^2 = xn2 (dlarfg): beta, tau and the factor `scal` of x.  The usual range
// takes one reciprocal square root and one reciprocal, each with its residual step; results that could
// leave the range of those take the square root and the divisions.
template <typename T>
__device__ __forceinline__ void householder(T alpha, T xn2, T &beta, T &tau, T &scal) {
    if (xn2 == T(0)) {
        beta = alpha;
        tau = scal = T(0);
        return;
    }
    constexpr T lo = sizeof(T) == 8 ? T(1e-280) : T(1e-30f), hi = sizeof(T) == 8 ? T(1e280) : T(1e30f);
    const T nn = alpha * alpha + xn2, a = fabs(alpha);
    if (nn > lo && nn < hi) {
        const T r = rsqrt_full(nn);
        T b = nn * r;
        b = fma(fma(-b, b, nn), T(0.5) * r, b);
        tau = fma(a, r, T(1));
        const T c = rcp_full(a + b);
        beta = alpha >= T(0) ? -b : b;
        scal = alpha >= T(0) ? c : -c;
    } else {
        beta = -dsign(sqrt(nn), alpha);
        tau = (beta - alpha) / beta;
        scal = T(1) / (alpha - beta);
    }
}

// LDS of the panel kernel.
template <typename T, int WAVES>
struct PanelLds {
    T red[2][WAVES][PQ_NB];       // partial products with the next column, per wave
    T xrow[2][PQ_NB];             // the next pivot row
    T t[PQ_NB][PQ_NB + 1];        // products of the reflectors, then the T factor
    T tau[PQ_NB];
    int piv[PQ_MAX_COLS];         // window pivoting: the trailing columns by position
    int vac[PQ_NB], disp[PQ_NB];  // chosen positions beyond the panel, and the panel's positions that were not chosen
    int inwin[PQ_NB];
    int stop;
};

// Householder factorisation of the panel p (rows x jb, jb <= 16; columns past jb and rows past the end
// zero).  One pass over the registers and one barrier per column: the pass of step j applies reflector j
// and accumulates, on the updated values, every column's product with column j + 1: summed, they give the
// next column's norm, the products of its (still unscaled) reflector with the later columns, and with the
// earlier reflectors, which T is built from.  The columns move one lane down per step, so that the current
// one is always in lane 0 of its row (a fixed broadcast in a short loop; a switch over 16 broadcasts
// measured the same).  On
// return lane (i16, k4) holds column (i16 + jb) % 16, its reflector still unscaled; the returned factor scales
// it.  tau receives jb values, l.t (upper triangle) the T factor.
//
// Bound by the chain of a column: two reductions' latency, a reciprocal square root and a reciprocal, one
// barrier: 0.7 us per column up to 512 rows.  Lanes along the columns need two exchanges per sum where a row
// per lane took six for 16 values.  A whole panel of the pivoted QR takes 20 us at 256 rows and 37 at 1024
// (50 and 47, for half as many columns, in LDS with a row per thread and four waves), its trailing update 7 and 18.
template <typename T, int WAVES, int GROUPS>
__device__ __forceinline__ T panel_factor(T (&p)[GROUPS][4], int jb, T *tau, PanelLds<T, WAVES> &l) {
    const int ln = lane_id(), i16 = ln & 15, k4 = ln >> 4, wv = wave_id();
    // the current column, rows below its pivot (0 elsewhere): kept from its products to the update after them where
    // the registers hold it beside p, broadcast twice in blocks of more than eight groups
    constexpr bool KEEP = GROUPS <= 8;
    T xs[KEEP ? GROUPS : 1][4];
    T myscal = T(0);
    int c = i16;      // this lane's column
    // column nj, which is in lane 0 of each row of lanes
    auto current = [&](int t, int s, int nj) {
        const T x = row_move<DPP_ROW_BCAST0>(p[t][s]);
        return (t == 0 && wv == 0 && 4 * k4 + s <= nj) ? T(0) : x;
    };
    // the products with it
    auto products = [&](int nj, int buf) {
        if constexpr (KEEP) {
#pragma unroll
            for (int t = 0; t < GROUPS; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) xs[t][s] = row_move<DPP_ROW_BCAST0>(p[t][s]);
        }
        if (wv == 0) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int r = 4 * k4 + s;
                if (r == nj) l.xrow[buf][c] = p[0][s];
                if (KEEP && r <= nj) xs[0][s] = T(0);
            }
        }
        T acc[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if constexpr (KEEP) acc[s] = fma(xs[t][s], p[t][s], acc[s]);
                else acc[s] = fma(current(t, s, nj), p[t][s], acc[s]);
            }
            group_end<GROUPS>();
        }
        const T sum = col_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
        if (k4 == 0) l.red[buf][wv][c] = sum;
    };
    products(0, 0);
    __syncthreads();
#pragma unroll 1
    for (int jj = 0; jj < jb; ++jj) {
        const int buf = jj & 1;
        T part[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) part[w] = l.red[buf][w][c];
#pragma unroll
        for (int h = WAVES / 2; h > 0; h >>= 1)
#pragma unroll
            for (int w = 0; w < h; ++w) part[w] += part[w + h];
        const T s = part[0], xk = l.xrow[buf][c];
        T beta, tj, scal;
        householder(read_lane(xk, 0), read_lane(s, 0), beta, tj, scal);
        // w_k = x_k[jj] + scal sum_{r > jj} x_jj[r] x_k[r]; x_k -= tau w_k v for the later columns
        const T wk = fma(scal, s, xk);
        const T gk = (c > jj && c < jb) ? tj * wk : T(0);
        const T gp = gk * scal;
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (KEEP) p[t][q] = fma(-gp, xs[t][q], p[t][q]);
                else p[t][q] = fma(-gp, current(t, q, jj), p[t][q]);
            }
            group_end<GROUPS>();
        }
        if (wv == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const T v = c == jj ? beta : p[0][q] - gk;
                p[0][q] = 4 * k4 + q == jj ? v : p[0][q];
            }
        }
        if (wv == WAVES - 1 && k4 == 0) {
            if (c < jj) l.t[c][jj] = myscal * wk;  // v_c . v_jj
            if (c == jj) l.tau[jj] = tj;
        }
        if (c == jj) myscal = scal;
#pragma unroll
        for (int t = 0; t < GROUPS; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) p[t][q] = row_move<DPP_ROW_DOWN1>(p[t][q]);
        myscal = row_move<DPP_ROW_DOWN1>(myscal);
        c = (c + 1) & 15;
        if (jj + 1 < jb) products(jj + 1, buf ^ 1);
        __syncthreads();
    }
    if (wv == WAVES - 1) {
        // T from the products G of the reflectors (dlarft): T[a][i] = -tau_i sum_{a <= b < i} T[a][b] G[b][i];
        // a lane per row a, which reads its own row only
        const int a = ln;
        if (a < PQ_NB) {
            T row[PQ_NB];
#pragma unroll
            for (int i = 0; i < PQ_NB; ++i) {
                T sum = T(0);
#pragma unroll
                for (int b = 0; b < i; ++b) sum = fma(b >= a ? row[b] : T(0), i < jb ? l.t[b][i] : T(0), sum);
                const T ti = i < jb ? l.tau[i] : T(0);
                row[i] = a < i ? -ti * sum : (a == i ? ti : T(0));
            }
            wave_fence();
#pragma unroll
            for (int i = 0; i < PQ_NB; ++i) l.t[a][i] = row[i];
            if (a < jb) tau[a] = l.tau[a];
        }
    }
    __syncthreads();
    return myscal;
}

// Sum of the squared norms cn[0..nt), by one wave.
template <typename T>
__device__ __forceinline__ T pivot_norm_sum(const T *cn, int nt) {
    T sum = T(0);
    for (int c = lane_id(); c < nt; c += WAVE) sum += cn[c];
    return wave_sum(sum);
}

// Ordering key of a squared norm: its bits, which order as the norms do, above 0 for "no column" and 1 for NaN, the lowest.
__device__ __forceinline__ unsigned long long norm_key(double v) {
    return v >= 0.0 ? (unsigned long long) __double_as_longlong(v) + 2u : 1u;
}
__device__ __forceinline__ unsigned norm_key(float v) { return v >= 0.f ? __float_as_uint(v) + 2u : 1u; }

// Largest key of the wave, in every lane.
__device__ __forceinline__ unsigned wave_max_key(unsigned k) { return wave_max_u32(k); }
__device__ __forceinline__ unsigned long long wave_max_key(unsigned long long k) {
    const unsigned hi = wave_max_u32((unsigned) (k >> 32));
    const unsigned lo = wave_max_u32((unsigned) (k >> 32) == hi ? (unsigned) k : 0u);
    return (unsigned long long) hi << 32 | lo;
}

// Window pivoting at a panel's start, by wave 0: the jb trailing columns of largest norm (cn[p], p in
// [0, nt), squared, by position) go to the panel, in decreasing norm, equal ones by position; the columns they displace
// take the positions they leave.  l.piv[0..nt) holds the columns by position and is permuted, and piv with it.
// A lane sorts its up to 12 columns once, and each round takes the largest head of the wave's lists.  (Rounds over
// the unsorted norms took 0.5 us each; a count of the larger norms per column, 768 x 768 reads of LDS, 10 us in all.)
template <typename T, int WAVES, int PER>
__device__ __forceinline__ void pivot_select(const T *cn, int nt, int jb, int32_t *piv, PanelLds<T, WAVES> &l) {
    using Key = decltype(norm_key(T(0)));
    const int ln = lane_id();
    Key key[PER];
    int col[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        col[t] = ln + WAVE * t;
        key[t] = col[t] < nt ? norm_key(cn[col[t]]) : Key(0);
    }
#pragma unroll
    for (int ph = 0; ph < PER; ++ph)
#pragma unroll
        for (int t = ph & 1; t + 1 < PER; t += 2) {
            const Key a = key[t], b = key[t + 1];
            const int ca = col[t], cb = col[t + 1];
            const bool keep = a >= b;  // equal ones stay in order
            key[t] = keep ? a : b;
            key[t + 1] = keep ? b : a;
            col[t] = keep ? ca : cb;
            col[t + 1] = keep ? cb : ca;
        }
    int mine = -1;  // lane r: the r-th choice
    for (int r = 0; r < jb; ++r) {
        const bool top = key[0] == wave_max_key(key[0]);
        unsigned long long tops = __ballot(top);
        if (tops & (tops - 1)) {
            const int first = PQ_MAX_COLS - (int) wave_max_u32(top ? (unsigned) (PQ_MAX_COLS - col[0]) : 0u);
            tops = __ballot(top && col[0] == first);
        }
        const int from = __ffsll(tops) - 1, c = __builtin_amdgcn_readlane(col[0], from);
        if (ln == r) mine = c;
        if (ln == from) {
#pragma unroll
            for (int t = 0; t + 1 < PER; ++t) {
                key[t] = key[t + 1];
                col[t] = col[t + 1];
            }
            key[PER - 1] = Key(0);
        }
    }
    if (ln < PQ_NB) l.inwin[ln] = 0;
    wave_fence();
    if (mine >= 0 && mine < jb) l.inwin[mine] = 1;
    wave_fence();
    const bool disp = ln < jb && l.inwin[ln] == 0, vac = mine >= jb;
    const unsigned long long md = __ballot(disp), mv = __ballot(vac), below = (1ull << ln) - 1ull;
    if (disp) l.disp[__popcll(md & below)] = ln;
    if (vac) l.vac[__popcll(mv & below)] = mine;
    const int nd = __popcll(md);
    wave_fence();
    const int to = ln < nd ? l.vac[ln] : 0;
    const int p0 = ln < jb ? l.piv[mine] : 0, p1 = ln < nd ? l.piv[l.disp[ln]] : 0;
    wave_fence();
    if (ln < jb) {
        l.piv[ln] = p0;
        piv[ln] = p0;
    }
    if (ln < nd) {
        l.piv[to] = p1;
        piv[to] = p1;
    }
    wave_fence();
}

// One panel of a QR at column j0 by one workgroup; for a pivoted one `stop(trail2)` may end the QR before the
// panel is formed.  Writes the reflectors (below the diagonal) and R to the panel's columns of A (R to J
// when pivoted), tau[j0..) and the T factor.
template <typename T, int WAVES, int GROUPS, typename STOP>
__device__ __forceinline__ void wg_panel(const PlainQr<T> &q, int j0, PanelLds<T, WAVES> &l, const STOP &stop) {
    const int ln = lane_id(), i16 = ln & 15, k4 = ln >> 4, wv = wave_id();
    const int nsteps = q.m < q.ncols ? q.m : q.ncols;
    const int jb = nsteps - j0 < PQ_NB ? nsteps - j0 : PQ_NB, rows = q.m - j0, nt = q.ncols - j0;
    if (q.pivot) {
        for (int c = threadIdx.x; c < nt; c += WAVES * WAVE) l.piv[c] = q.piv[j0 + c];
        __syncthreads();
        if (wv == 0) {
            const bool end = stop(pivot_norm_sum(q.cn + j0, nt));
            if (!end) {
                if (nt <= WAVE) pivot_select<T, WAVES, 1>(q.cn + j0, nt, jb, q.piv + j0, l);
                else if (nt <= 4 * WAVE) pivot_select<T, WAVES, 4>(q.cn + j0, nt, jb, q.piv + j0, l);
                else pivot_select<T, WAVES, PQ_MAX_COLS / WAVE>(q.cn + j0, nt, jb, q.piv + j0, l);
            }
            if (ln == 0) l.stop = end;
        }
        __syncthreads();
        if (l.stop) return;
    }
    const bool wide = wide_columns(q.A, q.m);
    auto column = [&](int c) { return q.A + (int64_t) (q.pivot ? l.piv[c] : j0 + c) * q.m + j0; };
    T p[GROUPS][4];
    load_block<WAVES>(column(i16 < jb ? i16 : 0), rows, i16 < jb, wide, p);
    const T scal = panel_factor<T, WAVES, GROUPS>(p, jb, q.tau + j0, l);
    const int c = (i16 + jb) & 15;
    T *dst = column(c < jb ? c : 0);
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        const int r = own_rows<GROUPS>(16 * (wv + WAVES * t) + 4 * k4);
        T v[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            v[s] = (t > 0 || r + s > c) ? scal * p[t][s] : p[t][s];
            // R[j0 + r, j0 + c] for the core
            if (t == 0 && q.pivot && c < jb && r + s <= c) q.J[l.piv[c] + (int64_t) (j0 + r + s) * q.ncols] = p[t][s];
        }
        store_rows<GROUPS>(dst, r, rows, c < jb, wide, v);
        group_end<GROUPS>();
    }
    T *ts = q.tsave + (int64_t) (j0 / PQ_NB) * PQ_NB * PQ_NB;
    for (int e = threadIdx.x; e < PQ_NB * PQ_NB; e += WAVES * WAVE) ts[e] = l.t[e % PQ_NB][e / PQ_NB];
}

// LDS of a block-reflector application.
template <typename T, int WAVES>
struct WyLds {
    T part[WAVES][PQ_NB * (PQ_NB + 1)];  // per wave: a group of P in turn, then the wave's share of P^T b
    T w[PQ_NB * (PQ_NB + 1)];
};

// Memory row, within a group, of output row i of the update's matrix-core product, chosen so that element
// v of lane (i16, k4) is row 4 k4 + v.
template <typename T>
__device__ __forceinline__ int pq_prow(int i) {
    return sizeof(T) == 8 ? 4 * (i & 3) + (i >> 2) : i;
}

// b <- (I - P op(T) P^T) b for a register block b, on the matrix cores; op(T) is T^T with `trans`.  pa(t, v) gives
// P, zero outside its rows: rows 16 G + 4 k4 .. + 3 of column i16, G = wave + WAVES t; groups below g0 are zero in P
// and skipped.  tm(i, j) gives T.  Two barriers; every wave of the workgroup calls it.  The second product takes P
// with its rows along the lanes, which each wave gets from its own LDS: reading both forms from memory, a CU moved P
// twice (update of 1024 rows 19.0 us, 17.9 now; reconstruction of 1024 rows and rank 341 435 us, 365 now).  Blocks of more
// than four groups turn a group as it is needed, blocks of more than eight read P again, for the registers.
template <typename T, int WAVES, int GROUPS, typename PA, typename TM>
__device__ __forceinline__ void wy_block(T (&b)[GROUPS][4], const PA &pa, const TM &tm, bool trans, int g0,
                                         WyLds<T, WAVES> &l) {
    using MF = Mfma16<T>;
    constexpr bool KEEP = GROUPS <= 8, EARLY = GROUPS <= 4;
    const int ln = lane_id(), i16 = ln & 15, k4 = ln >> 4, wv = wave_id();
    T a[KEEP ? GROUPS : 1][4], c[EARLY ? GROUPS : 1][4], top[4];
    if constexpr (KEEP) {
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) pa(t, a[t]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int k = MF::row(s, k4);
        top[s] = trans ? tm(k, i16) : tm(i16, k);
    }
    T *tile = l.part[wv];
    const int pr = pq_prow<T>(i16);
    auto turn = [&](const T (&x)[4], T (&y)[4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) tile[i16 * (PQ_NB + 1) + 4 * k4 + s] = x[s];
        wave_fence();
#pragma unroll
        for (int s = 0; s < 4; ++s) y[s] = tile[MF::row(s, k4) * (PQ_NB + 1) + pr];
        wave_fence();
    };
    if constexpr (EARLY) {
#pragma unroll
        for (int t = 0; t < GROUPS; ++t)
            if (wv + WAVES * t >= g0) turn(a[t], c[t]);
    }
    typename MF::acc acc = MF::zero();
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        if (wv + WAVES * t < g0) continue;
        if constexpr (!KEEP) pa(t, a[0]);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = MF::mma(a[KEEP ? t : 0][s], b[t][s], acc);
        group_end<GROUPS>();
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) l.part[wv][MF::row(v, k4) * PQ_NB + i16] = acc[v];
    __syncthreads();
    if (threadIdx.x < PQ_NB * PQ_NB) {
        T sum = T(0);
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += l.part[w][threadIdx.x];
        l.w[(threadIdx.x / PQ_NB) * (PQ_NB + 1) + threadIdx.x % PQ_NB] = sum;
    }
    __syncthreads();
    typename MF::acc wp = MF::zero();
#pragma unroll
    for (int s = 0; s < 4; ++s) wp = MF::mma(top[s], l.w[MF::row(s, k4) * (PQ_NB + 1) + i16], wp);
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        if (wv + WAVES * t < g0) continue;
        if constexpr (!KEEP) pa(t, a[0]);
        if constexpr (!EARLY) turn(a[KEEP ? t : 0], c[0]);
        typename MF::acc d = MF::zero();
#pragma unroll
        for (int s = 0; s < 4; ++s) d = MF::mma(c[EARLY ? t : 0][s], wp[s], d);
#pragma unroll
        for (int v = 0; v < 4; ++v) b[t][v] -= d[v];
        group_end<GROUPS>();
    }
}

}  // namespace hcamd
