// Triangular solve of up to 16 vectors by one workgroup, shared by the Cholesky tile solves
// (cholesky.hip) and the BLAS-style trsm (tileops.hip).
#pragma once

#include "device_common.hpp"

namespace hcamd {

constexpr int TS_NB = 32;    // rows per block step
constexpr int TS_NV = 16;    // vectors per workgroup
constexpr int TS_LDD = TS_NB + 1;
constexpr int TS_LDX = TS_NV + 1;
// LDS elements ahead of the vectors: the diagonal block and the waves' partial sums.
constexpr int TS_HEAD = TS_NB * TS_LDD + NWAVES * TS_NB * TS_LDX + TS_NB;
// Longest vectors that stay in LDS (two workgroups per CU).
template <typename T>
__host__ __device__ constexpr int ts_len_lds() {
    return (int) ((78 * 1024 / (int64_t) sizeof(T) - TS_HEAD) / TS_LDX);
}
template <typename T>
constexpr int64_t ts_lds_bytes(int len) {
    return (int64_t) sizeof(T) * (TS_HEAD + (len <= ts_len_lds<T>() ? (int64_t) len * TS_LDX : 0));
}

// b / d with r = 1 / d at hand: one residual step on b r, which the chain of a substitution waits for
// less than for a division; where that is not a number (infinities, r out of range) the division itself.
template <typename T>
__device__ __forceinline__ T divide(T b, T d, T r) {
    const T q = b * r;
    T x = fma(fma(-q, d, b), r, q);
    if (__any(!(x == x))) x = b / d;
    return x;
}

// x <- alpha M^{-1} x for vectors v in [0, nv), nv <= TS_NV, of `len` elements; element e of vector v is
// X[e es + v vs].  M(i, j) is A[i + j lda], or A[j + i lda] with `mt`; lower (forward substitution) or
// upper (backward); `unit`: the diagonal is not read.  lds: ts_lds_bytes<T>(len).
//
// Left-looking over blocks of 32 rows: the four waves share the product of the block's rows with the
// vectors' solved elements on the matrix cores (16 rows x 16 vectors x 4 per step), and one wave then
// solves the block, the vectors in its lanes and the rows in registers, 32 dependent steps of a
// broadcast, a division and eight updates.  The blocks are a serial chain (about 14 us each at 512 rows),
// so the work is split by vectors over the GPU, 16 per workgroup.  (One thread per vector, reading M
// from memory for every element, took 18 ms for 96 vectors of 512 elements; this takes 0.22 ms.)
template <typename T>
__device__ __forceinline__ void wg_trsm(T *X, int64_t es, int64_t vs, int nv, int len, const T *A, int64_t lda, bool mt,
                                        bool lower, bool unit, T alpha, T *lds) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4, w = wave_id();
    T *D = lds;                            // D[i * TS_LDD + j]: the diagonal block
    T *part = lds + TS_NB * TS_LDD;        // per wave: 32 rows x 16 vectors
    T *rd = part + NWAVES * TS_NB * TS_LDX;  // reciprocals of the diagonal
    T *xs = lds + TS_HEAD;                 // solved elements, in substitution order
    const bool in_lds = len <= ts_len_lds<T>();
    // index e of the substitution's order -> row of M
    auto row = [&](int e) { return lower ? e : len - 1 - e; };
    auto mat = [&](int e, int f) -> T {
        const int64_t i = row(e), j = row(f);
        return mt ? A[j + i * lda] : A[i + j * lda];
    };
    const int nblk = (len + TS_NB - 1) / TS_NB;
    for (int b = 0; b < nblk; ++b) {
        const int e0 = b * TS_NB, nb = len - e0 < TS_NB ? len - e0 : TS_NB;
        for (int q = threadIdx.x; q < TS_NB * TS_NB; q += NT) {
            const int i = mt ? q / TS_NB : q % TS_NB, j = mt ? q % TS_NB : q / TS_NB;
            const T m = (i < nb && j < nb && (j < i || (j == i && !unit))) ? mat(e0 + i, e0 + j) : T(i == j);
            D[i * TS_LDD + j] = m;
            if (i == j) rd[i] = T(1) / m;
        }
        // partial products over the solved elements, 32 at a time per wave
        typename MF::acc acc[2] = {MF::zero(), MF::zero()};
        for (int f0 = w * TS_NB; f0 < e0; f0 += NWAVES * TS_NB) {
            T a[2][8], x[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int f = f0 + 4 * s + k4;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int e = e0 + 16 * h + i16;
                    a[h][s] = e < len ? mat(e, f) : T(0);
                }
                x[s] = in_lds ? xs[f * TS_LDX + i16] : (i16 < nv ? X[(int64_t) row(f) * es + i16 * vs] : T(0));
            }
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int h = 0; h < 2; ++h) acc[h] = MF::mma(a[h][s], x[s], acc[h]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                part[(w * TS_NB + 16 * h + MF::row(v, k4)) * TS_LDX + i16] = acc[h][v];
        __syncthreads();
        if (w == 0) {
            T x[2][4];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * h + MF::row(v, k4);
                    T sum = T(0);
#pragma unroll
                    for (int ww = 0; ww < NWAVES; ++ww) sum += part[(ww * TS_NB + i) * TS_LDX + i16];
                    const T rhs = (i < nb && i16 < nv) ? alpha * X[(int64_t) row(e0 + i) * es + i16 * vs] : T(0);
                    x[h][v] = rhs - sum;
                }
#pragma unroll
            for (int i = 0; i < TS_NB; ++i) {
                // row i sits in register (oh, ov) of the lanes with k4 = ok
                const int oh = i / 16, ov = sizeof(T) == 8 ? (i % 16) / 4 : i % 4, ok = sizeof(T) == 8 ? i % 4 : (i % 16) / 4;
                T xi = x[oh][ov];
                if (!unit) xi = divide(xi, D[i * (TS_LDD + 1)], rd[i]);
                xi = lane_fetch(xi, 16 * ok + i16);
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int j = 16 * h + MF::row(v, k4);
                        if (16 * h + 15 < i) continue;
                        const T upd = x[h][v] - D[j * TS_LDD + i] * xi;
                        x[h][v] = j > i ? upd : (j == i ? xi : x[h][v]);
                    }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * h + MF::row(v, k4);
                    if (i < nb) {
                        if (in_lds) xs[(e0 + i) * TS_LDX + i16] = x[h][v];
                        if (i16 < nv) X[(int64_t) row(e0 + i) * es + i16 * vs] = x[h][v];
                    }
                }
        }
        __syncthreads();
    }
}

// The same for one vector of `len` elements by one thread.
template <typename T>
__device__ __forceinline__ void thread_trsm(T *x, int64_t es, int len, const T *A, int64_t lda, bool mt, bool lower,
                                            bool unit, T alpha) {
    auto row = [&](int e) { return lower ? e : len - 1 - e; };
    auto M = [&](int i, int j) { return mt ? A[j + i * lda] : A[i + j * lda]; };
    for (int e = 0; e < len; ++e) {
        const int i = row(e);
        T s = alpha * x[i * es];
        for (int f = 0; f < e; ++f) s -= M(i, row(f)) * x[row(f) * es];
        x[i * es] = unit ? s : s / M(i, i);
    }
}
// Whether `count` vectors of `len` elements are solved so, a thread each: where the vectors are very short, or short and so
// many that the 1280 workgroups that fit the GPU at once take several rounds of 16 (us, 16 per workgroup / a thread each: 4
// elements 47 / 43 at any count, 16 elements 60 / 60 at 16384 vectors, 80 / 61 at 32768, 207 / 69 at 131072; 32 elements 91 /
// 126 at 32768, 137 / 126 at 65536, 238 / 135 at 131072).  Up to 32 elements both have the same error; beyond, a thread's
// long sums have the larger one.
__host__ __device__ inline bool trsm_by_thread(int64_t len, int64_t count) {
    return len <= 8 || (len <= 32 && count >= 2048 * len);
}

// Rows of X (rows x n, column k at X + k ldx) <- X L^{-T} for lower-triangular L (n x n, ld ldl) by one workgroup, up to NT rows
// at a time: a thread owns a row, the columns go 16 at a time, with L staged through LDS in 16 x 16 pieces.  lds:
// RT_LDS elements.  Every thread of the workgroup must call it.
constexpr int RT_NB = 16;
constexpr int RT_LDS = RT_NB * (RT_NB + 1);
template <typename T>
__device__ __forceinline__ void wg_rows_trsm(T *X, int rows, int n, int64_t ldx, const T *L, int64_t ldl, T *lds) {
    const int tid = (int) threadIdx.x;
    for (int r0 = 0; r0 < rows; r0 += NT) {
        const int a = r0 + tid;
        const bool act = a < rows, wave = r0 + __builtin_amdgcn_readfirstlane(tid) < rows;  // this thread, this wave has rows
        T *x = X + (act ? a : 0);
        for (int j0 = 0; j0 < n; j0 += RT_NB) {
            const int jb = (n - j0) < RT_NB ? (n - j0) : RT_NB;
            T acc[RT_NB];
#pragma unroll
            for (int c = 0; c < RT_NB; ++c) acc[c] = (act && c < jb) ? x[(int64_t) (j0 + c) * ldx] : T(0);
            for (int k0 = 0; k0 <= j0; k0 += RT_NB) {
                // piece (j0, k0) of L; the last one is the diagonal block, 1 past its end
                __syncthreads();
                {
                    const int c = tid % RT_NB, k = tid / RT_NB;
                    lds[c * (RT_NB + 1) + k] = (c < jb && (k0 < j0 || k <= c)) ? L[(j0 + c) + (int64_t) (k0 + k) * ldl] : T(c == k);
                }
                __syncthreads();
                if (k0 < j0 && wave) {
                    T v[RT_NB];
#pragma unroll
                    for (int k = 0; k < RT_NB; ++k) v[k] = act ? x[(int64_t) (k0 + k) * ldx] : T(0);
#pragma unroll
                    for (int c = 0; c < RT_NB; ++c) {
                        T p = T(0);
#pragma unroll
                        for (int k = 0; k < RT_NB; ++k) p = fma(v[k], lds[c * (RT_NB + 1) + k], p);
                        acc[c] -= p;
                    }
                }
            }
            if (wave) {
#pragma unroll
                for (int c = 0; c < RT_NB; ++c) {
#pragma unroll
                    for (int k = 0; k < c; ++k) acc[c] = fma(-acc[k], lds[c * (RT_NB + 1) + k], acc[c]);
                    acc[c] /= lds[c * (RT_NB + 1) + c];
                    if (act && c < jb) x[(int64_t) (j0 + c) * ldx] = acc[c];
                }
            }
        }
    }
}
static_assert(RT_NB * RT_NB == NT, "a thread per element of a piece of L");

}  // namespace hcamd
