// Workgroup-level tiled GEMM for the factor products and dense tile updates
// (HCoreKernels::Gemm call sites: reference src/api/HCore.cpp:176-264 via
// src/operators/concrete/Dense.cpp:46-108).  One workgroup computes one
// 64x64 tile of C = alpha*op(A)*op(B) + beta*C with a K chunk (32 deep in FP64, 16 in FP32)
// staged in LDS; FP64 on the matrix cores, FP32 with a 4x4 register block per thread.
#pragma once

#include "device_common.hpp"

namespace hcamd {

constexpr int GT_M = 64, GT_N = 64, GT_K = 16;
// K chunk of the FP64 (matrix-core) form: 32 deep, so that each thread has 16 loads in flight
// per chunk and a tile takes half as many memory round trips (the FP32 form and the mixed split
// keep 16: the split's exactness bound counts 16-deep sums).
constexpr int GT_KD = 32;
constexpr int GT_LDS_ELEMS = GT_KD * (GT_M + 1) + GT_KD * (GT_N + 1);
template <typename T>
__host__ __device__ constexpr int gemm_kc() {
    return sizeof(T) == 8 ? GT_KD : GT_K;
}

// The K loop (chunks of gemm_kc<T>() = KC) is software-pipelined: the next chunk's elements are
// loaded into registers (KC / 4 of A and of B per thread) right after the current chunk is in LDS, so their memory latency
// overlaps the chunk's arithmetic.  `fa(i, k)` and `fb(k, j)` return op(A)[i, k] and op(B)[k, j]
// (zero outside the operands); A's chunk is read row-fastest when `a_rows_fast`, B's K-fastest
// unless `b_cols_fast`, so that consecutive threads read consecutive addresses.  `epi(i, j, v)`
// receives each element of the tile inside M x N.
// FP64 runs on the matrix cores (v_mfma_f64_16x16x4f64): wave w computes the 32 x 32 quarter at
// rows 32 (w / 2), columns 32 (w % 2) of the tile as 2 x 2 blocks of 16 x 16; per 4-deep K step
// a lane reads two values of A and two of B from LDS for four MFMAs (the VALU form, a 4 x 4
// block per thread, reads eight for sixteen FMAs).  MFMA lane layout: A[i][k] in lane i + 16 k,
// B[k][j] in lane j + 16 k, D[4 v + l / 16][l % 16] in element v of lane l.
// Only K chunks overlapping [k_lo, k_hi) are visited (operands known to vanish outside, as for
// triangular factors); k_lo is rounded down to a chunk boundary.
template <typename T, typename FA, typename FB, typename EPI>
__device__ __forceinline__ void wg_gemm_tile_core(int M, int N, int Kd, const FA &fa, const FB &fb, bool a_rows_fast,
                                                  bool b_cols_fast, const EPI &epi, int ti, int tj, T *lds,
                                                  int k_lo = 0, int k_hi = -1) {
    constexpr int KC = gemm_kc<T>();
    k_lo = (k_lo / KC) * KC;
    if (k_hi < 0 || k_hi > Kd) k_hi = Kd;
    T *As = lds;                    // [KC][GT_M + 1]  As[k][i]
    T *Bs = lds + KC * (GT_M + 1);  // [KC][GT_N + 1]  Bs[k][j]
    const int i0 = ti * GT_M, j0 = tj * GT_N;
    constexpr int PER = GT_M * KC / NT;  // elements of each operand chunk per thread
    static_assert(GT_M * KC == GT_N * KC && PER * NT == GT_M * KC, "tile shape");
    auto a_pos = [&](int e, int &i, int &k) {
        if (a_rows_fast) {
            i = e % GT_M;
            k = e / GT_M;
        } else {
            k = e % KC;
            i = e / KC;
        }
    };
    auto b_pos = [&](int e, int &j, int &k) {
        if (b_cols_fast) {
            j = e % GT_N;
            k = e / GT_N;
        } else {
            k = e % KC;
            j = e / KC;
        }
    };
    T ra[PER], rb[PER];
    auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = threadIdx.x + q * NT;
            int i, j, k, k2;
            a_pos(e, i, k);
            b_pos(e, j, k2);
            const int gi = i0 + i, gk = k0 + k, gj = j0 + j, gk2 = k0 + k2;
            ra[q] = (gi < M && gk < Kd) ? fa(gi, gk) : T(0);
            rb[q] = (gj < N && gk2 < Kd) ? fb(gk2, gj) : T(0);
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = threadIdx.x + q * NT;
            int i, j, k, k2;
            a_pos(e, i, k);
            b_pos(e, j, k2);
            As[k * (GT_M + 1) + i] = ra[q];
            Bs[k2 * (GT_N + 1) + j] = rb[q];
        }
    };
    if constexpr (sizeof(T) == 8) {
        const int l = lane_id(), i16 = l & 15, k4 = l >> 4, w = wave_id();
        const int qi = 32 * (w >> 1), qj = 32 * (w & 1);
        hcamd_doublex4 acc[2][2];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = hcamd_doublex4{0.0, 0.0, 0.0, 0.0};
        if (k_lo < k_hi) load(k_lo);
        for (int k0 = k_lo; k0 < k_hi; k0 += KC) {
            stage();
            __syncthreads();
            if (k0 + KC < k_hi) load(k0 + KC);
#pragma unroll
            for (int s = 0; s < KC / 4; ++s) {
                const int kr = 4 * s + k4;
                double av[2], bv[2];
#pragma unroll
                for (int bi = 0; bi < 2; ++bi) av[bi] = As[kr * (GT_M + 1) + qi + 16 * bi + i16];
#pragma unroll
                for (int bj = 0; bj < 2; ++bj) bv[bj] = Bs[kr * (GT_N + 1) + qj + 16 * bj + i16];
#pragma unroll
                for (int bi = 0; bi < 2; ++bi)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
                        acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[bi], bv[bj], acc[bi][bj], 0, 0, 0);
            }
            __syncthreads();
        }
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int gi = i0 + qi + 16 * bi + 4 * v + k4, gj = j0 + qj + 16 * bj + i16;
                    if (gi < M && gj < N) epi(gi, gj, acc[bi][bj][v]);
                }
    } else {
        const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
        T acc[4][4];
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[p][q] = T(0);
        if (k_lo < k_hi) load(k_lo);
        for (int k0 = k_lo; k0 < k_hi; k0 += KC) {
            stage();
            __syncthreads();
            if (k0 + KC < k_hi) load(k0 + KC);
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                T av[4], bv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    av[q] = As[k * (GT_M + 1) + ty + 16 * q];
                    bv[q] = Bs[k * (GT_N + 1) + tx + 16 * q];
                }
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[p][q] += av[p] * bv[q];
            }
            __syncthreads();
        }
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gi = i0 + ty + 16 * p, gj = j0 + tx + 16 * q;
                if (gi < M && gj < N) epi(gi, gj, acc[p][q]);
            }
    }
}

template <typename T>
__device__ void wg_gemm_tile(int M, int N, int Kd, T alpha, const T *A, int64_t lda, bool ta, const T *B,
                             int64_t ldb, bool tb, T beta, T *C, int64_t ldc, int ti, int tj, T *lds) {
    auto fa = [=](int i, int k) -> T { return ta ? A[k + (int64_t) i * lda] : A[i + (int64_t) k * lda]; };
    auto fb = [=](int k, int j) -> T { return tb ? B[j + (int64_t) k * ldb] : B[k + (int64_t) j * ldb]; };
    auto epi = [=](int gi, int gj, T v) {
        T *c = C + gi + (int64_t) gj * ldc;
        *c = (beta == T(0)) ? alpha * v : alpha * v + beta * *c;
    };
    wg_gemm_tile_core<T>(M, N, Kd, fa, fb, !ta, tb, epi, ti, tj, lds);
}

// One 64 x 64 tile of C (M x N, ld ldc) = sum_k fa(i, k) fb(k, j) for operands given as element
// functions (each returns zero outside its structure: triangles, gathered rows); K chunks are
// staged in LDS as in wg_gemm_tile.  A's chunk is read row-fastest, B's K-fastest.
template <typename T, typename FA, typename FB>
__device__ void wg_gemm_tile_fn(int M, int N, int Kd, const FA &fa, const FB &fb, T *C, int64_t ldc, int ti, int tj,
                                T *lds, int k_lo = 0, int k_hi = -1) {
    auto epi = [=](int gi, int gj, T v) { C[gi + (int64_t) gj * ldc] = v; };
    wg_gemm_tile_core<T>(M, N, Kd, fa, fb, true, false, epi, ti, tj, lds, k_lo, k_hi);
}

// Whole-matrix GEMM by one workgroup (loops over all 64x64 tiles).
template <typename T>
__device__ void wg_gemm(int M, int N, int Kd, T alpha, const T *A, int64_t lda, bool ta, const T *B, int64_t ldb,
                        bool tb, T beta, T *C, int64_t ldc, T *lds) {
    const int tm = (M + GT_M - 1) / GT_M, tn = (N + GT_N - 1) / GT_N;
    for (int t = 0; t < tm * tn; ++t) {
        wg_gemm_tile<T>(M, N, Kd, alpha, A, lda, ta, B, ldb, tb, beta, C, ldc, t % tm, t / tm, lds);
    }
}

// ---------------------------------------------------------------------------
// Products too small to fill the GPU with 64 x 64 tiles: one workgroup of 8 waves per 32 x 32 tile, the
// waves splitting K (16 at a time) and each holding the whole tile as 2 x 2 matrix-core blocks.  The operands
// go from memory to registers in the matrix cores' layout, four 16-deep chunks in flight per wave, without
// LDS or barriers until the waves' sums are added up at the end, so a K of 512 is one memory round trip.
// (The 64 x 64 form walks K in 16 staged chunks in one workgroup, 38 us for a 64 x 72 product of K = 512; the
// three products of C += (U V)(U V) with a dense 512 x 512 C took 62 us, 27 here.)  fa(i, k), fb(k, j) and
// epi(i, j, v) as in wg_gemm_tile_core; k_lo: the operands vanish before it.
// ---------------------------------------------------------------------------
constexpr int GS_T = 32, GS_WAVES = 8, GS_CH = 4;
constexpr int GS_LDS_ELEMS = GS_WAVES * 16 * (GS_T + 1);
template <typename T, typename FA, typename FB, typename EPI>
__device__ __forceinline__ void wg_gemm_small(int M, int N, int Kd, const FA &fa, const FB &fb, const EPI &epi, int ti,
                                              int tj, T *lds, int k_lo = 0) {
    using MF = Mfma16<T>;
    const int l = lane_id(), i16 = l & 15, k4 = l >> 4, w = wave_id();
    const int i0 = ti * GS_T, j0 = tj * GS_T;
    typename MF::acc acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = MF::zero();
    k_lo &= ~15;
    for (int k0 = k_lo + 16 * w; k0 < Kd; k0 += 16 * GS_WAVES * GS_CH) {
        T a[GS_CH][2][4], b[GS_CH][2][4];
#pragma unroll
        for (int c = 0; c < GS_CH; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // a chunk's 16 terms may be summed in any order: lane k4 takes k0 + 4 k4 .. + 3
                    const int k = k0 + 16 * GS_WAVES * c + 4 * k4 + s, i = i0 + 16 * h + i16, j = j0 + 16 * h + i16;
                    a[c][h][s] = (k < Kd && i < M) ? fa(i, k) : T(0);
                    b[c][h][s] = (k < Kd && j < N) ? fb(k, j) : T(0);
                }
#pragma unroll
        for (int c = 0; c < GS_CH; ++c) {
            if (k0 + 16 * GS_WAVES * c >= Kd) break;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int q = 0; q < 2; ++q) acc[p][q] = MF::mma(a[c][p][s], b[c][q][s], acc[p][q]);
        }
    }
    // the waves' sums, 16 rows of the tile at a time
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        if (p) __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) lds[(w * 16 + MF::row(v, k4)) * (GS_T + 1) + 16 * q + i16] = acc[p][q][v];
        __syncthreads();
        const int i = threadIdx.x % 16, j = threadIdx.x / 16;  // 512 threads: one element each
        T sum = T(0);
#pragma unroll
        for (int ww = 0; ww < GS_WAVES; ++ww) sum += lds[(ww * 16 + i) * (GS_T + 1) + j];
        const int gi = i0 + 16 * p + i, gj = j0 + j;
        if (gi < M && gj < N) epi(gi, gj, sum);
    }
}

// Whether a product takes that form.  Its 32 x 32 tiles run in rounds of 256, one per CU, and its time grows with them; the
// 64 x 64 form's does not while there is a tile per CU at most (225 of them: 18 us at K = 128, 74 at 960).  Times by rounds,
// 64 x 64 form / this one:
//   one      1.2-3.7 for every K and transpose;
//   two      1.14-2.0 from K = 48 on, 0.95-0.99 up to 32;
//   three    0.91 at K = 128, 0.97 at 512 and 1.1 at 8192; B transposed alone, both operands' lanes along memory, 0.91 at
//            64, 1.01 at 128, 1.35 from 512 on; A transposed alone 0.7;
//   four     0.56-0.84; B transposed alone 0.84 at 128, 1.07 from 512 on.
// FP32, whose 64 x 64 form has no matrix cores: 1.1-7 for all of them.
template <typename T>
__host__ __device__ inline bool gemm_is_small(int64_t M, int64_t N, int64_t K, bool ta, bool tb) {
    if (((M + GT_M - 1) / GT_M) * ((N + GT_N - 1) / GT_N) >= 256) return false;
    const int64_t rounds = (((M + GS_T - 1) / GS_T) * ((N + GS_T - 1) / GS_T) + 255) / 256;
    if (sizeof(T) == 4 || rounds <= 1) return true;
    if (rounds == 2) return K > 32;
    if (!ta && tb) return K >= (rounds == 3 ? 128 : 512);
    return rounds == 3 && K >= 8192 && ta == tb;
}

// ---------------------------------------------------------------------------
// Mixed-precision tile GEMM: C = op(A) op(B) (alpha = 1, beta = 0) for FP64 operands with the
// products formed on the FP16 matrix cores (v_mfma_f32_16x16x16_f16) with FP32 accumulation, made
// exact by an error-free split of the operands (the Ozaki scheme).  Each row i of op(A) is scaled
// by a power of two 2^ea_i above its largest magnitude and cut into MS_SLICES slices: integers
// x_s of at most MS_BITS bits with op(A)[i, k] = 2^ea_i sum_s x_s 2^(-MS_BITS (s+1)) + (a rest
// below 2^(ea_i - MS_BITS MS_SLICES - 1)); each column of op(B) likewise.  FP16 holds every such integer
// exactly (|x_0| <= 2^10, the later ones 2^9).  The products of the pairs (s, t) and (t, s) are summed in FP32 over one
// 16-deep K chunk, at most 16 * 2 * 2^10 * 2^9 = 2^24 and so exact in whatever order the matrix core sums, and each of
// the six sums with s + t < MS_SLICES is added to the FP64 result with its power-of-two weight.  (One sum for all pairs of
// a weight passes 2^24 where there are three or four of them, and lost units of 2^-40.)  The error is the dropped
// slices: about 2^-40 of 2^(ea_i + eb_j) per term (FP64 rounding for the rest), against 2^-24 for plain FP32
// operands.
// A 64 x 64 output tile per workgroup: wave w computes the 32 x 32 quarter at rows 32 (w / 2),
// columns 32 (w % 2) as 2 x 2 blocks of 16 x 16.  Every thread splits eight consecutive K of one row of op(A) and
// of one column of op(B) per stage of two chunks, loaded a stage ahead, and stores each slice's fours as 8-byte words,
// the words a lane of the matrix cores takes: A[i][4 g .. 4 g + 3] from lane i + 16 g, B likewise,
// D[4 (l / 16) + v][l % 16] in element v of lane l.
// (The slices as FP32 on v_mfma_f32_16x16x4f32, 40 of those and ten sums per chunk and block where there are ten
// and six now: the two products of an update of 512 rows and ranks near 190 took 3.6 ms in one workgroup, 1.0 now,
// with the same errors; four sums, one per weight, 0.8, but not exact.)
// ---------------------------------------------------------------------------
constexpr int MS_BITS = 10, MS_SLICES = 4;
constexpr int MS_KC = 2 * GT_K;                  // K staged at a time: two chunks per round trip and barrier pair
constexpr int MS_KT = MS_KC / 4;                 // of which a thread splits these for one row and one column
constexpr int MS_LD = MS_KC + 4;                 // halves per row of a slice: 8-byte words, banks spread
constexpr int MS_SLICE = GT_M * MS_LD;           // halves per slice of either operand
constexpr int GTM_LDS_FLOATS = MS_SLICES * MS_SLICE + GT_M + GT_N;
static_assert(GT_M == GT_N && GT_K == 16 && GT_M * 4 == NT, "a thread per row and four K");
static_assert(4 + 1 + MS_BITS + (MS_BITS - 1) <= 24, "two slice pairs over a 16-deep chunk must be exact in FP32");

typedef _Float16 hcamd_halfx4 __attribute__((ext_vector_type(4)));

// Exponent e with |v| < 2^e for the largest magnitude v of a row or column (0 for a zero one).
__device__ __forceinline__ int ms_exponent(double vmax) {
    return vmax > 0.0 ? ilogb(vmax) + 1 : 0;
}

// Slices of MS_KT values in [-1, 1] (divided by their row's or column's power-of-two scale), each slice's
// stored at dst + s MS_SLICE.
__device__ __forceinline__ void ms_split(const double (&v)[MS_KT], int e, _Float16 *dst) {
#pragma unroll
    for (int k0 = 0; k0 < MS_KT; k0 += 4) {
        float x[MS_SLICES][4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            double r = ldexp(v[k0 + k], MS_BITS - e);
#pragma unroll
            for (int s = 0; s < MS_SLICES; ++s) {
                const double q = rint(r);
                x[s][k] = (float) q;
                r = (r - q) * double(1 << MS_BITS);
            }
        }
#pragma unroll
        for (int s = 0; s < MS_SLICES; ++s) {
            // packed conversions (exact here); a cast of a rounded double to _Float16 becomes a software conversion
            const auto lo = __builtin_amdgcn_cvt_pkrtz(x[s][0], x[s][1]), hi = __builtin_amdgcn_cvt_pkrtz(x[s][2], x[s][3]);
            uint2 u;
            __builtin_memcpy(&u.x, &lo, 4);
            __builtin_memcpy(&u.y, &hi, 4);
            *reinterpret_cast<uint2 *>(dst + s * MS_SLICE + k0) = u;
        }
    }
}

__device__ inline void wg_gemm_tile_mixed(int M, int N, int Kd, const double *A, int64_t lda, bool ta,
                                          const double *B, int64_t ldb, bool tb, double *C, int64_t ldc, int ti,
                                          int tj, float *lds) {
    _Float16 *As = reinterpret_cast<_Float16 *>(lds);  // [slice][i][k]
    _Float16 *Bs = As + MS_SLICES * MS_SLICE;          // [slice][j][k]
    int *ea = reinterpret_cast<int *>(Bs + MS_SLICES * MS_SLICE);  // row exponents of op(A)
    int *eb = ea + GT_M;                                           // column exponents of op(B)
    const int l = lane_id(), w = wave_id(), t = (int) threadIdx.x;
    const int wr = 32 * (w / 2), wc = 32 * (w % 2), i16 = l & 15, g = l >> 4;
    // this thread's row of op(A) and column of op(B), and its K of every stage: along the memory order
    const int ai = ta ? t / 4 : t % GT_M, ak = MS_KT * (ta ? t % 4 : t / GT_M);
    const int bj = tb ? t % GT_N : t / 4, bk = MS_KT * (tb ? t / GT_N : t % 4);
    const int gi = ti * GT_M + ai, gj = tj * GT_N + bj;
    const double *pa = A + (gi < M ? (ta ? gi * lda : gi) : 0), *pb = B + (gj < N ? (tb ? gj : gj * ldb) : 0);
    const int64_t sa = ta ? 1 : lda, sb = tb ? ldb : 1;
    auto load_one = [&](const double *p, int64_t st, int left, double (&x)[MS_KT]) {
        if (left >= MS_KT) {
#pragma unroll
            for (int s = 0; s < MS_KT; ++s) x[s] = p[s * st];
        } else {
#pragma unroll
            for (int s = 0; s < MS_KT; ++s) x[s] = s < left ? p[s * st] : 0.0;
        }
    };
    auto load = [&](int k0, double (&a)[MS_KT], double (&b)[MS_KT]) {
        load_one(pa + (k0 + ak) * sa, sa, gi < M ? Kd - k0 - ak : 0, a);
        load_one(pb + (k0 + bk) * sb, sb, gj < N ? Kd - k0 - bk : 0, b);
    };
    // power-of-two scales: every thread's share of its row and column, then the four shares' largest
    {
        double amax = 0.0, bmax = 0.0;
#pragma unroll 2
        for (int k0 = 0; k0 < Kd; k0 += MS_KC) {
            double a[MS_KT], b[MS_KT];
            load(k0, a, b);
#pragma unroll
            for (int s = 0; s < MS_KT; ++s) {
                amax = fmax(amax, fabs(a[s]));
                bmax = fmax(bmax, fabs(b[s]));
            }
        }
        double *red = reinterpret_cast<double *>(lds);
        red[ai + GT_M * (ak / MS_KT)] = amax;
        red[NT + bj + GT_N * (bk / MS_KT)] = bmax;
        __syncthreads();
        if (t < GT_M + GT_N) {
            const double *r = red + (t < GT_M ? t : NT + t - GT_M);
            ea[t] = ms_exponent(fmax(fmax(r[0], r[GT_M]), fmax(r[2 * GT_M], r[3 * GT_M])));
        }
        __syncthreads();
    }
    const int ae = ea[ai], be = eb[bj];
    double acc[2][2][4];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[p][q][v] = 0.0;
    double na[MS_KT], nb[MS_KT];
    load(0, na, nb);
    for (int k0 = 0; k0 < Kd; k0 += MS_KC) {
        ms_split(na, ae, As + ai * MS_LD + ak);
        ms_split(nb, be, Bs + bj * MS_LD + bk);
        __syncthreads();
        if (k0 + MS_KC < Kd) load(k0 + MS_KC, na, nb);
#pragma unroll
        for (int c = 0; c < MS_KC; c += GT_K) {
            if (k0 + c >= Kd) break;
            hcamd_halfx4 a[2][MS_SLICES], b[2][MS_SLICES];
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int s = 0; s < MS_SLICES; ++s) {
                    const int o = s * MS_SLICE + (16 * p + i16) * MS_LD + c + 4 * g;
                    __builtin_memcpy(&a[p][s], __builtin_assume_aligned(As + wr * MS_LD + o, 8), 8);
                    __builtin_memcpy(&b[p][s], __builtin_assume_aligned(Bs + wc * MS_LD + o, 8), 8);
                }
#pragma unroll
            for (int d = 0; d < MS_SLICES; ++d) {
                const double wgt = 1.0 / double(int64_t(1) << (MS_BITS * (d + 2)));
#pragma unroll
                for (int s = 0; 2 * s <= d; ++s) {
                    const int t = d - s;
#pragma unroll
                    for (int p = 0; p < 2; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            hcamd_floatx4 part{0.f, 0.f, 0.f, 0.f};
                            part = __builtin_amdgcn_mfma_f32_16x16x16f16(a[p][s], b[q][t], part, 0, 0, 0);
                            if (s != t) part = __builtin_amdgcn_mfma_f32_16x16x16f16(a[p][t], b[q][s], part, 0, 0, 0);
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[p][q][v] = fma((double) part[v], wgt, acc[p][q][v]);
                        }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int ri = wr + 16 * p + 4 * g + v, cj = wc + 16 * q + i16;
                const int ci = ti * GT_M + ri, cc = tj * GT_N + cj;
                if (ci < M && cc < N) C[ci + (int64_t) cc * ldc] = ldexp(acc[p][q][v], ea[ri] + eb[cj]);
            }
    __syncthreads();
}

__device__ inline void wg_gemm_mixed(int M, int N, int Kd, const double *A, int64_t lda, bool ta, const double *B,
                                     int64_t ldb, bool tb, double *C, int64_t ldc, float *lds) {
    const int tm = (M + GT_M - 1) / GT_M, tn = (N + GT_N - 1) / GT_N;
    for (int t = 0; t < tm * tn; ++t)
        wg_gemm_tile_mixed(M, N, Kd, A, lda, ta, B, ldb, tb, C, ldc, t % tm, t / tm, lds);
}

}  // namespace hcamd
