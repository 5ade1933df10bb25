// Tile kernels of the TLR Cholesky factorisation A = L L^T (lower), in the engine's tile
// convention (compressed tile = U (m x r) V (r x n), stored [U | V], ld m and r):
//   potrf  dense diagonal tile A_kk = L_kk L_kk^T (in place, lower; the strict upper part is zeroed)
//   trsm   L_ik = A_ik L_kk^{-T}: only the V factor of a compressed A_ik changes, V <- V L_kk^{-T}
//   syrk   A_ii <- A_ii - L_ik L_ik^T = A_ii - U (V V^T) U^T for a compressed L_ik (dense A_ii)
//   transpose  compressed B = A^T: U_B = V_A^T, V_B = U_A^T (the B operand of the trailing
//              updates A_ij <- A_ij - L_ik L_jk^T, which then run as ordinary CCC recompressions)
// The trsm, syrk and transpose kernels handle a batch of independent tiles; potrf is blocked over several
// launches.
#include "kernels.hpp"
#include "cholesky.hpp"
#include "jacobi.hpp"
#include "trsm.hpp"

namespace hcamd {

constexpr int CB = 32;   // column block of the blocked potrf

// Row `i` of a CB-column block, zero past its jb columns.
template <typename T>
__device__ __forceinline__ void load_block_row(const T *A, int64_t lda, int jb, bool ok, T (&a)[CB]) {
#pragma unroll
    for (int c = 0; c < CB; ++c) a[c] = (ok && c < jb) ? A[(int64_t) c * lda] : T(0);
}

// Cholesky factor of the jb x jb diagonal block D (ld lda, lower triangle read) by one wave, row i in lane i's
// registers `a`; with PANEL also b <- b L^{-T} for a row `b` per lane.  Right-looking, every index known at
// compile time: step j broadcasts the column's elements from lane to lane through scalar registers, which
// both updates share.  Returns the first non-positive pivot (1-based) or 0; such a pivot is replaced by 1 so that
// the factorisation runs to the end.
//
// One wave, because the steps are a chain of a square root and a division each and a barrier per step
// (256 threads on a block in LDS) cost more than the whole of it: the block took 29 us and the solve below it 18
// (a row per thread, the columns in LDS).
template <typename T, bool PANEL>
__device__ __forceinline__ int factor_block(const T *D, int64_t lda, int jb, T (&a)[CB], T (&b)[CB]) {
    const int l = lane_id();
    load_block_row(D + l, lda, l + 1 < jb ? l + 1 : jb, l < jb, a);
#pragma unroll
    for (int c = 0; c < CB; ++c) a[c] = (c >= jb && l == c) ? T(1) : a[c];
    constexpr T lo = sizeof(T) == 8 ? T(1e-280) : T(1e-30f), hi = sizeof(T) == 8 ? T(1e280) : T(1e30f);
    int bad = 0;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const T v = read_lane(a[j], j);
        T p = T(1), r = T(1);
        if (v > lo && v < hi) {
            // square root and reciprocal from one reciprocal square root, with its residual step
            r = rsqrt_full(v);
            p = v * r;
            p = fma(fma(-p, p, v), T(0.5) * r, p);
        } else if (v > T(0)) {
            p = sqrt(v);
            r = T(1) / p;
        } else if (bad == 0) {
            bad = j + 1;
        }
        const T q = divide(a[j], p, r);
        a[j] = l == j ? p : q;
        if constexpr (PANEL) b[j] = divide(b[j], p, r);
#pragma unroll
        for (int c = j + 1; c < CB; ++c) {
            const T lc = read_lane(a[j], c);
            a[c] = fma(-a[j], lc, a[c]);
            if constexpr (PANEL) b[c] = fma(-b[j], lc, b[c]);
        }
    }
    return bad;
}

// Diagonal block of the blocked potrf in place.  info[0] receives the first non-positive pivot (1-based,
// whole-tile numbering) unless already set.
template <typename T>
__device__ __forceinline__ void write_diag(T *A, int64_t lda, int j0, int jb, int *info) {
    T a[CB], none[CB];
    T *D = A + j0 + (int64_t) j0 * lda;
    const int l = lane_id(), bad = factor_block<T, false>(D, lda, jb, a, none);
    if (l == 0 && bad && info[0] == 0) info[0] = j0 + bad;
#pragma unroll
    for (int c = 0; c < CB; ++c)
        if (l < jb && c <= l) D[l + (int64_t) c * lda] = a[c];
}

template <typename T>
__global__ void __launch_bounds__(WAVE) k_potrf_diag(T *A, int64_t lda, int j0, int jb, int *info) {
    write_diag(A, lda, j0, jb, info);
}

// Sub-diagonal panel of the blocked potrf: A[j0+CB:n, j0:j0+CB] <- (that) L_jj^{-T}, 64 rows per workgroup of
// one wave, each of which factors the diagonal block for itself (A_jj stays as it is until the trailing update's
// launch): the factor's broadcasts serve the rows as well, and a launch is saved.
template <typename T>
__global__ void __launch_bounds__(WAVE) k_potrf_panel(T *A, int n, int64_t lda, int j0) {
    const int r = j0 + CB + (int) blockIdx.x * WAVE + lane_id();
    T *row = A + (r < n ? r : n - 1) + (int64_t) j0 * lda;
    T a[CB], b[CB];
    load_block_row(row, lda, CB, true, b);
    factor_block<T, true>(A + j0 + (int64_t) j0 * lda, lda, CB, a, b);
    if (r < n)
#pragma unroll
        for (int c = 0; c < CB; ++c) row[(int64_t) c * lda] = b[c];
}

// Trailing update A22 -= L21 L21^T, the 32 x 32 tiles of the lower triangle only, one per wave on the matrix
// cores; the first workgroup's first wave writes the diagonal block's factor instead.
template <typename T>
__global__ void HCAMD_KERNEL k_potrf_trail(T *A, int n, int64_t lda, int j0, int *info) {
    using MF = Mfma16<T>;
    int t = (int) blockIdx.x * NWAVES + wave_id() - 1;
    if (t < 0) {
        write_diag(A, lda, j0, CB, info);
        return;
    }
    const int i1 = j0 + CB, rest = n - i1, nt = (rest + 31) / 32;
    int tj = 0;
    while (tj < nt && t >= nt - tj) t -= nt - tj++;
    if (tj >= nt) return;
    const int i0 = 32 * (tj + t), c0 = 32 * tj, l = lane_id(), i16 = l & 15, k4 = l >> 4;
    const T *L = A + i1 + (int64_t) j0 * lda;
    T *C = A + i1 + (int64_t) i1 * lda;
    typename MF::acc acc[2][2];
    T a[2][CB / 4], b[2][CB / 4], old[2][2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < CB / 4; ++s) {
            const int i = i0 + 16 * h + i16, j = c0 + 16 * h + i16;
            a[h][s] = i < rest ? L[i + (int64_t) (4 * s + k4) * lda] : T(0);
            b[h][s] = j < rest ? L[j + (int64_t) (4 * s + k4) * lda] : T(0);
        }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            acc[p][q] = MF::zero();
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + 16 * p + MF::row(v, k4), j = c0 + 16 * q + i16;
                old[p][q][v] = (i < rest && j < rest) ? C[i + (int64_t) j * lda] : T(0);
            }
        }
#pragma unroll
    for (int s = 0; s < CB / 4; ++s)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[p][q] = MF::mma(a[p][s], b[q][s], acc[p][q]);
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + 16 * p + MF::row(v, k4), j = c0 + 16 * q + i16;
                if (i < rest && j < rest) C[i + (int64_t) j * lda] = old[p][q][v] - acc[p][q][v];
            }
}

template <typename T>
__global__ void HCAMD_KERNEL k_zero_upper(T *A, int n, int64_t lda) {
    for (int64_t e = (int64_t) blockIdx.x * NT + threadIdx.x; e < (int64_t) n * n; e += (int64_t) gridDim.x * NT) {
        const int i = (int) (e % n), c = (int) (e / n);
        if (i < c) A[i + (int64_t) c * lda] = T(0);
    }
}

__global__ void k_zero_int(int *p) {
    if (threadIdx.x == 0) *p = 0;
}

// V (r x n, ld r) <- V L^{-T} for lower-triangular L (n x n, ld ldl): the rows of V solve L x^T = v^T,
// 16 rows of one tile per workgroup.  (One workgroup per tile with a row per thread took 358 us for tiles
// of 256 columns.)
__global__ void HCAMD_KERNEL k_trsm_v(const CholTrsm *jobs) {
    extern __shared__ unsigned char smem_raw[];
    const CholTrsm jb = jobs[blockIdx.y];
    const int r0 = (int) blockIdx.x * TS_NV, left = (int) jb.rank - r0;
    if (left <= 0) return;
    wg_trsm<double>(jb.v + r0, jb.rank, 1, left < TS_NV ? left : TS_NV, (int) jb.n, jb.l, jb.ldl, false, true, false,
                    1.0, reinterpret_cast<double *>(smem_raw));
}

// The same with a workgroup per tile and a row per thread.
__global__ void HCAMD_KERNEL k_trsm_v_rows(const CholTrsm *jobs) {
    __shared__ double lds[RT_LDS];
    const CholTrsm jb = jobs[blockIdx.x];
    wg_rows_trsm<double>(jb.v, (int) jb.rank, (int) jb.n, jb.rank, jb.l, jb.ldl, lds);
}

// A (n x n dense) <- A - U (V V^T) U^T, with scratch W (r x r) and T (n x r); the strict upper triangle of A is
// then set to 0, as the reference's Syrk does for a lower update.  Three launches of 32 x 32 tiles over all
// tiles' jobs (W and A by their lower triangles): a workgroup per job, which walked its three products alone,
// took 336 us for 11 tiles of 256 and left 245 CUs idle.
// Tile (ti, tj <= ti) of a lower triangle, column by column: tile `t` of nt (nt + 1) / 2.
__device__ __forceinline__ void lower_tile(int t, int nt, int &ti, int &tj) {
    tj = 0;
    while (t >= nt - tj) t -= nt - tj++;
    ti = tj + t;
}
__global__ void __launch_bounds__(GS_WAVES *WAVE) k_syrk_w(const CholSyrk *jobs) {
    __shared__ double lds[GS_LDS_ELEMS];
    const CholSyrk jb = jobs[blockIdx.y];
    const int n = (int) jb.n, r = (int) jb.rank, nt = (r + GS_T - 1) / GS_T;
    if ((int) blockIdx.x >= nt * (nt + 1) / 2) return;
    int ti, tj;
    lower_tile(blockIdx.x, nt, ti, tj);
    auto fa = [=](int i, int k) -> double { return jb.v[i + (int64_t) k * r]; };
    auto fb = [=](int k, int j) -> double { return jb.v[j + (int64_t) k * r]; };
    auto epi = [=](int i, int j, double v) {
        if (i >= j) jb.w[i + (int64_t) j * r] = jb.w[j + (int64_t) i * r] = v;
    };
    wg_gemm_small<double>(r, r, n, fa, fb, epi, ti, tj, lds);
}
__global__ void __launch_bounds__(GS_WAVES *WAVE) k_syrk_t(const CholSyrk *jobs) {
    __shared__ double lds[GS_LDS_ELEMS];
    const CholSyrk jb = jobs[blockIdx.y];
    const int n = (int) jb.n, r = (int) jb.rank, nt = (n + GS_T - 1) / GS_T, t = (int) blockIdx.x;
    if (t >= nt * ((r + GS_T - 1) / GS_T)) return;
    auto fa = [=](int i, int k) -> double { return jb.u[i + (int64_t) k * n]; };
    auto fb = [=](int k, int j) -> double { return jb.w[k + (int64_t) j * r]; };
    auto epi = [=](int i, int j, double v) { jb.t[i + (int64_t) j * n] = v; };
    wg_gemm_small<double>(n, r, r, fa, fb, epi, t % nt, t / nt, lds);
}
__global__ void __launch_bounds__(GS_WAVES *WAVE) k_syrk_a(const CholSyrk *jobs) {
    __shared__ double lds[GS_LDS_ELEMS];
    const CholSyrk jb = jobs[blockIdx.y];
    const int n = (int) jb.n, r = (int) jb.rank, nt = (n + GS_T - 1) / GS_T;
    if ((int) blockIdx.x >= nt * (nt + 1) / 2) return;
    int ti, tj;
    lower_tile(blockIdx.x, nt, ti, tj);
    auto fa = [=](int i, int k) -> double { return jb.t[i + (int64_t) k * n]; };
    auto fb = [=](int k, int j) -> double { return jb.u[j + (int64_t) k * n]; };
    auto epi = [=](int i, int j, double v) {
        double *a = jb.a + i + (int64_t) j * jb.lda;
        if (i >= j) *a -= v;
        if (i > j) jb.a[j + (int64_t) i * jb.lda] = 0.0;
    };
    wg_gemm_small<double>(n, n, r, fa, fb, epi, ti, tj, lds);
}

// The same with a workgroup per tile for its three products of 64 x 64 tiles.
__global__ void HCAMD_KERNEL k_syrk(const CholSyrk *jobs) {
    __shared__ double lds[GT_LDS_ELEMS];
    const CholSyrk jb = jobs[blockIdx.x];
    const int n = (int) jb.n, r = (int) jb.rank;
    if (r > 0) {
        wg_gemm<double>(r, r, n, 1.0, jb.v, r, false, jb.v, r, true, 0.0, jb.w, r, lds);
        __syncthreads();
        wg_gemm<double>(n, r, r, 1.0, jb.u, n, false, jb.w, r, false, 0.0, jb.t, n, lds);
        __syncthreads();
        wg_gemm<double>(n, n, r, -1.0, jb.t, n, false, jb.u, n, true, 1.0, jb.a, jb.lda, lds);
        __syncthreads();
    }
    if (n < 1) return;
    for (ColWalk p(threadIdx.x, NT, n); p.c < n; p.next())
        if (p.i < p.c) jb.a[p.i + (int64_t) p.c * jb.lda] = 0.0;
}

// dst (compressed, [U n x r | V r x m], max_rank cap) = src^T for src [U m x r | V r x n].
__global__ void HCAMD_KERNEL k_transpose_factors(const CholTrans *jobs) {
    const CholTrans jb = jobs[blockIdx.x];
    const int64_t m = jb.m, n = jb.n, r = jb.rank;
    const double *su = jb.src, *sv = jb.src + m * jb.src_max_rank;
    double *du = jb.dst, *dv = jb.dst + n * jb.dst_max_rank;
    for (int64_t e = threadIdx.x; e < n * r; e += NT) {  // du[j, a] = sv[a, j]
        const int64_t j = e % n, a = e / n;
        du[e] = sv[a + j * r];
    }
    for (int64_t e = threadIdx.x; e < r * m; e += NT) {  // dv[a, i] = su[i, a]
        const int64_t a = e % r, i = e / r;
        dv[e] = su[i + a * m];
    }
}

// Blocked right-looking potrf, two launches per block column: the panel below the diagonal block, then
// the trailing update of the lower triangle with the diagonal block's factor beside it.  The last block column
// has no panel.  The strict upper part is cleared at the end.  (Three launches before: the block, the panel,
// and the trailing product as a general one over both triangles.)  A 512 x 512 tile operation sequence, potrf, three
// trsm, three syrk and the updates, went from 8.2 to 7.4 ms, a factorisation of 12 x 12 tiles of 256 from 93.3 to
// 86.6 ms, with the syrk below the row solves in three launches as well.
template <typename T>
hipError_t launch_potrf(hipStream_t s, T *A, int n, int64_t lda, int *info) {
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, s, info);
    for (int j0 = 0; j0 < n; j0 += CB) {
        const int rest = n - j0 - CB;
        if (rest <= 0) {
            hipLaunchKernelGGL(k_potrf_diag<T>, dim3(1), dim3(WAVE), 0, s, A, lda, j0, n - j0, info);
            break;
        }
        hipLaunchKernelGGL(k_potrf_panel<T>, dim3((rest + WAVE - 1) / WAVE), dim3(WAVE), 0, s, A, n, lda, j0);
        const int nt = (rest + 31) / 32, waves = nt * (nt + 1) / 2 + 1;
        hipLaunchKernelGGL(k_potrf_trail<T>, dim3((waves + NWAVES - 1) / NWAVES), dim3(NT), 0, s, A, n, lda, j0, info);
    }
    int64_t work = (int64_t) n * n;
    int grid = (int) ((work + NT - 1) / NT);
    if (grid > 1024) grid = 1024;
    hipLaunchKernelGGL(k_zero_upper<T>, dim3(grid > 0 ? grid : 1), dim3(NT), 0, s, A, n, lda);
    return hipGetLastError();
}
template hipError_t launch_potrf<double>(hipStream_t, double *, int, int64_t, int *);
template hipError_t launch_potrf<float>(hipStream_t, float *, int, int64_t, int *);
hipError_t launch_trsm_v(hipStream_t s, const CholTrsm *jobs, int n, int max_rank, int len) {
    // Workgroups of 16 vectors: the time grows with their number, at about n / 1000 us each from 500 on.  A workgroup per
    // tile: a latency of about n us (1.3 n from 256 columns on), up to 1000 tiles of up to 256 rows at a time.  (us, 16
    // vectors each / a tile each: 32 columns 33 / 31, with 32 vectors 120 / 50 for 2048 tiles; 64 columns 45 / 48 for 512
    // tiles of 16 vectors, 114 / 87 for 2048; 128 columns with 64 vectors 73 / 110 for 128 tiles, 206 / 115 for 512, 742 / 241
    // for 2048; 256 columns with 200 vectors 445 / 380 for 128, 5906 / 1858 for 2048; 512 columns with 48 722 / 1200 for 512.)
    const int64_t groups = (max_rank + TS_NV - 1) / TS_NV;
    const bool rows_form = len <= 32 || groups * (n < 1000 ? n : 1000) >= 10 * (int64_t) len;
    if (n > 0 && rows_form) {
        hipLaunchKernelGGL(k_trsm_v_rows, dim3(n), dim3(NT), 0, s, jobs);
        return hipGetLastError();
    }
    // jobs along y (at most 65535 per launch)
    for (int j0 = 0; j0 < n; j0 += 65535) {
        const int nj = n - j0 < 65535 ? n - j0 : 65535;
        hipLaunchKernelGGL(k_trsm_v, dim3((max_rank + TS_NV - 1) / TS_NV, nj), dim3(NT), (size_t) ts_lds_bytes<double>(len),
                           s, jobs + j0);
    }
    return hipGetLastError();
}
hipError_t set_cholesky_lds_limits() {
    return hipFuncSetAttribute((const void *) k_trsm_v, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int) ts_lds_bytes<double>(ts_len_lds<double>()));
}
hipError_t launch_syrk(hipStream_t s, const CholSyrk *jobs, int n, int max_n, int max_rank) {
    const int nn = (max_n + GS_T - 1) / GS_T, nr = (max_rank + GS_T - 1) / GS_T;
    if (nn < 1) return hipSuccess;
    // A workgroup per tile from about one per CU on, where the three launches' tiles no longer find idle CUs (us, three
    // launches / one workgroup per tile: 48 rows 40 / 45 for 128 tiles, 48 / 47 for 256, 68 / 57 for 512, 371 / 274 for 4000;
    // 128 rows of rank 128 123 / 172 for 128, 407 / 289 for 512; 512 rows of rank 48 797 / 841 for 256, 1168 / 1145 for 384,
    // 1548 / 1202 for 512).  A tile of 32 rows is one workgroup's in the three launches as well (126 / 142 for 2048).
    const bool per_tile = max_n > 32 && n > (max_n <= 128 ? 256 : 384);
    if (per_tile) {
        hipLaunchKernelGGL(k_syrk, dim3(n), dim3(NT), 0, s, jobs);
        return hipGetLastError();
    }
    const dim3 wg(GS_WAVES * WAVE);
    // jobs along y (at most 65535 per launch)
    for (int j0 = 0; j0 < n; j0 += 65535) {
        const int nj = n - j0 < 65535 ? n - j0 : 65535;
        if (nr > 0) {
            hipLaunchKernelGGL(k_syrk_w, dim3(nr * (nr + 1) / 2, nj), wg, 0, s, jobs + j0);
            hipLaunchKernelGGL(k_syrk_t, dim3(nn * nr, nj), wg, 0, s, jobs + j0);
        }
        hipLaunchKernelGGL(k_syrk_a, dim3(nn * (nn + 1) / 2, nj), wg, 0, s, jobs + j0);
    }
    return hipGetLastError();
}
hipError_t launch_transpose_factors(hipStream_t s, const CholTrans *jobs, int n) {
    if (n > 0) hipLaunchKernelGGL(k_transpose_factors, dim3(n), dim3(NT), 0, s, jobs);
    return hipGetLastError();
}

}  // namespace hcamd
