// HIP kernels of the TLR recompression engine (gfx950).  Each kernel is a thin
// wrapper that maps workgroups onto the workgroup-level phases of
// recompress.hpp / gemm.hpp; the batched persistent kernel runs every phase of
// one update in one workgroup and pulls updates from a device work queue.
#include "kernels.hpp"

#include <cstring>
#include <type_traits>

#include "plain_qr.hpp"

namespace hcamd {


// Phase timestamps of the batched kernel (100 MHz constant clock), recorded only in builds
// with HCAMD_PHASE_TIMING; read back with hcorepp_batch_phase_times.
#ifdef HCAMD_PHASE_TIMING
#define HCAMD_TSTAMP() ((uint64_t) wall_clock64())
#else
#define HCAMD_TSTAMP() ((uint64_t) 0)
#endif

template <typename T>
__global__ void HCAMD_KERNEL k_gemm(int M, int N, int Kd, T alpha, const T *A, int64_t lda, int ta,
                                             const T *B, int64_t ldb, int tb, T beta, T *C, int64_t ldc) {
    __shared__ T lds[GT_LDS_ELEMS];
    wg_gemm_tile<T>(M, N, Kd, alpha, A, lda, ta != 0, B, ldb, tb != 0, beta, C, ldc, blockIdx.x, blockIdx.y, lds);
}

template <typename T>
__global__ void __launch_bounds__(GS_WAVES *WAVE) k_gemm_small(int M, int N, int Kd, T alpha, const T *A, int64_t lda,
                                                              int ta, const T *B, int64_t ldb, int tb, T beta, T *C,
                                                              int64_t ldc) {
    __shared__ T lds[GS_LDS_ELEMS];
    auto fa = [=](int i, int k) -> T { return ta ? A[k + (int64_t) i * lda] : A[i + (int64_t) k * lda]; };
    auto fb = [=](int k, int j) -> T { return tb ? B[j + (int64_t) k * ldb] : B[k + (int64_t) j * ldb]; };
    auto epi = [=](int gi, int gj, T v) {
        T *c = C + gi + (int64_t) gj * ldc;
        *c = (beta == T(0)) ? alpha * v : alpha * v + beta * *c;
    };
    wg_gemm_small<T>(M, N, Kd, fa, fb, epi, blockIdx.x, blockIdx.y, lds);
}

template <typename T>
__global__ void HCAMD_KERNEL k_stack(RecompDesc<T> d) {
    ph_stack<T>(d, blockIdx.x, gridDim.x);
}

template <typename T>
__global__ void HCAMD_KERNEL k_y(RecompDesc<T> d) {
    __shared__ T lds[GT_LDS_ELEMS];
    ph_y<T>(d, blockIdx.x, gridDim.x, lds);
}

// The same by 32 x 32 tiles (wg_gemm_small), where gemm_is_small says so.
template <typename T>
__global__ void __launch_bounds__(GS_WAVES *WAVE) k_y_small(RecompDesc<T> d, int K, int mu) {
    __shared__ T lds[GS_LDS_ELEMS];
    const WsLayout L = ws_layout<T>(d.m, d.n, d.kmax, d.max_rank);
    const StackedV<T> fa = stacked_v(d, K);
    const T *us = d.ws + L.us;
    T *y = d.ws + L.y;
    const int64_t ldu = d.m, ldy = d.n;
    auto fb = [=](int k, int j) -> T { return k < j ? T(0) : us[j + (int64_t) k * ldu]; };  // R_U^T
    auto epi = [=](int gi, int gj, T v) { y[gi + (int64_t) gj * ldy] = v; };
    wg_gemm_small<T>(d.n, mu, K, fa, fb, epi, blockIdx.x, blockIdx.y, lds, (int) blockIdx.y * GS_T);
}

// ---------------------------------------------------------------------------
// Blocked QR of the plain form (plain_qr.hpp): one launch factors a panel (one workgroup, window pivoting
// included for the QR of Y); the next applies its block reflector to the trailing columns, 4 or 16 columns
// per workgroup over the whole GPU.  The operand's pointers and sizes come as arguments: the host knows
// them, and a read of the workspace header at the start of every launch took 2 us.
// ---------------------------------------------------------------------------

// Set-up of the QR of Y: squared column norms (one wave per column, eight loads in flight: 9.4 us for columns of 2048 rows with
// one, 3.5 now), the identity permutation and J = 0.
template <typename T>
__global__ void HCAMD_KERNEL k_qr_setup(PlainQr<T> q, int kk) {
    const int l = lane_id();
    for (int c = blockIdx.x * NWAVES + wave_id(); c < q.ncols; c += gridDim.x * NWAVES) {
        const T *col = q.A + (int64_t) c * q.m;
        T sum = T(0);
#pragma unroll 8
        for (int r = l; r < q.m; r += WAVE) sum += col[r] * col[r];
        sum = wave_sum(sum);
        if (l == 0) {
            q.cn[c] = sum;
            q.piv[c] = c;
        }
    }
    const int64_t tot = (int64_t) q.ncols * kk;
    for (int64_t e = (int64_t) blockIdx.x * NT + threadIdx.x; e < tot; e += (int64_t) gridDim.x * NT) q.J[e] = T(0);
}

template <typename T, int WAVES, int GROUPS>
__global__ void __launch_bounds__(WAVES *WAVE) k_qr_panel(PlainQr<T> q, RecompDesc<T> d, int kk, int j0) {
    __shared__ PanelLds<T, WAVES> lds;
    // the QR of Y stops at the first panel whose trailing matrix is below the core-truncation
    // level (as ph_qr_y); the launches after that return at once
    if (q.pivot && q.hdr[HDR_KQ] > 0) return;
    wg_panel<T, WAVES, GROUPS>(q, j0, lds, [&](T trail2) {
        if (j0 == 0) {
            if (threadIdx.x == 0) q.hdr[HDR_STOP2] = __double_as_longlong((double) qr_y_stop2<T>(d, trail2, kk));
            return false;
        }
        if (!(trail2 <= (T) __longlong_as_double(q.hdr[HDR_STOP2]))) return false;
        if (threadIdx.x == 0) {
            q.hdr[HDR_KQ] = j0;
            q.hdr[HDR_TRAIL2] = __double_as_longlong((double) trail2);
        }
        return true;
    });
}

// Trailing update: workgroup x takes the uc <= 16 columns at positions j0 + jb + uc x on.  The block is read
// once, kept in registers through both products and written back; pivoted, its rows of R go to J and the
// squared norms below them to cn for the next panel's pivoting.
template <typename T, int WAVES, int GROUPS>
__global__ void __launch_bounds__(WAVES *WAVE) k_qr_update(PlainQr<T> q, int j0, int uc) {
    __shared__ WyLds<T, WAVES> lds;
    const int ln = lane_id(), i16 = ln & 15, k4 = ln >> 4, wv = wave_id();
    const int rows = q.m - j0;
    const int nsteps = q.m < q.ncols ? q.m : q.ncols;
    const int jb = nsteps - j0 < PQ_NB ? nsteps - j0 : PQ_NB;
    const int pos = j0 + jb + uc * (int) blockIdx.x + i16;
    const bool cok = i16 < uc && pos < q.ncols, wide = wide_columns(q.A, q.m);
    auto column = [&](int p) { return q.pivot ? q.piv[p] : p; };
    const int c = column(cok ? pos : j0);
    const T *pcol = q.A + (int64_t) column(j0 + (i16 < jb ? i16 : 0)) * q.m + j0;
    if (q.pivot && q.hdr[HDR_KQ] > 0) return;  // the QR of Y stopped early
    T *col = q.A + (int64_t) c * q.m + j0;
    T b[GROUPS][4];
    load_block<WAVES>(col, rows, cok, wide, b);
    const T *ts = q.tsave + (int64_t) (j0 / PQ_NB) * PQ_NB * PQ_NB;
    // the panel's columns hold R on and above the diagonal: unit lower in the first group of rows
    wy_block<T, WAVES, GROUPS>(
            b,
            [&](int t, T (&v)[4]) {
                const int g = wv + WAVES * t;
                load_rows<GROUPS>(pcol, own_rows<GROUPS>(16 * g + 4 * k4), rows, i16 < jb, wide, v);
                if (g == 0) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int r = 4 * k4 + s;
                        v[s] = r > i16 ? v[s] : T(r == i16 && i16 < jb);
                    }
                }
            },
            [&](int i, int j) { return i <= j ? ts[i + PQ_NB * j] : T(0); }, true, 0, lds);
    T nsq = T(0);
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        const int r = own_rows<GROUPS>(16 * (wv + WAVES * t) + 4 * k4);
        if (q.pivot) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if (t == 0 && cok && r + s < jb) q.J[c + (int64_t) (j0 + r + s) * q.ncols] = b[t][s];
                if (cok && (t > 0 || r + s >= jb) && r + s < rows) nsq = fma(b[t][s], b[t][s], nsq);
            }
        }
        store_rows<GROUPS>(col, r, rows, cok, wide, b[t]);
        group_end<GROUPS>();
    }
    if (q.pivot) {
        nsq = col_sum(nsq);
        if (k4 == 0) lds.part[wv][i16] = nsq;  // the partial products were read before the last barrier
        __syncthreads();
        if (threadIdx.x < PQ_NB && cok) {
            T sum = T(0);
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) sum += lds.part[ww][i16];
            q.cn[pos] = sum;
        }
    }
}

// Waves and 16-row groups per wave for a block of `rows` rows (2048 at most).  Eight waves, whose 256 registers hold the
// FP64 blocks of 1024 rows with both operands of an update and those of 2048 rows alone (sixteen waves' 128 spilled all of
// it); FP32 blocks take half and sixteen waves beyond 1024 rows.
template <typename T, typename F>
static void pq_shape(int rows, F f) {
    const int g = (rows + 15) / 16;
    if (g <= 8) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
    else if (g <= 16) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 2>{});
    else if (g <= 32) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 4>{});
    else if (g <= 64) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 8>{});
    else if constexpr (sizeof(T) == 8) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 16>{}, std::integral_constant<int, 8>{});
}

template <typename T>
static hipError_t launch_qr(hipStream_t s, const RecompDesc<T> &d, const PlainQr<T> &q, int kk) {
    const int nsteps = q.m < q.ncols ? q.m : q.ncols;
    if (q.pivot) {
        const int grid = (q.ncols + NWAVES - 1) / NWAVES;
        hipLaunchKernelGGL(k_qr_setup<T>, dim3(grid), dim3(NT), 0, s, q, kk);
    }
    for (int j0 = 0; j0 < nsteps; j0 += PQ_NB) {
        const int jb = nsteps - j0 < PQ_NB ? nsteps - j0 : PQ_NB, trail = q.ncols - (j0 + jb);
        pq_shape<T>(q.m - j0, [&](auto waves, auto groups) {
            constexpr int WV = decltype(waves)::value, GR = decltype(groups)::value;
            hipLaunchKernelGGL((k_qr_panel<T, WV, GR>), dim3(1), dim3(WV * WAVE), 0, s, q, d, kk, j0);
            // four columns per workgroup while that is one workgroup per CU at most: an update is bound by what one CU
            // moves of its columns, not by the matrix cores, which 16 would fill (1024 rows 24.8 us with 16, 20.9 with
            // 8, 19.0 with 4; 512 rows 13.8, 11.9, 11.0; 256 rows 8.4, 7.6, 7.1; 17.9, 10.5 and 7.0 since P is read once).
            // Beyond, either is within 1 % of the whole update: 600 rows, 1200 stacked columns 10.61 ms with 16, 10.68 with 4,
            // 700 rows and 1400 columns 14.07 and 14.19
            const int uc = trail <= 4 * 256 ? 4 : PQ_NB;
            if (trail > 0)
                hipLaunchKernelGGL((k_qr_update<T, WV, GR>), dim3((trail + uc - 1) / uc), dim3(WV * WAVE), 0, s, q, j0, uc);
        });
    }
    return hipGetLastError();
}

template <typename T>
__global__ void HCAMD_KERNEL k_fill_identity(T *I, int64_t n) {
    for (int64_t e = (int64_t) blockIdx.x * NT + threadIdx.x; e < n * n; e += (int64_t) gridDim.x * NT)
        I[e] = ((e % n) == (e / n)) ? T(1) : T(0);
}

template <typename T>
hipError_t launch_fill_identity(hipStream_t s, T *I, int64_t n) {
    int64_t grid = (n * n + NT - 1) / NT;
    if (grid > 1024) grid = 1024;
    hipLaunchKernelGGL(k_fill_identity<T>, dim3((unsigned) (grid > 0 ? grid : 1)), dim3(NT), 0, s, I, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Core SVD of the plain (one update per launch sequence) form: the core build, the Jacobi with V
// accumulated, the rank rule.  Narrow cores run the Jacobi in one workgroup; a core of MW_MIN_COLS
// columns or more is spread over the GPU, one launch per step of the round-robin ordering of
// super-blocks (jacobi.hpp).  flags[s] records whether sweep s saw a pair far from orthogonal; the
// launches of a later sweep return at once when it did not.
// ---------------------------------------------------------------------------
constexpr int JW_THREADS = 512;                  // the one-workgroup Jacobi
constexpr int64_t JW_LDS_BYTES = 150 * 1024;     // its LDS: the workgroup has the CU to itself

// Squared norms of the core's columns (the rows of R_Y), one wave per column.
template <typename T>
__global__ void HCAMD_KERNEL k_core_norms(const T *J, int mu, int kk, T *rn) {
    for (int j = blockIdx.x * NWAVES + wave_id(); j < kk; j += gridDim.x * NWAVES) {
        T sum = T(0);
        for (int r = lane_id(); r < mu; r += WAVE) {
            const T v = J[r + (int64_t) j * mu];
            sum += v * v;
        }
        sum = wave_sum(sum);
        if (lane_id() == 0) rn[j] = sum;
    }
}

// Core width from those norms (ph_core_width), ||J||_F^2, and the Jacobi's flags.
template <typename T>
__global__ void HCAMD_KERNEL k_core_size(RecompDesc<T> d, const T *norms, int32_t *flags) {
    __shared__ T rn[CORE_LDS_ELEMS];
    Ws<T> w = ws_of(d);
    const Dims z = dims_of(d, w);
    for (int j = threadIdx.x; j < z.kk; j += NT) rn[j] = norms[j];
    for (int i = threadIdx.x; i < JACOBI_MAX_SWEEPS; i += NT) flags[i] = 0;
    __syncthreads();
    ph_core_width<T>(d, rn);
    if (threadIdx.x == 0) {
        // rn[j] = ||R_Y[j:, :]||_F^2 now, so ||J||_F^2 = rn[0] - rn[kt]
        const int kt = (int) w.hdr[HDR_KT];
        const T fro2 = z.kk > 0 ? rn[0] - (kt < z.kk ? rn[kt] : T(0)) : T(0);
        w.hdr[HDR_JFRO2] = __double_as_longlong((double) fro2);
    }
}

// One-workgroup Jacobi; J, and V beside it, move into LDS where they fit (ld odd).
template <typename T>
__global__ void __launch_bounds__(JW_THREADS) k_jacobi_wg(RecompDesc<T> d) {
    extern __shared__ unsigned char smem_raw[];
    T *lds = reinterpret_cast<T *>(smem_raw);
    constexpr int NW = JW_THREADS / WAVE;
    constexpr int64_t cap = JW_LDS_BYTES / (int64_t) sizeof(T) - gram_jacobi_lds<T>(NW);
    Ws<T> w = ws_of(d);
    const Dims z = dims_of(d, w);
    const int rows = z.mu, nc = z.kt, ldj = rows | 1, ldv = nc | 1;
    const T fro2 = (T) __longlong_as_double(w.hdr[HDR_JFRO2]), stop = JacobiStopCos<T>::tight;
    T *Jl = lds + gram_jacobi_lds<T>(NW), *Vl = Jl + (int64_t) ldj * nc;
    const bool jin = (int64_t) ldj * nc <= cap, vin = (int64_t) (ldj + ldv) * nc <= cap;
    int sweeps;
    if (!vin)
        for (ColWalk p(threadIdx.x, JW_THREADS, nc); p.c < nc; p.next()) w.v1[p.i + (int64_t) p.c * nc] = T(p.i == p.c);
    if (nc < 1) {
        sweeps = 0;
    } else if (jin) {
        for (ColWalk p(threadIdx.x, JW_THREADS, rows); p.c < nc; p.next())
            Jl[p.i + p.c * ldj] = w.j[p.i + (int64_t) p.c * rows];
        if (vin) {
            for (ColWalk p(threadIdx.x, JW_THREADS, nc); p.c < nc; p.next()) Vl[p.i + p.c * ldv] = T(p.i == p.c);
            __syncthreads();
            sweeps = wg_gram_jacobi<T>(Jl, ldj, rows, nc, Vl, ldv, nc, fro2, stop, JACOBI_MAX_SWEEPS, NW, lds);
        } else {
            __syncthreads();
            sweeps = wg_gram_jacobi<T>(Jl, ldj, rows, nc, w.v1, nc, nc, fro2, stop, JACOBI_MAX_SWEEPS, NW, lds);
        }
        __syncthreads();
        for (ColWalk p(threadIdx.x, JW_THREADS, rows); p.c < nc; p.next())
            w.j[p.i + (int64_t) p.c * rows] = Jl[p.i + p.c * ldj];
        if (vin)
            for (ColWalk p(threadIdx.x, JW_THREADS, nc); p.c < nc; p.next())
                w.v1[p.i + (int64_t) p.c * nc] = Vl[p.i + p.c * ldv];
    } else {
        __syncthreads();
        sweeps = wg_gram_jacobi<T>(w.j, rows, rows, nc, w.v1, nc, nc, fro2, stop, JACOBI_MAX_SWEEPS, NW, lds);
    }
    if (threadIdx.x == 0) w.hdr[HDR_SWEEPS] = sweeps;
}

// What the steps of one multi-workgroup Jacobi work on.  The host knows the core's width and norm by
// then, so a step starts on its columns at once instead of after two dependent reads of the header (7.2 ->
// 6.6 us per step of a 128-column core).  rec: the records of two launches (npair each, alternating),
// then their flags; they sit in the core-QR region of the workspace (j2 and what follows), which the
// plain form does not use otherwise.
template <typename T>
struct MwJacobi {
    T *j, *v, *rec;
    int32_t *flags;
    int rows, ncols, nbp;  // nbp: blocks, rounded up to even
    T fro2;
};

// Step `step` of sweep `sweep` (blockIdx.y 0), and V's part of the step before it (blockIdx.y >= 1);
// `last`: only V's part, after the last step launched.  GROUPS: 16-row groups per wave.
template <typename T, int GROUPS>
__global__ void __launch_bounds__(MW_WAVES *WAVE) k_jacobi_step(MwJacobi<T> m, int sweep, int step, int last) {
    __shared__ T lds[MW_LDS];
    const int npair = m.nbp / 2, steps = m.nbp - 1;
    const bool rotate = blockIdx.y == 0;
    int launch = sweep * steps + step;  // the launch whose pair this workgroup works on
    if (rotate) {
        if (last) return;
    } else {
        if (launch == 0) return;
        --launch;
    }
    const int sw = launch / steps, st = launch % steps, bp = (int) blockIdx.x;
    int cI, cJ;
    if (!jacobi_pair_cols(bp, st, m.nbp, GJ_B, m.ncols, cI, cJ)) return;
    if (st > 0 && cJ >= m.ncols) return;
    const int32_t live = sw > 0 ? m.flags[sw - 1] : 1;  // 0: converged in an earlier sweep
    T *rec = m.rec + (int64_t) ((launch & 1) * npair + bp) * MW_REC;
    int32_t *used = reinterpret_cast<int32_t *>(m.rec + (int64_t) 2 * npair * MW_REC) + (launch & 1) * npair + bp;
    if (rotate) {
        const GramTol<T> g(m.fro2, m.rows, JacobiStopCos<T>::tight);
        const int any =
                mw_rotate_tile<T, GROUPS>(m.j, m.rows, m.ncols, cI, cJ, st == 0, live != 0, g, rec, used, lds);
        if ((any & JROT_LARGE) && threadIdx.x == 0) m.flags[sw] = 1;
    } else if (live && *used) {
        mw_apply_v<T>(m.v, m.ncols, m.ncols, cI, cJ, rec, ((int) blockIdx.y - 1) * MW_VROWS);
    }
}

template <typename T>
static void launch_jacobi_step(hipStream_t s, const MwJacobi<T> &m, int sweep, int step, int last) {
    const dim3 wg(MW_WAVES * WAVE), grid(m.nbp / 2, 1 + (m.ncols + MW_VROWS - 1) / MW_VROWS);
    const int groups = (m.rows + 16 * MW_WAVES - 1) / (16 * MW_WAVES);
    if (groups <= 1) hipLaunchKernelGGL((k_jacobi_step<T, 1>), grid, wg, 0, s, m, sweep, step, last);
    else if (groups <= 2) hipLaunchKernelGGL((k_jacobi_step<T, 2>), grid, wg, 0, s, m, sweep, step, last);
    else if (groups <= 4) hipLaunchKernelGGL((k_jacobi_step<T, 4>), grid, wg, 0, s, m, sweep, step, last);
    else hipLaunchKernelGGL((k_jacobi_step<T, 6>), grid, wg, 0, s, m, sweep, step, last);
}
static_assert(JACOBI_ROWS_MAX <= 16 * MW_WAVES * 6, "the widest k_jacobi_step holds the tallest core");

// Singular values (column norms of the orthogonalised core), one wave per column.
template <typename T>
__global__ void HCAMD_KERNEL k_svd_sigma(RecompDesc<T> d) {
    Ws<T> w = ws_of(d);
    const Dims z = dims_of(d, w);
    const int j = blockIdx.x * NWAVES + wave_id();
    if (j >= z.kt) return;
    const T *zj = w.j + (int64_t) j * z.mu;
    T s = T(0);
    for (int r = lane_id(); r < z.mu; r += WAVE) s += zj[r] * zj[r];
    s = wave_sum(s);
    if (lane_id() == 0) w.sig[j] = sqrt(s);
}

// Their descending order, four threads per column, and (workgroup 0) the rank rule.  `launched` sweeps of
// the multi-workgroup Jacobi, or -1 after the one-workgroup one.
template <typename T>
__global__ void HCAMD_KERNEL k_svd_rank(RecompDesc<T> d, const int32_t *flags, int launched) {
    __shared__ T sig[JACOBI_ROWS_MAX];
    Ws<T> w = ws_of(d);
    const Dims z = dims_of(d, w);
    const int kt = z.kt;
    for (int j = threadIdx.x; j < kt; j += NT) sig[j] = w.sig[j];
    __syncthreads();
    const int j = (int) blockIdx.x * (NT / 4) + (int) threadIdx.x / 4, part = threadIdx.x % 4;
    int pos = 0;
    if (j < kt) {
        const T sj = order_key(sig[j]);
        for (int k = part; k < kt; k += 4) {
            const T sk = order_key(sig[k]);
            pos += (sk > sj) || (sk == sj && k < j);
        }
    }
    pos += __shfl_xor(pos, 1, WAVE);
    pos += __shfl_xor(pos, 2, WAVE);
    if (j < kt && part == 0) {
        w.perm[pos] = j;
        if (d.sigma_out) d.sigma_out[pos] = (double) sig[j];
    }
    if (blockIdx.x != 0) return;
    if (d.sigma_out)
        for (int i = kt + threadIdx.x; i < z.kk; i += NT) d.sigma_out[i] = 0.0;
    int sweeps = launched < 0 ? (int) w.hdr[HDR_SWEEPS] : launched;
    for (int s = 0; s < launched; ++s)
        if (flags[s] == 0) {
            sweeps = s;
            break;
        }
    ph_rank<T>(d, sig, sweeps);
}

// The whole core SVD.  Cores that may be wide (kk columns are known here) have their width read back
// once, so that the steps are launched for the columns there are: the core is cut at the rounding
// level, often at half of kk, and a launch that finds nothing to do costs as much as a tenth of a step.
// The sweeps are launched in chunks; the host reads the last sweep's flag between chunks.
template <typename T>
static hipError_t launch_core_svd(hipStream_t s, const RecompDesc<T> &d, int mu, int kk, int32_t *flags,
                                  volatile int64_t *host, T *scratch) {
    const WsLayout L = ws_layout<T>(d.m, d.n, d.kmax, d.max_rank);
    auto finish = [&](int kt, int launched) {
        hipLaunchKernelGGL(k_svd_sigma<T>, dim3((kt + NWAVES - 1) / NWAVES), dim3(NT), 0, s, d);
        hipLaunchKernelGGL(k_svd_rank<T>, dim3((kt + NT / 4 - 1) / (NT / 4)), dim3(NT), 0, s, d, flags, launched);
        return hipGetLastError();
    };
    hipLaunchKernelGGL(k_core_norms<T>, dim3((kk + NWAVES - 1) / NWAVES), dim3(NT), 0, s, (const T *) (d.ws + L.j), mu,
                       kk, scratch);
    hipLaunchKernelGGL(k_core_size<T>, dim3(1), dim3(NT), 0, s, d, (const T *) scratch, flags);
    hipError_t e;
    int kt = kk;
    T fro2 = T(0);
    if (kk >= MW_MIN_COLS) {
        static_assert(HDR_JFRO2 == HDR_KT + 1, "read together");
        const int64_t *hdr = reinterpret_cast<const int64_t *>(d.ws);
        e = hipMemcpyAsync((void *) host, hdr + HDR_KT, 2 * sizeof(int64_t), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        kt = (int) host[0];
        const int64_t bits = host[1];
        double f;
        memcpy(&f, &bits, sizeof(f));
        fro2 = (T) f;
    }
    if (kt < MW_MIN_COLS) {
        hipLaunchKernelGGL(k_jacobi_wg<T>, dim3(1), dim3(JW_THREADS), JW_LDS_BYTES, s, d);
        return finish(kt, -1);
    }
    const int nblk = (kt + GJ_B - 1) / GJ_B, nbp = nblk + (nblk & 1);
    const MwJacobi<T> m{d.ws + L.j, d.ws + L.v1, d.ws + L.j2, flags, mu, kt, nbp, fro2};
    e = launch_fill_identity<T>(s, m.v, kt);
    if (e != hipSuccess) return e;
    // most cores converge within 5 to 8 sweeps: the first five are launched at once, then one at a time
    int launched = 0, chunk = 5;
    while (launched < JACOBI_MAX_SWEEPS) {
        const int end = launched + chunk < JACOBI_MAX_SWEEPS ? launched + chunk : JACOBI_MAX_SWEEPS;
        for (int sw = launched; sw < end; ++sw)
            for (int st = 0; st < nbp - 1; ++st) launch_jacobi_step<T>(s, m, sw, st, 0);
        launched = end;
        e = hipGetLastError();
        if (e == hipSuccess)
            e = hipMemcpyAsync((void *) host, flags + launched - 1, sizeof(int32_t), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        if (*reinterpret_cast<volatile int32_t *>(host) == 0) break;
        chunk = 1;
    }
    launch_jacobi_step<T>(s, m, launched, 0, 1);
    return finish(kt, launched);
}

// Reconstruction of the plain form, 16 columns of the new rank per workgroup, side blockIdx.y:
//   0: C_U[:, c] = Q_U [z_perm(c) / sigma; 0]  (z: column of J = P R_Y^T after the Jacobi; P, the pivoting of
//      the QR of Y, is applied when J is built)
//   1: C_V[c, :] = (Q_Y [v1_perm(c) sigma; 0])^T
// The block stays in registers from its first to its last reflector panel and goes straight to the tile
// (C_V transposed: 16 consecutive elements per store).
template <typename T, int WAVES, int GROUPS>
__global__ void __launch_bounds__(WAVES *WAVE) k_recon(RecompDesc<T> d) {
    __shared__ WyLds<T, WAVES> lds;
    __shared__ int32_t cols[PQ_MAX_COLS];  // the columns that hold the reflectors
    Ws<T> w = ws_of(d);
    const Dims z = dims_of(d, w);
    const int r = (int) w.hdr[HDR_RANK], side = (int) blockIdx.y;
    const int ln = lane_id(), i16 = ln & 15, k4 = ln >> 4, wv = wave_id();
    const int c = PQ_NB * (int) blockIdx.x + i16;
    const bool cok = c < r && c < z.kt;
    const int rows = side ? d.n : d.m, filled = side ? z.kt : z.mu;
    const T *src = side ? w.v1 : w.j;
    const int j = cok ? w.perm[c] : 0;
    const T sg = cok ? w.sig[j] : T(0);
    T b[GROUPS][4];
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        const int r0 = own_rows<GROUPS>(16 * (wv + WAVES * t) + 4 * k4);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int row = r0 + s;
            const T v = (cok && row < filled) ? src[row + (int64_t) j * filled] : T(0);
            b[t][s] = side ? v * sg : (sg > T(0) ? v / sg : T(0));
        }
        group_end<GROUPS>();
    }
    const T *A = side ? w.y : w.us, *tsave = side ? w.t_y : w.t_u;  // ld rows
    // [v1 sigma; 0] vanishes below row kt, where reflectors kt.. of Q_Y act as the identity (each is zero
    // above its own row), so only the first kt are applied
    const int nref = side ? (z.kt < z.kk ? z.kt : z.kk) : z.mu;
    const bool wide = wide_columns(A, rows);
    for (int i = threadIdx.x; i < nref; i += WAVES * WAVE) cols[i] = side ? w.piv[i] : i;
    __syncthreads();
    for (int p = (nref + PQ_NB - 1) / PQ_NB - 1; p >= 0; --p) {
        const int j0 = p * PQ_NB, jb = nref - j0 < PQ_NB ? nref - j0 : PQ_NB;
        const T *ts = tsave + (int64_t) p * PQ_NB * PQ_NB;
        const T *pcol = A + (int64_t) cols[j0 + (i16 < jb ? i16 : 0)] * rows;
        // the panel is unit lower from row j0 on (a multiple of 16: one mixed group)
        wy_block<T, WAVES, GROUPS>(
                b,
                [&](int t, T (&v)[4]) {
                    const int g = wv + WAVES * t;
                    load_rows<GROUPS>(pcol, own_rows<GROUPS>(16 * g + 4 * k4), rows, i16 < jb && g >= p, wide, v);
                    if (g == p) {
#pragma unroll
                        for (int s = 0; s < 4; ++s) {
                            const int rr = 4 * k4 + s;
                            v[s] = rr > i16 ? v[s] : T(rr == i16 && i16 < jb);
                        }
                    }
                },
                [&](int i, int jj) { return (i <= jj && jj < jb) ? ts[i + PQ_NB * jj] : T(0); }, false, p, lds);
    }
    if (c >= r) return;
    T *cu = d.cdata, *cv = d.cdata + (int64_t) d.m * d.max_rank;
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
        const int r0 = own_rows<GROUPS>(16 * (wv + WAVES * t) + 4 * k4);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int row = r0 + s;
            if (row < rows) {
                if (side) cv[c + (int64_t) row * r] = b[t][s];
                else cu[row + (int64_t) c * d.m] = b[t][s];
            }
        }
        group_end<GROUPS>();
    }
}

__global__ void k_set_i64(int64_t *p, int64_t v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

// Fill V (n x n, ld n) with the identity (FillIdentityMatrix, reference omp/kernels.cpp:144-151,
// on a zeroed buffer) and copy U = W (m x n): the DDC ReadjustTile (Compressed.cpp:696-734).
template <typename T>
__global__ void HCAMD_KERNEL k_readjust_ddc(const T *W, int64_t m, int64_t n, T *cdata) {
    const int64_t tot = m * n + n * n;
    for (int64_t e = (int64_t) blockIdx.x * NT + threadIdx.x; e < tot; e += (int64_t) gridDim.x * NT) {
        if (e < m * n) {
            cdata[e] = W[e];
        } else {
            const int64_t f = e - m * n;
            cdata[e] = ((f % n) == (f / n)) ? T(1) : T(0);
        }
    }
}

// ---------------------------------------------------------------------------
// Batched persistent kernel.
// ---------------------------------------------------------------------------
static_assert(GTM_LDS_FLOATS * sizeof(float) <= (size_t) BATCH_LDS_BYTES, "mixed tile GEMM LDS");

// Factor products of one update (C.Gemm's temporaries).  mixed: FP16 matrix-core products of
// the operands' error-free slices with FP32 accumulation (FP64 operands and results,
// wg_gemm_mixed), otherwise FP64.
template <typename T>
__device__ void run_temp_gemms(const BatchEntry<T> &e, T *lds, int mixed) {
    for (int g = 0; g < e.ngemm; ++g) {
        const GemmSpec<T> &s = e.gemm[g];
        if constexpr (sizeof(T) == 8) {
            if (mixed) {
                wg_gemm_mixed(s.m, s.n, s.k, s.a, s.lda, s.ta, s.b, s.ldb, s.tb, s.c, s.ldc,
                              reinterpret_cast<float *>(lds));
                __syncthreads();
                continue;
            }
        }
        wg_gemm<T>(s.m, s.n, s.k, T(1), s.a, s.lda, s.ta, s.b, s.ldb, s.tb, T(0), s.c, s.ldc, lds);
        __syncthreads();
    }
}

// The rebased copy of one batch entry: pointers named by `rel` are byte offsets into `slot`.
template <typename P>
__device__ __forceinline__ P rebase(P p, int32_t rel, int32_t bit, char *slot) {
    return (rel & bit) ? reinterpret_cast<P>(slot + reinterpret_cast<uintptr_t>(p)) : p;
}

template <typename T, int PB>
__global__ void HCAMD_KERNEL k_batched(const BatchEntry<T> *entries, const int32_t *order, int64_t n,
                                       BatchCounters *ctr, int mixed, char *slots, int64_t slot_bytes,
                                       int64_t *hdrs) {
    extern __shared__ unsigned char smem_raw[];
    T *lds = reinterpret_cast<T *>(smem_raw);
    __shared__ int64_t s_item;
    __shared__ BatchEntry<T> s_ent;  // the current update, its pointers rebased onto this slot
    char *slot = slots + (int64_t) blockIdx.x * slot_bytes;
    for (;;) {
        if (threadIdx.x == 0) s_item = (int64_t) atomicAdd(&ctr->next, 1ULL);
        __syncthreads();
        const int64_t item = s_item;
        if (item >= n) break;
        const int32_t idx = order[item];
        if (threadIdx.x == 0) {
            BatchEntry<T> e = entries[idx];
            const int32_t rel = e.rel;
            e.gemm[0].a = rebase(e.gemm[0].a, rel, REL_G0A, slot);
            e.gemm[0].b = rebase(e.gemm[0].b, rel, REL_G0B, slot);
            e.gemm[0].c = rebase(e.gemm[0].c, rel, REL_G0C, slot);
            e.gemm[1].a = rebase(e.gemm[1].a, rel, REL_G1A, slot);
            e.gemm[1].b = rebase(e.gemm[1].b, rel, REL_G1B, slot);
            e.gemm[1].c = rebase(e.gemm[1].c, rel, REL_G1C, slot);
            e.rd.afin = rebase(e.rd.afin, rel, REL_AFIN, slot);
            e.rd.bfin = rebase(e.rd.bfin, rel, REL_BFIN, slot);
            e.rd.ws = rebase(e.rd.ws, rel, REL_WS, slot);
            s_ent = e;
        }
        __syncthreads();
        const BatchEntry<T> &e = s_ent;
        const RecompDesc<T> &d = e.rd;
        Ws<T> w = ws_of(d);
        // the slot's header still holds the previous update's words: start from zero
        for (int k = threadIdx.x; k < HDR_WORDS; k += NT) w.hdr[k] = 0;
        __syncthreads();
        const uint64_t t_start = HCAMD_TSTAMP();
        run_temp_gemms<T>(e, lds, mixed);
        const uint64_t t_gemm = HCAMD_TSTAMP();
        // FP64 with 16-column panels: the QR of U_s reads U_s beyond its first panel in place
        // (StackedU); only the first panel's 16 columns are stacked
        constexpr bool u_in_place = PB == 16 && sizeof(T) == 8;
        ph_stack<T, !u_in_place>(d, 0, 1);
        __syncthreads();
        const Dims z = dims_of(d, w);
        // features for the rank model, and in the exact form, whose runs are its training data;
        // the tolerance rule without a model reads the core width off R_Y and needs none
        if (z.K <= d.kmax && (d.rank_model || !(d.model_tol > 0.0))) ph_features<T>(d, lds);
        uint64_t t_qru = 0, t_y = 0, t_qry = 0, t_svd = 0, t_ru = 0;
        if (z.K <= d.kmax) {
            wg_geqrf<T, PB>(d.m, z.K, w.us, d.m, w.tau_u, w.t_u, lds, w.hdr, u_in_place, stacked_u(d, z.K));
            __syncthreads();
            t_qru = HCAMD_TSTAMP();
            ph_y<T>(d, 0, 1, lds);
            __syncthreads();
            t_y = HCAMD_TSTAMP();
            ph_qr_y<T, PB>(d, lds);
            __syncthreads();
            ph_core_size<T>(d, lds);
            ph_learned_size<T>(d, lds);
            ph_core_build<T>(d);
            ph_core_qr<T, PB>(d, lds);
            t_qry = HCAMD_TSTAMP();
            ph_svd_nov<T>(d);
            __syncthreads();
            t_svd = HCAMD_TSTAMP();
        }
        // A core beyond the Jacobi's limit, or NaN/Inf in the factors, leaves C as it was: its
        // factors and rank are kept and the status word reports the update.
        const bool keep_c = (z.K > d.kmax) || (w.hdr[HDR_STATUS] & (STATUS_TOO_BIG | STATUS_NAN)) != 0;
        const int r = keep_c ? (int) *d.crank : (int) w.hdr[HDR_RANK];
        if (!keep_c) {
            ph_recon_nov<T, PB>(d, lds);
            __syncthreads();
            t_ru = HCAMD_TSTAMP();
            ph_finish<T>(d, 0, 1);
            __syncthreads();
        }
#ifdef HCAMD_PHASE_TIMING
        if (threadIdx.x == 0) {
            const uint64_t ts[8] = {t_start, t_gemm, t_qru, t_y, t_qry, t_svd, t_ru, HCAMD_TSTAMP()};
            for (int k = 0; k < 8; ++k) w.hdr[HDR_T0 + k] = (int64_t) ts[k];
        }
        __syncthreads();
#else
        (void) t_start; (void) t_gemm; (void) t_qru; (void) t_y; (void) t_qry; (void) t_svd; (void) t_ru;
#endif
        if (threadIdx.x == 0) {
            *d.crank = r;
            const int64_t st = w.hdr[HDR_STATUS];
            if (st) atomicOr(&ctr->status, (unsigned long long) st);
            if (z.K <= d.kmax && w.hdr[HDR_LEARNED] == 2) atomicAdd(&ctr->fallbacks, 1ULL);
            atomicMax(&ctr->max_sweeps, (unsigned long long) w.hdr[HDR_SWEEPS]);
        }
        // the header outlives the slot: diagnostics read it per update
        for (int k = threadIdx.x; k < HDR_WORDS; k += NT) hdrs[(int64_t) idx * HDR_WORDS + k] = w.hdr[k];
        __syncthreads();
    }
}

__global__ void k_reset_counters(BatchCounters *c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        c->next = 0;
        c->status = 0;
        c->max_sweeps = 0;
        c->fallbacks = 0;
    }
}

// ---------------------------------------------------------------------------
// Host launch wrappers
// ---------------------------------------------------------------------------
template <typename T>
hipError_t launch_gemm(hipStream_t s, int M, int N, int Kd, T alpha, const T *A, int64_t lda, bool ta, const T *B,
                       int64_t ldb, bool tb, T beta, T *C, int64_t ldc) {
    if (M <= 0 || N <= 0) return hipSuccess;
    if (gemm_is_small<T>(M, N, Kd, ta, tb)) {
        dim3 grid((M + GS_T - 1) / GS_T, (N + GS_T - 1) / GS_T);
        hipLaunchKernelGGL(k_gemm_small<T>, grid, dim3(GS_WAVES * WAVE), 0, s, M, N, Kd, alpha, A, lda, (int) ta, B, ldb,
                           (int) tb, beta, C, ldc);
        return hipGetLastError();
    }
    dim3 grid((M + GT_M - 1) / GT_M, (N + GT_N - 1) / GT_N);
    hipLaunchKernelGGL(k_gemm<T>, grid, dim3(NT), 0, s, M, N, Kd, alpha, A, lda, (int) ta, B, ldb, (int) tb, beta,
                       C, ldc);
    return hipGetLastError();
}

// Householder panel width for a QR of `rows` rows: the widest panel whose register tile in
// apply_wy (rows/256 row chunks x PB per lane) stays within 32 values and whose LDS fits.
int pick_pb(int64_t rows, int64_t lds_elems) {
    for (int p = 16; p >= 4; p /= 2)
        if (pb_fits(rows, p, lds_elems)) return p;
    return 0;
}

// Whether a panel of pb columns is valid for a QR of `rows` rows: an instantiated width, at most
// 32 panel values per lane in apply_wy, and the panel workspace within lds_elems.
bool pb_fits(int64_t rows, int pb, int64_t lds_elems) {
    if (pb != 4 && pb != 8 && pb != 16) return false;
    if (rows > 2048 * 4 / pb) return false;
    return qr_lds_elems(rows, pb) <= lds_elems;
}

static int clamp_grid(int64_t work) {
    int64_t g = (work + NT - 1) / NT;
    if (g > 1024) g = 1024;
    if (g < 1) g = 1;
    return (int) g;
}

template <typename T>
hipError_t launch_recomp_pre(hipStream_t s, const RecompDesc<T> &d, int64_t K, int32_t *jflags, int64_t *host,
                             T *cn) {
    const int64_t m = d.m, n = d.n;
    const int64_t mu = m < K ? m : K;
    const int64_t kk = n < mu ? n : mu;
    hipLaunchKernelGGL(k_stack<T>, dim3(clamp_grid(m * K)), dim3(NT), 0, s, d);
    const WsLayout L = ws_layout<T>(m, n, d.kmax, d.max_rank);
    int64_t *hdr = reinterpret_cast<int64_t *>(d.ws + L.hdr);
    const PlainQr<T> qu{d.ws + L.us, d.ws + L.tau_u, d.ws + L.t_u, nullptr, nullptr, nullptr, hdr, (int) m, (int) K, 0};
    const PlainQr<T> qy{d.ws + L.y, d.ws + L.tau_y, d.ws + L.t_y, d.ws + L.j, cn,
                        reinterpret_cast<int32_t *>(d.ws + L.piv), hdr, (int) n, (int) mu, 1};
    hipError_t e = launch_qr<T>(s, d, qu, (int) kk);
    if (e != hipSuccess) return e;
    const int ytiles = (int) (((n + GT_M - 1) / GT_M) * ((mu + GT_N - 1) / GT_N));
    if (gemm_is_small<T>(n, mu, K, true, true))  // V_s and R_U^T are read as transposed operands are
        hipLaunchKernelGGL(k_y_small<T>, dim3((unsigned) ((n + GS_T - 1) / GS_T), (unsigned) ((mu + GS_T - 1) / GS_T)),
                           dim3(GS_WAVES * WAVE), 0, s, d, (int) K, (int) mu);
    else
        hipLaunchKernelGGL(k_y<T>, dim3(ytiles), dim3(NT), 0, s, d);
    e = launch_qr<T>(s, d, qy, (int) kk);
    if (e != hipSuccess) return e;
    return launch_core_svd<T>(s, d, (int) mu, (int) kk, jflags, host, cn);
}

template <typename T>
hipError_t launch_recomp_post(hipStream_t s, const RecompDesc<T> &d, int64_t r) {
    pq_shape<T>(d.m > d.n ? d.m : d.n, [&](auto waves, auto groups) {
        constexpr int WV = decltype(waves)::value, GR = decltype(groups)::value;
        hipLaunchKernelGGL((k_recon<T, WV, GR>), dim3((unsigned) ((r + PQ_NB - 1) / PQ_NB), 2), dim3(WV * WAVE), 0, s, d);
    });
    return hipGetLastError();
}

hipError_t launch_set_i64(hipStream_t s, int64_t *p, int64_t v) {
    hipLaunchKernelGGL(k_set_i64, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_readjust_ddc(hipStream_t s, const T *W, int64_t m, int64_t n, T *cdata) {
    int nwg = (int) ((m * n + n * n + NT - 1) / NT);
    if (nwg > 1024) nwg = 1024;
    hipLaunchKernelGGL(k_readjust_ddc<T>, dim3(nwg), dim3(NT), 0, s, W, m, n, cdata);
    return hipGetLastError();
}

hipError_t launch_reset_counters(hipStream_t s, BatchCounters *c) {
    hipLaunchKernelGGL(k_reset_counters, dim3(1), dim3(64), 0, s, c);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_batched(hipStream_t s, const BatchEntry<T> *entries, const int32_t *order, int64_t n,
                          BatchCounters *ctr, int grid, int64_t lds_bytes, int pb, int mixed, char *slots,
                          int64_t slot_bytes, int64_t *hdrs) {
    switch (pb) {
        case 16:
            hipLaunchKernelGGL((k_batched<T, 16>), dim3(grid), dim3(NT), lds_bytes, s, entries, order, n, ctr, mixed,
                               slots, slot_bytes, hdrs);
            break;
        case 8:
            hipLaunchKernelGGL((k_batched<T, 8>), dim3(grid), dim3(NT), lds_bytes, s, entries, order, n, ctr, mixed,
                               slots, slot_bytes, hdrs);
            break;
        default:
            hipLaunchKernelGGL((k_batched<T, 4>), dim3(grid), dim3(NT), lds_bytes, s, entries, order, n, ctr, mixed,
                               slots, slot_bytes, hdrs);
            break;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t set_kernel_lds_limits(int64_t lds_bytes) {
    // Allow the dynamic-LDS kernels to use more than the default 64 KB.
    if constexpr (sizeof(T) == 8) {  // the batched form is FP64
        const void *fns[] = {
                (const void *) k_batched<T, 16>, (const void *) k_batched<T, 8>, (const void *) k_batched<T, 4>,
        };
        for (const void *f : fns) {
            hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds_bytes);
            if (e != hipSuccess) return e;
        }
    }
    return hipFuncSetAttribute((const void *) k_jacobi_wg<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int) JW_LDS_BYTES);
}

#define HCAMD_INSTANTIATE(T)                                                                                     \
    template hipError_t launch_gemm<T>(hipStream_t, int, int, int, T, const T *, int64_t, bool, const T *,      \
                                       int64_t, bool, T, T *, int64_t);                                          \
    template hipError_t launch_recomp_pre<T>(hipStream_t, const RecompDesc<T> &, int64_t, int32_t *, int64_t *,  \
                                             T *);                                                               \
    template hipError_t launch_recomp_post<T>(hipStream_t, const RecompDesc<T> &, int64_t);                      \
    template hipError_t launch_readjust_ddc<T>(hipStream_t, const T *, int64_t, int64_t, T *);                   \
    template hipError_t launch_fill_identity<T>(hipStream_t, T *, int64_t);                                      \
    template hipError_t set_kernel_lds_limits<T>(int64_t);

HCAMD_INSTANTIATE(double)
HCAMD_INSTANTIATE(float)
template hipError_t launch_batched<double>(hipStream_t, const BatchEntry<double> *, const int32_t *, int64_t,
                                           BatchCounters *, int, int64_t, int, int, char *, int64_t, int64_t *);

}  // namespace hcamd
