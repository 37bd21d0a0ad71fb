// solve.hip -- multi-RHS solve with the LU factors and FP64 iterative
// refinement.  Replaces cuSOLVER Zgetrs (solver.cu:51-84, 125-128).
//
// Right-hand sides and solutions are planar FP64, row-major n x ldr (one RHS
// per column), resident on the device.  A solve with the factors of P Z = L U:
//   Y = P B;  Y <- L^{-1} Y;  Y <- U^{-1} Y
// in blocks of rows: the diagonal block (FP32 factors: by its inverse; FP64: by
// substitution, trsm.h), then the update of the remaining rows on the matrix
// cores (cmul.h; gemm.h), for all right-hand sides at once.
//
// Mixed precision (factors in FP32): X_0 = 0, R_0 = B, and per sweep
//   D = solve32(fp32(P R));  X += D;  R = B - Z X   (with the FP64 Z: zmul.hip)
// until max_j ||R_j|| / ||B_j|| <= tol.  Norm reductions use a fixed order.
#include <algorithm>
#include <cmath>

#include "../bem_internal.h"
#include "cmul.h"
#include "gemm.h"
#include "trsm.h"

namespace {

constexpr int NB = 256;

template <typename T>
__global__ __launch_bounds__(256) void k_gather_rows(int n, int ncol, const int* __restrict__ perm,
                                                     const double* __restrict__ Br, const double* __restrict__ Bi,
                                                     long ldb, T* __restrict__ Yr, T* __restrict__ Yi, long ldy) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)n * ncol) return;
    const int i = (int)(idx / ncol), j = (int)(idx % ncol);
    const long src = (long)perm[i] * ldb + j;
    Yr[(long)i * ldy + j] = (T)Br[src];
    Yi[(long)i * ldy + j] = (T)Bi[src];
}

template <typename T>
__global__ __launch_bounds__(256) void k_accumulate(long count, const T* __restrict__ Dr, const T* __restrict__ Di,
                                                    double* __restrict__ Xr, double* __restrict__ Xi, int assign) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    if (assign) {
        Xr[i] = (double)Dr[i];
        Xi[i] = (double)Di[i];
    } else {
        Xr[i] += (double)Dr[i];
        Xi[i] += (double)Di[i];
    }
}

// M, N and K multiples of 16.  The column tiles are split into the groups that need the
// fewest rounds of workgroups (one per CU), each of a time of about 2 NT + 1: one tile
// per workgroup while those fit the chip at once (768 x 64, K = 1024: 8.7 us; four tiles
// 18), several after that (17408 x 128: 217 us; 137).
constexpr int kCmulTiles = 5;
void cmul(bem_ctx* c, int M, int N, int K, int tri, const float* Ar, const float* Ai, long lda, const float* Br,
          const float* Bi, long ldb, float* Cr, float* Ci, long ldc, int mode) {
    if (M <= 0) return;
    const int kt = kt_mark(c, KS_GEMM32, c->stream);
    const int tiles = N / 16, rows = M / 16;
    auto cost = [&](int nt, int ngrp) { return ngrp ? (2 * nt + 1) * (((long)rows * ngrp + c->cus - 1) / c->cus) : 0L; };
    int G = tiles;
    long least = cost(1, tiles);
    for (int g = tiles - 1; g * kCmulTiles >= tiles && g > 0; g--) {
        const int wide = tiles % g;
        const long t = cost(tiles / g + 1, wide) + cost(tiles / g, g - wide);
        if (t <= least) {
            least = t;
            G = g;
        }
    }
    const int nt = tiles / G, wide = tiles % G;
    for (int p = 0; p < 2; p++) {
        const int t = p ? nt : nt + 1, ngrp = p ? G - wide : wide, c0 = p ? 16 * (nt + 1) * wide : 0;
        if (ngrp == 0) continue;
        auto k = t == 1 ? k_cmul<1> : t == 2 ? k_cmul<2> : t == 3 ? k_cmul<3> : t == 4 ? k_cmul<4> : k_cmul<5>;
        hipLaunchKernelGGL(k, dim3((unsigned)((rows * ngrp + 7) / 8 * 8)), dim3(256), 0, c->stream, rows * ngrp, ngrp,
                           c0, K, tri, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode);
    }
    kt_close(c, kt, (tri ? 3.0 : 6.0) * (double)M * N * K,
             2.0 * sizeof(float) * ((tri ? 0.5 : 1.0) * (double)M * K + (double)K * N + (mode == 0 ? 2.0 : 1.0) * M * N));
}

// Y <- U^{-1} L^{-1} Y for the FP32 factors at (Fr, Fi), Y planar n x ncol (ld ncol), with
// the inverses of the IB x IB diagonal blocks at inv (L blocks, then U blocks; n x IB per
// plane), which refinement corrects:
//   forward   W_I = L_II^{-1} Y_I;   Y_{>I} -= L_{>I,I} W_I
//   backward  Y_I = U_II^{-1} W_I;   W_{<I} -= U_{<I,I} Y_I
// from kTwoLevel rows on in two levels: the blocks of a superblock of kSuper update the
// rows inside it only, then one update brings its solution into all rows beyond it
// (17408 rows, 80 columns: 107 + 14 us instead of 4 x 34; with 2816 rows 25 + 15 instead of
// 4 x 9.5).  Below, two levels would be faster for many columns (256 at 7000 unknowns 1.22
// ms, 1.38) and slower for few (16: 0.65, 0.61), and sums of 1024 terms instead of 256
// leave an unrefined residual 1.15 - 1.3 times as large.  W is a work buffer of Y's shape;
// the result is left in Y.
constexpr int kSuper = 4, kTwoLevel = 8192;
void lu_apply32(bem_ctx* c, const float* Fr, const float* Fi, const void* inv, float* Yr, float* Yi, float* Wr,
                float* Wi, int ncol) {
    const int n = c->npad;
    const long ld = n;
    const float* Lir = static_cast<const float*>(inv);
    const float* Lii = Lir + (size_t)n * IB;
    const float* Uir = Lii + (size_t)n * IB;
    const float* Uii = Uir + (size_t)n * IB;
    const int super = n >= kTwoLevel ? kSuper * IB : IB;
    // rows [r0, r0 + rows) of C -= F[rows, [k0, k0 + K)] X[[k0, k0 + K), :]
    auto update = [&](int r0, int rows, int k0, int K, const float* xr, const float* xi, float* cr, float* ci) {
        const long a = (long)r0 * ld + k0, x = (long)k0 * ncol, o = (long)r0 * ncol;
        cmul(c, rows, ncol, K, 0, Fr + a, Fi + a, ld, xr + x, xi + x, ncol, cr + o, ci + o, ncol, 0);
    };
    for (int s0 = 0; s0 < n; s0 += super) {
        const int s1 = std::min(s0 + super, n);
        for (int r = s0; r < s1; r += IB) {
            const long y = (long)r * ncol, io = (long)r * IB;
            cmul(c, IB, ncol, IB, 1, Lir + io, Lii + io, IB, Yr + y, Yi + y, ncol, Wr + y, Wi + y, ncol, 1);
            update(r + IB, s1 - r - IB, r, IB, Wr, Wi, Yr, Yi);
        }
        update(s1, n - s1, s0, s1 - s0, Wr, Wi, Yr, Yi);
    }
    for (int s1 = n; s1 > 0; s1 = std::max(s1 - super, 0)) {
        const int s0 = std::max(s1 - super, 0);
        for (int r = s1 - IB; r >= s0; r -= IB) {
            const long y = (long)r * ncol, io = (long)r * IB;
            cmul(c, IB, ncol, IB, 2, Uir + io, Uii + io, IB, Wr + y, Wi + y, ncol, Yr + y, Yi + y, ncol, 1);
            update(s0, r - s0, r, IB, Yr, Yi, Wr, Wi);
        }
        update(0, s0, s0, s1 - s0, Yr, Yi, Wr, Wi);
    }
}

// FP64 short-K products, K = NB: C -= A B with one 16 x 16 output tile
// per block and the block's four waves each taking a quarter of K.  The last
// updates of the triangular solves have too few output tiles and too short a K
// for the LDS-staged kernel to hide its load latency; here every wave issues
// all its loads at once, straight into MFMA operand registers.  Lane (r, g) =
// (lane % 16, lane / 16) holds A[m0 + r][k + 4g + i] (one 32-byte row chunk)
// and B[k + 4g + i][n0 + r] for MFMA i = 0..3 of each 16-wide K step: A and
// B see the same order of k.  The four wave tiles are summed through LDS in
// wave order.  Blocks b with one value of b % 8 (one XCD) take a contiguous
// run of the row-major tile order, so the column tiles of a row share that
// XCD's L2 copy of A's rows.  4M form (as k_cgemm).
constexpr int kShortKW = NB / 4;  // K per wave

__global__ __launch_bounds__(256) void k_cgemm_short(int M, int N, const double* __restrict__ Ar,
                                                     const double* __restrict__ Ai, long lda,
                                                     const double* __restrict__ Br, const double* __restrict__ Bi,
                                                     long ldb, double* __restrict__ Cr, double* __restrict__ Ci,
                                                     long ldc) {
    constexpr int NS = kShortKW / 16;  // K steps per wave
    __shared__ double red[4][2][16][17];
    const int nct = N / 16, G = (M / 16) * nct;
    const int per = (G + 7) / 8;
    const int f = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (f >= G) return;
    const int m0 = (f / nct) * 16, n0 = (f % nct) * 16;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    double ar[NS][4], ai[NS][4], br[NS][4], bi[NS][4];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = w * kShortKW + 16 * s + 4 * g;
        const long oa = (long)(m0 + r) * lda + k;
        load_row4<double>(Ar + oa, ar[s]);
        load_row4<double>(Ai + oa, ai[s]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long ob = (long)(k + i) * ldb + n0 + r;
            br[s][i] = Br[ob];
            bi[s][i] = Bi[ob];
        }
    }
    // every load in flight before the first MFMA waits on its operands
    __builtin_amdgcn_sched_barrier(0);
    v4d re{}, im{};
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            re = mfma16x16x4(ar[s][i], br[s][i], re);
            re = mfma16x16x4(ai[s][i], -bi[s][i], re);
            im = mfma16x16x4(ar[s][i], bi[s][i], im);
            im = mfma16x16x4(ai[s][i], br[s][i], im);
        }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        red[w][0][g + 4 * q][r] = re[q];
        red[w][1][g + 4 * q][r] = im[q];
    }
    __syncthreads();
    const int row = threadIdx.x / 16, col = threadIdx.x % 16;
    const long o = (long)(m0 + row) * ldc + n0 + col;
    Cr[o] -= ((red[0][0][row][col] + red[1][0][row][col]) + red[2][0][row][col]) + red[3][0][row][col];
    Ci[o] -= ((red[0][1][row][col] + red[1][1][row][col]) + red[2][1][row][col]) + red[3][1][row][col];
}

// C -= A B for K = NB, M and N multiples of 16 and 16-byte aligned rows of A, on the
// context stream with per-launch timing.
void cgemm_short_ctx(bem_ctx* c, int M, int N, const double* Ar, const double* Ai, long lda, const double* Br,
                     const double* Bi, long ldb, double* Cr, double* Ci, long ldc) {
    constexpr int K = NB;
    const int k = kt_mark(c, KS_GEMM64, c->stream);
    const long tiles = (long)(M / 16) * (N / 16);
    const unsigned grid = (unsigned)(((tiles + 7) / 8) * 8);
    hipLaunchKernelGGL(k_cgemm_short, dim3(grid), dim3(256), 0, c->stream, M, N, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc);
    kt_close(c, k, 8.0 * (double)M * N * K, 16.0 * ((double)M * K + (double)K * N + 2.0 * M * N));
}

// Updates of at most this many rows go to the short-K kernel (below it the
// tiled GEMM's launches are load-latency bound at K = 256).
constexpr int kShortRows = 4096;

// The same with the FP64 factors, in blocks of NB rows, whose diagonal blocks are solved by
// substitution (k_trsm_rhs): the unrefined FP64 solve stays backward stable as Zgetrs is.
void lu_apply64(bem_ctx* c, const double* Fr, const double* Fi, double* Yr, double* Yi, double* Wr, double* Wi,
                int ncol) {
    const int n = c->npad, nb = n / NB;
    const long ld = n;
    auto update = [&](int rows, const double* ar, const double* ai, const double* br, const double* bi, double* cr,
                      double* ci) {
        if (rows <= kShortRows)
            cgemm_short_ctx(c, rows, ncol, ar, ai, ld, br, bi, ncol, cr, ci, ncol);
        else
            cgemm_ctx(c, rows, ncol, NB, ar, ai, ld, br, bi, ncol, cr, ci, ncol, 0);
    };
    for (int I = 0; I < nb; I++) {
        const long y = (long)I * NB * ncol, dg = (long)I * NB * (ld + 1);
        trsm_rhs<double>(c->stream, true, Fr + dg, Fi + dg, ld, Yr + y, Yi + y, ncol, Wr + y, Wi + y, ncol, ncol);
        const int rest = n - (I + 1) * NB;
        if (rest > 0) {
            const long a = (long)(I + 1) * NB * ld + (long)I * NB, yc = (long)(I + 1) * NB * ncol;
            update(rest, Fr + a, Fi + a, Wr + y, Wi + y, Yr + yc, Yi + yc);
        }
    }
    for (int I = nb - 1; I >= 0; I--) {
        const long y = (long)I * NB * ncol, dg = (long)I * NB * (ld + 1);
        trsm_rhs<double>(c->stream, false, Fr + dg, Fi + dg, ld, Wr + y, Wi + y, ncol, Yr + y, Yi + y, ncol, ncol);
        if (I > 0) {
            const long a = (long)I * NB;  // rows 0 .. I*NB-1, columns of block I
            update(I * NB, Fr + a, Fi + a, Yr + y, Yi + y, Wr, Wi);
        }
    }
}

// |r| / |b| of one column from the squares (|r| itself for b = 0).
double ratio(double r2, double b2) { return b2 == 0.0 ? std::sqrt(r2) : std::sqrt(r2 / b2); }

constexpr double kTiny = 0x1p-540;  // the squares of all doubles times this, and their sums, are finite

// The same where a square is not finite, from the squares of the columns times kTiny.
double ratio_scaled(double r2, double b2, double r2s, double b2s) {
    const double r = std::isfinite(r2) ? kTiny * std::sqrt(r2) : std::sqrt(r2s);
    const double b = std::isfinite(b2) ? kTiny * std::sqrt(b2) : std::sqrt(b2s);
    return r / b;
}

}  // namespace

size_t lu_precond_work_bytes(const bem_ctx* c) {
    const size_t ysz = c->factored == BEM_F32_3M ? sizeof(float) : sizeof(double);
    return 4 * (size_t)c->npad * c->ldr * ysz;
}

int lu_precond_apply(bem_ctx* c, const double* Sr, const double* Si, double* Dr, double* Di, void* work) {
    const int n = c->npad, ncol = c->ldr;
    const long cnt = (long)n * ncol;
    hipStream_t s = c->stream;
    const dim3 g1((unsigned)((cnt + 255) / 256));
    if (c->factored == BEM_F32_3M) {
        float* Yr = static_cast<float*>(work);
        float* Yi = Yr + cnt;
        float* Qr = Yi + cnt;
        float* Qi = Qr + cnt;
        hipLaunchKernelGGL(k_gather_rows<float>, g1, dim3(256), 0, s, n, ncol, c->perm, Sr, Si, (long)ncol, Yr, Yi,
                           (long)ncol);
        lu_apply32(c, c->Wr, c->Wi, c->inv32, Yr, Yi, Qr, Qi, ncol);
        hipLaunchKernelGGL(k_accumulate<float>, g1, dim3(256), 0, s, cnt, Yr, Yi, Dr, Di, 1);
    } else if (c->factored == BEM_F64) {
        double* Yr = static_cast<double*>(work);
        double* Yi = Yr + cnt;
        double* Qr = Yi + cnt;
        double* Qi = Qr + cnt;
        hipLaunchKernelGGL(k_gather_rows<double>, g1, dim3(256), 0, s, n, ncol, c->perm, Sr, Si, (long)ncol, Yr, Yi,
                           (long)ncol);
        lu_apply64(c, c->Vr, c->Vi, Yr, Yi, Qr, Qi, ncol);
        hipLaunchKernelGGL(k_accumulate<double>, g1, dim3(256), 0, s, cnt, Yr, Yi, Dr, Di, 1);
    } else {
        return bem_fail(c, BEM_ERR_STATE, "preconditioner: no factorisation");
    }
    BEM_HIP(c, hipGetLastError());
    return 0;
}

int lu_solve_launch(bem_ctx* c, int nrhs, double tol, int maxit, int* iters, double* res0, double* res,
                    double* t_solve_ms, double* t_ir_ms) {
    const int n = c->npad, ldr = c->ldr, ncol = ldr;
    const long cnt = (long)n * ldr;
    hipStream_t s = c->stream;
    const bool f32 = c->factored == BEM_F32_3M;
    const bool can_refine = c->has_Z64;
    // scratch: R (FP64 planar), Y and W (working precision planar), norms
    const size_t ysz = f32 ? sizeof(float) : sizeof(double);
    const size_t npart = col_norm2_work(c->n, ldr);  // column-norm partial sums
    const size_t bytes = 2 * cnt * sizeof(double) + 4 * cnt * ysz + (2 * (size_t)ldr + npart) * sizeof(double) +
                         256;
    void* scr = nullptr;
    if (int rc = ctx_scratch(c, bytes, &scr)) return rc;
    double* Rr = static_cast<double*>(scr);
    double* Ri = Rr + cnt;
    char* yp = reinterpret_cast<char*>(Ri + cnt);
    char* wp = yp + 2 * cnt * ysz;
    double* nb2 = reinterpret_cast<double*>(wp + 2 * cnt * ysz);
    double* nr2 = nb2 + ldr;
    double* npt = nr2 + ldr;
    hipEvent_t e[4];
    for (auto& x : e) BEM_HIP(c, hipEventCreate(&x));
    const dim3 g1((unsigned)((cnt + 255) / 256));
    const dim3 gr((unsigned)(((long)n * ncol + 255) / 256));
    float ts = 0.0f, ti = 0.0f;
    std::vector<double> b2(ldr), r2(ldr);

    auto solve_into_X = [&](const double* Sr, const double* Si, int assign) {
        if (f32) {
            float* Yr = reinterpret_cast<float*>(yp);
            float* Yi = Yr + cnt;
            float* Wr = reinterpret_cast<float*>(wp);
            float* Wi = Wr + cnt;
            hipLaunchKernelGGL(k_gather_rows<float>, gr, dim3(256), 0, s, n, ncol, c->perm, Sr, Si, (long)ldr, Yr, Yi,
                               (long)ldr);
            lu_apply32(c, c->Wr, c->Wi, c->inv32, Yr, Yi, Wr, Wi, ncol);
            hipLaunchKernelGGL(k_accumulate<float>, g1, dim3(256), 0, s, cnt, Yr, Yi, c->Xr, c->Xi, assign);
        } else {
            double* Yr = reinterpret_cast<double*>(yp);
            double* Yi = Yr + cnt;
            double* Wr = reinterpret_cast<double*>(wp);
            double* Wi = Wr + cnt;
            hipLaunchKernelGGL(k_gather_rows<double>, gr, dim3(256), 0, s, n, ncol, c->perm, Sr, Si, (long)ldr, Yr,
                               Yi, (long)ldr);
            lu_apply64(c, c->Vr, c->Vi, Yr, Yi, Wr, Wi, ncol);
            hipLaunchKernelGGL(k_accumulate<double>, g1, dim3(256), 0, s, cnt, Yr, Yi, c->Xr, c->Xi, assign);
        }
    };
    auto residual = [&](bool first) -> int {  // R = B - Z X and *res, with B's norms at first
        if (int rc = z_product(c, ncol, c->Xr, c->Xi, c->Br, c->Bi, Rr, Ri)) return rc;
        col_norm2(s, c->n, nrhs, Rr, Ri, (long)ldr, npt, nr2);
        const size_t nb = nrhs * sizeof(double);
        if (int rc = first ? ctx_fetch(c, {{r2.data(), nr2, nb}, {b2.data(), nb2, nb}})
                           : ctx_fetch(c, {{r2.data(), nr2, nb}}))
            return rc;
        auto finite = [&](int j) { return std::isfinite(r2[j]) && std::isfinite(b2[j]); };
        int bad = 0;
        while (bad < nrhs && finite(bad)) bad++;
        std::vector<double> r2s, b2s;
        if (bad < nrhs) {  // values above 1e154, or no numbers at all
            r2s.resize(nrhs);
            b2s.resize(nrhs);
            col_norm2(s, c->n, nrhs, Rr, Ri, (long)ldr, npt, nr2, kTiny);
            col_norm2(s, c->n, nrhs, c->Br, c->Bi, (long)ldr, npt, nb2, kTiny);
            if (int rc = ctx_fetch(c, {{r2s.data(), nr2, nb}, {b2s.data(), nb2, nb}})) return rc;
        }
        *res = 0.0;
        for (int j = 0; j < nrhs; j++) {
            const double v = finite(j) ? ratio(r2[j], b2[j]) : ratio_scaled(r2[j], b2[j], r2s[j], b2s[j]);
            if (!(v <= *res)) *res = v;
            if (std::isnan(v)) break;  // (std::max would drop it, and a solution of NaN would count as converged)
        }
        return 0;
    };

    // plain solve
    BEM_HIP(c, hipEventRecord(e[0], s));
    solve_into_X(c->Br, c->Bi, 1);
    BEM_HIP(c, hipEventRecord(e[1], s));
    BEM_HIP(c, hipEventSynchronize(e[1]));
    BEM_HIP(c, hipEventElapsedTime(&ts, e[0], e[1]));
    *iters = 0;
    *res0 = *res = 0.0;
    int rc = 0;
    if (can_refine && (maxit > 0 || f32)) {
        BEM_HIP(c, hipEventRecord(e[2], s));
        col_norm2(s, c->n, nrhs, c->Br, c->Bi, (long)ldr, npt, nb2);
        if (int e2 = residual(true)) return e2;
        *res0 = *res;
        int it = 0;
        float ts_loop = 0.0f;  // triangular solves inside the sweeps
        while (it < maxit && *res > tol) {
            float t0 = 0.0f;
            BEM_HIP(c, hipEventRecord(e[0], s));
            solve_into_X(Rr, Ri, 0);
            BEM_HIP(c, hipEventRecord(e[1], s));
            if (int e2 = residual(false)) return e2;
            BEM_HIP(c, hipEventElapsedTime(&t0, e[0], e[1]));
            ts_loop += t0;
            it++;
        }
        *iters = it;
        BEM_HIP(c, hipEventRecord(e[3], s));
        BEM_HIP(c, hipEventSynchronize(e[3]));
        float tall = 0.0f;
        BEM_HIP(c, hipEventElapsedTime(&tall, e[2], e[3]));
        ts += ts_loop;          // all triangular solves
        ti = tall - ts_loop;    // residual GEMMs, norms, updates
        if (maxit > 0 && !(*res <= tol)) rc = BEM_ERR_NOCONV;  // a residual of NaN, too
    }
    BEM_HIP(c, hipGetLastError());
    for (auto& x : e) (void)hipEventDestroy(x);
    *t_solve_ms = ts;
    *t_ir_ms = std::max(0.0f, ti);
    return rc;
}
