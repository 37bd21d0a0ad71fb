// zmul.hip -- products of the FP64 matrix with a block of vectors (the refinement
// residual, the GMRES product) and column norms of such blocks.
#include <algorithm>

#include "../bem_internal.h"
#include "gemm.h"

namespace {

// P_s = A[:, K_s] X[K_s, :] for the columns c0 + 16 NT (0 .. ngrp - 1) .. of X and the
// splits K_s of Ks columns of A each; A is M x M (ld M), X and every P_s M x N, planar.
// FP64 in the 3M form (Re = Ar Xr - Ai Xi, Im = (Ar + Ai)(Xr + Xi) - Ar Xr - Ai Xi).
//
// A wave owns 16 rows and 16 NT columns and feeds the matrix cores straight from global
// memory, one step of 8 U columns of A ahead: no LDS and no barrier, since A is used by
// one wave only and a matrix-core product takes 64 cycles here.  In a step lane (r, g)
// holds A[row r][2 U g ..] (U 16-byte loads per plane) and X[2 U g ..][column r]; the
// four waves of a workgroup take consecutive rows and the same columns, so three of
// four X loads hit the L1.  Workgroups b with one value of b % 8 (one XCD) take a
// contiguous run of the order (split, rows, column groups): the groups reuse the rows of
// A from that XCD's L2, and its X comes from one or two splits.
//
// Bound by reading A for few columns and by the FP64 matrix cores (72 TFLOP/s) for
// many.  On assembled matrices, instead of with operands staged through LDS in tiles of
// 32 x 32 or 64 x 64: M = 4608, 16 columns 87 us (A at 3.9 TB/s) instead of 138, 128
// columns 0.30 ms instead of 0.40; M = 18432, 80 columns 2.78 ms instead of 4.25, 128
// columns 4.55 (57 TFLOP/s) instead of 4.79.  The accumulators have to stay out of the
// accumulation registers (two waves per SIMD as the bound): there the compiler copies
// them in and out in every step (128 columns 6.0 ms).
template <int NT, int U>
__global__ __launch_bounds__(256, 2) void k_zmul(int M, int N, int c0, int ngrp, int Ks, int nblk,
                                              const double* __restrict__ Ar, const double* __restrict__ Ai,
                                              const double* __restrict__ Xr, const double* __restrict__ Xi,
                                              double* __restrict__ P) {
    const int per = (nblk + 7) / 8;
    const int f = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (f >= nblk || (int)blockIdx.x / 8 >= per) return;
    const int nrow = M / 64, grp = f % ngrp, rb = f / ngrp % nrow, split = f / (ngrp * nrow);
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int m0 = 64 * rb + 16 * (threadIdx.x >> 6), n0 = c0 + 16 * NT * grp, k0 = split * Ks;
    constexpr int E = 2 * U, STEP = 8 * U, NP = NT / 2;
    const double* ar = Ar + (long)(m0 + r) * M + k0 + E * g;
    const double* ai = Ai + (long)(m0 + r) * M + k0 + E * g;
    const double* xr = Xr + (long)(k0 + E * g) * N + n0;
    const double* xi = Xi + (long)(k0 + E * g) * N + n0;
    struct Step {
        v2d a[2][U];
        double x[2][E][NT];
    } cur, nxt;
    auto load = [&](Step& s, int k) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            s.a[0][u] = *reinterpret_cast<const v2d*>(ar + k + 2 * u);
            s.a[1][u] = *reinterpret_cast<const v2d*>(ai + k + 2 * u);
        }
#pragma unroll
        for (int e = 0; e < E; e++)
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const double* x = (p ? xi : xr) + (long)(k + e) * N;
#pragma unroll
                for (int t = 0; t < NP; t++) {
                    const v2d v = *reinterpret_cast<const v2d*>(x + 32 * t + 2 * r);
                    s.x[p][e][2 * t] = v[0];
                    s.x[p][e][2 * t + 1] = v[1];
                }
                if constexpr (NT % 2) s.x[p][e][NT - 1] = x[32 * NP + r];
            }
    };
    v4d t1[NT], t2[NT], t3[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) t1[t] = t2[t] = t3[t] = v4d{};
    auto multiply = [&](const Step& s) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            const double a0 = s.a[0][e / 2][e % 2], a1 = s.a[1][e / 2][e % 2], a2 = a0 + a1;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const double x0 = s.x[0][e][t], x1 = s.x[1][e][t];
                t1[t] = mfma16x16x4(a0, x0, t1[t]);
                t2[t] = mfma16x16x4(a1, x1, t2[t]);
                t3[t] = mfma16x16x4(a2, x0 + x1, t3[t]);
            }
        }
    };
    load(cur, 0);
#pragma unroll 1
    for (int k = 0; k < Ks; k += 2 * STEP) {
        load(nxt, k + STEP);
        __builtin_amdgcn_sched_barrier(0);  // the next step's loads in flight before this one's products
        multiply(cur);
        __builtin_amdgcn_sched_barrier(0);
        load(cur, k + 2 * STEP < Ks ? k + 2 * STEP : k);  // (the last ones are not used)
        __builtin_amdgcn_sched_barrier(0);
        multiply(nxt);
        __builtin_amdgcn_sched_barrier(0);
    }
    const long count = (long)M * N;
    double* p = P + 2 * split * count + (long)(m0 + g) * N + n0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        double* o = p + (long)(4 * q) * N;
#pragma unroll
        for (int t = 0; t < NP; t++) {
            const int u = 2 * t, w = 2 * t + 1;
            *reinterpret_cast<v2d*>(o + 32 * t + 2 * r) = v2d{t1[u][q] - t2[u][q], t1[w][q] - t2[w][q]};
            *reinterpret_cast<v2d*>(o + count + 32 * t + 2 * r) =
                v2d{t3[u][q] - t1[u][q] - t2[u][q], t3[w][q] - t1[w][q] - t2[w][q]};
        }
        if constexpr (NT % 2) {
            constexpr int t = NT - 1;
            o[32 * NP + r] = t1[t][q] - t2[t][q];
            o[count + 32 * NP + r] = t3[t][q] - t1[t][q] - t2[t][q];
        }
    }
}

// O = B - sum_s P_s, or sum_s P_s without B, in split order; two values per thread.
__global__ __launch_bounds__(256) void k_zmul_sum(long count, int S, const double* __restrict__ P,
                                                  const double* __restrict__ Br, const double* __restrict__ Bi,
                                                  double* __restrict__ Or, double* __restrict__ Oi) {
    const long i = 2 * ((long)blockIdx.x * 256 + threadIdx.x);
    if (i >= count) return;
    v2d vr{}, vi{};
#pragma unroll 4
    for (int s = 0; s < S; s++) {
        vr += *reinterpret_cast<const v2d*>(P + 2 * s * count + i);
        vi += *reinterpret_cast<const v2d*>(P + (2 * s + 1) * count + i);
    }
    if (Br) {
        vr = *reinterpret_cast<const v2d*>(Br + i) - vr;
        vi = *reinterpret_cast<const v2d*>(Bi + i) - vi;
    }
    *reinterpret_cast<v2d*>(Or + i) = vr;
    *reinterpret_cast<v2d*>(Oi + i) = vi;
}

// Columns per wave: at most kTiles tiles of 16 (more do not fit the registers of two waves
// per SIMD; 80 columns at M = 18432 as 48 + 32, reading A twice, 3.66 ms).  Steps of 16
// columns of A for one or two tiles, where reading A is the bound (whole 128-byte lines
// of it per step: 16 columns at M = 18432 take 1.17 ms, in steps of 8 1.35), of 8 for
// more, where the longer step does not fit (64 columns: 2.11, 3.11).
constexpr int kTiles = 5;

// Splits of A's columns: the fewest of 1, 2, 4, 8, 16 that load the compute units evenly
// (95 % of the last one's blocks), else the most even.  A split is a multiple of 32 columns,
// two of the long steps.
int zmul_splits(int cus, int M, int N) {
    const int tiles = N / 16, grps = (tiles + kTiles - 1) / kTiles;
    const long rows = (long)(M / 64) * grps;
    int best = 1;
    double best_eff = 0.0;
    for (int S = 1; S <= 16 && M % (32 * S) == 0; S *= 2) {
        const long blocks = rows * S;
        const double eff = (double)blocks / (double)(cus * ((blocks + cus - 1) / cus));
        if (eff > best_eff + 1e-9) {
            best = S;
            best_eff = eff;
        }
        if (eff >= 0.95) break;
    }
    return best;
}

void zmul_launch(hipStream_t s, int nt, int M, int N, int c0, int ngrp, int S, const double* Ar, const double* Ai,
                 const double* Xr, const double* Xi, double* P) {
    const int nblk = ngrp * (M / 64) * S, Ks = M / S;
    const dim3 grid((unsigned)((nblk + 7) / 8 * 8));
    auto k = nt == 1 ? k_zmul<1, 2> : nt == 2 ? k_zmul<2, 2> : nt == 3 ? k_zmul<3, 1> : nt == 4 ? k_zmul<4, 1> : k_zmul<5, 1>;
    hipLaunchKernelGGL(k, grid, dim3(256), 0, s, M, N, c0, ngrp, Ks, nblk, Ar, Ai, Xr, Xi, P);
}

// part[b][j] = sum of |scale A[i][j]|^2 over the rows i of block b (kNormRows of them), j <
// ncol.  cw columns (a power of two, at most 64) side by side, the rows in 256 / cw
// lanes, summed in a fixed order.
constexpr int kNormRows = 128;
__global__ __launch_bounds__(256) void k_colnorm2_part(int n, int ncol, int cw, const double* __restrict__ Ar,
                                                       const double* __restrict__ Ai, long ld, double scale,
                                                       double* __restrict__ part) {
    __shared__ double red[256];
    const int tx = threadIdx.x % cw, ty = threadIdx.x / cw, lanes = 256 / cw;
    const int r0 = blockIdx.x * kNormRows, r1 = min(n, r0 + kNormRows), j = blockIdx.y * cw + tx;
    double s = 0.0;
    if (j < ncol)
#pragma unroll 8
        for (int i = r0 + ty; i < r1; i += lanes) {
            const double a = scale * Ar[(long)i * ld + j], b = scale * Ai[(long)i * ld + j];
            s += a * a + b * b;
        }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = lanes / 2; w > 0; w /= 2) {
        if (ty < w) red[threadIdx.x] += red[threadIdx.x + w * cw];
        __syncthreads();
    }
    if (ty == 0 && j < ncol) part[(long)blockIdx.x * ncol + j] = red[tx];
}

// out[j] = the sum of the parts of column j = blockIdx.x: by 64 lanes, then across them.
__global__ __launch_bounds__(64) void k_colnorm2_sum(int nblk, int ncol, const double* __restrict__ part,
                                                     double* __restrict__ out) {
    const int j = blockIdx.x;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 64) s += part[(long)b * ncol + j];
    for (int w = 32; w > 0; w /= 2) s += __shfl_xor(s, w);
    if (threadIdx.x == 0) out[j] = s;
}

int norm_blocks(int n) { return (n + kNormRows - 1) / kNormRows; }

}  // namespace

int z_product(bem_ctx* c, int N, const double* Xr, const double* Xi, const double* Br, const double* Bi, double* Or,
              double* Oi) {
    const int M = c->npad;
    const long count = (long)M * N;
    const int S = zmul_splits(c->cus, M, N);
    const size_t bytes = 2 * (size_t)S * count * sizeof(double);
    if (c->part_bytes < bytes) {
        if (c->part) (void)hipFree(c->part);
        c->part = nullptr;
        c->part_bytes = 0;
        if (hipMalloc(&c->part, bytes) != hipSuccess) return bem_fail(c, BEM_ERR_NOMEM, "split-K partial products");
        c->part_bytes = bytes;
    }
    double* P = static_cast<double*>(c->part);
    const int k = kt_mark(c, KS_GEMM64, c->stream);
    // groups of nearly equal width
    const int tiles = N / 16, G = (tiles + kTiles - 1) / kTiles, nt = tiles / G, wide = tiles % G;
    if (wide) zmul_launch(c->stream, nt + 1, M, N, 0, wide, S, c->Zr, c->Zi, Xr, Xi, P);
    zmul_launch(c->stream, nt, M, N, 16 * (nt + 1) * wide, G - wide, S, c->Zr, c->Zi, Xr, Xi, P);
    hipLaunchKernelGGL(k_zmul_sum, dim3((unsigned)((count / 2 + 255) / 256)), dim3(256), 0, c->stream, count, S, P, Br,
                       Bi, Or, Oi);
    kt_close(c, k, 6.0 * (double)M * N * M, 16.0 * ((double)M * M + (double)M * N * (2.0 * S + 2.0)));
    BEM_HIP(c, hipGetLastError());
    return 0;
}

size_t col_norm2_work(int n, int ncol) { return (size_t)norm_blocks(n) * ncol; }

void col_norm2(hipStream_t s, int n, int ncol, const double* Ar, const double* Ai, long ld, double* part, double* out,
               double scale) {
    int cw = 1;
    while (cw < ncol && cw < 64) cw *= 2;
    hipLaunchKernelGGL(k_colnorm2_part, dim3(norm_blocks(n), (ncol + cw - 1) / cw), dim3(256), 0, s, n, ncol, cw, Ar,
                       Ai, ld, scale, part);
    hipLaunchKernelGGL(k_colnorm2_sum, dim3(ncol), dim3(64), 0, s, norm_blocks(n), ncol, (const double*)part, out);
}
