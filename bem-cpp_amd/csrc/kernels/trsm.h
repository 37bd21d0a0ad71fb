// trsm.h -- triangular solves of a block of right-hand sides by substitution, for
// the FP64 solve phase.
#pragma once

#include <hip/hip_runtime.h>

__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }

// a / b.  In FP32 with b brought to [1/2, 1) by a power of two: the square of a divisor
// below 5e-20 or above 1.8e19 leaves the range (that of a double below 1e-154).
template <typename T>
__device__ __forceinline__ void cdiv(T ar, T ai, T br, T bi, T& qr, T& qi) {
    int e = 0;
    if constexpr (sizeof(T) == 4) {
        e = -__builtin_amdgcn_frexp_expf(fmaxf(fabsf(br), fabsf(bi)));
        br = ldexpf(br, e);
        bi = ldexpf(bi, e);
    }
    const T d = br * br + bi * bi;
    qr = (ar * br + ai * bi) / d;
    qi = (ai * br - ar * bi) / d;
    if constexpr (sizeof(T) == 4) {
        qr = ldexpf(qr, e);
        qi = ldexpf(qi, e);
    }
}

// Value of lane l (uniform) of the wave, broadcast through the scalar unit.
__device__ __forceinline__ double wave_bcast(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Solves T X = B by substitution for one 256 x 256 triangular block T (unit
// lower: forward; non-unit upper: backward) and the columns of B, CW columns
// per block (blockIdx.x; the column count a multiple of CW).  This is the
// backward-stable form of the FP64 solves (no explicit inverse is formed).
//   Thread t keeps row t of X (CW columns) and, slab by slab, its own row of
// T (S columns) in registers; the next slab's row is loaded while the
// current one is used, so the triangle never passes through LDS.  Inside a
// slab the S rows are solved by the one wave that holds them: the finished
// row of each step goes to every lane of the wave through the scalar unit
// (readlane), with no LDS round trip and no barrier.  Then the slab's rows go
// to LDS, one barrier publishes them (the LDS rows are double buffered by slab
// parity, so that is the only barrier of a slab) and every row outside the
// slab subtracts their contribution.  The upper case scales the pivot row by
// the reciprocal of its diagonal entry, formed by every lane of the slab for
// its own row before the steps (off the critical path of the steps).  B and X
// may be the same array (each block reads its columns before it writes them).
template <typename T, int CW, int S, bool LOWER>
__global__ __launch_bounds__(256) void k_trsm_rhs(const T* __restrict__ Tr, const T* __restrict__ Ti, long ldt,
                                                  const T* Br, const T* Bi, long ldb, T* Xr, T* Xi, long ldx) {
    constexpr int R = 256, NS = R / S;
    static_assert(S <= 64 && 64 % S == 0, "a slab lies inside one wave");
    __shared__ T pr[2][S][CW], pi[2][S][CW];
    const int t = threadIdx.x, c0 = blockIdx.x * CW;
    const T* rowr = Tr + (long)t * ldt;
    const T* rowi = Ti + (long)t * ldt;
    T xr[CW], xi[CW];
#pragma unroll
    for (int c = 0; c < CW; c++) {
        xr[c] = Br[(long)t * ldb + c0 + c];
        xi[c] = Bi[(long)t * ldb + c0 + c];
    }
    auto slab0 = [](int sI) { return LOWER ? sI * S : R - S * (sI + 1); };
    T ar[S], ai[S], nr[S], ni[S];
#pragma unroll
    for (int q = 0; q < S; q++) {
        ar[q] = rowr[slab0(0) + q];
        ai[q] = rowi[slab0(0) + q];
    }
#pragma unroll 1
    for (int sI = 0; sI < NS; sI++) {
        const int s = slab0(sI), buf = sI & 1;
        if (sI + 1 < NS) {
            const int sn = slab0(sI + 1);
#pragma unroll
            for (int q = 0; q < S; q++) {
                nr[q] = rowr[sn + q];
                ni[q] = rowi[sn + q];
            }
        }
        if ((t >> 6) == (s >> 6)) {  // the wave that holds rows s .. s + S - 1
            T rr = T(1), ri = T(0);   // upper: 1 / T[t][t] for the rows of the slab
            if (!LOWER) {
                T dr = T(1), di = T(0);
#pragma unroll
                for (int q = 0; q < S; q++)
                    if (t == s + q) {
                        dr = ar[q];
                        di = ai[q];
                    }
                const T inv = T(1) / (dr * dr + di * di);
                rr = dr * inv;
                ri = -di * inv;
            }
#pragma unroll
            for (int k = 0; k < S; k++) {
                const int q = LOWER ? k : S - 1 - k, l = s + q;
                if (!LOWER && t == l) {
#pragma unroll
                    for (int c = 0; c < CW; c++) {
                        const T a = xr[c], b = xi[c];
                        xr[c] = a * rr - b * ri;
                        xi[c] = a * ri + b * rr;
                    }
                }
                T ur[CW], ui[CW];
#pragma unroll
                for (int c = 0; c < CW; c++) {
                    ur[c] = wave_bcast(xr[c], l & 63);
                    ui[c] = wave_bcast(xi[c], l & 63);
                }
                if (LOWER ? (t > l && t < s + S) : (t >= s && t < l)) {
                    const T a = ar[q], b = ai[q];
                    const T na = -a, nb = -b;
#pragma unroll
                    for (int c = 0; c < CW; c++) {
                        xr[c] = fmadd(na, ur[c], xr[c]);
                        xr[c] = fmadd(b, ui[c], xr[c]);
                        xi[c] = fmadd(na, ui[c], xi[c]);
                        xi[c] = fmadd(nb, ur[c], xi[c]);
                    }
                }
            }
            if (t >= s && t < s + S) {
#pragma unroll
                for (int c = 0; c < CW; c++) {
                    pr[buf][t - s][c] = xr[c];
                    pi[buf][t - s][c] = xi[c];
                }
            }
        }
        __syncthreads();  // pr[buf] holds the slab's S solved rows
        if (LOWER ? (t >= s + S) : (t < s)) {
#pragma unroll
            for (int q = 0; q < S; q++) {
                const T a = ar[q], b = ai[q];
                const T na = -a, nb = -b;
#pragma unroll
                for (int c = 0; c < CW; c++) {
                    const T ur = pr[buf][q][c], ui = pi[buf][q][c];
                    xr[c] = fmadd(na, ur, xr[c]);
                    xr[c] = fmadd(b, ui, xr[c]);
                    xi[c] = fmadd(na, ui, xi[c]);
                    xi[c] = fmadd(nb, ur, xi[c]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < S; q++) {
            ar[q] = nr[q];
            ai[q] = ni[q];
        }
    }
#pragma unroll
    for (int c = 0; c < CW; c++) {
        Xr[(long)t * ldx + c0 + c] = xr[c];
        Xi[(long)t * ldx + c0 + c] = xi[c];
    }
}

// T X = B for the 256 x 256 triangle at (Tr, Ti) and ncols columns (a
// multiple of 8) on stream s.  Up to 512 right-hand sides: 2 columns and 16-row
// slabs per block, so the latency-bound chain of steps is as short as it gets
// (lower / upper 48 / 61 us at 128 columns); more: 8 columns and 8-row slabs, where
// throughput counts (274 / 322 us at 9216).
template <typename T>
inline void trsm_rhs(hipStream_t s, bool lower, const T* Tr, const T* Ti, long ldt, const T* Br, const T* Bi,
                     long ldb, T* Xr, T* Xi, long ldx, int ncols) {
    if (ncols <= 512) {
        const dim3 grid((unsigned)(ncols / 2));
        if (lower)
            hipLaunchKernelGGL((k_trsm_rhs<T, 2, 16, true>), grid, dim3(256), 0, s, Tr, Ti, ldt, Br, Bi, ldb, Xr, Xi,
                               ldx);
        else
            hipLaunchKernelGGL((k_trsm_rhs<T, 2, 16, false>), grid, dim3(256), 0, s, Tr, Ti, ldt, Br, Bi, ldb, Xr, Xi,
                               ldx);
    } else {
        const dim3 grid((unsigned)(ncols / 8));
        if (lower)
            hipLaunchKernelGGL((k_trsm_rhs<T, 8, 8, true>), grid, dim3(256), 0, s, Tr, Ti, ldt, Br, Bi, ldb, Xr, Xi,
                               ldx);
        else
            hipLaunchKernelGGL((k_trsm_rhs<T, 8, 8, false>), grid, dim3(256), 0, s, Tr, Ti, ldt, Br, Bi, ldb, Xr, Xi,
                               ldx);
    }
}
