// cmul.h -- FP32 complex products of a tall or small matrix with a block of columns, for
// the solves and the inverses of the diagonal blocks.
//
// C (op)= A B, planar complex FP32 in the 3M form (T1 = Ar Br, T2 = Ai Bi, T3 = (Ar + Ai)
// (Br + Bi); Re = T1 - T2, Im = T3 - T1 - T2), A, B and C row-major.  A workgroup owns a
// tile of 16 rows and 16 NT columns; its four waves take a quarter of k each, straight
// from memory into the matrix cores, one step of 16 k ahead, and are added through LDS
// in wave order.  In a step lane (r, g) holds A[row r][4 g .. 4 g + 3] (one 16-byte load per
// plane) and B[4 g + e][its columns], as 16-, 8- or 4-byte loads: of every 4 (2, 1) tiles
// lane r holds columns 4 r .. 4 r + 3 (2 r, 2 r + 1; r), so that its results are
// adjacent, too.
//
// Bound by load latency for few tiles, by the FP32 matrix cores (153 TFLOP/s) for many:
// K = 1024, 17408 rows: 128 columns 139 us (99 TFLOP/s), 80 columns 109, 16 columns 49;
// 256 rows, K = 256: 4.8 us in a solve.  The same waves side by side on rows instead of
// k leave SIMDs idle at the end (128 columns 182 us); longer steps of 32 or 64 k need
// registers of other waves (142 us).  Two solves at n = 18432, 80 columns: 8.4 ms with
// tiled products that wanted multiples of 32 columns for their fast path, now 6.6.
#pragma once

#include <hip/hip_runtime.h>

#include "gemm.h"

// Rows of the diagonal blocks that the FP32 solves apply as inverses: the padded size is a
// multiple of 256 and of nothing larger.
constexpr int IB = 256;

typedef float v2f __attribute__((ext_vector_type(2)));

// Loads / stores the NT values of one row that lane r owns.
template <int NT>
__device__ __forceinline__ void cmul_load(const float* __restrict__ p, int r, float (&o)[NT]) {
    constexpr int Q = NT / 4, R = NT % 4;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const v4f v = *reinterpret_cast<const v4f*>(p + 64 * q + 4 * r);
#pragma unroll
        for (int i = 0; i < 4; i++) o[4 * q + i] = v[i];
    }
    if constexpr (R >= 2) {
        const v2f v = *reinterpret_cast<const v2f*>(p + 64 * Q + 2 * r);
        o[4 * Q] = v[0];
        o[4 * Q + 1] = v[1];
    }
    if constexpr (R % 2) o[NT - 1] = p[16 * (NT - 1) + r];
}
template <int NT>
__device__ __forceinline__ void cmul_store(float* __restrict__ p, int r, const float (&o)[NT]) {
    constexpr int Q = NT / 4, R = NT % 4;
#pragma unroll
    for (int q = 0; q < Q; q++)
        *reinterpret_cast<v4f*>(p + 64 * q + 4 * r) = v4f{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
    if constexpr (R >= 2) *reinterpret_cast<v2f*>(p + 64 * Q + 2 * r) = v2f{o[4 * Q], o[4 * Q + 1]};
    if constexpr (R % 2) p[16 * (NT - 1) + r] = o[NT - 1];
}

// The workgroup's tile at (m0, n0) over k = [k0, k1) (multiples of 16).  mode 0: C -= A B,
// 1: C = A B, 3: C = -A B.  C may not overlap A or B.  red: 4 x 2 x 16 x 16 NT floats of LDS.
template <int NT>
__device__ __forceinline__ void cmul_tile(int m0, int n0, int k0, int k1, const float* __restrict__ Ar,
                                          const float* __restrict__ Ai, long lda, const float* __restrict__ Br,
                                          const float* __restrict__ Bi, long ldb, float* __restrict__ Cr,
                                          float* __restrict__ Ci, long ldc, int mode, float* red) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ns = (k1 - k0) / 16, first = k0 + 16 * (ns * wave / 4), end = k0 + 16 * (ns * (wave + 1) / 4);
    const float* ar = Ar + (long)(m0 + r) * lda + 4 * g;
    const float* ai = Ai + (long)(m0 + r) * lda + 4 * g;
    const float* br = Br + (long)(4 * g) * ldb + n0;
    const float* bi = Bi + (long)(4 * g) * ldb + n0;
    struct Step {
        v4f a[2];
        float b[2][4][NT];
    } cur, nxt;
    auto load = [&](Step& s, int k) {
        s.a[0] = *reinterpret_cast<const v4f*>(ar + k);
        s.a[1] = *reinterpret_cast<const v4f*>(ai + k);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            cmul_load<NT>(br + (long)(k + e) * ldb, r, s.b[0][e]);
            cmul_load<NT>(bi + (long)(k + e) * ldb, r, s.b[1][e]);
        }
    };
    // the thread's values of C
    const int row = threadIdx.x / 16, c = threadIdx.x % 16;
    const long o = (long)(m0 + row) * ldc + n0;
    float old[2][NT] = {};
    if (mode == 0) {
        cmul_load<NT>(Cr + o, c, old[0]);
        cmul_load<NT>(Ci + o, c, old[1]);
    }
    v4f t1[NT], t2[NT], t3[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) t1[t] = t2[t] = t3[t] = v4f{};
    auto multiply = [&](const Step& s) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float a0 = s.a[0][e], a1 = s.a[1][e], a2 = a0 + a1;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float b0 = s.b[0][e][t], b1 = s.b[1][e][t];
                t1[t] = mfma16x16x4(a0, b0, t1[t]);
                t2[t] = mfma16x16x4(a1, b1, t2[t]);
                t3[t] = mfma16x16x4(a2, b0 + b1, t3[t]);
            }
        }
    };
    if (first < end) {
        load(cur, first);
        int k = first;
        // every load unconditional: the compiler would move others to their use
#pragma unroll 1
        for (; k + 32 <= end; k += 32) {
            load(nxt, k + 16);
            __builtin_amdgcn_sched_barrier(0);
            multiply(cur);
            __builtin_amdgcn_sched_barrier(0);
            load(cur, k + 32 < end ? k + 32 : k);  // (past the end: loaded again, not used)
            __builtin_amdgcn_sched_barrier(0);
            multiply(nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (k < end) multiply(cur);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float re[NT], im[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            re[t] = t1[t][q] - t2[t][q];
            im[t] = t3[t][q] - t1[t][q] - t2[t][q];
        }
        float* w = red + (wave * 32 + 4 * g + q) * 16 * NT;
        cmul_store<NT>(w, r, re);
        cmul_store<NT>(w + 256 * NT, r, im);
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; p++) {
        float v[NT], u[NT];
        cmul_load<NT>(red + (p * 16 + row) * 16 * NT, c, v);
#pragma unroll
        for (int w = 1; w < 4; w++) {
            cmul_load<NT>(red + (w * 32 + p * 16 + row) * 16 * NT, c, u);
#pragma unroll
            for (int t = 0; t < NT; t++) v[t] += u[t];
        }
#pragma unroll
        for (int t = 0; t < NT; t++) v[t] = mode == 0 ? old[p][t] - v[t] : mode == 1 ? v[t] : -v[t];
        cmul_store<NT>((p ? Ci : Cr) + o, c, v);
    }
}

// C (op)= A B on k_cmul, tri 0: all of A, 1: A lower, 2: A upper triangular (its 16 x 16
// diagonal tiles are read whole).  Workgroups b with one value of b % 8 (one XCD) take a
// contiguous run of the order (rows, column groups), so that the column groups reuse the
// rows of A from that XCD's L2.
template <int NT>
__global__ __launch_bounds__(256, 2) void k_cmul(int ntile, int ngrp, int c0, int K, int tri,
                                                 const float* __restrict__ Ar, const float* __restrict__ Ai, long lda,
                                                 const float* __restrict__ Br, const float* __restrict__ Bi, long ldb,
                                                 float* __restrict__ Cr, float* __restrict__ Ci, long ldc, int mode) {
    __shared__ __align__(16) float red[4 * 2 * 16 * 16 * NT];
    const int per = (ntile + 7) / 8, f = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (f >= ntile) return;
    const int m0 = f / ngrp * 16, n0 = c0 + f % ngrp * 16 * NT;
    cmul_tile<NT>(m0, n0, tri == 2 ? m0 : 0, tri == 1 ? m0 + 16 : K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, red);
}
