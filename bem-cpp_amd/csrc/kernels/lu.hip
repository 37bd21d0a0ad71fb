// lu.hip -- blocked complex LU with row pivoting on gfx950, FP64 and FP32.
//
// Replaces cuSOLVER Zgetrf (solver.cu:7-48, 87-113).  The reference factors
// the column-major view of its row-major Z (i.e. Z^T) and solves with OP_T;
// this library factors P Z = L U directly on the row-major matrix (rows are
// contiguous, so row interchanges are contiguous copies) and solves Z X = B.
// The pivots differ from cuSOLVER's; the solution does not.
//
// Right-looking two-level blocking on the padded matrix (npad = 256 k):
//   outer panel of NB = 256 columns, factored in 8 inner steps of PB = 32, two
//   launches each:
//     1. pivot selection for the 32 columns over all remaining rows by a
//        tournament (communication-avoiding "TSLU": Grigori, Demmel & Xiang,
//        SIAM J. Matrix Anal. Appl. 32 (2011)): sets of 256 rows (512 where that
//        saves a level) each choose 32 candidate rows by partial pivoting in
//        registers; the last block of every group of sets to finish (integer
//        arrival counter) merges the group's candidates, up to the root, whose
//        pivot order becomes LAPACK-style swaps ipiv[j0 .. j0+31] and the
//        factored 32 x 32 diagonal block.  No block ever waits.
//     2. (k_step) the swaps in the panel, L21 = A21 U11^{-1}, U12 = L11^{-1} A12
//        and the rank-32 update of the next 32 columns on the matrix cores; the
//        update of the panel's other columns rides in the next tournament's
//        launch
//   then the panel's net row interchanges in the other columns, U12 = L11^{-1} A12 by
//   blocked substitution (k_u12_strip) and the rank-256 trailing update A22 -= L21 U12
//   as matrix-core GEMMs (gemm_nt.h in FP32, 3M form; gemm.h).  The inverses of all
//   256 x 256 L and U diagonal blocks are formed after the last panel for the
//   GEMM-based multi-RHS solves (FP32 only).
#include <cstdlib>
#include <vector>

#include "../bem_internal.h"
#include "cmul.h"
#include "gemm.h"
#include "gemm_nt.h"
#include "trsm.h"

namespace {

constexpr int NB = 256;  // outer panel width = solve block size
constexpr int PB = 32;   // inner panel width (pivot block)

template <typename T>
__device__ __forceinline__ T mag2(T r, T i) {
    return fmadd(r, r, i * i);
}

// 16-byte vector type of T (4 floats or 2 doubles).
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
    using type = float4;
};
template <>
struct Vec16<double> {
    using type = double2;
};

// The same as a native vector (arrays of it stay in registers).
template <typename T>
using Nat16 = T __attribute__((ext_vector_type(16 / sizeof(T))));

// 1 / d for the pivot scaling: the hardware reciprocal in FP32 (1 ulp), an
// IEEE division in FP64.
__device__ __forceinline__ float recip(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double recip(double d) { return 1.0 / d; }

// Maximum over the wave, in a scalar register (DPP within rows of 16, then
// across the rows).
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned max_dpp(unsigned v) {
    return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ unsigned wave_max(unsigned v) {
    v = max_dpp<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v = max_dpp<0x112, 0xf>(v);
    v = max_dpp<0x114, 0xf>(v);
    v = max_dpp<0x118, 0xf>(v);
    v = max_dpp<0x142, 0xa>(v);  // row_bcast 15, 31
    v = max_dpp<0x143, 0xc>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Order-preserving 32-bit keys of |r + i i|; 0 is "no candidate".  The row is found by a
// ballot: with the lane in the key's low bits instead (2N = 3840 10.14 ms, now 10.23) 17 (14)
// mantissa bits are left, and a zero ties with a small entry.
// FP64: sign (that of a NaN masked), exponent and 20 mantissa bits of |x|^2; rows closer
// than that tie.
// FP32: all of |2^e x|^2 with the exponent counted from 2^-253, so that the keys of e = 0,
// 63 (for squares below the range) and -64 (above) compare with each other.
__device__ __forceinline__ unsigned mag_key(double r, double i) {
    return ((unsigned)((unsigned long long)__double_as_longlong(mag2(r, i)) >> 32) & 0x7fffffffu) + 1u;
}
template <int E>
__device__ __forceinline__ unsigned mag_key(float r, float i) {
    if constexpr (E != 0) {
        r = ldexpf(r, E);
        i = ldexpf(i, E);
    }
    return (__float_as_uint(mag2(r, i)) & 0x7fffffffu) + ((126u - 2 * E) << 23) + 1u;
}

// FP32 values whose squares and their reciprocals are normal numbers: those within these
// bounds.  The tournament computes with the squares; where a pivot turns out to lie outside,
// the factorisation is done again with WIDE set, which scales such values by powers of two
// first (in every tournament that costs 7 % at 2N = 3840, 10.2 -> 10.8 ms).
constexpr float kSquareMin = 0x1p-62f, kSquareMax = 0x1p62f;

// The largest key of the wave's open rows into wk, and the lane that has it (ties: the
// lowest; a wave without open rows: lane 0, key 0).
template <bool WIDE>
__device__ __forceinline__ int best_lane(bool open, double r, double i, unsigned& wk) {
    const unsigned key = open ? mag_key(r, i) : 0u;
    wk = wave_max(key);
    return __ffsll((long long)__ballot(key == wk)) - 1;
}
template <bool WIDE>
__device__ __forceinline__ int best_lane(bool open, float r, float i, unsigned& wk) {
    constexpr unsigned kLow = ((27u + 126u) << 23) + 1u, kHigh = ((254u + 126u) << 23) + 1u;  // 2^-100, 2^127
    unsigned key = open ? mag_key<0>(r, i) : 0u;
    wk = wave_max(key);
    if constexpr (WIDE) {
        if (wk - 1u < kLow - 1u) {
            key = open ? mag_key<63>(r, i) : 0u;
            wk = wave_max(key);
        } else if (wk >= kHigh) {
            key = open ? mag_key<-64>(r, i) : 0u;
            wk = wave_max(key);
        }
    }
    return __ffsll((long long)__ballot(key == wk)) - 1;
}

// l = x / u by the reciprocal of u (the rows scale by it, as zgetf2 does), 0 for u = 0;
// returns whether u is not 0.  WIDE: x and u by the power of two that brings u to [1/2, 1)
// first; otherwise rounded the same.
template <bool WIDE, typename T>
__device__ __forceinline__ bool scale_row(T xr, T xi, T ur, T ui, T& lr, T& li) {
    if constexpr (WIDE) {
        const int e = -__builtin_amdgcn_frexp_expf(fmaxf(fabsf(ur), fabsf(ui)));
        xr = ldexpf(xr, e);
        xi = ldexpf(xi, e);
        ur = ldexpf(ur, e);
        ui = ldexpf(ui, e);
    }
    const T d = mag2(ur, ui);
    const T inv = d > T(0) ? recip(d) : T(0);
    const T qr = ur * inv, qi = -ui * inv;
    lr = fmadd(xr, qr, -(xi * qi));
    li = fmadd(xr, qi, xi * qr);
    return d > T(0);
}

// v of lane l (l the same for the whole wave) as a scalar.
__device__ __forceinline__ float from_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double from_lane(double v, int l) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)u, l), hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

constexpr int EW = 4;        // columns of an elimination window
constexpr int NG = PB / EW;  // windows of a row
template <typename T>
using Grp = T __attribute__((ext_vector_type(EW)));  // a row's entries of a window

template <typename T>
__device__ __forceinline__ void load_groups(const T* __restrict__ p, Grp<T> (&x)[NG]) {
    constexpr int E = 16 / sizeof(T);
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int c = 0; c < EW; c += E) {
            const Nat16<T> a = *reinterpret_cast<const Nat16<T>*>(p + g * EW + c);
#pragma unroll
            for (int e = 0; e < E; e++) x[g][c + e] = a[e];
        }
}
template <typename T>
__device__ __forceinline__ void store_group(T* p, const Grp<T>& x, int from = 0) {
    constexpr int E = 16 / sizeof(T);
#pragma unroll
    for (int c = 0; c < EW; c += E)
        if (c + E - 1 >= from) {
            Nat16<T> a;
#pragma unroll
            for (int e = 0; e < E; e++) a[e] = x[c + e];
            *reinterpret_cast<Nat16<T>*>(p + c) = a;
        }
}

// Exchange area of the register-resident elimination (W waves).
template <typename T, int W>
struct ElimLds {
    alignas(16) T win[2][W][2][EW];  // [step parity][wave][plane]: the wave's best row, window columns
    alignas(16) unsigned key[2][W];  // its key
    alignas(16) T raw[EW][2][PB];    // the window's pivot rows before the window's updates right of it
    alignas(16) T u[sizeof(T) == 8 ? W : 1][EW][2][PB];  // FP64: the same as rows of U, one copy per wave
    alignas(16) int oid[PB];         // chosen rows in pivot order
    int osrc[PB];
    alignas(16) int sw[2][PB];       // root_swaps
    int last;
    int zmin;  // first zero pivot of the root (1-based)
};

// Group G of the row takes the window's EW pivots and moves to G - 1, from G = 1 on:
// with the window at the end, the row has rotated by one group then.  Groups beyond
// ng only move.  (vr, vi): lane l's values of the window's pivot rows in column EW + l.
// Per element and pivot the four multiply-adds are those of the column-by-column
// elimination, in its order.
// FP32: v_mfma_f32_4x4x1 with one block's A operand broadcast to all 16 is a rank-1
// update of four columns with a row per lane, and that block is group G's lanes of vr
// and vi as they lie.
template <int G>
__device__ __forceinline__ void window_update(Grp<float> (&xr)[NG], Grp<float> (&xi)[NG], const float (&lr)[EW],
                                              const float (&li)[EW], const float (&vr)[EW], const float (&vi)[EW],
                                              int ng) {
    if constexpr (G < NG) {
        if (G <= ng) {
            v4f a = xr[G], b = xi[G];
#pragma unroll
            for (int q = 0; q < EW; q++) {
                const float nl = -lr[q];
                a = __builtin_amdgcn_mfma_f32_4x4x1f32(vr[q], nl, a, 4, G - 1, 0);
                b = __builtin_amdgcn_mfma_f32_4x4x1f32(vi[q], nl, b, 4, G - 1, 0);
                a = __builtin_amdgcn_mfma_f32_4x4x1f32(vi[q], li[q], a, 4, G - 1, 0);
                b = __builtin_amdgcn_mfma_f32_4x4x1f32(-vr[q], li[q], b, 4, G - 1, 0);
            }
            xr[G - 1] = a;
            xi[G - 1] = b;
        } else {
            xr[G - 1] = xr[G];
            xi[G - 1] = xi[G];
        }
        window_update<G + 1>(xr, xi, lr, li, vr, vi, ng);
    }
}
// FP64 has no such form: the values come from LDS (u, the wave's copy), two columns
// read ahead; the scheduling barriers keep more from being hoisted, which would not
// fit in the registers.
struct WindowCols {
    v2d r[EW], i[EW];
};
__device__ __forceinline__ void window_read(const double (*u)[2][PB], int c, WindowCols& w) {
#pragma unroll
    for (int q = 0; q < EW; q++) {
        w.r[q] = *reinterpret_cast<const v2d*>(&u[q][0][c]);
        w.i[q] = *reinterpret_cast<const v2d*>(&u[q][1][c]);
    }
}
template <int G>
__device__ __forceinline__ void window_update(Grp<double> (&xr)[NG], Grp<double> (&xi)[NG], const double (&lr)[EW],
                                              const double (&li)[EW], const double (*u)[2][PB], WindowCols& cur,
                                              int ng) {
    if constexpr (G < NG) {
        if (G <= ng) {
            WindowCols nxt;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 0)
                    window_read(u, G * EW + 2, nxt);
                else if (G + 1 < NG)
                    window_read(u, (G + 1) * EW, cur);  // (unused beyond group ng)
                __builtin_amdgcn_sched_barrier(0);
                const WindowCols now = h ? nxt : cur;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    double a = xr[G][2 * h + e], b = xi[G][2 * h + e];
#pragma unroll
                    for (int q = 0; q < EW; q++) {
                        a = fmadd(li[q], double(now.i[q][e]), fmadd(-lr[q], double(now.r[q][e]), a));
                        b = fmadd(-li[q], double(now.r[q][e]), fmadd(-lr[q], double(now.i[q][e]), b));
                    }
                    xr[G - 1][2 * h + e] = a;
                    xi[G - 1][2 * h + e] = b;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            xr[G - 1] = xr[G];
            xi[G - 1] = xi[G];
        }
        window_update<G + 1>(xr, xi, lr, li, u, cur, ng);
    }
}

// Partial pivoting over the block's rows, one per thread in registers (rows at
// nrows and beyond take no part; nrows >= PB), with implicit row interchanges: rows
// stay with their thread and a chosen row is only marked.  Step jc: the largest
// |x_jc|^2 among the rows not chosen yet (by mag_key; ties: lowest wave, lane)
// becomes pivot jc, and the remaining rows are eliminated (multiplier stored in
// x_jc).  An all-zero column chooses the lowest open row and eliminates nothing.
// Afterwards mine is the pivot number of the thread's row (the thread holds that row
// of L11 \ U11), -1 for rows not chosen; oid/osrc list the chosen rows in pivot order.
//
// The chain of 32 steps is bound by the exchange between the waves and by
// instruction fetch, so:
// - a step has one exchange: every wave's best row goes to LDS with its key
//   before one barrier, but only the columns of the current window of EW, which
//   is also all that is updated within the window.  The columns right of it take
//   the window's EW pivots at once: their rows go to LDS, each wave solves them
//   against the window's unit triangle, one column per lane, and updates its
//   rows (window_update).
// - the windows are a loop, not unrolled code: the row registers rotate by a
//   group after each window, so the window is always group 0 and the eighth
//   rotation brings every column home.  (Unrolled, the 32 steps are 40 KB of code.)
// One level of 256 rows takes 22.1 us (FP64 31.3), of 512 31.0, alone; with the
// products of window_update as multiply-adds on operands from LDS and the rows rotated
// by copies it took 24.5 (31.5), and 35.8 with two rows per thread of 4 waves.
template <typename T, int W, bool WIDE>
__device__ __forceinline__ void elim_rows(ElimLds<T, W>& L, Grp<T> (&xr)[NG], Grp<T> (&xi)[NG], int id, int src,
                                          int nrows, int& mine) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool valid = t < nrows;
    // Of 8 waves, one without rows only keeps the barriers (and its key, 0): 256 rows
    // 23.4 us instead of 27.0.  (With 4 waves the branches cost full sets 1.3 us.)
    const bool active = W == 4 || __builtin_amdgcn_readfirstlane(wave) * 64 < nrows;
    if (!active && lane < 2) L.key[lane][wave] = 0u;
    mine = -1;
#pragma unroll 1
    for (int w = 0; w < NG; w++) {
        const int s = w * EW, ng = NG - 1 - w;  // first column; groups right of the window
        T lr[EW], li[EW];                       // the window's multipliers (0: row not eliminated)
        Grp<T> hr = xr[0], hi = xi[0];          // the window
#pragma unroll
        for (int q = 0; q < EW; q++) {
            const int par = q & 1;
            int wl = 0;  // the wave's best lane (ties: the lowest)
            if (active) {
                unsigned wk;
                wl = best_lane<WIDE>(valid && mine < 0, T(hr[q]), T(hi[q]), wk);
                if (lane == wl) {
                    store_group<T>(L.win[par][wave][0], hr, q);
                    store_group<T>(L.win[par][wave][1], hi, q);
                    L.key[par][wave] = wk;
                }
            }
            __syncthreads();
            if (!active) continue;
            // lane l reads wave l % W's entry; the maximum over W lanes then
            // names the wave whose window the scalar registers take (one LDS
            // latency instead of the keys' and then the window's)
            const unsigned kw = L.key[par][lane & (W - 1)];
            T cr[EW], ci[EW];
            constexpr int E = 16 / sizeof(T);
#pragma unroll
            for (int c = 0; c < EW; c += E)
                if (c + E - 1 >= q) {
                    const Nat16<T> a = *reinterpret_cast<const Nat16<T>*>(&L.win[par][lane & (W - 1)][0][c]);
                    const Nat16<T> d = *reinterpret_cast<const Nat16<T>*>(&L.win[par][lane & (W - 1)][1][c]);
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        cr[c + e] = a[e];
                        ci[c + e] = d[e];
                    }
                }
            unsigned best = max_dpp<0xb1, 0xf>(kw);  // quad_perm [1, 0, 3, 2], then [2, 3, 0, 1]
            best = max_dpp<0x4e, 0xf>(best);
            if constexpr (W == 8) best = max_dpp<0x141, 0xf>(best);  // row_half_mirror
            const int wv = __ffsll((long long)__ballot(kw == best)) - 1;  // ties: the lower wave
            T ur[EW], ui[EW];
#pragma unroll
            for (int c = q; c < EW; c++) {
                ur[c] = from_lane(cr[c], wv);
                ui[c] = from_lane(ci[c], wv);
            }
            const bool won = wave == wv && lane == wl;
            T a, b;
            const bool nonzero = scale_row<WIDE>(T(hr[q]), T(hi[q]), ur[q], ui[q], a, b);
            if (won) mine = s + q;
            // branch-free update: rows that are not eliminated use multiplier 0
            const bool upd = valid && mine < 0 && nonzero;
            lr[q] = upd ? a : T(0);
            li[q] = upd ? b : T(0);
            hr[q] = upd ? a : T(hr[q]);
            hi[q] = upd ? b : T(hi[q]);
            const T nlr = -lr[q], nli = -li[q];
#pragma unroll
            for (int c = q + 1; c < EW; c++) {
                hr[c] = fmadd(li[q], ui[c], fmadd(nlr, ur[c], T(hr[c])));
                hi[c] = fmadd(nli, ur[c], fmadd(nlr, ui[c], T(hi[c])));
            }
        }
        // the window's pivot rows (window columns final, the others without the
        // window's updates); the last window has no others, the rows only rotate
        if (ng > 0 && mine >= s) {
            T *pr = L.raw[mine - s][0], *pi = L.raw[mine - s][1];
            store_group<T>(pr, hr);
            store_group<T>(pi, hi);
#pragma unroll
            for (int g = 1; g < NG; g++)
                if (g <= ng) {
                    store_group<T>(pr + g * EW, xr[g]);
                    store_group<T>(pi + g * EW, xi[g]);
                }
        }
        __syncthreads();
        if (!active) continue;
        // lane l solves column EW + l against the window's unit triangle
        // (beyond the groups left, some value)
        const int cl = EW + min(lane, PB - EW - 1);
        T vr[EW], vi[EW];
#pragma unroll
        for (int q = 0; q < EW; q++) {
            vr[q] = L.raw[q][0][cl];
            vi[q] = L.raw[q][1][cl];
        }
#pragma unroll
        for (int q = 0; q < EW; q++)
#pragma unroll
            for (int k = 0; k < q; k++) {
                const T mr = L.raw[q][0][k], mi = L.raw[q][1][k];
                vr[q] = fmadd(-mr, vr[k], vr[q]);
                vr[q] = fmadd(mi, vi[k], vr[q]);
                vi[q] = fmadd(-mr, vi[k], vi[q]);
                vi[q] = fmadd(-mi, vr[k], vi[q]);
            }
        if constexpr (sizeof(T) == 4) {
            window_update<1>(xr, xi, lr, li, vr, vi, ng);
        } else {
            if (lane < ng * EW) {
#pragma unroll
                for (int q = 0; q < EW; q++) {
                    L.u[wave][q][0][EW + lane] = vr[q];
                    L.u[wave][q][1][EW + lane] = vi[q];
                }
            }
            __builtin_amdgcn_wave_barrier();  // the wave's own copy: LDS operations of a wave stay in order
            WindowCols cur;
            window_read(L.u[wave], EW, cur);
            window_update<1>(xr, xi, lr, li, L.u[wave], cur, ng);
        }
        xr[NG - 1] = hr;
        xi[NG - 1] = hi;
    }
    if (mine >= 0) {
        L.oid[mine] = id;
        L.osrc[mine] = src;
    }
    __syncthreads();
}

// Root of the tournament, one wave: pivot order -> LAPACK-style swaps
// ipiv[j0 .. j0+31], and their net effect on the touched rows as a list of
// (destination, source) row pairs: pl[0] = count, pl[1 + 2k] = destination,
// pl[2 + 2k] = source (at most 2 PB pairs).
// Step c swaps row j0 + c with the row y_c where the c-th chosen row is by
// then.  A row moves only when its slot is swapped: chosen row o_c stays put
// unless it started in a slot k < c, whose content went to y_k, and so on, so y_c
// is the end of the chain v <- o_{slot of v} while v is in a slot below c.  The
// content of slot c at step c is the row j0 + c unless an earlier step put its
// own content there; the last such step's content, and so on (cont below).
// Row j0 + c ends as o_c, and a row y outside the slots as the content of the
// last step that swaps with it.  All lanes follow their chains side by side
// (the 32 swaps one after the other took 13 500 cycles, 5.5 us of each
// tournament).
__device__ void root_swaps(const int* __restrict__ oid, int* __restrict__ y, int* __restrict__ lastw, int j0,
                           int* __restrict__ ipiv, int* __restrict__ pl) {
    const int lane = threadIdx.x, c = lane & (PB - 1);  // both halves of the wave hold step c
    const int o = oid[c];
    int v = o;
    while (v - j0 < c && v >= j0) v = oid[v - j0];
    if (lane < PB) {
        y[c] = v;
        ipiv[j0 + c] = v;
    }
    __builtin_amdgcn_wave_barrier();
    int lw = -1;        // the last step below c that puts its content into slot c
    bool final = true;  // no later step swaps with the same row
#pragma unroll
    for (int k = 0; k < PB; k++) {
        const int yk = y[k];
        if (k < c && yk == j0 + c) lw = k;
        if (k > c && yk == v) final = false;
    }
    if (lane < PB) lastw[c] = lw;
    __builtin_amdgcn_wave_barrier();
    int cont = c;
    for (int k = lw; k >= 0; k = lastw[k]) cont = k;
    // lanes below PB: the slots; the others: the rows outside them
    const int dst = lane < PB ? j0 + c : v, from = lane < PB ? o : j0 + cont;
    const bool moved = lane < PB ? dst != from : v >= j0 + PB && final;
    const unsigned long long mm = __ballot(moved);
    const int k = __popcll(mm & ((1ull << lane) - 1ull));
    if (moved) {
        pl[1 + 2 * k] = dst;
        pl[2 + 2 * k] = from;
    }
    if (lane == 0) pl[0] = __popcll(mm);
}

// What the columns of the panel beyond the next 32 still need from the step at
// columns jp: the rank-32 update of the columns [c0, c0 + ncol), rows from jp +
// 32 on (16 x 16 tiles, one per wave), and U12 of the next 32 columns put
// in place (one workgroup).  It rides in the launch of the next tournament,
// whose few workgroups leave the device idle, instead of on a stream of its own
// with an event each way.
struct FarUpdate {
    int jp, c0, ncol, blocks;  // blocks: workgroups of the launch that do this
};

// One 16 x 16 tile of C -= L21 U12 per wave with K = 32, operands straight from
// memory to the matrix cores, every load issued before the first product.
template <typename T, int W>
__device__ __forceinline__ void far_update(T* __restrict__ Ar, T* __restrict__ Ai, long ld, int n, FarUpdate f,
                                           int block, const T* __restrict__ Ur, const T* __restrict__ Ui) {
    if (block == f.blocks - 1) {
        for (int e = threadIdx.x; e < PB * PB; e += 64 * W) {
            const long o = (long)(f.jp + e / PB) * ld + f.jp + PB + e % PB;
            Ar[o] = Ur[e];
            Ai[o] = Ui[e];
        }
        return;
    }
    const int i0 = f.jp + PB, nct = f.ncol / 16, ntiles = (n - i0) / 16 * nct;
    const int tile = block * W + (threadIdx.x >> 6);
    if (tile >= ntiles) return;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int m0 = i0 + tile / nct * 16, n0 = f.c0 + tile % nct * 16;
    T a0[2][4], a1[2][4], b0[2][4], b1[2][4];
    const long oa = (long)(m0 + r) * ld + f.jp + 4 * g;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        load_row4<T>(Ar + oa + 16 * q, a0[q]);
        load_row4<T>(Ai + oa + 16 * q, a1[q]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const long ob = (long)(f.jp + 16 * q + 4 * g + e) * ld + n0 + r;
            b0[q][e] = Ar[ob];
            b1[q][e] = Ai[ob];
        }
    }
    if constexpr (sizeof(T) == 4) {
        const long oc = (long)(m0 + r) * ld + n0 + 4 * g;
        const v4f cr = *reinterpret_cast<const v4f*>(Ar + oc), ci = *reinterpret_cast<const v4f*>(Ai + oc);
        __builtin_amdgcn_sched_barrier(0);
        v4f t1 = v4f{0.f, 0.f, 0.f, 0.f}, t2 = t1, t3 = t1;
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                t1 = mfma16x16x4(b0[q][e], a0[q][e], t1);
                t2 = mfma16x16x4(b1[q][e], a1[q][e], t2);
                t3 = mfma16x16x4(b0[q][e] + b1[q][e], a0[q][e] + a1[q][e], t3);
            }
        *reinterpret_cast<v4f*>(Ar + oc) = cr - (t1 - t2);
        *reinterpret_cast<v4f*>(Ai + oc) = ci - (t3 - t1 - t2);
    } else {
        const long oc = (long)(m0 + g) * ld + n0 + r;
        v4d cr, ci, re{}, im{};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            cr[q] = Ar[oc + 4 * q * ld];
            ci[q] = Ai[oc + 4 * q * ld];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                re = mfma16x16x4(a0[q][e], b0[q][e], re);
                re = mfma16x16x4(a1[q][e], -b1[q][e], re);
                im = mfma16x16x4(a0[q][e], b1[q][e], im);
                im = mfma16x16x4(a1[q][e], b0[q][e], im);
            }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            Ar[oc + 4 * q * ld] = cr[q] - re[q];
            Ai[oc + 4 * q * ld] = ci[q] - im[q];
        }
    }
}

// ---------------------------------------------------------------------------
// Pivot tournament for columns j0..j0+31 over rows j0..n-1, one launch; row i
// of the columns at S + i lds.  Sets of CH = 64 W rows (one per thread) choose 32
// candidates each, groups of G = CH / 32 sets merge.
// Candidate sets of level L live at set index off[L] + i; a set is 32 ids and
// the 32 x 32 original values per plane.  cnt: one arrival counter per group
// per level (zero on entry; reset by the merging block).  The root writes
// ipiv, the row-pair list pl, the factored diagonal block d11 (32 x 32 per
// plane), the first zero pivot into *info and whether a pivot asks for WIDE into
// info[1].  The last f.blocks workgroups do
// the previous step's far update instead (A, U; other columns than S's).
// ---------------------------------------------------------------------------
template <typename T, int W, bool WIDE = false>
__global__ __launch_bounds__(64 * W, sizeof(T) == 4 ? 2 : 1) void k_tslu(const T* __restrict__ Sr, const T* __restrict__ Si, long lds, int j0,
                                              int n, int* __restrict__ cid, T* __restrict__ cvr, T* __restrict__ cvi,
                                              int* __restrict__ cnt, int* __restrict__ ipiv, int* __restrict__ pl,
                                              T* __restrict__ d11r, T* __restrict__ d11i, int* __restrict__ info,
                                              T* __restrict__ Ar, T* __restrict__ Ai, long ld, FarUpdate f,
                                              const T* __restrict__ Ur, const T* __restrict__ Ui) {
    __builtin_amdgcn_s_setprio(3);  // latency-bound: win issue slots over co-resident GEMM waves
    constexpr int CH = 64 * W, G = CH / PB;
    if (blockIdx.x >= gridDim.x - f.blocks) {
        far_update<T, W>(Ar, Ai, ld, n, f, blockIdx.x - (gridDim.x - f.blocks), Ur, Ui);
        return;
    }
    __shared__ ElimLds<T, W> L;
    const int t = threadIdx.x;
    // level 0: rows j0 + b*CH .. (n - j0 is a multiple of PB, so every set is full)
    const int r0 = j0 + blockIdx.x * CH;
    int nrows = min(CH, n - r0);
    Grp<T> xr[NG], xi[NG];
    int id = r0 + t, src = r0 + t, mine;
    if (t < nrows) {
        load_groups(Sr + (long)(r0 + t) * lds, xr);
        load_groups(Si + (long)(r0 + t) * lds, xi);
    }
    int level_sets = (n - j0 + CH - 1) / CH;  // sets at this level
    int set = blockIdx.x, off = 0, cnt_off = 0;
    bool from_matrix = true;
    for (;;) {
        elim_rows<T, W, WIDE>(L, xr, xi, id, src, nrows, mine);
        if (level_sets <= 1) break;
        // candidate set = original values of the chosen rows
        for (int e = t; e < PB * PB; e += 64 * W) {
            const int r = e / PB, c = e % PB;
            const long o = ((long)(off + set) * PB + r) * PB + c;
            if (from_matrix) {
                const long g = (long)L.osrc[r] * lds + c;
                cvr[o] = Sr[g];
                cvi[o] = Si[g];
            } else {
                const long g = (long)L.osrc[r] * PB + c;
                cvr[o] = cvr[g];
                cvi[o] = cvi[g];
            }
        }
        if (t < PB) cid[(off + set) * PB + t] = L.oid[t];
        // arrive at the group counter; the last arrival merges the group
        const int grp = set / G;
        const int gsize = min(G, level_sets - grp * G);
        __threadfence();
        __syncthreads();
        if (t == 0) {
            const int prev = atomicAdd(&cnt[cnt_off + grp], 1);
            L.last = prev == gsize - 1;
            if (L.last) cnt[cnt_off + grp] = 0;  // ready for the next launch
        }
        __syncthreads();
        if (!L.last) return;
        __threadfence();
        const int s0 = off + grp * G;
        nrows = gsize * PB;
        id = -1;
        src = s0 * PB + t;
        if (t < nrows) {
            load_groups(cvr + ((long)s0 * PB + t) * PB, xr);
            load_groups(cvi + ((long)s0 * PB + t) * PB, xi);
            id = cid[s0 * PB + t];
        }
        from_matrix = false;
        cnt_off += (level_sets + G - 1) / G;
        off += level_sets;
        set = grp;
        level_sets = (level_sets + G - 1) / G;
    }
    // root: the factored diagonal block, swaps, row-pair list, zero pivot
    if (t == 0) L.zmin = 0x7fffffff;
    __syncthreads();
    if (mine >= 0) {
        T dr = T(0), di = T(0);
#pragma unroll
        for (int g = 0; g < NG; g++) {
            store_group<T>(d11r + mine * PB + g * EW, xr[g]);
            store_group<T>(d11i + mine * PB + g * EW, xi[g]);
#pragma unroll
            for (int c = 0; c < EW; c++)
                if (g * EW + c == mine) {
                    dr = xr[g][c];
                    di = xi[g][c];
                }
        }
        if (dr == T(0) && di == T(0)) atomicMin(&L.zmin, j0 + mine + 1);
        if constexpr (sizeof(T) == 4 && !WIDE) {
            const float m = fmaxf(fabsf(dr), fabsf(di));
            if (m < kSquareMin || m > kSquareMax) info[1] = 1;
        }
    }
    __syncthreads();
    if (t == 0 && L.zmin != 0x7fffffff && *info == 0) *info = L.zmin;
    if (t < 64) root_swaps(L.oid, L.sw[0], L.sw[1], j0, ipiv, pl);
}

constexpr int kWideSetRows = 4096;

// Levels of the tournament over m rows with w waves per set.
int tslu_levels(int m, int w) {
    int l = 1;
    for (int sets = (m + 64 * w - 1) / (64 * w); sets > 1; sets = (sets + 2 * w - 1) / (2 * w)) l++;
    return l;
}

constexpr int PLS = 256;  // ints per row-pair list

// Triangular solves of the panel steps: a row x of 32 is spread over the four
// lanes of a quad, lane j holding x[4 k + j] in x[k] (cyclic, so the work stays
// even to the last column).  The triangle lies in LDS as M[l][j][k] = M_l,4k+j
// with zeros at and left of the diagonal, so a lane reads its part of row l in
// 16-byte pieces and needs no mask.
constexpr int QK = PB / 4;  // elements of a row per lane
__device__ __forceinline__ int tri_index(int l, int c) { return l * PB + (c & 3) * QK + c / 4; }

// Lane JL's value of each quad.
template <int JL>
__device__ __forceinline__ float quad_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), JL * 0x55, 0xf, 0xf, false));
}
template <int JL>
__device__ __forceinline__ double quad_bcast(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, JL * 0x55, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), JL * 0x55, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <typename T, int L>
__device__ __forceinline__ void solve_step(T (&xr)[QK], T (&xi)[QK], const T* mr, const T* mi, bool scale,
                                           const T* rr, const T* ri) {
    using V = typename Vec16<T>::type;
    constexpr int E = 16 / sizeof(T), K0 = L / 4, JL = L % 4;
    const int j = threadIdx.x & 3;
    if (scale) {
        const T a = xr[K0], b = xi[K0], sr = rr[L], si = ri[L];
        xr[K0] = j == JL ? a * sr - b * si : a;
        xi[K0] = j == JL ? a * si + b * sr : b;
    }
    if constexpr (L < PB - 1) {
        const T lr = quad_bcast<JL>(xr[K0]), li = quad_bcast<JL>(xi[K0]);
#pragma unroll
        for (int k0 = K0 / E * E; k0 < QK; k0 += E) {
            T ur[E], ui[E];
            const V a = *reinterpret_cast<const V*>(mr + L * PB + j * QK + k0);
            const V d = *reinterpret_cast<const V*>(mi + L * PB + j * QK + k0);
            __builtin_memcpy(ur, &a, 16);
            __builtin_memcpy(ui, &d, 16);
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int k = k0 + e;
                if (k < K0) continue;
                xr[k] = fmadd(-lr, ur[e], xr[k]);
                xr[k] = fmadd(li, ui[e], xr[k]);
                xi[k] = fmadd(-lr, ui[e], xi[k]);
                xi[k] = fmadd(-li, ur[e], xi[k]);
            }
        }
        solve_step<T, L + 1>(xr, xi, mr, mi, scale, rr, ri);
    }
}

// Solves x M = x in place for the upper triangle M: x_l is scaled by the
// reciprocal (rr, ri)[l] of the diagonal when `scale` (else unit diagonal), then
// x_c -= x_l M_lc for c > l (four fused multiply-adds per element).
template <typename T>
__device__ __forceinline__ void solve_tri(T (&xr)[QK], T (&xi)[QK], const T* mr, const T* mi, bool scale, const T* rr,
                                          const T* ri) {
    solve_step<T, 0>(xr, xi, mr, mi, scale, rr, ri);
}

// The 32 columns from c on: the row pairs of a step's list pl (np of them)
// interchanged in place, one workgroup for all rows, and with u12 the rows j0 ..
// j0+31 replaced by U12 = L11^{-1} A12 (L11 transposed at lr, li; top: the rows
// they come from).  Every source is in registers before the first store.
template <typename T>
__device__ __forceinline__ void swap_strip(T* __restrict__ Ar, T* __restrict__ Ai, long ld, int j0, int c, bool u12,
                                           const int* __restrict__ pl, int np, const int* top, const T* lr,
                                           const T* li) {
    constexpr int RG = 256 / PB, PER = 2 * PB / RG;  // row groups; pairs per thread
    const int t = threadIdx.x, tx = t % PB, ty = t / PB, i = t / 4, j = t & 3;
    T vr[PER], vi[PER], xr[QK], xi[QK];
    int dst[PER], src[PER];  // unconditional loads stay in flight together
#pragma unroll
    for (int u = 0; u < PER; u++) {
        dst[u] = pl[1 + 2 * (ty + RG * u)];
        src[u] = pl[2 + 2 * (ty + RG * u)];
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const bool in = ty + RG * u < np;
        dst[u] = in ? dst[u] : -1;
        const long o = (long)(in ? src[u] : j0) * ld + c + tx;
        vr[u] = Ar[o];
        vi[u] = Ai[o];
    }
    const bool solve = u12 && t < 4 * PB;  // a column per quad of lanes
    if (solve) {
#pragma unroll
        for (int k = 0; k < QK; k++) {
            const long o = (long)top[4 * k + j] * ld + c + i;
            xr[k] = Ar[o];
            xi[k] = Ai[o];
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++)
        if (dst[u] >= (u12 ? j0 + PB : 0)) {
            const long o = (long)dst[u] * ld + c + tx;
            Ar[o] = vr[u];
            Ai[o] = vi[u];
        }
    if (solve) {
        solve_tri<T>(xr, xi, lr, li, false, lr, li);
#pragma unroll
        for (int k = 0; k < QK; k++) {
            const long o = (long)(j0 + 4 * k + j) * ld + c + i;
            Ar[o] = xr[k];
            Ai[o] = xi[k];
        }
    }
}

// The net effect of an outer panel's row interchanges: net[i] (i < NB) is the
// row that ends in row k0 + i, net[NB] the number of (destination, source) pairs
// that follow for the rows below the panel's top NB (at most NB of them).
constexpr int NETS = 3 * NB + 64;  // ints per net list

// Composes the NB / PB row-pair lists of a panel (list l at pl + l PLS, applied in
// order) into net: the last list with a row as destination names its source, whose
// content before that list is followed through the earlier lists.  One workgroup.
// A list's pairs lie in a table of their own, kListSlots places probed in order from a
// hash of the destination, so that a row is found in a list in one or two steps: the
// chain is what bounds it (each entry going through all pairs of the lists, k_step of a
// panel's last step took 60 - 80 us for a random matrix and 22 for an assembled one, now 17 and 9).
constexpr int kListSlots = 128;  // twice the pairs of a list, so a probe always ends
struct PairTable {
    int *dst, *src;  // NB / PB tables; dst -1: empty
    __device__ __forceinline__ static int first(int row) { return (int)((unsigned)row * 0x9e3779b1u >> 25); }
    __device__ __forceinline__ void insert(int l, int row, int from) const {
        int h = first(row);
        while (atomicCAS(&dst[l * kListSlots + h], -1, row) != -1) h = (h + 1) % kListSlots;
        src[l * kListSlots + h] = from;
    }
    // the source of `row` in list l, -1 if it is no destination there
    __device__ __forceinline__ int find(int l, int row) const {
        for (int h = first(row);; h = (h + 1) % kListSlots) {
            const int d = dst[l * kListSlots + h];
            if (d == row) return src[l * kListSlots + h];
            if (d == -1) return -1;
        }
    }
};
__device__ void compose_lists(const int* __restrict__ pl, int k0, int* __restrict__ net, PairTable tab, int* top,
                              int* count) {
    constexpr int NL = NB / PB, PER = NL * 2 * PB / 256;
    const int t = threadIdx.x;
    static_assert(kListSlots == 128 && kListSlots >= 4 * PB, "the hash gives 7 bits; half of the places stay empty");
    int2 pair[PER];
    bool in[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int e = t + 256 * u, l = e / (2 * PB), k = e % (2 * PB);
        pair[u] = make_int2(pl[l * PLS + 1 + 2 * k], pl[l * PLS + 2 + 2 * k]);  // beyond the count: not used
        in[u] = k < pl[l * PLS];
    }
    for (int e = t; e < NL * kListSlots; e += 256) tab.dst[e] = -1;
    top[t] = k0 + t;
    if (t == 0) *count = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++)
        if (in[u]) tab.insert((t + 256 * u) / (2 * PB), pair[u].x, pair[u].y);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const int l = (t + 256 * u) / (2 * PB), dst = pair[u].x;
        if (!in[u]) continue;
        bool last = true;
        for (int m = l + 1; m < NL && last; m++) last = tab.find(m, dst) < 0;
        if (!last) continue;
        int src = pair[u].y;
        for (int m = l - 1; m >= 0; m--) {
            const int from = tab.find(m, src);
            src = from < 0 ? src : from;
        }
        if (dst < k0 + NB) {
            top[dst - k0] = src;
        } else if (src != dst) {
            const int i = atomicAdd(count, 1);
            net[NB + 1 + 2 * i] = dst;
            net[NB + 2 + 2 * i] = src;
        }
    }
    __syncthreads();
    net[t] = top[t];
    if (t == 0) net[NB] = *count;
}

// Panel step after the tournament of columns J = j0..j0+31, for 32 rows per
// workgroup (rows from j0 + 32 on): the step's row interchanges, L21 = A21
// U11^{-1}, and for the next 32 columns J' (with_next) U12 = L11^{-1} A12 and the
// rank-32 update, all that the next tournament waits for.
//
// Nothing is interchanged in place: a row is read from where the step's
// row-pair list pl says it comes from.  The columns J are read from S (row i at
// S + 32 i, a compact copy) and L21 goes to the matrix; the columns J' are read
// from the matrix and go, updated, to the compact copy D that the next
// tournament and step read.  U12 of J' goes to U (32 x 32), not over the rows
// other workgroups still read.  The other columns of the panel follow in the
// next tournament's launch.
//
// Waves 0 and 1 form L21 (one row per quad of lanes), waves 2 and 3 U12 (one
// column per quad) at the same time, then each wave multiplies one 16 x 16 tile
// on the matrix cores (3M in FP32, as the products of the other columns).
// Latency-bound: the loads that depend on nothing are issued first, and the
// quads cut the substitution's chain to a quarter of the multiply-adds of a
// whole row per lane (3840 rows: 10 us for what three launches of 7, 14 and 5 us
// did).  It needs few enough registers and little
// enough LDS to start beside the trailing update as soon as one of its
// workgroups ends.  A zero pivot leaves its column unscaled.
template <typename T>
__global__ __launch_bounds__(256) void k_step(T* __restrict__ Ar, T* __restrict__ Ai, long ld,
                                              const T* __restrict__ Sr, const T* __restrict__ Si, int k0, int j0,
                                              int n, int with_next, const int* __restrict__ pl,
                                              const T* __restrict__ d11r, const T* __restrict__ d11i,
                                              T* __restrict__ Dr, T* __restrict__ Di, T* __restrict__ Ur,
                                              T* __restrict__ Ui, int* __restrict__ net) {
    __builtin_amdgcn_s_setprio(3);
    constexpr int SL = PB + 4;  // row stride of L21 and U12 in LDS
    __shared__ __align__(16) T ur[PB * PB], ui[PB * PB], lr[PB * PB], li[PB * PB];  // U11; L11 transposed
    __shared__ __align__(16) T pr[PB * SL], pi[PB * SL], vr[PB * SL], vi[PB * SL];  // L21, U12
    __shared__ T rr[PB], ri[PB];
    __shared__ int map[PB], top[PB];  // source rows of this workgroup's rows and of rows j0 .. j0+31
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nrow = max(1, (n - j0 - PB) / PB), strip = (int)blockIdx.x - nrow;  // strip >= 0: other columns
    const int r0 = j0 + PB + blockIdx.x * PB;
    if (strip == NB / PB - 1 && !with_next) {  // beside the panel's last step
        static_assert(sizeof(ur) >= NB / PB * kListSlots * sizeof(int), "a table's half fits");
        compose_lists(pl - (NB / PB - 1) * PLS, k0, net, PairTable{reinterpret_cast<int*>(ur), reinterpret_cast<int*>(ui)},
                      reinterpret_cast<int*>(lr), map);
        return;
    }
    const int np = pl[0];
    int2 pair = make_int2(-1, -1);
    if (t < 2 * PB) pair = make_int2(pl[1 + 2 * t], pl[2 + 2 * t]);  // beyond np: not used
    T da[4], db[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        da[u] = d11r[t + 256 * u];
        db[u] = d11i[t + 256 * u];
    }
    if (t < PB)
        map[t] = min(r0 + t, n - 1);
    else if (t < 2 * PB)
        top[t - PB] = j0 + t - PB;
    __syncthreads();
    if (t < np) {  // np <= 2 PB
        if (pair.x < j0 + PB)
            top[pair.x - j0] = pair.y;
        else if (strip < 0 && pair.x >= r0 && pair.x < r0 + PB)
            map[pair.x - r0] = pair.y;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int e = t + 256 * u, r = e / PB, c = e % PB;
        const T a = da[u], b = db[u];
        ur[tri_index(r, c)] = c > r ? a : T(0);
        ui[tri_index(r, c)] = c > r ? b : T(0);
        lr[tri_index(c, r)] = r > c ? a : T(0);
        li[tri_index(c, r)] = r > c ? b : T(0);
        if (r == c) {
            if (a == T(0) && b == T(0)) {
                rr[r] = T(1);
                ri[r] = T(0);
            } else {
                cdiv(T(1), T(0), a, b, rr[r], ri[r]);
            }
        }
        if (blockIdx.x == 0) {
            Ar[(long)(j0 + r) * ld + j0 + c] = a;
            Ai[(long)(j0 + r) * ld + j0 + c] = b;
        }
    }
    __syncthreads();
    if (strip >= 0) {
        const int nleft = (j0 - k0) / PB;
        const bool left = strip < nleft;
        swap_strip<T>(Ar, Ai, ld, j0, left ? k0 + strip * PB : j0 + 2 * PB + (strip - nleft) * PB, !left, pl, np, top,
                      lr, li);
        return;
    }
    const bool rows = wave < 2;
    const int i = (wave & 1) * 16 + lane / 4, j = lane & 3;  // row of L21 or column of U12; part of it
    const int r16 = lane & 15, g = lane >> 4, m0 = (wave >> 1) * 16, n0 = (wave & 1) * 16;
    const bool inside = r0 < n;  // n - r0 is a multiple of 32
    T xr[QK], xi[QK];
    if (rows) {
        const long o = (long)map[i] * PB + j;
#pragma unroll
        for (int k = 0; k < QK; k++) {
            xr[k] = Sr[o + 4 * k];
            xi[k] = Si[o + 4 * k];
        }
    } else if (with_next) {
#pragma unroll
        for (int k = 0; k < QK; k++) {
            const long o = (long)top[4 * k + j] * ld + j0 + PB + i;
            xr[k] = Ar[o];
            xi[k] = Ai[o];
        }
    }
    // this wave's 16 x 16 tile of J' before the update: FP32 row m0 + r16,
    // columns n0 + 4 g .. + 3; FP64 rows m0 + g + 4 q, column n0 + r16
    typedef typename std::conditional<sizeof(T) == 4, v4f, v4d>::type acc_t;
    acc_t cr{}, ci{};
    if (with_next) {
        if constexpr (sizeof(T) == 4) {
            const long o = (long)map[m0 + r16] * ld + j0 + PB + n0 + 4 * g;
            cr = *reinterpret_cast<const v4f*>(Ar + o);
            ci = *reinterpret_cast<const v4f*>(Ai + o);
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long o = (long)map[m0 + g + 4 * q] * ld + j0 + PB + n0 + r16;
                cr[q] = Ar[o];
                ci[q] = Ai[o];
            }
        }
    }
    if (rows || with_next) solve_tri<T>(xr, xi, rows ? ur : lr, rows ? ui : li, rows, rr, ri);
    if (rows) {
        if (inside) {
            const long o = (long)(r0 + i) * ld + j0 + j;
#pragma unroll
            for (int k = 0; k < QK; k++) {
                Ar[o + 4 * k] = xr[k];
                Ai[o + 4 * k] = xi[k];
            }
        }
#pragma unroll
        for (int k = 0; k < QK; k++) {
            pr[i * SL + 4 * k + j] = xr[k];
            pi[i * SL + 4 * k + j] = xi[k];
        }
    } else if (with_next) {
#pragma unroll
        for (int k = 0; k < QK; k++) {
            vr[(4 * k + j) * SL + i] = xr[k];
            vi[(4 * k + j) * SL + i] = xi[k];
            if (blockIdx.x == 0) {
                Ur[(4 * k + j) * PB + i] = xr[k];
                Ui[(4 * k + j) * PB + i] = xi[k];
            }
        }
    }
    if (!with_next || !inside) return;
    __syncthreads();
    if constexpr (sizeof(T) == 4) {
        v4f t1 = v4f{0.f, 0.f, 0.f, 0.f}, t2 = t1, t3 = t1;
#pragma unroll
        for (int q = 0; q < PB / 16; q++) {
            const v4f a0 = *reinterpret_cast<const v4f*>(pr + (m0 + r16) * SL + 16 * q + 4 * g);
            const v4f a1 = *reinterpret_cast<const v4f*>(pi + (m0 + r16) * SL + 16 * q + 4 * g);
            const v4f a2 = a0 + a1;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int o = (16 * q + 4 * g + e) * SL + n0 + r16;
                const float b0 = vr[o], b1 = vi[o];
                t1 = mfma16x16x4(b0, a0[e], t1);
                t2 = mfma16x16x4(b1, a1[e], t2);
                t3 = mfma16x16x4(b0 + b1, a2[e], t3);
            }
        }
        const long o = (long)(r0 + m0 + r16) * PB + n0 + 4 * g;
        *reinterpret_cast<v4f*>(Dr + o) = cr - (t1 - t2);
        *reinterpret_cast<v4f*>(Di + o) = ci - (t3 - t1 - t2);
    } else {
        v4d re{}, im{};
#pragma unroll
        for (int q = 0; q < PB / 4; q++) {
            const int k = 4 * q + g;
            const T a0 = pr[(m0 + r16) * SL + k], a1 = pi[(m0 + r16) * SL + k];
            const T b0 = vr[k * SL + n0 + r16], b1 = vi[k * SL + n0 + r16];
            re = mfma16x16x4(a0, b0, re);
            re = mfma16x16x4(a1, -b1, re);
            im = mfma16x16x4(a0, b1, im);
            im = mfma16x16x4(a1, b0, im);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const long o = (long)(r0 + m0 + g + 4 * q) * PB + n0 + r16;
            Dr[o] = cr[q] - re[q];
            Di[o] = ci[q] - im[q];
        }
    }
}

// The first 32 columns of an outer panel, rows [k0, n), into the compact copy D
// (row i at D + 32 i).
template <typename T>
__global__ __launch_bounds__(256) void k_compact(const T* __restrict__ Ar, const T* __restrict__ Ai, long ld, int k0,
                                                 int n, T* __restrict__ Dr, T* __restrict__ Di) {
    using V = typename Vec16<T>::type;
    constexpr int E = 16 / sizeof(T), W = PB / E;
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int i = k0 + e / W, q = (e % W) * E;
    if (i >= n) return;
    *reinterpret_cast<V*>(Dr + (long)i * PB + q) = *reinterpret_cast<const V*>(Ar + (long)i * ld + k0 + q);
    *reinterpret_cast<V*>(Di + (long)i * PB + q) = *reinterpret_cast<const V*>(Ai + (long)i * ld + k0 + q);
}

// A panel's row interchanges (net, see compose_lists) in place in the columns
// c0, c0 + 16, ...: 16 columns per workgroup, every source read before the first
// store.
template <typename T>
__global__ __launch_bounds__(256) void k_swap_net(T* __restrict__ Ar, T* __restrict__ Ai, long ld, int k0, int c0,
                                                  const int* __restrict__ net) {
    using V = Nat16<T>;
    constexpr int E = 16 / sizeof(T), W = 16 / E;  // 16-byte pieces per row
    const int t = threadIdx.x;
    const long c = c0 + 16 * (long)blockIdx.x;
    int dst[2], src[2];
    dst[0] = k0 + t;
    src[0] = net[t];
    dst[1] = src[1] = 0;
    if (t < net[NB]) {
        dst[1] = net[NB + 1 + 2 * t];
        src[1] = net[NB + 2 + 2 * t];
    }
    V vr[2][W], vi[2][W];
#pragma unroll
    for (int u = 0; u < 2; u++)
        if (dst[u] != src[u])
#pragma unroll
            for (int k = 0; k < W; k++) {
                vr[u][k] = *reinterpret_cast<const V*>(Ar + (long)src[u] * ld + c + k * E);
                vi[u][k] = *reinterpret_cast<const V*>(Ai + (long)src[u] * ld + c + k * E);
            }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; u++)
        if (dst[u] != src[u])
#pragma unroll
            for (int k = 0; k < W; k++) {
                *reinterpret_cast<V*>(Ar + (long)dst[u] * ld + c + k * E) = vr[u][k];
                *reinterpret_cast<V*>(Ai + (long)dst[u] * ld + c + k * E) = vi[u][k];
            }
}

// Columns right of outer panel k0, 16 per workgroup (c0, c0 + 16, ...): the
// panel's row interchanges (net) and U12 = L11^{-1} A12 (256 x 16), by blocked
// substitution with L11 itself.  U12 goes to the matrix and, for the FP32
// trailing update, transposed to Ut (row = column c0 + i, ld NB).
//
// The strip stays in registers as the accumulators of 16 x 16 matrix-core tiles,
// wave w holding the 32-row block w.  Step j: wave j solves its block against the
// 32 x 32 unit triangle (quads of lanes per column, the block through LDS), one
// barrier, then every later wave subtracts L_wj X_j from its block.  What does not
// depend on X is loaded ahead: a wave's triangle at the start (to LDS one step
// before its turn), the rows of L before the barrier.
//
// Latency-bound for the next panel's 256 columns (16 workgroups), which the
// next panel waits for.  Before, those took eight row-pair lists one after the
// other (15 us), the explicit inverse of L11 (seven launches, 67 us), a product
// (15 us) and a transposing copy (5 us); now one launch of 37 us (FP64, before
// by substitution in 62 us behind the lists: 51).
template <typename T>
__global__ __launch_bounds__(512) void k_u12_strip(T* __restrict__ Ar, T* __restrict__ Ai, long ld, int k0, int c0,
                                                   const int* __restrict__ net, T* __restrict__ Utr,
                                                   T* __restrict__ Uti) {
    __builtin_amdgcn_s_setprio(3);
    using V = Nat16<T>;
    constexpr int E = 16 / sizeof(T), W = 16 / E, NJ = NB / PB, XS = 16 + E;  // XS: row stride of a block in LDS
    __shared__ __align__(16) T tri[2][2][PB * PB];  // [step parity][plane]: the triangle, transposed
    __shared__ __align__(16) T xb[2][2][PB * XS];   // [step parity][plane]: block j, then X_j
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const long c = c0 + 16 * (long)blockIdx.x;
    typedef typename std::conditional<sizeof(T) == 4, v4f, v4d>::type acc_t;
    // tile i: rows 32 wave + 16 i + .. of the panel.  FP32: row r16, columns 4 g ..
    // + 3; FP64: rows g + 4 q, column r16
    acc_t cr[2], ci[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = PB * wave + 16 * i;
        if constexpr (sizeof(T) == 4) {
            const long o = (long)net[row + r16] * ld + c + 4 * g;
            cr[i] = *reinterpret_cast<const v4f*>(Ar + o);
            ci[i] = *reinterpret_cast<const v4f*>(Ai + o);
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long o = (long)net[row + g + 4 * q] * ld + c + r16;
                cr[i][q] = Ar[o];
                ci[i][q] = Ai[o];
            }
        }
    }
    // the rows below the panel: half a row per thread
    int dst = -1;
    V vr[W / 2], vi[W / 2];
    const long half = c + (t & 1) * 8;
    if (t / 2 < net[NB]) {
        dst = net[NB + 1 + t / 2 * 2];
        const long o = (long)net[NB + 2 + t / 2 * 2] * ld + half;
#pragma unroll
        for (int k = 0; k < W / 2; k++) {
            vr[k] = *reinterpret_cast<const V*>(Ar + o + k * E);
            vi[k] = *reinterpret_cast<const V*>(Ai + o + k * E);
        }
    }
    T ta[PB * PB / 64], tb[PB * PB / 64];  // this wave's triangle
    {
        const T* lr = Ar + (long)(k0 + PB * wave) * (ld + 1);
        const T* li = Ai + (long)(k0 + PB * wave) * (ld + 1);
#pragma unroll
        for (int u = 0; u < PB * PB / 64; u++) {
            const int e = lane + 64 * u;
            ta[u] = lr[(long)(e / PB) * ld + e % PB];
            tb[u] = li[(long)(e / PB) * ld + e % PB];
        }
    }
    auto put_tri = [&](int par) {
#pragma unroll
        for (int u = 0; u < PB * PB / 64; u++) {
            const int e = lane + 64 * u, r = e / PB, q = e % PB;
            tri[par][0][tri_index(q, r)] = q < r ? ta[u] : T(0);
            tri[par][1][tri_index(q, r)] = q < r ? tb[u] : T(0);
        }
    };
    if (wave == 0) put_tri(0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // every source has been read
    if (dst >= 0) {
#pragma unroll
        for (int k = 0; k < W / 2; k++) {
            *reinterpret_cast<V*>(Ar + (long)dst * ld + half + k * E) = vr[k];
            *reinterpret_cast<V*>(Ai + (long)dst * ld + half + k * E) = vi[k];
        }
    }
#pragma unroll 1
    for (int j = 0; j < NJ; j++) {
        const int par = j & 1;
        T(*x)[PB * XS] = xb[par];
        T la[2][2][4], lb[2][2][4];  // element k = 16 q + 4 g + e of row r16 of the wave's tiles
        if (wave > j) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const long o = (long)(k0 + PB * wave + 16 * i + r16) * ld + k0 + PB * j + 16 * q + 4 * g;
                    load_row4<T>(Ar + o, la[i][q]);
                    load_row4<T>(Ai + o, lb[i][q]);
                }
            if (wave == j + 1) put_tri(par ^ 1);
        } else if (wave == j) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if constexpr (sizeof(T) == 4) {
                    *reinterpret_cast<v4f*>(&x[0][(16 * i + r16) * XS + 4 * g]) = cr[i];
                    *reinterpret_cast<v4f*>(&x[1][(16 * i + r16) * XS + 4 * g]) = ci[i];
                } else {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        x[0][(16 * i + g + 4 * q) * XS + r16] = cr[i][q];
                        x[1][(16 * i + g + 4 * q) * XS + r16] = ci[i][q];
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();  // the wave's own data: its LDS operations stay in order
            T yr[QK], yi[QK];
#pragma unroll
            for (int k = 0; k < QK; k++) {
                yr[k] = x[0][(4 * k + (lane & 3)) * XS + lane / 4];
                yi[k] = x[1][(4 * k + (lane & 3)) * XS + lane / 4];
            }
            solve_tri<T>(yr, yi, tri[par][0], tri[par][1], false, yr, yi);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < QK; k++) {
                x[0][(4 * k + (lane & 3)) * XS + lane / 4] = yr[k];
                x[1][(4 * k + (lane & 3)) * XS + lane / 4] = yi[k];
            }
        }
        __syncthreads();
        if (wave > j) {
            if constexpr (sizeof(T) == 4) {
                v4f t1[2], t2[2], t3[2];
#pragma unroll
                for (int i = 0; i < 2; i++) t1[i] = t2[i] = t3[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int o = (16 * q + 4 * g + e) * XS + r16;
                        const float b0 = x[0][o], b1 = x[1][o], b2 = b0 + b1;
#pragma unroll
                        for (int i = 0; i < 2; i++) {
                            t1[i] = mfma16x16x4(b0, la[i][q][e], t1[i]);
                            t2[i] = mfma16x16x4(b1, lb[i][q][e], t2[i]);
                            t3[i] = mfma16x16x4(b2, la[i][q][e] + lb[i][q][e], t3[i]);
                        }
                    }
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    cr[i] -= t1[i] - t2[i];
                    ci[i] -= t3[i] - t1[i] - t2[i];
                }
            } else {
                v4d re[2], im[2];
#pragma unroll
                for (int i = 0; i < 2; i++) re[i] = im[i] = v4d{};
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int o = (16 * q + 4 * g + e) * XS + r16;
                        const T b0 = x[0][o], b1 = x[1][o];
#pragma unroll
                        for (int i = 0; i < 2; i++) {
                            re[i] = mfma16x16x4(la[i][q][e], b0, re[i]);
                            re[i] = mfma16x16x4(lb[i][q][e], -b1, re[i]);
                            im[i] = mfma16x16x4(la[i][q][e], b1, im[i]);
                            im[i] = mfma16x16x4(lb[i][q][e], b0, im[i]);
                        }
                    }
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    cr[i] -= re[i];
                    ci[i] -= im[i];
                }
            }
        } else {  // the waves that are done: X_j to the matrix by rows and to Ut by columns
            for (int e = t; e < PB * 16; e += (j + 1) * 64) {
                const int r = e / 16, q = e % 16;
                const long o = (long)(k0 + PB * j + r) * ld + c + q;
                Ar[o] = x[0][r * XS + q];
                Ai[o] = x[1][r * XS + q];
                if constexpr (sizeof(T) == 4) {
                    const int n = e / PB, k = e % PB;
                    const long u = (16 * (long)blockIdx.x + n) * NB + PB * j + k;
                    Utr[u] = x[0][k * XS + n];
                    Uti[u] = x[1][k * XS + n];
                }
            }
        }
    }
}

// Inverses of the 32 x 32 diagonal triangles of the factors at F into the diagonals of
// the blocks L, U (block p at p IB IB, ld IB), with their zeros: blockIdx.x = triangle,
// blockIdx.y = 0 unit lower, 1 upper.  One wave each, the triangle staged in LDS, lane j forms column j by
// substitution in registers.
template <typename T>
__global__ __launch_bounds__(64) void k_inv_tri32(const T* __restrict__ Fr, const T* __restrict__ Fi, long ldf,
                                                  T* __restrict__ Lr, T* __restrict__ Li, T* __restrict__ Ur,
                                                  T* __restrict__ Ui) {
    __shared__ T sr[PB][PB + 1], si[PB][PB + 1];
    const int lane = threadIdx.x, p = blockIdx.x / (IB / PB), d = blockIdx.x % (IB / PB);
    const long f = (long)blockIdx.x * PB * (ldf + 1), o = (long)p * IB * IB + (long)d * PB * (IB + 1);
#pragma unroll
    for (int u = 0; u < PB * PB / 64; u++) {
        const int e = lane + 64 * u, r = e / PB, q = e % PB;
        sr[r][q] = Fr[f + r * ldf + q];
        si[r][q] = Fi[f + r * ldf + q];
    }
    __syncthreads();
    const int j = lane & (PB - 1);
    T xr[PB], xi[PB];
    const bool lower = blockIdx.y == 0;
#pragma unroll
    for (int v = 0; v < PB; v++) {  // lower: rows 0, 1, ..; upper: rows 31, 30, ..
        // x_i = delta_ij - sum_k t_ik x_k over the rows k done before
        const int i = v, iu = PB - 1 - v;
        const int row = lower ? i : iu;
        T ar = row == j ? T(1) : T(0), ai = T(0);
#pragma unroll
        for (int w = 0; w < v; w++) {
            const int k = lower ? w : PB - 1 - w;
            const T a = sr[row][k], b = si[row][k];
            ar = fmadd(-a, xr[w], ar);
            ar = fmadd(b, xi[w], ar);
            ai = fmadd(-a, xi[w], ai);
            ai = fmadd(-b, xr[w], ai);
        }
        if (!lower) {
            T qr, qi;
            cdiv(ar, ai, sr[row][row], si[row][row], qr, qi);
            ar = qr;
            ai = qi;
        }
        xr[v] = ar;
        xi[v] = ai;
    }
    if (lane >= PB) return;
    T* outr = lower ? Lr : Ur;
    T* outi = lower ? Li : Ui;
#pragma unroll
    for (int v = 0; v < PB; v++) {
        const int row = lower ? v : PB - 1 - v;
        outr[o + (long)row * IB + j] = xr[v];
        outi[o + (long)row * IB + j] = xi[v];
    }
}

// One product of joining the diagonal inverses of all IB x IB blocks in pairs of h rows:
//   lower [X11 0; X21 X22]  with X21 = -X22 (L21 X11),
//   upper [X11 X12; 0 X22]  with X12 = -X11 (U12 X22)
// (blockIdx.z = 0, 1; blockIdx.y = pair of all blocks; stage 0: the inner product W, to the
// unused triangle of the block, 1: the outer one).  The upper ones then take one step of
// correction: W <- U12 X22 + U11 X12 (k_tri_residual), 2: X12 <- X12 - X11 W.  The sums
// run over the triangles only, so that no value beside them is read; the 32 x 32 triangles
// at the start are stored with their zeros.
__global__ __launch_bounds__(256, 2) void k_tri_join(int stage, int h, const float* __restrict__ Fr,
                                                     const float* __restrict__ Fi, long ldf, float* Lr, float* Li,
                                                     float* Ur, float* Ui) {
    constexpr int NT = 2;
    __shared__ __align__(16) float red[4 * 2 * 16 * 16 * NT];
    const bool lower = stage < 2 && blockIdx.z == 0;
    const int nct = h / (16 * NT), m0 = blockIdx.x / nct * 16, n0 = blockIdx.x % nct * 16 * NT;
    const int np = IB / (2 * h), blk = blockIdx.y / np, d = blockIdx.y % np * 2 * h;
    const long f = ((long)blk * IB + d) * (ldf + 1), x = (long)blk * IB * IB + (long)d * (IB + 1);
    float* Xr = (lower ? Lr : Ur) + x;
    float* Xi = (lower ? Li : Ui) + x;
    const long x22 = (long)h * (IB + 1), x21 = (long)h * IB, x12 = h;
    const long o = lower ? x21 : x12, w = lower ? x12 : x21;
    if (stage == 0) {
        const long a = f + (lower ? (long)h * ldf : h), b = lower ? 0 : x22;
        cmul_tile<NT>(m0, n0, lower ? n0 : 0, lower ? h : n0 + 16 * NT, Fr + a, Fi + a, ldf, Xr + b, Xi + b, IB, Xr + w,
                      Xi + w, IB, 1, red);
    } else if (stage == 1) {
        const long a = lower ? x22 : 0;
        cmul_tile<NT>(m0, n0, lower ? 0 : m0, lower ? m0 + 16 : h, Xr + a, Xi + a, IB, Xr + w, Xi + w, IB, Xr + o,
                      Xi + o, IB, 3, red);
    } else {
        cmul_tile<NT>(m0, n0, m0, h, Xr, Xi, IB, Xr + w, Xi + w, IB, Xr + o, Xi + o, IB, 0, red);
    }
}

// The residual of a join of upper triangles (h, blockIdx.y as in k_tri_join): W = U12 X22 +
// U11 X12, to the unused triangle of the block, with products and sums in FP64, so that the
// corrected X12 is good to its own rounding given X11 and X22: U X = I has to hold to the
// rounding of |U||X|, as by substitution.  The joined products alone leave |U11||X11||W|,
// which on meshes with triangles of very different sizes made the first solve's residual
// 3 - 30 times as large (7200 edges: 1e-2, 6 sweeps instead of 3).  With W in FP32 X12 keeps
// cond(U11) roundings (an ellipsoid of 10440 unknowns: 2e-2 before and 4e-5 after the
// first sweep, 4 sweeps; now 1e-2, 3e-6 and 3, by substitution 2e-2, 3e-5 and 3).
// A workgroup takes 16 x 32 values, its waves a quarter of k each, as in cmul_tile.
__global__ __launch_bounds__(256, 2) void k_tri_residual(int h, const float* __restrict__ Fr,
                                                         const float* __restrict__ Fi, long ldf, float* Ur,
                                                         float* Ui) {
    constexpr int NT = 2;
    __shared__ double red[4][2][16][16 * NT];
    const int nct = h / (16 * NT), m0 = blockIdx.x / nct * 16, n0 = blockIdx.x % nct * 16 * NT;
    const int np = IB / (2 * h), blk = blockIdx.y / np, d = blockIdx.y % np * 2 * h;
    const long f = ((long)blk * IB + d) * (ldf + 1), x = (long)blk * IB * IB + (long)d * (IB + 1);
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    v4d re[NT], im[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) re[t] = im[t] = v4d{};
    // U11 X12 over k = m0 .. h, then U12 X22 over k = h .. h + n0 + 16 NT (columns of U, rows of X)
    const int n1 = (h - m0) / 16, ns = n1 + n0 / 16 + NT;
    const float* ar = Fr + f + (long)(m0 + r) * ldf;
    const float* ai = Fi + f + (long)(m0 + r) * ldf;
    const float* br = Ur + x + h + n0 + r;
    const float* bi = Ui + x + h + n0 + r;
    for (int q = wave; q < ns; q += 4) {
        const int k = (q < n1 ? m0 + 16 * q : h + 16 * (q - n1)) + 4 * g;
        float a0[4], a1[4];
        load_row4<float>(ar + k, a0);
        load_row4<float>(ai + k, a1);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool in = k + e >= m0 + r;  // left of the diagonal lies L
            const double p = in ? a0[e] : 0.f, s = in ? a1[e] : 0.f;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const double b0 = br[(long)(k + e) * IB + 16 * t], b1 = bi[(long)(k + e) * IB + 16 * t];
                re[t] = mfma16x16x4(p, b0, re[t]);
                re[t] = mfma16x16x4(s, -b1, re[t]);
                im[t] = mfma16x16x4(p, b1, im[t]);
                im[t] = mfma16x16x4(s, b0, im[t]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            red[wave][0][g + 4 * q][16 * t + r] = re[t][q];
            red[wave][1][g + 4 * q][16 * t + r] = im[t][q];
        }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 16 * NT; e += 256) {
        const int row = e / (16 * NT), col = e % (16 * NT);
        const long o = x + (long)(h + m0 + row) * IB + n0 + col;
        Ur[o] = (float)(((red[0][0][row][col] + red[1][0][row][col]) + red[2][0][row][col]) + red[3][0][row][col]);
        Ui[o] = (float)(((red[0][1][row][col] + red[1][1][row][col]) + red[2][1][row][col]) + red[3][1][row][col]);
    }
}

// Work buffers of one factorisation (device).
template <typename T>
struct LuWork {
    int* info;       // first zero pivot (1-based), 0 if none; whether a pivot lies outside kSquareMin .. kSquareMax
    int* cnt;        // tournament arrival counters
    int* cid;        // candidate row ids
    T *cvr, *cvi;    // candidate values
    int* pl;         // row-pair lists of the 8 steps of an outer panel (PLS ints each)
    T* d11;          // factored 32 x 32 diagonal block (2 planes), two sets by step parity
    T *cpr, *cpi;    // compact copies (n x 32 per plane) of the columns being factored, two sets by step parity
    T *sur, *sui;    // U12 of the next 32 columns (32 x 32)
    T *utr, *uti;    // n x 256 transpose of U12 (FP32 trailing update)
    int* net;        // net row interchanges of an outer panel, two sets
};

// The net row interchanges of outer panel k0.  Two sets, by panel parity: the
// update stream applies panel K's while panel K+1 composes its own.
template <typename T>
int* panel_net(const LuWork<T>& w, int k0) {
    return w.net + ((k0 / NB) & 1) * NETS;
}

// L^{-1} and U^{-1} of the IB x IB diagonal blocks of the n x n FP32 factors at F into the
// blocks at L and U (ld IB, block b at b IB IB), all blocks in each launch: the 32 x 32
// diagonal triangles by substitution, then joined in pairs.  For the solves; the
// factorisation itself does not use them.
void invert_blocks(hipStream_t s, int n, const float* Fr, const float* Fi, long ldf, float* Lr, float* Li, float* Ur,
                   float* Ui) {
    hipLaunchKernelGGL(k_inv_tri32<float>, dim3(n / PB, 2), dim3(64), 0, s, Fr, Fi, ldf, Lr, Li, Ur, Ui);
    for (int h = PB; h < IB; h *= 2) {
        const unsigned tiles = h / 16 * (h / 32), pairs = n / (2 * h);
        for (int stage = 0; stage < 3; stage++) {
            if (stage == 2)
                hipLaunchKernelGGL(k_tri_residual, dim3(tiles, pairs), dim3(256), 0, s, h, Fr, Fi, ldf, Ur, Ui);
            hipLaunchKernelGGL(k_tri_join, dim3(tiles, pairs, stage < 2 ? 2 : 1), dim3(256), 0, s, stage, h, Fr, Fi, ldf, Lr,
                               Li, Ur, Ui);
        }
    }
}

// Factors the outer panel of columns k0 .. k0+NB-1 (rows k0 .. n-1) on stream
// s: 8 steps of 32 columns, two launches each.  k_step finishes the step's own
// columns, the next 32 and the swaps of the others; the rank-32 update of the
// columns beyond the next 32 rides in the launch of the next tournament, which
// does not need them.  (With that update and the other columns' swaps on a third
// stream, behind an event each way, and the next 32 columns' swaps, panel solve
// and update as three launches a step took 115 us at 3840 rows; now 75.)  The
// swaps of the steps end as one net list for the columns outside the panel.
// The FP32 tournament takes sets of 512 rows (8 waves) where they save a level: 3840
// rows 54.9 us against 65.0 (59.2 with two rows per thread of 4 waves); 1920 rows, where
// they save none, 51.8 against 44.5.
// Up to kWideSetRows only: 8 waves start beside the trailing update later than 4, when
// two of its workgroups on a CU have ended.  In FP64 8 waves do not fit the registers.
template <typename T>
void factor_panel(bem_ctx* c, hipStream_t s, T* Ar, T* Ai, int k0, const LuWork<T>& w, bool wide) {
    const int n = c->npad;
    const long ld = n, cp = (long)n * PB;
    const int k1 = k0 + NB, first = ((n - k0) * (PB * (int)sizeof(T) / 16) + 255) / 256;
    int kt = kt_mark(c, KS_OTHER, s);
    hipLaunchKernelGGL(k_compact<T>, dim3(first), dim3(256), 0, s, Ar, Ai, ld, k0, n, w.cpr, w.cpi);
    kt_close(c, kt, 0.0, 4.0 * sizeof(T) * (double)(n - k0) * PB);
    FarUpdate far{0, 0, 0, 0};
    int far_tiles = -1;  // -1: nothing left to do
    for (int j0 = k0; j0 < k1; j0 += PB) {
        const int m = n - j0, par = ((j0 - k0) / PB) & 1;
        T *Sr = w.cpr + par * cp, *Si = w.cpi + par * cp;
        T *Dr = w.cpr + (par ^ 1) * cp, *Di = w.cpi + (par ^ 1) * cp;
        T *d11r = w.d11 + par * 2 * PB * PB, *d11i = d11r + PB * PB;
        int* pl = w.pl + ((j0 - k0) / PB) * PLS;
        kt = kt_mark(c, KS_TSLU, s);
        auto tslu = k_tslu<T, 4>;
        int waves = 4;
        if constexpr (sizeof(T) == 4) {
            if (m <= kWideSetRows && tslu_levels(m, 8) < tslu_levels(m, 4)) waves = 8;
            tslu = waves == 8 ? (wide ? k_tslu<T, 8, true> : k_tslu<T, 8>) : wide ? k_tslu<T, 4, true> : k_tslu<T, 4>;
        }
        const int set = 64 * waves;
        far.blocks = far_tiles < 0 ? 0 : (far_tiles + waves - 1) / waves + 1;
        hipLaunchKernelGGL(tslu, dim3((m + set - 1) / set + far.blocks), dim3(set), 0, s, Sr, Si, (long)PB, j0, n,
                           w.cid, w.cvr, w.cvi, w.cnt, c->ipiv, pl, d11r, d11i, w.info, Ar, Ai, ld, far, w.sur, w.sui);
        kt_close(c, kt, (sizeof(T) == 4 ? 6.0 : 8.0) * far.ncol * (double)m * PB,
                 2.0 * sizeof(T) * (double)m * (PB + 2 * far.ncol));
        const int next = j0 + PB < k1, others = NB / PB - 1 - next;
        kt = kt_mark(c, KS_PANEL, s);
        hipLaunchKernelGGL(k_step<T>, dim3(std::max(1, (m - PB) / PB) + others + !next), dim3(256), 0, s, Ar, Ai, ld,
                           Sr, Si, k0, j0, n, next, pl, d11r, d11i, Dr, Di, w.sur, w.sui, panel_net(w, k0));
        kt_close(c, kt, (next ? 10.0 : 4.0) * (double)m * PB * PB, (next ? 8.0 : 4.0) * sizeof(T) * (double)m * PB);
        const int c0 = std::min(k1, j0 + 2 * PB), ncol = k1 - c0;  // columns beyond the next 32
        far = FarUpdate{j0, c0, ncol, 0};
        far_tiles = next ? (m - PB) / 16 * (ncol / 16) : -1;
    }
}

// The swaps of outer panel k0, U12 = L11^{-1} A12 and A22 -= L21 U12 for the
// columns [c0, c0 + nc) right of the panel, on stream us; cap > 0: the update on that many
// workgroups.
template <typename T>
void update_columns(bem_ctx* c, hipStream_t us, T* Ar, T* Ai, int k0, int c0, int nc, const LuWork<T>& w,
                    long cap) {
    const int n = c->npad;
    const long ld = n;
    const int nr = n - (k0 + NB);
    const long o12 = (long)k0 * ld + c0, o21 = (long)(k0 + NB) * ld + k0, o22 = (long)(k0 + NB) * ld + c0;
    T *utr = nullptr, *uti = nullptr;
    if constexpr (sizeof(T) == 4) {
        utr = w.utr + (long)(c0 - (k0 + NB)) * NB;
        uti = w.uti + (long)(c0 - (k0 + NB)) * NB;
    }
    int kt = kt_mark(c, KS_TRSM, us);
    hipLaunchKernelGGL(k_u12_strip<T>, dim3(nc / 16), dim3(512), 0, us, Ar, Ai, ld, k0, c0, panel_net(w, k0), utr, uti);
    kt_close(c, kt, 4.0 * (double)NB * NB * nc, (sizeof(T) == 4 ? 8.0 : 6.0) * sizeof(T) * (double)NB * nc);
    if constexpr (sizeof(T) == 4) {  // on the k-contiguous kernel; nr and nc are multiples of 256
        const GemmPlan& plan = c->gemm_plan[0];
        kt = kt_mark(c, KS_UPDATE32, us);
        cupdate_nt(plan.nt, us, nr, nc, NB, Ar + o21, Ai + o21, ld, utr, uti, NB, Ar + o22, Ai + o22, ld,
                   cap);
        kt_close(c, kt, 6.0 * (double)nr * nc * NB,
                 2.0 * sizeof(T) * ((double)nr * NB + (double)NB * nc + 2.0 * nr * nc));
    } else {
        cgemm_ctx(c, nr, nc, NB, Ar + o21, Ai + o21, ld, Ar + o12, Ai + o12, ld, Ar + o22, Ai + o22, ld, 0, us, true,
                  cap);
    }
}

// Blocked right-looking factorisation of the padded npad x npad matrix with
// look-ahead of depth one: outer panel K+1 is factored on the panel stream
// while the trailing update of panel K runs on the update stream.  Panel K+1
// only touches its own columns; its swaps reach the other columns on the
// update stream.  After panel K, the critical path to panel K+1 is the swaps, U12
// and the update of those 256 columns, on the panel stream too, which then waits for
// no event between panels once the chain is the longer part (18 us a panel less than with
// that part on the update stream: 2N = 3840 10.21 -> 10.08 ms); the swaps and the
// update of all other columns follow on the update stream while panel K+1 is factored.
// Stream layout (c->lu_streams): 0 = everything on the context stream (no
// overlap); 1 = panel stream and context stream over all CUs.
template <typename T>
void factor(bem_ctx* c, T* Ar, T* Ai, T* Lir, T* Lii, T* Uir, T* Uii, const LuWork<T>& w, bool wide) {
    const int n = c->npad, nb = n / NB;
    const long ld = n;
    hipStream_t us = c->stream, ps = c->stream2;
    if (c->lu_streams == 0) ps = us;
    hipEvent_t e_rest = c->lu_ev[0], e_next = c->lu_ev[1], e_start = c->lu_ev[2];
    (void)hipEventRecord(e_start, us);  // the matrix and work buffers are ready
    (void)hipStreamWaitEvent(ps, e_start, 0);
    auto swap_left = [&](int k0) {
        if (k0 == 0) return;
        const int kt = kt_mark(c, KS_LASWP, us);
        hipLaunchKernelGGL(k_swap_net<T>, dim3(k0 / 16), dim3(256), 0, us, Ar, Ai, ld, k0, 0, panel_net(w, k0));
        kt_close(c, kt, 0.0, 4.0 * sizeof(T) * (double)k0 * 2 * NB);
    };
    factor_panel<T>(c, ps, Ar, Ai, 0, w, wide);
    for (int K = 0; K < nb; K++) {
        const int k0 = K * NB;
        const int nr = n - (k0 + NB);
        if (nr <= 0) {
            (void)hipEventRecord(e_next, ps);
            (void)hipStreamWaitEvent(us, e_next, 0);
            swap_left(k0);
            break;
        }
        // columns of panel K+1 first, on the panel stream, once the update of panel K-1
        // has left them
        if (K > 0) (void)hipStreamWaitEvent(ps, e_rest, 0);
        update_columns<T>(c, ps, Ar, Ai, k0, k0 + NB, NB, w, 0);
        (void)hipEventRecord(e_next, ps);
        (void)hipStreamWaitEvent(us, e_next, 0);
        // the rest of the update is enqueued before panel K+1's launches, so a
        // host that enqueues slowly (under a profiler, say) does not hold the
        // update stream back
        swap_left(k0);
        if (nr > NB)
            update_columns<T>(c, us, Ar, Ai, k0, k0 + 2 * NB, nr - NB, w,
                              ps != us ? c->gemm_plan[sizeof(T) == 4 ? 0 : 1].cap : 0);
        (void)hipEventRecord(e_rest, us);
        factor_panel<T>(c, ps, Ar, Ai, k0 + NB, w, wide);
    }
    // the inverses of all diagonal blocks (FP32; the FP64 solves substitute with
    // the diagonal blocks themselves)
    if constexpr (sizeof(T) == 4) {
        const int kt = kt_mark(c, KS_TRSM, us);
        invert_blocks(us, n, Ar, Ai, ld, Lir, Lii, Uir, Uii);
        kt_close(c, kt, 16.0 * (double)n * IB * IB / 6.0, 8.0 * sizeof(T) * (double)n * IB);
    }
}

template <typename T>
__global__ void k_convert(const double* __restrict__ a, T* __restrict__ b, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (T)a[i];
}

template <typename T>
int factor_prec(bem_ctx* c, T* Ar, T* Ai, void*& inv, size_t& inv_bytes, bool wide = false) {
    const int n = c->npad;
    // diagonal-block inverses (FP32 only): L and U, npad x NB per plane each
    constexpr bool with_inv = sizeof(T) == 4;
    const size_t ib = 4 * (size_t)n * IB * sizeof(T);
    if (with_inv && inv_bytes < ib) {
        if (inv) (void)hipFree(inv);
        inv = nullptr;
        inv_bytes = 0;
        if (hipMalloc(&inv, ib) != hipSuccess) return bem_fail(c, BEM_ERR_NOMEM, "LU: diagonal-block inverses");
        inv_bytes = ib;
    }
    T* Lir = with_inv ? static_cast<T*>(inv) : nullptr;
    T* Lii = with_inv ? Lir + (size_t)n * IB : nullptr;
    T* Uir = with_inv ? Lii + (size_t)n * IB : nullptr;
    T* Uii = with_inv ? Uir + (size_t)n * IB : nullptr;
    // work: info, counters, row-pair list, candidate ids, candidate values,
    // diagonal blocks, compact columns, U12 buffers
    const int nsets0 = (n + 255) / 256;
    const size_t ncnt = 2 * (size_t)nsets0 + 64;
    const size_t nint = 64 + ncnt + (NB / PB) * PLS + 2 * NETS + 2 * (size_t)nsets0 * PB;
    const size_t bytes = nint * sizeof(int) + 256 + 4 * (size_t)nsets0 * PB * PB * sizeof(T) +
                         6 * (size_t)PB * PB * sizeof(T) + 4 * (size_t)PB * n * sizeof(T) +
                         (with_inv ? 2 * (size_t)NB * n * sizeof(T) : 0) + 256;
    void* scr = nullptr;
    if (int rc = ctx_scratch(c, bytes, &scr)) return rc;
    LuWork<T> w;
    w.info = static_cast<int*>(scr);
    w.cnt = w.info + 64;
    w.pl = w.cnt + ncnt;
    w.net = w.pl + (NB / PB) * PLS;
    w.cid = w.net + 2 * NETS;
    char* p = reinterpret_cast<char*>(w.info + nint);
    p += (256 - reinterpret_cast<uintptr_t>(p) % 256) % 256;
    w.cvr = reinterpret_cast<T*>(p);
    w.cvi = w.cvr + 2 * (size_t)nsets0 * PB * PB;
    w.d11 = w.cvi + 2 * (size_t)nsets0 * PB * PB;
    w.sur = w.d11 + 4 * PB * PB;
    w.sui = w.sur + PB * PB;
    w.cpr = w.sui + PB * PB;
    w.cpi = w.cpr + 2 * (size_t)PB * n;
    w.utr = w.cpi + 2 * (size_t)PB * n;
    w.uti = w.utr + (size_t)NB * n;
    BEM_HIP(c, hipMemsetAsync(w.info, 0, (64 + ncnt) * sizeof(int), c->stream));
    factor<T>(c, Ar, Ai, Lir, Lii, Uir, Uii, w, wide);
    return 0;
}

}  // namespace

namespace {

// Notes the time at its start and end in at[0], at[1] and lasts `ticks` of the
// constant clock (bounded besides by the number of looks at it).
__global__ void k_interval(long long ticks, long long* at) {
    const long long t0 = wall_clock64();
    long long t1 = t0;
    for (int i = 0; i < 100000 && t1 - t0 < ticks; i++) {
        __builtin_amdgcn_s_sleep(8);
        t1 = wall_clock64();
    }
    at[0] = t0;
    at[1] = t1;
}

// Whether kernels of the two streams run side by side.
bool streams_overlap(hipStream_t a, hipStream_t b, long long* at, long long ticks) {
    long long h[4] = {0, 0, 0, 0};
    for (int warm = 1; warm >= 0; warm--) {  // a stream's first launch can take long
        hipLaunchKernelGGL(k_interval, dim3(1), dim3(1), 0, a, warm ? 0 : ticks, at);
        hipLaunchKernelGGL(k_interval, dim3(1), dim3(1), 0, b, warm ? 0 : ticks, at + 2);
        if (hipStreamSynchronize(a) != hipSuccess || hipStreamSynchronize(b) != hipSuccess) return true;
    }
    if (hipMemcpy(h, at, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return true;
    return h[0] < h[3] && h[2] < h[1];
}

}  // namespace

// The panel stream has to run beside the context stream.  The runtime spreads a
// process's streams over a few hardware queues (four by default) by their load,
// and two streams of one queue run one after the other: a second context's pair
// can end on one (the factorisation at n = 18432 then takes 176 instead of 141
// ms).  So the first factorisation large enough to gain looks whether the two
// overlap (~0.1 ms) and otherwise takes another panel stream.
int lu_setup_streams(bem_ctx* c) {
    // (A layout with the panel stream on CUs reserved by a CU mask ended in a
    // host-side crash in its first run, cause not established; it was removed.)
    if (c->lu_streams < 0) {
        const char* e1 = std::getenv("BEM_LU_STREAMS");
        c->lu_streams = e1 && std::atoi(e1) == 0 ? 0 : 1;
    }
    constexpr int kOverlapMinN = 2048, kTries = 4;
    if (c->lu_streams == 0 || c->lu_streams_checked || c->npad < kOverlapMinN) return 0;
    c->lu_streams_checked = true;
    void* scr = nullptr;
    if (int rc = ctx_scratch(c, 4 * sizeof(long long), &scr)) return rc;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device) != hipSuccess || khz <= 0) return 0;
    const long long ticks = khz / 25;  // 40 us
    hipStream_t tried[kTries] = {};
    for (int i = 0; i < kTries && !streams_overlap(c->stream, c->stream2, static_cast<long long*>(scr), ticks); i++) {
        hipStream_t other = nullptr;
        if (hipStreamCreateWithFlags(&other, hipStreamNonBlocking) != hipSuccess) break;
        tried[i] = c->stream2;  // kept until the end: its queue stays the more loaded one
        c->stream2 = other;
    }
    for (hipStream_t s : tried)
        if (s) (void)hipStreamDestroy(s);
    (void)hipGetLastError();
    return 0;
}

namespace {

// Systems from this size on choose the trailing-update tile by whole trial
// factorisations: how well the update GEMM overlaps the panel stream decides
// the factorisation time, and a GEMM timed alone does not show that.
constexpr int kTrialMinN = 8192;

// The working copy of precision T from the FP64 matrix Z.
template <typename T>
int load_working_copy(bem_ctx* c, T* Ar, T* Ai) {
    const size_t nn = (size_t)c->npad * c->npad;
    if constexpr (sizeof(T) == 8) {
        BEM_HIP(c, hipMemcpyAsync(Ar, c->Zr, nn * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
        BEM_HIP(c, hipMemcpyAsync(Ai, c->Zi, nn * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    } else {
        const size_t blocks = (nn + 255) / 256;
        hipLaunchKernelGGL(k_convert<float>, dim3(blocks), dim3(256), 0, c->stream, c->Zr, Ar, nn);
        hipLaunchKernelGGL(k_convert<float>, dim3(blocks), dim3(256), 0, c->stream, c->Zi, Ai, nn);
    }
    return 0;
}

// One timed factorisation of the context's matrix per tile configuration;
// the fastest becomes the plan's trailing-update tile.  Every configuration
// gives the same factors (same accumulation order), so the trials change
// nothing but the choice.  Sets *ran when the working copy was overwritten.
template <typename T>
int factor_trials(bem_ctx* c, T* Ar, T* Ai, void*& inv, size_t& inv_bytes, bool* ran) {
    GemmPlan& plan = c->gemm_plan[sizeof(T) == 4 ? 0 : 1];
    *ran = false;
    if (plan.trialed) return 0;
    if (c->npad < kTrialMinN) {
        plan.trialed = true;
        return 0;
    }
    if (!c->has_Z64) return 0;  // no source to restore the working copy from
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        return bem_fail(c, BEM_ERR_HIP, "LU trials: events");
    }
    *ran = true;
    int rc = 0;
    // FP32 tries the configurations of its trailing-update kernel (k_cupdate_nt),
    // FP64 the large tile of k_cgemm
    constexpr bool f32 = sizeof(T) == 4;
    const int ncfg = f32 ? kNtCfgs : kGemmTrialCfgs;
    for (int cfg = 0; cfg < ncfg && !rc; cfg++) {
        (f32 ? plan.nt : plan.large) = cfg;
        if ((rc = load_working_copy<T>(c, Ar, Ai))) break;
        (void)hipEventRecord(e0, c->stream);
        if ((rc = factor_prec<T>(c, Ar, Ai, inv, inv_bytes))) break;
        (void)hipEventRecord(e1, c->stream);
        if (hipEventSynchronize(e1) != hipSuccess) {
            rc = bem_fail(c, BEM_ERR_HIP, "LU trials: factorisation");
            break;
        }
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        plan.trial_ms[cfg] = ms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    // the fastest trial; among trials within 1 % of it (run-to-run noise),
    // FP64 takes the configuration with the higher rate timed alone, FP32 the
    // first (configuration 0 is the fastest alone).  (A 3 % band once took
    // the FP64 64 x 64 / K 8 tile at 368 ms over the 64 x 64 tile at 358 ms,
    // and its factorisations then took 372 ms against 361.)
    int best = 0;
    for (int cfg = 1; cfg < ncfg; cfg++)
        if (plan.trial_ms[cfg] < plan.trial_ms[best]) best = cfg;
    const double lim = 1.01 * plan.trial_ms[best];
    int pick = best;
    for (int cfg = 0; cfg < ncfg; cfg++) {
        if (plan.trial_ms[cfg] > lim) continue;
        if (f32 ? cfg < pick : plan.alone_tflops[cfg] > plan.alone_tflops[pick]) pick = cfg;
    }
    (f32 ? plan.nt : plan.large) = pick;
    if (rc) return rc;
    plan.trialed = true;
    gemm_cache_store(c, sizeof(T) == 4);
    return 0;
}

}  // namespace

int lu_factor_launch(bem_ctx* c, int precision) {
    const int n = c->npad;
    int rc = gemm_ensure_tuned(c, precision != BEM_F64);
    if (rc) return rc;
    if ((rc = lu_setup_streams(c))) return rc;
    bool trials = false;
    if (precision == BEM_F64) {
        void* no_inv = nullptr;  // FP64 factors keep no diagonal-block inverses
        size_t no_inv_bytes = 0;
        if ((rc = factor_trials<double>(c, c->Vr, c->Vi, no_inv, no_inv_bytes, &trials))) return rc;
        if ((rc = load_working_copy<double>(c, c->Vr, c->Vi))) return rc;
        rc = factor_prec<double>(c, c->Vr, c->Vi, no_inv, no_inv_bytes);
    } else {
        if ((rc = factor_trials<float>(c, c->Wr, c->Wi, c->inv32, c->inv32_bytes, &trials))) return rc;
        if (!c->has_Z32 || trials)
            if ((rc = load_working_copy<float>(c, c->Wr, c->Wi))) return rc;
        rc = factor_prec<float>(c, c->Wr, c->Wi, c->inv32, c->inv32_bytes);
    }
    if (rc) return rc;
    int info[2] = {0, 0};
    // swap sequence -> row permutation (row i of P Z is row perm[i] of Z)
    std::vector<int> ip(n), perm(n);
    auto fetch = [&]() -> int {
        BEM_HIP(c, hipGetLastError());
        void* scr = nullptr;
        if (int e = ctx_scratch(c, 256, &scr)) return e;
        return ctx_fetch(c, {{info, scr, sizeof(info)}, {ip.data(), c->ipiv, n * sizeof(int)}});
    };
    if ((rc = fetch())) return rc;
    if (info[1] && c->has_Z64) {  // FP32 pivots whose squares leave the range
        if ((rc = load_working_copy<float>(c, c->Wr, c->Wi))) return rc;
        if ((rc = factor_prec<float>(c, c->Wr, c->Wi, c->inv32, c->inv32_bytes, true))) return rc;
        if ((rc = fetch())) return rc;
    }
    for (int i = 0; i < n; i++) perm[i] = i;
    for (int i = 0; i < n; i++)
        if (ip[i] != i) std::swap(perm[i], perm[ip[i]]);
    if (int e = ctx_put(c, c->perm, perm.data(), n * sizeof(int))) return e;
    return info[0] > c->n ? 0 : info[0];  // a zero pivot inside the identity padding cannot occur
}
