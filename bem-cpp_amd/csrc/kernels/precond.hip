// precond.hip -- block-Jacobi / restricted additive Schwarz preconditioner
// on the dense matrix (precond.cu:407-895 build, 1303-1410 apply).
//
// The reference assembles each block's 2B x 2B PMCHWT matrix on the CPU
// from its own near-field quadrature, factors it with an unblocked
// partial-pivoting LU (precond.cu:636-868) and applies the factors with one
// warp per block (precond.cu:1303-1410).  On the dense path the block
// matrices are sub-matrices of Z, which is already on the device, and the
// apply has to serve all right-hand sides of an iteration at once, so here:
//   k_bj_gather  copies rows/columns {rwg_j, N + rwg_j : j in the extended
//                block} of the FP64 Z into a zero-padded n2max x n2max slot
//                per block (one launch for all blocks);
//   k_bj_panel, k_bj_inner, k_bj_rows, k_bj_update
//                invert every block in place by blocked Gauss-Jordan
//                elimination with the reference's pivoting (the largest
//                |a_ik| of the rows not used yet, precond.cu:842-851; a pivot
//                below 1e-30 in magnitude is replaced by 1e-15,
//                precond.cu:858-859);
//   apply        gathers each block's extended part of r into a padded slot,
//                multiplies the slots by their inverses on the matrix cores
//                (k_bj_mult), and scatters only the block's own unknowns
//                (restricted additive Schwarz; without overlap plain
//                block-Jacobi).
// The inverse gives the same M^{-1} r as the reference's LU solve up to
// rounding, at three times the factorisation work, and turns the apply into
// one matrix-core product instead of sequential substitutions.
#include <algorithm>
#include <cmath>
#include <vector>

#include "../bem_internal.h"
#include "../host/bem_host.h"
#include "gemm.h"

namespace {

// Block b: own size B[b], extended size Be[b] (own first), RWG list at
// rwg + roff[b], pivots at piv + poff[b]; its matrix (then inverse) is slot b
// of ld x ld (row-major per plane, zero beyond 2 Be).
struct BjView {
    const int *B, *Be, *rwg, *roff, *poff;
};

__device__ __forceinline__ int bj_row(const int* rwg, int Be, int N, int p) {
    return p < Be ? rwg[p] : N + rwg[p - Be];
}

__global__ __launch_bounds__(256) void k_bj_gather(BjView v, int N, int ld, const double* __restrict__ Zr,
                                                   const double* __restrict__ Zi, long ldz, double* __restrict__ Ar,
                                                   double* __restrict__ Ai) {
    const int b = blockIdx.x;
    const int Be = v.Be[b], n2 = 2 * Be;
    const int* rwg = v.rwg + v.roff[b];
    double* ar = Ar + (long)b * ld * ld;
    double* ai = Ai + (long)b * ld * ld;
    for (int p = blockIdx.y; p < n2; p += gridDim.y) {
        const long zr = (long)bj_row(rwg, Be, N, p) * ldz;
        for (int q = threadIdx.x; q < n2; q += blockDim.x) {
            const int zc = bj_row(rwg, Be, N, q);
            ar[(long)p * ld + q] = Zr[zr + zc];
            ai[(long)p * ld + q] = Zi[zr + zc];
        }
    }
}

// ---------------------------------------------------------------------------
// Inverse of every block by blocked Gauss-Jordan elimination in place, all
// blocks in each launch.  Rows are not interchanged: column k takes its pivot
// among the rows not used yet and remembers it in prow[k].  With slot k then
// holding the column of b_{prow[k]}, the result M at the end gives
//   x_k = sum_j M[prow_k][j] b_{prow_j},
// so the apply gathers r and scatters the result through prow and no row or
// column is ever moved.  For a set K of columns whose panel G (all rows of
// the columns K after their elimination) is known, every other column c is
//   a_ic <- (i in prow_K ? 0 : a_ic) + sum_{k in K} G_ik a_{prow_k, c}:
// an outer panel of 64 columns is eliminated in four inner panels of 16
// (k_bj_panel, then k_bj_inner for the other 48 columns of the panel), then
// the rest of the matrix takes one rank-64 product (k_bj_rows, k_bj_update).
//
// What bounds it: the rank-64 FP64 products (186 us each) and the panels' serial
// chain of pivot steps (44 us per 16 columns at 1107 unknowns, blocks side by
// side).  27 blocks of up to 1107 unknowns: 9.0 ms, where one
// workgroup sweeping its whole block from memory at every pivot step (the
// earlier form) took 1600 ms, n2^2 complex values moved per step.
// ---------------------------------------------------------------------------
constexpr int BJ_W = 16;   // inner panel
constexpr int BJ_O = 64;   // outer panel
constexpr int BJ_T = 512;  // threads of k_bj_panel (256 threads with twice the rows each measured the same)
constexpr int BJ_MAXR = 3; // rows per thread it can hold in registers (64 registers each)

// |z|^2, 0 for a NaN: a column always has a pivot.
__device__ __forceinline__ double bj_mag(double r, double i) { return fmax(r * r + i * i, 0.0); }

extern "C" __device__ unsigned __ockl_wfred_max_u32(unsigned);
// Maximum over the eight lanes of each row half (DPP).
__device__ __forceinline__ unsigned bj_max8(unsigned v) {
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, false));  // quad_perm [1, 0, 3, 2]
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, false));  // [2, 3, 0, 1]
    return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));  // row_half_mirror
}

// A lane's candidate: the upper word of its |z|^2 plus one (0: none), the lower word, its row.
struct BjCand {
    unsigned hi, lo, row;
};
// The first lane with the largest candidate (ties: the lowest row) of the wave, or of its
// first eight lanes: by the upper word, which mostly decides, then the lower, then the row.
template <bool EIGHT>
__device__ __forceinline__ int bj_best_lane(const BjCand& k) {
    auto top = [](unsigned v) { return EIGHT ? bj_max8(v) : __ockl_wfred_max_u32(v); };
    constexpr unsigned long long kLanes = EIGHT ? 0xffull : ~0ull;
    unsigned long long mask = __ballot(k.hi == top(k.hi)) & kLanes;
    if (__popcll(mask) > 1) {
        const int lane = threadIdx.x & 63;
        const unsigned lo = (mask >> lane) & 1ull ? k.lo : 0u;
        mask &= __ballot(lo == top(lo));
        const unsigned low = (mask >> lane) & 1ull ? ~k.row : 0u;
        mask &= __ballot(low == top(low));
    }
    return __ffsll((long long)mask) - 1;
}

// Columns of unrolled elimination steps; the registers rotate by so many after them.
// (All 16 steps unrolled, each row read ahead whole and with two selects per value
// for the pivot row, took 98 us per panel of 1107 rows, 44 now.  With three rows per
// thread, those rows' included, the kernel takes all 256 registers and spills eight.)
constexpr int BJ_S = 4;

// Entries BJ_S .. to the front, the first BJ_S to the end.
__device__ __forceinline__ void bj_rotate(double (&x)[BJ_W]) {
    double h[BJ_S];
#pragma unroll
    for (int c = 0; c < BJ_S; c++) h[c] = x[c];
#pragma unroll
    for (int c = 0; c < BJ_W - BJ_S; c++) x[c] = x[c + BJ_S];
#pragma unroll
    for (int c = 0; c < BJ_S; c++) x[BJ_W - BJ_S + c] = h[c];
}

// The BJ_W columns of rows i0 .. i0+63 from / to memory (rows n2 and beyond: some other
// row, nothing), row i0 + lane in the lane's registers.  Four lanes take 64 bytes of a row
// side by side and the wave's part of LDS turns them (a lane read its own row, 16
// bytes of 64 lines per load).  The LDS operations of a wave
// stay in order, so the buffer needs no barrier.
struct alignas(16) BjStage {
    double x[64][BJ_W / 2 + 2];
};
__device__ __forceinline__ void bj_load_rows(const double* __restrict__ a, int ld, int i0, int n2, BjStage& st,
                                             double (&x)[BJ_W]) {
    const int lane = threadIdx.x & 63, r = lane / 4, c = 2 * (lane % 4);
    v2d v[2][4];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = min(i0 + 16 * u + r, n2 - 1);
            v[h][u] = *reinterpret_cast<const v2d*>(a + (long)i * ld + 8 * h + c);
        }
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int u = 0; u < 4; u++) *reinterpret_cast<v2d*>(&st.x[16 * u + r][c]) = v[h][u];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const v2d y = *reinterpret_cast<const v2d*>(&st.x[lane][2 * k]);
            x[8 * h + 2 * k] = y[0];
            x[8 * h + 2 * k + 1] = y[1];
        }
        __builtin_amdgcn_wave_barrier();
    }
}
__device__ __forceinline__ void bj_store_rows(double* __restrict__ a, int ld, int i0, int n2, BjStage& st,
                                              const double (&x)[BJ_W]) {
    const int lane = threadIdx.x & 63, r = lane / 4, c = 2 * (lane % 4);
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            *reinterpret_cast<v2d*>(&st.x[lane][2 * k]) = v2d{x[8 * h + 2 * k], x[8 * h + 2 * k + 1]};
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + 16 * u + r;
            if (i < n2)
                *reinterpret_cast<v2d*>(a + (long)i * ld + 8 * h + c) = *reinterpret_cast<const v2d*>(&st.x[16 * u + r][c]);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Elimination of columns c0 .. c0+15 of every block, one workgroup each.
// RPT > 0: the panel's rows in registers, rows t + BJ_T r, r < RPT (n2 <= RPT
// BJ_T); RPT == 0: the panel stays in memory (any n2).  step[row] is the
// column a row is the pivot of (-1: none yet).  The pivot is the largest |a|^2
// (ties: the lowest row) of the unused rows; a pivot below 1e-30 in modulus is
// replaced by 1e-15 (precond.cu:842-859).
// At the end the pivot rows' entries in the outer panel's 64 columns (from k0)
// go to Bin (16 x 64 per plane and block).
template <int RPT>
__global__ __launch_bounds__(BJ_T) void k_bj_panel(BjView v, int ld, int c0, int k0, double* __restrict__ Ar,
                                                   double* __restrict__ Ai, int* __restrict__ step,
                                                   int* __restrict__ prow, double* __restrict__ Bin) {
    constexpr int NW = BJ_T / 64, R = RPT > 0 ? RPT : 1;
    __shared__ BjCand kb[NW];  // the waves' candidates
    __shared__ double row_r[BJ_W], row_i[BJ_W];
    __shared__ int prows[BJ_W];
    __shared__ BjStage stage[RPT > 0 ? NW : 1];
    const int b = blockIdx.x, t = threadIdx.x, wave = t >> 6;
    const int n2 = 2 * v.Be[b];
    if (c0 >= n2) return;
    const int w = min(BJ_W, n2 - c0);
    double* ar = Ar + (long)b * ld * ld + c0;
    double* ai = Ai + (long)b * ld * ld + c0;
    int* st = step + (long)b * ld;
    double xr[R][BJ_W], xi[R][BJ_W];
    int used[R];
    if constexpr (RPT > 0) {
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int i = t + BJ_T * q;
            used[q] = i < n2 ? st[i] : 0;
            bj_load_rows(ar, ld, i - (t & 63), n2, stage[wave], xr[q]);
            bj_load_rows(ai, ld, i - (t & 63), n2, stage[wave], xi[q]);
        }
    }
#pragma unroll 1
    for (int s = 0; s < BJ_W; s += BJ_S) {
        // register c holds column (c + s) % BJ_W of the panel
#pragma unroll
        for (int j = 0; j < BJ_S; j++) {
            if (s + j < w) {  // the same for the whole workgroup; a break would keep the loop from unrolling
                double big = -1.0;
                int best = 0x7fffffff;
                if constexpr (RPT > 0) {
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        const double m = used[q] < 0 ? bj_mag(xr[q][j], xi[q][j]) : -1.0;
                        if (m > big) {
                            big = m;
                            best = t + BJ_T * q;
                        }
                    }
                } else {
                    for (int i = t; i < n2; i += BJ_T) {
                        const double m = st[i] < 0 ? bj_mag(ar[(long)i * ld + s + j], ai[(long)i * ld + s + j]) : -1.0;
                        if (m > big) {
                            big = m;
                            best = i;
                        }
                    }
                }
                const unsigned long long u = (unsigned long long)__double_as_longlong(big);
                const BjCand mine{big >= 0.0 ? (unsigned)(u >> 32) + 1u : 0u, (unsigned)u, (unsigned)best};
                if ((t & 63) == bj_best_lane<false>(mine)) kb[wave] = mine;
                __syncthreads();
                const BjCand all = kb[t & (NW - 1)];
                static_assert(NW == 8, "a wave's first eight lanes hold every wave's candidate");
                // some row is unused: n2 pivots over n2 steps
                const int p = __builtin_amdgcn_readlane((int)all.row, bj_best_lane<true>(all));
                if (p % BJ_T == t) {
                    if constexpr (RPT > 0) {
#pragma unroll
                        for (int q = 0; q < R; q++)
                            if (p == t + BJ_T * q) {
                                used[q] = c0 + s + j;
#pragma unroll
                                for (int c = 0; c < BJ_W; c++) {
                                    row_r[c] = xr[q][c];
                                    row_i[c] = xi[q][c];
                                    xr[q][c] = xi[q][c] = 0.0;
                                }
                            }
                    } else {
#pragma unroll
                        for (int c = 0; c < BJ_W; c++) {
                            const long o = (long)p * ld + (c + s) % BJ_W;
                            row_r[c] = ar[o];
                            row_i[c] = ai[o];
                            ar[o] = ai[o] = 0.0;
                        }
                    }
                    st[p] = c0 + s + j;
                    prows[s + j] = p;
                }
                __syncthreads();
                double dr = row_r[j], di = row_i[j];
                if (dr * dr + di * di < 1e-60) {
                    dr = 1e-15;
                    di = 0.0;
                }
                const double inv = 1.0 / (dr * dr + di * di), qr = dr * inv, qi = -di * inv;  // 1 / pivot
                // row i: a_ic -= g u_c (c != j), a_ij = -g, g = a_ij / pivot; the pivot
                // row, cleared above, the same with g = -1 / pivot: a_pc = u_c / pivot,
                // a_pj = 1 / pivot
                auto eliminate = [&](int i0, double (&yr)[R][BJ_W], double (&yi)[R][BJ_W]) {
                    double gr[R], gi[R];
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        const bool piv = i0 + BJ_T * q == p;
                        const double fr = yr[q][j], fi = yi[q][j];
                        gr[q] = piv ? -qr : fr * qr - fi * qi;
                        gi[q] = piv ? -qi : fr * qi + fi * qr;
                    }
#pragma unroll
                    for (int c = 0; c < BJ_W; c++) {
                        if (c != j) {
                            const double ur = row_r[c], ui = row_i[c];
#pragma unroll
                            for (int q = 0; q < R; q++) {
                                yr[q][c] = fma(gi[q], ui, fma(-gr[q], ur, yr[q][c]));
                                yi[q][c] = fma(-gi[q], ur, fma(-gr[q], ui, yi[q][c]));
                            }
                        }
                        // (more of the row read ahead does not fit in the registers)
                        if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        yr[q][j] = -gr[q];
                        yi[q][j] = -gi[q];
                    }
                };
                if constexpr (RPT > 0) {
                    eliminate(t, xr, xi);
                } else {
                    for (int i = t; i < n2; i += BJ_T) {
#pragma unroll
                        for (int c = 0; c < BJ_W; c++) {
                            xr[0][c] = ar[(long)i * ld + (c + s) % BJ_W];
                            xi[0][c] = ai[(long)i * ld + (c + s) % BJ_W];
                        }
                        eliminate(i, xr, xi);
#pragma unroll
                        for (int c = 0; c < BJ_W; c++) {
                            ar[(long)i * ld + (c + s) % BJ_W] = xr[0][c];
                            ai[(long)i * ld + (c + s) % BJ_W] = xi[0][c];
                        }
                    }
                }
                // (a thread reads the row before it reaches the next step's first
                // barrier, the keys before this step's second)
            }
        }
        if constexpr (RPT > 0) {
#pragma unroll
            for (int q = 0; q < R; q++) {
                bj_rotate(xr[q]);
                bj_rotate(xi[q]);
            }
        }
    }
    if constexpr (RPT > 0) {
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int i = t + BJ_T * q;
            bj_store_rows(ar, ld, i - (t & 63), n2, stage[wave], xr[q]);
            bj_store_rows(ai, ld, i - (t & 63), n2, stage[wave], xi[q]);
        }
    }
    if (t < w) prow[v.poff[b] + c0 + t] = prows[t];
    if (!Bin) return;
    double* br = Bin + (long)b * 2 * BJ_W * BJ_O;
    double* bi = br + BJ_W * BJ_O;
    const int off = k0 - c0;  // the outer panel's first column relative to c0
    for (int e = t; e < BJ_W * BJ_O; e += BJ_T) {
        const int k = e / BJ_O, c = e % BJ_O;
        const bool in = k < w && !(c + off >= 0 && c + off < BJ_W);  // the panel's own columns are not used
        br[e] = in ? ar[(long)prows[k] * ld + off + c] : 0.0;
        bi[e] = in ? ai[(long)prows[k] * ld + off + c] : 0.0;
    }
}

// The other columns of the outer panel [k0, k0 + 64) after the inner panel at
// c0: 32 rows per workgroup (blockIdx.y), one column and 8 rows per thread, G
// and the pivot rows from LDS.
__global__ __launch_bounds__(256) void k_bj_inner(BjView v, int ld, int c0, int k0, double* __restrict__ Ar,
                                                  double* __restrict__ Ai, const int* __restrict__ step,
                                                  const double* __restrict__ Bin) {
    __shared__ double gr[32][BJ_W + 1], gi[32][BJ_W + 1], ur[BJ_W][BJ_O], ui[BJ_W][BJ_O];
    const int b = blockIdx.x, t = threadIdx.x, i0 = blockIdx.y * 32;
    const int n2 = 2 * v.Be[b];
    if (c0 >= n2 || i0 >= n2) return;
    double* ar = Ar + (long)b * ld * ld;
    double* ai = Ai + (long)b * ld * ld;
    const double* br = Bin + (long)b * 2 * BJ_W * BJ_O;
    for (int e = t; e < BJ_W * BJ_O; e += 256) {
        ur[e / BJ_O][e % BJ_O] = br[e];
        ui[e / BJ_O][e % BJ_O] = br[BJ_W * BJ_O + e];
    }
    for (int e = t; e < 32 * BJ_W; e += 256) {
        const int i = e / BJ_W, k = e % BJ_W;
        const bool in = i0 + i < n2;
        gr[i][k] = in ? ar[(long)(i0 + i) * ld + c0 + k] : 0.0;
        gi[i][k] = in ? ai[(long)(i0 + i) * ld + c0 + k] : 0.0;
    }
    // the rows' values and steps all in flight before the first is used (one row after
    // the other waited for memory twice each: 20.7 us per panel of 27 blocks of 1107 unknowns, 17.1 now; 60 MB, 12 us)
    constexpr int LANES = 256 / BJ_O, RW = 32 / LANES;
    const int col = t % BJ_O, c = k0 + col, r0 = t / BJ_O;  // rows i0 + r0 + LANES u
    const bool mine = c < n2 && !(c >= c0 && c < c0 + BJ_W);
    double sr[RW], si[RW];
    int st[RW];
#pragma unroll
    for (int u = 0; u < RW; u++) {
        const int i = min(i0 + r0 + LANES * u, n2 - 1);
        const long o = (long)i * ld + c;  // (c < ld)
        st[u] = step[(long)b * ld + i];
        sr[u] = ar[o];
        si[u] = ai[o];
    }
    __syncthreads();
    if (!mine) return;
#pragma unroll
    for (int u = 0; u < RW; u++) {
        const bool piv = st[u] >= c0 && st[u] < c0 + BJ_W;
        sr[u] = piv ? 0.0 : sr[u];
        si[u] = piv ? 0.0 : si[u];
    }
#pragma unroll 4
    for (int k = 0; k < BJ_W; k++) {
        const double pr = ur[k][col], pi = ui[k][col];
#pragma unroll
        for (int u = 0; u < RW; u++) {
            const double a = gr[r0 + LANES * u][k], d = gi[r0 + LANES * u][k];
            sr[u] += a * pr - d * pi;
            si[u] += a * pi + d * pr;
        }
    }
#pragma unroll
    for (int u = 0; u < RW; u++) {
        const int i = i0 + r0 + LANES * u;
        if (i < n2) {
            ar[(long)i * ld + c] = sr[u];
            ai[(long)i * ld + c] = si[u];
        }
    }
}

// The outer panel's pivot rows before its rank-64 product: Bo (64 x ld per
// plane and block), rows beyond n2 zero.
__global__ __launch_bounds__(256) void k_bj_rows(BjView v, int ld, int k0, const double* __restrict__ Ar,
                                                 const double* __restrict__ Ai, const int* __restrict__ prow,
                                                 double* __restrict__ Bo) {
    const int b = blockIdx.x, k = blockIdx.y;
    const int n2 = 2 * v.Be[b];
    if (k0 >= n2) return;
    const bool in = k0 + k < n2;
    const long src = (long)b * ld * ld + (in ? (long)prow[v.poff[b] + k0 + k] * ld : 0);
    double* br = Bo + (long)b * 2 * BJ_O * ld + (long)k * ld;
    double* bi = br + (long)BJ_O * ld;
    for (int c = threadIdx.x; c < ld; c += 256) {
        br[c] = in ? Ar[src + c] : 0.0;
        bi[c] = in ? Ai[src + c] : 0.0;
    }
}

// The columns outside the outer panel [k0, k0 + 64): 64 x 64 tiles
// (workgroup = block + nb (tile column + nt tile row)), each of the four waves a 32 x 32 sub-tile.  The operands go straight from memory to
// the registers of v_mfma_f64_16x16x4f64 (K is only 64 and the tiles' rows are
// shared through the caches): lane (r, g) holds G[row r][4g + s] and
// Bo[4g + s][col r] for product s = 0..3 of a 16-wide piece of K.  Tiles
// beyond a block's own size end at once.
__global__ __launch_bounds__(256) void k_bj_update(BjView v, int nb, int ld, int k0, int nt,
                                                   double* __restrict__ Ar, double* __restrict__ Ai,
                                                   const int* __restrict__ step, const double* __restrict__ Bo) {
    const int b = blockIdx.x % nb, tile = blockIdx.x / nb, tm = tile / nt, tn = tile % nt;
    const int n2 = 2 * v.Be[b];
    if (k0 >= n2 || tm * 64 >= n2 || tn * 64 >= n2 || tn * 64 == k0) return;
    double* ar = Ar + (long)b * ld * ld;
    double* ai = Ai + (long)b * ld * ld;
    const double* br = Bo + (long)b * 2 * BJ_O * ld;
    const double* bi = br + (long)BJ_O * ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int m0 = tm * 64 + (wave >> 1) * 32, n0 = tn * 64 + (wave & 1) * 32;
    v4d acc[2][2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[p][i][j] = v4d{};
#pragma unroll
    for (int kk = 0; kk < BJ_O; kk += 16) {
        double a[2][2][4], u[2][2][4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const long oa = (long)(m0 + 16 * i + r) * ld + k0 + kk + 4 * g;
            load_row4<double>(ar + oa, a[0][i]);
            load_row4<double>(ai + oa, a[1][i]);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const long ob = (long)(kk + 4 * g + s) * ld + n0 + 16 * i + r;
                u[0][i][s] = br[ob];
                u[1][i][s] = bi[ob];
            }
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    acc[0][i][j] = mfma16x16x4(a[0][i][s], u[0][j][s], acc[0][i][j]);
                    acc[0][i][j] = mfma16x16x4(a[1][i][s], -u[1][j][s], acc[0][i][j]);
                    acc[1][i][j] = mfma16x16x4(a[0][i][s], u[1][j][s], acc[1][i][j]);
                    acc[1][i][j] = mfma16x16x4(a[1][i][s], u[0][j][s], acc[1][i][j]);
                }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int row = m0 + 16 * i + g + 4 * q;
            if (row >= n2) continue;
            const int s = step[(long)b * ld + row];
            const bool clear = s >= k0 && s < k0 + BJ_O;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const long o = (long)row * ld + n0 + 16 * j + r;
                ar[o] = (clear ? 0.0 : ar[o]) + acc[0][i][j][q];
                ai[o] = (clear ? 0.0 : ai[o]) + acc[1][i][j][q];
            }
        }
}

// Slot b of S (ld x ncol per plane) = the extended block of r in pivot order
// (row k: r at row prow[k] of the block; rows beyond 2 Be stay zero); rows
// blockIdx.y, blockIdx.y + gridDim.y, ... of a block per workgroup.
__global__ __launch_bounds__(256) void k_bj_gather_vec(BjView v, int N, int ld, int ncol,
                                                       const int* __restrict__ prow, const double* __restrict__ Rr,
                                                       const double* __restrict__ Ri, double* __restrict__ Sr,
                                                       double* __restrict__ Si) {
    const int b = blockIdx.x;
    const int Be = v.Be[b], n2 = 2 * Be;
    const int* rwg = v.rwg + v.roff[b];
    const int* pr = prow + v.poff[b];
    double* sr = Sr + (long)b * ld * ncol;
    double* si = Si + (long)b * ld * ncol;
    for (long e = (long)blockIdx.y * 256 + threadIdx.x; e < (long)ld * ncol; e += 256L * gridDim.y) {
        const int p = (int)(e / ncol), j = (int)(e % ncol);
        const long g = p < n2 ? (long)bj_row(rwg, Be, N, pr[p]) * ncol + j : 0;
        sr[e] = p < n2 ? Rr[g] : 0.0;
        si[e] = p < n2 ? Ri[g] : 0.0;
    }
}

// Y_b = M_b S_b for every block (rows in the storage order of M): one 16 x
// (16 NT) tile per workgroup (blockIdx.x = block + nb row tile, columns
// blockIdx.y), the four waves each a quarter of K in 16-wide pieces straight
// from memory, summed through LDS in wave order.  Bound by reading M once per
// 16 NT columns; a tile beyond the block's own size ends at once and K stops
// there (16 columns, the blocks above: 90 us; the batched 64 x 64 tile product
// over the padded slots took 527 us).
template <int NT>
__global__ __launch_bounds__(256) void k_bj_mult(BjView v, int nb, int ld, int ncol,
                                                 const double* __restrict__ Ar, const double* __restrict__ Ai,
                                                  const double* __restrict__ Sr,
                                                 const double* __restrict__ Si, double* __restrict__ Yr,
                                                 double* __restrict__ Yi) {
    __shared__ double red[4][2][16][17];
    const int b = blockIdx.x % nb, m0 = blockIdx.x / nb * 16, n0 = blockIdx.y * 16 * NT;
    const int n2 = 2 * v.Be[b];
    if (m0 >= n2) return;
    const double* ar = Ar + (long)b * ld * ld;
    const double* ai = Ai + (long)b * ld * ld;
    const double* sr = Sr + (long)b * ld * ncol;
    const double* si = Si + (long)b * ld * ncol;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    v4d acc[2][NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[0][j] = acc[1][j] = v4d{};
    for (int kk = wave * 16; kk < n2; kk += 64) {  // rows and columns up to ld (a multiple of 64) are zero beyond n2
        double a[2][4], u[NT][2][4];
        const long oa = (long)(m0 + r) * ld + kk + 4 * g;
        load_row4<double>(ar + oa, a[0]);
        load_row4<double>(ai + oa, a[1]);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const long ob = (long)(kk + 4 * g + s) * ncol + n0 + 16 * j + r;
                u[j][0][s] = sr[ob];
                u[j][1][s] = si[ob];
            }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                acc[0][j] = mfma16x16x4(a[0][s], u[j][0][s], acc[0][j]);
                acc[0][j] = mfma16x16x4(a[1][s], -u[j][1][s], acc[0][j]);
                acc[1][j] = mfma16x16x4(a[0][s], u[j][1][s], acc[1][j]);
                acc[1][j] = mfma16x16x4(a[1][s], u[j][0][s], acc[1][j]);
            }
    }
    const int row = threadIdx.x / 16, col = threadIdx.x % 16;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        if (j) __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            red[wave][0][g + 4 * q][r] = acc[0][j][q];
            red[wave][1][g + 4 * q][r] = acc[1][j][q];
        }
        __syncthreads();
        const long o = (long)b * ld * ncol + (long)(m0 + row) * ncol + n0 + 16 * j + col;
        Yr[o] = ((red[0][0][row][col] + red[1][0][row][col]) + red[2][0][row][col]) + red[3][0][row][col];
        Yi[o] = ((red[0][1][row][col] + red[1][1][row][col]) + red[2][1][row][col]) + red[3][1][row][col];
    }
}

// z at the block's own unknowns k in {0..B-1, Be..Be+B-1} = row prow[k] of slot b of Y.
__global__ __launch_bounds__(256) void k_bj_scatter(BjView v, int N, int ld, int ncol,
                                                    const int* __restrict__ prow, const double* __restrict__ Yr,
                                                    const double* __restrict__ Yi, double* __restrict__ Zr,
                                                    double* __restrict__ Zi) {
    const int b = blockIdx.x;
    const int B = v.B[b], Be = v.Be[b];
    const int* rwg = v.rwg + v.roff[b];
    const double* yr = Yr + (long)b * ld * ncol;
    const double* yi = Yi + (long)b * ld * ncol;
    const int* pr = prow + v.poff[b];
    for (long e = (long)blockIdx.y * 256 + threadIdx.x; e < 2L * B * ncol; e += 256L * gridDim.y) {
        const int q = (int)(e / ncol), j = (int)(e % ncol);
        const int p = q < B ? q : Be + (q - B);
        const long g = (long)bj_row(rwg, Be, N, p) * ncol + j;
        Zr[g] = yr[(long)pr[p] * ncol + j];
        Zi[g] = yi[(long)pr[p] * ncol + j];
    }
}

// rows [n, npad) of the padded system: the identity
__global__ __launch_bounds__(256) void k_copy_tail(long from, long count, const double* __restrict__ Rr,
                                                   const double* __restrict__ Ri, double* __restrict__ Zr,
                                                   double* __restrict__ Zi) {
    const long e = from + (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    Zr[e] = Rr[e];
    Zi[e] = Ri[e];
}

template <typename E>
int upload(bem_ctx* c, E*& dst, const std::vector<E>& src, const char* what) {
    if (hipMalloc((void**)&dst, std::max<size_t>(1, src.size()) * sizeof(E)) != hipSuccess) {
        dst = nullptr;
        return bem_fail(c, BEM_ERR_NOMEM, std::string("block_jacobi: ") + what);
    }
    BEM_HIP(c, hipMemcpy((void*)dst, src.data(), src.size() * sizeof(E), hipMemcpyHostToDevice));
    return 0;
}

}  // namespace

void bj_free(bem_ctx* c) {
    BlockJacobi& J = c->bj;
    for (void* p : {(void*)J.rwg, (void*)J.B, (void*)J.Be, (void*)J.roff, (void*)J.poff, (void*)J.Ar, (void*)J.Ai,
                    (void*)J.piv})
        if (p) (void)hipFree(p);
    J = BlockJacobi{};
}

int bj_build_launch(bem_ctx* c, double radius_mult, int max_block_rwg, int overlap_layers, double* t_ms) {
    Timer tm;
    const int N = c->rwg.N;
    const BlockPartition P = block_partition(c->mesh, c->rwg, c->quad, radius_mult, max_block_rwg, overlap_layers);
    const int nb = (int)P.own.size();
    if (nb == 0) return bem_fail(c, BEM_ERR_MESH, "block_jacobi: no unknowns");
    std::vector<int> B(nb), Be(nb), roff(nb), poff(nb), rwg;
    long piv_total = 0;
    int n2max = 0;
    for (int b = 0; b < nb; b++) {
        B[b] = (int)P.own[b].size();
        Be[b] = (int)P.ext[b].size();
        if (B[b] < 1 || Be[b] < B[b]) return bem_fail(c, BEM_ERR_STATE, "block_jacobi: inconsistent partition");
        roff[b] = (int)rwg.size();
        for (int m : P.ext[b]) {
            if (m < 0 || m >= N) return bem_fail(c, BEM_ERR_STATE, "block_jacobi: RWG index out of range");
            rwg.push_back(m);
        }
        poff[b] = (int)piv_total;
        piv_total += 2L * Be[b];
        n2max = std::max(n2max, 2 * Be[b]);
    }
    const int ld = (n2max + 63) / 64 * 64;  // slot side: a multiple of the GEMM tile
    const size_t slot = (size_t)ld * ld;
    bj_free(c);
    BlockJacobi& J = c->bj;
    int rc = upload(c, J.rwg, rwg, "RWG lists");
    if (!rc) rc = upload(c, J.B, B, "sizes");
    if (!rc) rc = upload(c, J.Be, Be, "sizes");
    if (!rc) rc = upload(c, J.roff, roff, "offsets");
    if (!rc) rc = upload(c, J.poff, poff, "offsets");
    if (rc) {
        bj_free(c);
        return rc;
    }
    if (hipMalloc((void**)&J.Ar, nb * slot * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&J.Ai, nb * slot * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&J.piv, piv_total * sizeof(int)) != hipSuccess) {
        bj_free(c);
        return bem_fail(c, BEM_ERR_NOMEM, "block_jacobi: inverses (" + std::to_string(nb * slot * 16) + " bytes)");
    }
    // scratch of the elimination: pivot rows of an inner and of an outer panel,
    // and per row the column it is the pivot of
    // (none where one panel holds every block)
    const size_t nbin = n2max > BJ_W ? 2 * (size_t)nb * BJ_W * BJ_O : 0;
    const size_t nbo = n2max > BJ_O ? 2 * (size_t)nb * BJ_O * ld : 0;
    void* scr = nullptr;
    if (int e = ctx_scratch(c, (nbin + nbo) * sizeof(double) + (size_t)nb * ld * sizeof(int), &scr)) {
        bj_free(c);
        return e;
    }
    double* Bin = static_cast<double*>(scr);
    double* Bo = Bin + nbin;
    int* step = reinterpret_cast<int*>(Bo + nbo);
    J.nb = nb;
    J.n2max = n2max;
    J.ld = ld;
    J.bytes = nb * slot * 16;
    J.N = N;
    J.own = P.own;
    J.ext = P.ext;
    const BjView v{J.B, J.Be, J.rwg, J.roff, J.poff};
    hipStream_t s = c->stream;
    BEM_HIP(c, hipMemsetAsync(J.Ar, 0, nb * slot * sizeof(double), s));
    BEM_HIP(c, hipMemsetAsync(J.Ai, 0, nb * slot * sizeof(double), s));
    hipLaunchKernelGGL(k_bj_gather, dim3(nb, 64), dim3(256), 0, s, v, N, ld, c->Zr, c->Zi, (long)c->npad, J.Ar,
                       J.Ai);
    BEM_HIP(c, hipMemsetAsync(step, 0xff, (size_t)nb * ld * sizeof(int), s));
    // rows per thread of the panel kernel: in registers up to BJ_MAXR BJ_T
    // rows, from memory beyond
    const int rpt = (n2max + BJ_T - 1) / BJ_T, nt = ld / 64;
    for (int k0 = 0; k0 < n2max; k0 += BJ_O) {
        for (int c0 = k0; c0 < std::min(n2max, k0 + BJ_O); c0 += BJ_W) {
            auto panel = rpt == 1 ? k_bj_panel<1> : rpt == 2 ? k_bj_panel<2> : rpt <= BJ_MAXR ? k_bj_panel<3>
                                                                                                 : k_bj_panel<0>;
            hipLaunchKernelGGL(panel, dim3(nb), dim3(BJ_T), 0, s, v, ld, c0, k0, J.Ar, J.Ai, step, J.piv,
                               nbin ? Bin : nullptr);
            if (nbin)
                hipLaunchKernelGGL(k_bj_inner, dim3(nb, (n2max + 31) / 32), dim3(256), 0, s, v, ld, c0, k0, J.Ar,
                                   J.Ai, (const int*)step, (const double*)Bin);
        }
        if (n2max <= BJ_O) break;
        hipLaunchKernelGGL(k_bj_rows, dim3(nb, BJ_O), dim3(256), 0, s, v, ld, k0, (const double*)J.Ar,
                           (const double*)J.Ai, (const int*)J.piv, Bo);
        hipLaunchKernelGGL(k_bj_update, dim3(nb * nt * nt), dim3(256), 0, s, v, nb, ld, k0, nt, J.Ar, J.Ai,
                           (const int*)step, (const double*)Bo);
    }
    BEM_HIP(c, hipGetLastError());
    BEM_HIP(c, hipStreamSynchronize(s));
    J.valid = true;
    *t_ms = tm.elapsed_ms();
    return nb;
}

size_t bj_work_bytes(const bem_ctx* c) {
    return 4 * (size_t)c->bj.nb * c->bj.ld * c->ldr * sizeof(double);
}

int bj_apply(bem_ctx* c, const double* Rr, const double* Ri, double* Zr, double* Zi, void* work) {
    BlockJacobi& J = c->bj;
    if (!J.valid || J.N * 2 != c->n) return bem_fail(c, BEM_ERR_STATE, "block_jacobi: not built for this system");
    const int ncol = c->ldr, ld = J.ld, nb = J.nb;
    const size_t vs = (size_t)nb * ld * ncol;
    double* Sr = static_cast<double*>(work);
    double* Si = Sr + vs;
    double* Yr = Si + vs;
    double* Yi = Yr + vs;
    hipStream_t s = c->stream;
    const BjView v{J.B, J.Be, J.rwg, J.roff, J.poff};
    const unsigned gy = (unsigned)std::min<long>(64, ((long)ld * ncol + 1023) / 1024);
    hipLaunchKernelGGL(k_bj_gather_vec, dim3(nb, gy), dim3(256), 0, s, v, J.N, ld, ncol, (const int*)J.piv, Rr, Ri,
                       Sr, Si);
    const int tiles = ncol / 16;  // ldr is a multiple of 16
    const unsigned mt = (unsigned)((J.n2max + 15) / 16);
    if (tiles % 4 == 0)
        hipLaunchKernelGGL(k_bj_mult<4>, dim3(nb * mt, tiles / 4), dim3(256), 0, s, v, nb, ld, ncol, (const double*)J.Ar,
                           (const double*)J.Ai, (const double*)Sr, (const double*)Si, Yr, Yi);
    else if (tiles % 2 == 0)
        hipLaunchKernelGGL(k_bj_mult<2>, dim3(nb * mt, tiles / 2), dim3(256), 0, s, v, nb, ld, ncol, (const double*)J.Ar,
                           (const double*)J.Ai, (const double*)Sr, (const double*)Si, Yr, Yi);
    else
        hipLaunchKernelGGL(k_bj_mult<1>, dim3(nb * mt, tiles), dim3(256), 0, s, v, nb, ld, ncol, (const double*)J.Ar,
                           (const double*)J.Ai, (const double*)Sr, (const double*)Si, Yr, Yi);
    hipLaunchKernelGGL(k_bj_scatter, dim3(nb, gy), dim3(256), 0, s, v, J.N, ld, ncol, (const int*)J.piv, Yr, Yi, Zr,
                       Zi);
    const long from = (long)c->n * ncol, count = (long)c->npad * ncol;
    if (count > from)
        hipLaunchKernelGGL(k_copy_tail, dim3((unsigned)((count - from + 255) / 256)), dim3(256), 0, s, from, count,
                           Rr, Ri, Zr, Zi);
    BEM_HIP(c, hipGetLastError());
    return 0;
}
