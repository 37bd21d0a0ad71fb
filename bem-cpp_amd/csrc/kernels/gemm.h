// gemm.h -- complex GEMM on CDNA4 matrix cores, planar operands.
//
//   C = C - A B   (mode 0)     C = A B   (mode 1)
//
// A is M x K, B is K x N, C is M x N; every matrix is stored as two planes
// (real, imaginary) in row-major order with its own leading dimension.
//
// FP32 uses the 3M form: three real products T1 = Ar Br, T2 = Ai Bi,
// T3 = (Ar + Ai)(Br + Bi) accumulate on v_mfma_f32_16x16x4f32, and the
// epilogue forms Re = T1 - T2, Im = T3 - T1 - T2 (3/4 of the real flops of the
// 4M form).  FP64 uses the 4M form on v_mfma_f64_16x16x4f64 with two
// accumulators (Re += Ar Br - Ai Bi, Im += Ar Bi + Ai Br).
//
// Tiling: 256 threads = 4 waves of 64 in a 2 x 2 arrangement; a K slice of BK
// is staged through LDS (k-major, double buffered, one barrier per slice);
// each wave owns a WM x WN sub-tile made of 16 x 16 MFMA tiles.
// MFMA 16x16x4 operand layout (wave64): A[i][k] in lane i + 16k, B[k][j] in
// lane j + 16k.  Result D[i][j]: f32 form in lane j + 16 (i / 4), register
// i % 4; f64 form in lane j + 16 (i % 4), register i / 4 (measured on gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

__device__ __forceinline__ v4f mfma16x16x4(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4d mfma16x16x4(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Tile configurations, indexed per precision (0, 1, 2): block BM x BN, wave
// tile WM x WN (4 waves in 2 x 2), K slice BK.  MINB: workgroups per CU the
// register allocation must allow (two per CU let one block's prologue and C
// update overlap another's MFMA stream).  Which configuration a launch uses
// is decided by the context's plan (gemm_plan in bem_ctx), set by the
// autotuner from measured times at the context's shapes.  FP64 products run
// here; the FP32 tiles are for the autotuner's report only.
template <typename T, int CFG>
struct GemmCfg;
template <>
struct GemmCfg<float, 0> {
    static constexpr int BM = 128, BN = 128, BK = 16, WM = 64, WN = 64, PAD = 16, MINB = 1;
    typedef v4f acc_t;
    typedef float4 vec_t;  // 16-byte global loads
    static constexpr int VEC = 4;
};
template <>
struct GemmCfg<float, 1> {
    static constexpr int BM = 128, BN = 64, BK = 16, WM = 64, WN = 32, PAD = 16, MINB = 2;
    typedef v4f acc_t;
    typedef float4 vec_t;
    static constexpr int VEC = 4;
};
template <>
struct GemmCfg<float, 2> {
    static constexpr int BM = 64, BN = 64, BK = 16, WM = 32, WN = 32, PAD = 16, MINB = 2;
    typedef v4f acc_t;
    typedef float4 vec_t;
    static constexpr int VEC = 4;
};
template <>
struct GemmCfg<double, 0> {
    static constexpr int BM = 128, BN = 64, BK = 16, WM = 64, WN = 32, PAD = 8, MINB = 1;
    typedef v4d acc_t;
    typedef double2 vec_t;
    static constexpr int VEC = 2;
};
template <>
struct GemmCfg<double, 1> {
    static constexpr int BM = 64, BN = 64, BK = 16, WM = 32, WN = 32, PAD = 8, MINB = 2;
    typedef v4d acc_t;
    typedef double2 vec_t;
    static constexpr int VEC = 2;
};
template <>
struct GemmCfg<double, 2> {
    static constexpr int BM = 64, BN = 32, BK = 16, WM = 32, WN = 16, PAD = 8, MINB = 2;
    typedef v4d acc_t;
    typedef double2 vec_t;
    static constexpr int VEC = 2;
};
// 64 x 64 with a K slice of 8: half the LDS of configuration 2 / 1, so more
// blocks fit on a CU beside the latency-bound panel kernels.
template <>
struct GemmCfg<float, 3> {
    static constexpr int BM = 64, BN = 64, BK = 8, WM = 32, WN = 32, PAD = 16, MINB = 2;
    typedef v4f acc_t;
    typedef float4 vec_t;
    static constexpr int VEC = 4;
};
template <>
struct GemmCfg<double, 3> {
    static constexpr int BM = 64, BN = 64, BK = 8, WM = 32, WN = 32, PAD = 8, MINB = 2;
    typedef v4d acc_t;
    typedef double2 vec_t;
    static constexpr int VEC = 2;
};
// 32 x 32 (one 16 x 16 MFMA tile per wave): products too small to give the
// device one block per CU with the other tiles.
template <>
struct GemmCfg<float, 4> {
    static constexpr int BM = 32, BN = 32, BK = 16, WM = 16, WN = 16, PAD = 16, MINB = 4;
    typedef v4f acc_t;
    typedef float4 vec_t;
    static constexpr int VEC = 4;
};
template <>
struct GemmCfg<double, 4> {
    static constexpr int BM = 32, BN = 32, BK = 16, WM = 16, WN = 16, PAD = 8, MINB = 4;
    typedef v4d acc_t;
    typedef double2 vec_t;
    static constexpr int VEC = 2;
};
constexpr int kGemmCfgs = 5;
constexpr int kGemmSmall = 4;       // the 32 x 32 configuration
constexpr int kGemmTrialCfgs = 4;   // configurations tried for the trailing update

template <typename T>
__device__ __forceinline__ void vec_split(const typename GemmCfg<T, 0>::vec_t& v, T* out);
template <>
__device__ __forceinline__ void vec_split<float>(const float4& v, float* o) {
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
template <>
__device__ __forceinline__ void vec_split<double>(const double2& v, double* o) {
    o[0] = v.x; o[1] = v.y;
}

// ROLE 1 only names the instantiation (the LU trailing updates, so a
// profiler lists them apart from the other products of the same tile).
template <typename T, int CFG, int ROLE = 0>
__global__ __launch_bounds__(256, (GemmCfg<T, CFG>::MINB)) void k_cgemm(int M, int N, int K, const T* __restrict__ Ar,
                                               const T* __restrict__ Ai, long lda, const T* __restrict__ Br,
                                               const T* __restrict__ Bi, long ldb, T* __restrict__ Cr,
                                               T* __restrict__ Ci, long ldc, int mode) {
    typedef GemmCfg<T, CFG> C;
    constexpr int BM = C::BM, BN = C::BN, BK = C::BK, WM = C::WM, WN = C::WN, VEC = C::VEC;
    constexpr int TM = WM / 16, TN = WN / 16;
    constexpr int SA = BM + C::PAD, SB = BN + C::PAD;
    constexpr int AVT = BM * BK / VEC, BVT = BK * BN / VEC;  // 16-byte vectors per plane per slice
    constexpr int AV = (AVT + 255) / 256, BV = (BVT + 255) / 256;  // per thread
    typedef typename C::vec_t vec_t;
    typedef typename C::acc_t acc_t;
    constexpr bool M3 = sizeof(T) == 4;  // 3M form
    constexpr int NACC = M3 ? 3 : 2;

    __shared__ T sA[2][2][BK][SA];
    __shared__ T sB[2][2][BK][SB];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;
    const int ntx = (N + BN - 1) / BN, nty = (M + BM - 1) / BM;
    const int ntiles = ntx * nty;
    const int nk = K / BK;

    // Tiles in row-major order; a grid smaller than the tile count makes every
    // block loop (persistent launch).
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int row0 = (tile / ntx) * BM, col0 = (tile % ntx) * BN;

        vec_t ga[2][AV], gb[2][BV];
        auto load = [&](int k0) {
#pragma unroll
            for (int u = 0; u < AV; u++) {
                const int v = tid + 256 * u;
                const int r = v / (BK / VEC), kv = (v % (BK / VEC)) * VEC;
                const bool ok = (AVT % 256 == 0 || v < AVT) && row0 + r < M;
                const long o = (long)(row0 + r) * lda + k0 + kv;
                ga[0][u] = ok ? *reinterpret_cast<const vec_t*>(Ar + o) : vec_t{};
                ga[1][u] = ok ? *reinterpret_cast<const vec_t*>(Ai + o) : vec_t{};
            }
#pragma unroll
            for (int u = 0; u < BV; u++) {
                const int v = tid + 256 * u;
                const int kr = v / (BN / VEC), nv = (v % (BN / VEC)) * VEC;
                const bool ok = (BVT % 256 == 0 || v < BVT) && col0 + nv < N;
                const long o = (long)(k0 + kr) * ldb + col0 + nv;
                gb[0][u] = ok ? *reinterpret_cast<const vec_t*>(Br + o) : vec_t{};
                gb[1][u] = ok ? *reinterpret_cast<const vec_t*>(Bi + o) : vec_t{};
            }
        };
        auto store = [&](int buf) {
#pragma unroll
            for (int u = 0; u < AV; u++) {
                const int v = tid + 256 * u;
                if (AVT % 256 != 0 && v >= AVT) continue;
                const int r = v / (BK / VEC), kv = (v % (BK / VEC)) * VEC;
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    T e[VEC];
                    vec_split<T>(ga[p][u], e);
#pragma unroll
                    for (int q = 0; q < VEC; q++) sA[buf][p][kv + q][r] = e[q];
                }
            }
#pragma unroll
            for (int u = 0; u < BV; u++) {
                const int v = tid + 256 * u;
                if (BVT % 256 != 0 && v >= BVT) continue;
                const int kr = v / (BN / VEC), nv = (v % (BN / VEC)) * VEC;
#pragma unroll
                for (int p = 0; p < 2; p++) *reinterpret_cast<vec_t*>(&sB[buf][p][kr][nv]) = gb[p][u];
            }
        };

        acc_t acc[NACC][TM][TN];
#pragma unroll
        for (int a = 0; a < NACC; a++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[a][i][j] = acc_t{};

        load(0);
        store(0);
        __syncthreads();
        for (int kt = 0; kt < nk; kt++) {
            const int buf = kt & 1;
            if (kt + 1 < nk) load((kt + 1) * BK);
#pragma unroll
            for (int kk = 0; kk < BK; kk += 4) {
                const int ka = kk + (lane >> 4);
                T ar[TM], ai[TM], br[TN], bi[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    ar[i] = sA[buf][0][ka][wm0 + i * 16 + (lane & 15)];
                    ai[i] = sA[buf][1][ka][wm0 + i * 16 + (lane & 15)];
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    br[j] = sB[buf][0][ka][wn0 + j * 16 + (lane & 15)];
                    bi[j] = sB[buf][1][ka][wn0 + j * 16 + (lane & 15)];
                }
                if constexpr (M3) {
                    T as[TM], bs[TN];
#pragma unroll
                    for (int i = 0; i < TM; i++) as[i] = ar[i] + ai[i];
#pragma unroll
                    for (int j = 0; j < TN; j++) bs[j] = br[j] + bi[j];
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++) {
                            acc[0][i][j] = mfma16x16x4(ar[i], br[j], acc[0][i][j]);
                            acc[1][i][j] = mfma16x16x4(ai[i], bi[j], acc[1][i][j]);
                            acc[2][i][j] = mfma16x16x4(as[i], bs[j], acc[2][i][j]);
                        }
                } else {
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++) {
                            acc[0][i][j] = mfma16x16x4(ar[i], br[j], acc[0][i][j]);
                            acc[0][i][j] = mfma16x16x4(ai[i], -bi[j], acc[0][i][j]);
                            acc[1][i][j] = mfma16x16x4(ar[i], bi[j], acc[1][i][j]);
                            acc[1][i][j] = mfma16x16x4(ai[i], br[j], acc[1][i][j]);
                        }
                }
            }
            if (kt + 1 < nk) store(buf ^ 1);
            __syncthreads();  // also ends the reads of this tile before the next tile's first store
        }

#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int col = col0 + wn0 + j * 16 + (lane & 15);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = row0 + wm0 + i * 16 + (sizeof(T) == 4 ? 4 * (lane >> 4) + r : (lane >> 4) + 4 * r);
                    if (row >= M || col >= N) continue;
                    T vr, vi;
                    if constexpr (M3) {
                        vr = acc[0][i][j][r] - acc[1][i][j][r];
                        vi = acc[2][i][j][r] - acc[0][i][j][r] - acc[1][i][j][r];
                    } else {
                        vr = acc[0][i][j][r];
                        vi = acc[1][i][j][r];
                    }
                    const long o = (long)row * ldc + col;
                    if (mode == 0) {
                        Cr[o] -= vr;
                        Ci[o] -= vi;
                    } else {
                        Cr[o] = vr;
                        Ci[o] = vi;
                    }
                }
            }
    }
}

// Host launcher of configuration cfg.  K must be a multiple of BK; N a
// multiple of the vector width (4 floats / 2 doubles) and every leading
// dimension a multiple of it.  cap > 0 limits the grid to cap blocks, which
// then loop over the tiles.
template <typename T, int CFG>
inline void cgemm_cfg(hipStream_t s, int M, int N, int K, const T* Ar, const T* Ai, long lda, const T* Br,
                      const T* Bi, long ldb, T* Cr, T* Ci, long ldc, int mode, long cap, int role) {
    typedef GemmCfg<T, CFG> C;
    const long tiles = (long)((N + C::BN - 1) / C::BN) * ((M + C::BM - 1) / C::BM);
    const long grid = cap > 0 && cap < tiles ? cap : tiles;
    auto k = role == 1 ? k_cgemm<T, CFG, sizeof(T) == 8 ? 1 : 0> : k_cgemm<T, CFG, 0>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(256), 0, s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode);
}

template <typename T>
inline void cgemm_any(int cfg, hipStream_t s, int M, int N, int K, const T* Ar, const T* Ai, long lda, const T* Br,
                      const T* Bi, long ldb, T* Cr, T* Ci, long ldc, int mode, long cap = 0, int role = 0) {
    if (M <= 0 || N <= 0 || K <= 0) return;
    switch (cfg) {
        case 1: cgemm_cfg<T, 1>(s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, role); break;
        case 2: cgemm_cfg<T, 2>(s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, role); break;
        case 3: cgemm_cfg<T, 3>(s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, role); break;
        case 4: cgemm_cfg<T, 4>(s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, role); break;
        default: cgemm_cfg<T, 0>(s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, role); break;
    }
}
static_assert(kGemmCfgs <= GemmPlan::kMaxCfgs, "GemmPlan holds one trial time per configuration");

// Blocks of configuration cfg for an M x N product.
template <typename T>
inline long gemm_blocks(int cfg, int M, int N) {
    int bm, bn;
    switch (cfg) {
        case 1: bm = GemmCfg<T, 1>::BM; bn = GemmCfg<T, 1>::BN; break;
        case 2: bm = GemmCfg<T, 2>::BM; bn = GemmCfg<T, 2>::BN; break;
        case 3: bm = GemmCfg<T, 3>::BM; bn = GemmCfg<T, 3>::BN; break;
        case 4: bm = GemmCfg<T, 4>::BM; bn = GemmCfg<T, 4>::BN; break;
        default: bm = GemmCfg<T, 0>::BM; bn = GemmCfg<T, 0>::BN; break;
    }
    return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

// The plan's configuration for an M x N product: the large-product tile when
// it still gives at least `fill` blocks, else the skinny-product tile while
// that gives one block per CU, else the 32 x 32 tile.
inline int gemm_choose(const bem_ctx* c, int M, int N) {
    const GemmPlan& p = c->gemm_plan[1];
    if (gemm_blocks<double>(p.large, M, N) >= p.fill) return p.large;
    return gemm_blocks<double>(p.skinny, M, N) >= c->cus ? p.skinny : kGemmSmall;
}

// FP64 GEMM with optional per-launch timing, on stream s (default: the context
// stream), tile configuration from the context's plan; update: an LU trailing
// update (its own kernel symbol and timing class); cap as in cgemm_cfg.
// Counted work: 8 M N K real flops; bytes = operands read once plus C read and
// written.
inline void cgemm_ctx(bem_ctx* c, int M, int N, int K, const double* Ar, const double* Ai, long lda, const double* Br,
                      const double* Bi, long ldb, double* Cr, double* Ci, long ldc, int mode, hipStream_t s = nullptr,
                      bool update = false, long cap = 0) {
    if (M <= 0 || N <= 0 || K <= 0) return;
    if (!s) s = c->stream;
    const int k = kt_mark(c, update ? KS_UPDATE64 : KS_GEMM64, s);
    cgemm_any<double>(gemm_choose(c, M, N), s, M, N, K, Ar, Ai, lda, Br, Bi, ldb, Cr, Ci, ldc, mode, cap, update ? 1 : 0);
    kt_close(c, k, 8.0 * M * N * (double)K,
             16.0 * ((double)M * K + (double)K * N + (mode == 1 ? 1.0 : 2.0) * M * N));
}

// Four consecutive values of a row, by 16-byte loads.
template <typename T>
__device__ __forceinline__ void load_row4(const T* __restrict__ p, T o[4]);
template <>
__device__ __forceinline__ void load_row4<float>(const float* __restrict__ p, float o[4]) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
template <>
__device__ __forceinline__ void load_row4<double>(const double* __restrict__ p, double o[4]) {
    const double2 v0 = *reinterpret_cast<const double2*>(p), v1 = *reinterpret_cast<const double2*>(p + 2);
    o[0] = v0.x; o[1] = v0.y; o[2] = v1.x; o[3] = v1.y;
}
