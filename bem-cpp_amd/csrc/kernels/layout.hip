// layout.hip -- interleaved complex matrices of the caller (host) to and from the
// device's planar padded ones.  The host copies bytes only; the planes are split,
// joined, transposed and padded on the device.
#include <algorithm>

#include "../bem_internal.h"

namespace {

constexpr int TS = 32;  // tile edge

// Lines [l0, l0 + nl) of a matrix, `len` complex values each at S (line by line), to or
// from the planes P: line l is row l of P, or its column l (TR).  UP: S to P, otherwise
// P times `scale` to S.  A workgroup moves 32 x 32 values, transposed ones through LDS,
// so that both sides are read and written in runs of 32.  The calls are bound by the
// host's copy: set_Z, factor and solve of 1999 unknowns and 33 right-hand sides take 9.75
// ms, of which the device works 6.9; with the host splitting and padding the
// planes, 25.2 ms.
template <bool UP, bool TR>
__global__ __launch_bounds__(256) void k_lines(double2* __restrict__ S, int l0, int nl, int len,
                                               double* __restrict__ Pr, double* __restrict__ Pi, long ld,
                                               double scale) {
    __shared__ double2 tile[TR ? TS : 1][TS + 1];
    const int tx = threadIdx.x & (TS - 1), ty = threadIdx.x / TS;
    const int e0 = blockIdx.x * TS, b0 = blockIdx.y * TS;  // first value, first line of the tile
    if constexpr (!TR) {
        const int e = e0 + tx;
        for (int k = ty; k < TS; k += 256 / TS) {
            if (b0 + k >= nl || e >= len) continue;
            const long s = (long)(b0 + k) * len + e, p = (long)(l0 + b0 + k) * ld + e;
            if constexpr (UP) {
                const double2 v = S[s];
                Pr[p] = v.x;
                Pi[p] = v.y;
            } else {
                S[s] = make_double2(scale * Pr[p], scale * Pi[p]);
            }
        }
    } else {
        // tile[k][m]: value e0 + k of line b0 + m (down) or value e0 + m of line b0 + k (up)
        for (int k = ty; k < TS; k += 256 / TS) {
            if constexpr (UP) {
                if (b0 + k < nl && e0 + tx < len) tile[k][tx] = S[(long)(b0 + k) * len + e0 + tx];
            } else {
                const long p = (long)(e0 + k) * ld + l0 + b0 + tx;
                if (e0 + k < len && b0 + tx < nl) tile[k][tx] = make_double2(scale * Pr[p], scale * Pi[p]);
            }
        }
        __syncthreads();
        for (int k = ty; k < TS; k += 256 / TS) {
            if constexpr (UP) {
                if (e0 + k >= len || b0 + tx >= nl) continue;
                const long p = (long)(e0 + k) * ld + l0 + b0 + tx;
                Pr[p] = tile[tx][k].x;
                Pi[p] = tile[tx][k].y;
            } else {
                if (b0 + k < nl && e0 + tx < len) S[(long)(b0 + k) * len + e0 + tx] = tile[tx][k];
            }
        }
    }
}

// The padding of the planes (prows x ld) around rows x cols values: zero, and one on
// the diagonal if asked.
__global__ __launch_bounds__(256) void k_pad(double* __restrict__ Pr, double* __restrict__ Pi, long ld, int rows,
                                             int cols, int identity) {
    const int r = blockIdx.x;
    for (int j = (r < rows ? cols : 0) + threadIdx.x; j < ld; j += 256) {
        Pr[r * ld + j] = identity && r == j ? 1.0 : 0.0;
        Pi[r * ld + j] = 0.0;
    }
}

// Device staging of whole lines of `len` values: kStage bytes, or less where the device
// has no room left (a single line at least).
constexpr size_t kStage = (size_t)32 << 20;
int staging(bem_ctx* c, int lines, int len, int& chunk, double2*& S) {
    const size_t line = (size_t)len * sizeof(double2);
    chunk = (int)std::min<size_t>(lines, std::max<size_t>(1, kStage / line));
    void* s = nullptr;
    int rc = ctx_scratch(c, chunk * line, &s);
    while (rc && chunk > 1) {
        (void)hipGetLastError();
        chunk = (chunk + 1) / 2;
        rc = ctx_scratch(c, chunk * line, &s);
    }
    S = static_cast<double2*>(s);
    return rc;
}

template <bool UP>
void lines_launch(hipStream_t s, bool row_major, double2* S, int l0, int nl, int len, double* Pr, double* Pi, long ld,
                  double scale) {
    const dim3 grid((len + TS - 1) / TS, (nl + TS - 1) / TS);
    if (row_major)
        hipLaunchKernelGGL((k_lines<UP, false>), grid, dim3(256), 0, s, S, l0, nl, len, Pr, Pi, ld, scale);
    else
        hipLaunchKernelGGL((k_lines<UP, true>), grid, dim3(256), 0, s, S, l0, nl, len, Pr, Pi, ld, scale);
}

}  // namespace

int planes_upload(bem_ctx* c, const double* src, int rows, int cols, bool row_major, double* Pr, double* Pi, int prows,
                  int ld, bool identity) {
    const int lines = row_major ? rows : cols, len = row_major ? cols : rows;
    int chunk = 0;
    double2* S = nullptr;
    if (int rc = staging(c, lines, len, chunk, S)) return rc;
    for (int l0 = 0; l0 < lines; l0 += chunk) {
        const int nl = std::min(chunk, lines - l0);
        BEM_HIP(c, hipMemcpyAsync(S, src + 2 * (size_t)l0 * len, (size_t)nl * len * sizeof(double2),
                                  hipMemcpyHostToDevice, c->stream));
        lines_launch<true>(c->stream, row_major, S, l0, nl, len, Pr, Pi, ld, 1.0);
    }
    hipLaunchKernelGGL(k_pad, dim3(prows), dim3(256), 0, c->stream, Pr, Pi, (long)ld, rows, cols, (int)identity);
    BEM_HIP(c, hipGetLastError());
    BEM_HIP(c, hipStreamSynchronize(c->stream));  // the caller's memory is its own again
    return 0;
}

int planes_download(bem_ctx* c, const double* Pr, const double* Pi, int ld, int rows, int cols, bool row_major,
                    double scale, double* dst) {
    const int lines = row_major ? rows : cols, len = row_major ? cols : rows;
    int chunk = 0;
    double2* S = nullptr;
    if (int rc = staging(c, lines, len, chunk, S)) return rc;
    for (int l0 = 0; l0 < lines; l0 += chunk) {
        const int nl = std::min(chunk, lines - l0);
        lines_launch<false>(c->stream, row_major, S, l0, nl, len, const_cast<double*>(Pr), const_cast<double*>(Pi), ld,
                            scale);
        BEM_HIP(c, hipGetLastError());
        BEM_HIP(c, hipMemcpyAsync(dst + 2 * (size_t)l0 * len, S, (size_t)nl * len * sizeof(double2),
                                  hipMemcpyDeviceToHost, c->stream));
    }
    BEM_HIP(c, hipStreamSynchronize(c->stream));
    return 0;
}
