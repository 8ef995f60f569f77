// adjoint.hip -- eigenvalue gradients on the sparsity pattern (gfx950).
//
// For a simple eigenvalue lambda_k of the symmetric A with unit eigenvector
// x_k, d lambda_k / d A_ij = x_k(i) x_k(j).  The loss sum_k w_k lambda_k
// therefore has, on the stored upper-triangle CSR (each off-diagonal entry
// stands for A_ij and A_ji), the gradient
//     g[e(i,j)] = c_ij * sum_k w_k x_k(i) x_k(j),   c_ij = 2 (i != j), 1 (i == j),
// and for a diagonal potential A = H + diag(V):  g_V[i] = sum_k w_k x_k(i)^2.
// Valid while each lambda_k is separated from the rest of the spectrum.
// No reference counterpart (the reference has no derivatives).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/jadamilu_amd.h"
#include "reduce.hpp"
#include "xcd.hpp"

namespace jdhip {

constexpr int kAB = 256;
constexpr int kMaxK = 64;

struct Weights {
    double w[kMaxK];
};

// One wave per 64 rows of the 1-based upper CSR.  What bounds it is the L1's
// one line a clock: with four lanes per row, neighbouring lanes read X at
// unrelated places and a load took 27 lines.  While its rows are short, a wave
// therefore gives each lane a row and goes through the rows' entries side by
// side: in a matrix with structure, the t-th entries of 64 consecutive rows
// refer to almost consecutive places.  Columns and results, which lie row after
// row, pass through LDS (written from the lanes directly they took 3.7 times
// their bytes).  x(i) stays in registers for all of a row's entries, and the
// loads of an entry (NC vectors) are all issued before the first use.  Waves
// with longer rows, and more than 16 vectors, keep the four lanes a row, which
// read their entries together.  Every XCD takes one
// contiguous range of rows, whose neighbours' entries of X its L2 then holds.
// Ten vectors, Anderson L = 100 (4M entries): 80.2 -> 49.0 us with three operands in
// turn (132 MB), 67 -> 36 us with two.
constexpr int kLaneRow = 16;   // longest row that a lane takes by itself
constexpr int kLaneWave = 512; // most entries of such a wave's 64 rows

template <int NC>
__global__ __launch_bounds__(kAB) void k_adjoint_csr(int n, const int *__restrict__ ia,
                                                     const int *__restrict__ ja,
                                                     const double *__restrict__ X, long ldx,
                                                     int k, Weights w, double *__restrict__ g) {
    const int lane = threadIdx.x & 63;
    const long r0 = (logical_block(1) * (kAB / 64) + (threadIdx.x >> 6)) * 64;
    if (r0 >= n) return;
    const long i = r0 + lane;
    const int b = i < n ? ia[i] - 1 : 0, e = i < n ? ia[i + 1] - 1 : 0;
    int longest = e - b;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o, 64));
    longest = __builtin_amdgcn_readfirstlane(longest);
    const int first = __builtin_amdgcn_readfirstlane(b);
    const int total = __shfl(e, (int)min((long)n - 1 - r0, 63L), 64) - first;
    if (longest <= kLaneRow && total <= kLaneWave && k <= NC) {
        __shared__ int cols[kAB / 64][kLaneWave];
        __shared__ double grad[kAB / 64][kLaneWave];
        int *cw = cols[threadIdx.x >> 6];
        double *gw = grad[threadIdx.x >> 6];
        for (int t = lane; t < total; t += 64) cw[t] = ja[first + t] - 1;
        wave_lds_sync();
        const long ii = min(i, (long)n - 1);
        double xi[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) xi[c] = c < k ? X[c * ldx + ii] : 0.0;
        for (int t = 0; t < longest; ++t) {
            const bool mine = b + t < e;
            const int j = mine ? cw[b - first + t] : (int)ii;
            double xj[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) xj[c] = c < k ? X[c * ldx + j] : 0.0;
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (c < k) s += w.w[c] * xi[c] * xj[c];
            if (mine) gw[b - first + t] = (j == i) ? s : 2.0 * s;
        }
        wave_lds_sync();
        for (int t = lane; t < total; t += 64) g[first + t] = gw[t];
        return;
    }
    const int q = lane >> 2, l = lane & 3;
    for (int r = q; r < 64; r += 16) {
        const long row = r0 + r;
        const int rb = __shfl(b, r, 64), re = __shfl(e, r, 64);
        for (int t = rb + l; t < re; t += 4) {
            const int j = ja[t] - 1;
            double s = 0.0;
            for (int c0 = 0; c0 < k; c0 += NC) {
                double xi[NC], xj[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const double *x = X + min(c0 + c, k - 1) * ldx;
                    xi[c] = x[row];
                    xj[c] = x[j];
                }
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    if (c0 + c < k) s += w.w[c0 + c] * xi[c] * xj[c];
            }
            g[t] = (j == row) ? s : 2.0 * s;
        }
    }
}

__global__ __launch_bounds__(kAB) void k_adjoint_diag(int n, const double *__restrict__ X,
                                                      long ldx, int k, Weights w,
                                                      double *__restrict__ g) {
    for (long i = blockIdx.x * (long)kAB + threadIdx.x; i < n; i += (long)gridDim.x * kAB) {
        double s = 0.0;
        for (int c = 0; c < k; ++c) {
            double v = X[c * ldx + i];
            s += w.w[c] * v * v;
        }
        g[i] = s;
    }
}

// f(NC): the vectors of a step, all of them up to 16
template <typename F>
static void by_vectors(int k, F &&f) {
    if (k <= 1) f(std::integral_constant<int, 1>{});
    else if (k <= 2) f(std::integral_constant<int, 2>{});
    else if (k <= 4) f(std::integral_constant<int, 4>{});
    else if (k <= 6) f(std::integral_constant<int, 6>{});
    else if (k <= 8) f(std::integral_constant<int, 8>{});
    else if (k <= 10) f(std::integral_constant<int, 10>{});
    else if (k <= 12) f(std::integral_constant<int, 12>{});
    else f(std::integral_constant<int, 16>{});
}

}  // namespace jdhip

extern "C" {

int jdhip_adjoint_csr(void *stream, int n, const int *ia_dev, const int *ja_dev,
                      const double *x_dev, long ldx, int k, const double *w, double *g_dev) {
    if (k <= 0 || k > jdhip::kMaxK || n <= 0) return -1;
    jdhip::Weights W{};
    for (int c = 0; c < k; ++c) W.w[c] = w[c];
    const int blocks = (int)(((long)n + jdhip::kAB - 1) / jdhip::kAB);
    jdhip::by_vectors(k, [&](auto nc) {
        jdhip::k_adjoint_csr<nc.value><<<blocks, jdhip::kAB, 0, (hipStream_t)stream>>>(
            n, ia_dev, ja_dev, x_dev, ldx, k, W, g_dev);
    });
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int jdhip_adjoint_diag(void *stream, int n, const double *x_dev, long ldx, int k,
                       const double *w, double *g_dev) {
    if (k <= 0 || k > jdhip::kMaxK || n <= 0) return -1;
    jdhip::Weights W{};
    for (int c = 0; c < k; ++c) W.w[c] = w[c];
    int blocks = (int)std::min<long>(8192, ((long)n + jdhip::kAB - 1) / jdhip::kAB);
    jdhip::k_adjoint_diag<<<std::max(blocks, 1), jdhip::kAB, 0, (hipStream_t)stream>>>(
        n, x_dev, ldx, k, W, g_dev);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // extern "C"
