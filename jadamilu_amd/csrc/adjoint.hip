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

// Any matrix, any k: four lanes a row of the 1-based upper CSR.
__global__ __launch_bounds__(kAB) void k_adjoint_rows(int n, const int *__restrict__ ia,
                                                      const int *__restrict__ ja,
                                                      const double *__restrict__ X, long ldx,
                                                      int k, Weights w, double *__restrict__ g) {
    const long i = blockIdx.x * (long)(kAB / 4) + (threadIdx.x >> 2);
    if (i >= n) return;
    const int e = ia[i + 1] - 1;
    for (int t = ia[i] - 1 + (threadIdx.x & 3); t < e; t += 4) {
        const int j = ja[t] - 1;
        double s = 0.0;
        for (int c = 0; c < k; ++c) s += w.w[c] * X[c * ldx + i] * X[c * ldx + j];
        g[t] = (j == i) ? s : 2.0 * s;
    }
}

// Up to NC vectors, 64 rows a wave.  What bounds it is the L1's one line a
// clock: with four lanes per row, neighbouring lanes read X at unrelated places
// and a load took 27 lines.  While its rows are short, a wave therefore gives
// each lane a row and goes through the rows' entries side by side: in a matrix
// with structure, the t-th entries of 64 consecutive rows refer to almost
// consecutive places.  Columns and results, which lie row after row, pass
// through LDS (written from the lanes directly they took 3.7 times their
// bytes).  x(i) stays in registers for all of a row's entries, and the loads of
// an entry (NC vectors) are all issued before the first use.  The entries of a
// wave with longer rows are taken by the whole block, one a thread, whatever rows
// they belong to.  Every XCD takes one contiguous range of rows, whose neighbours' entries of X its L2 then holds.
// Against k_adjoint_rows, ten vectors: Anderson L = 100 (4M entries) 80.2 -> 49.0
// us with three operands in turn (132 MB), 67.9 -> 36.9 with two; rows of 14
// entries, which the block shares (80^3, 27 points) 120 -> 103; rows of up to
// thousands of entries (a power-law graph of 200,000 rows) 1,354 -> 635.  One
// vector: 17.9 -> 18.4, 35.6 -> 30.5, 133 -> 75.
// The limits: longer rows by lanes need more LDS; with 32 and 1,024, Anderson L =
// 100 takes 28.7 us instead of 18.4 for one vector and 46.1 instead of 39.4 for
// ten.
constexpr int kLaneRow = 16;    // longest row that a lane takes by itself
constexpr int kLaneWave = 512;  // most entries of such a wave's 64 rows

template <int NC>
__global__ __launch_bounds__(kAB) void k_adjoint_csr(int n, const int *__restrict__ ia,
                                                     const int *__restrict__ ja,
                                                     const double *__restrict__ X, long ldx,
                                                     int k, Weights w, double *__restrict__ g) {
    __shared__ int cols[kAB / 64][kLaneWave];
    __shared__ double grad[kAB / 64][kLaneWave];
    __shared__ int done[kAB / 64], row_of[kAB / 64][65];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long b0 = logical_block(1) * kAB, r0 = b0 + 64 * wave;
    const long i = r0 + lane;
    const int b = i < n ? ia[i] - 1 : 0, e = i < n ? ia[i + 1] - 1 : 0;
    int longest = e - b;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o, 64));
    longest = __builtin_amdgcn_readfirstlane(longest);
    const int first = __builtin_amdgcn_readfirstlane(b);
    // (a wave past the last row has nothing to do: its total is not read)
    const int total = __shfl(e, (int)max(0L, min((long)n - 1 - r0, 63L)), 64) - first;
    const bool by_lanes = r0 >= n || (longest <= kLaneRow && total <= kLaneWave);
    if (lane == 0) done[wave] = by_lanes;
    if (!by_lanes) {
        row_of[wave][lane] = i < n ? b : first + total;
        if (lane == 0) row_of[wave][64] = first + total;
    }
    if (by_lanes && r0 < n) {
        int *cw = cols[wave];
        double *gw = grad[wave];
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
    }
    __syncthreads();
    for (int q = 0; q < kAB / 64; ++q) {
        if (done[q]) continue;
        const int *start = row_of[q];
        for (long t = start[0] + (int)threadIdx.x; t < start[64]; t += kAB) {
            int r = 0;  // the last row that starts at t or before
#pragma unroll
            for (int step = 32; step > 0; step >>= 1)
                if (start[r + step] <= t) r += step;
            const long row = b0 + 64 * q + r, j = ja[t] - 1;
            double xi[NC], xj[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                xi[c] = c < k ? X[c * ldx + row] : 0.0;
                xj[c] = c < k ? X[c * ldx + j] : 0.0;
            }
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (c < k) s += w.w[c] * xi[c] * xj[c];
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

// f(NC): room for k <= kMaxLaneK vectors
constexpr int kMaxLaneK = 16;
template <typename F>
static void by_vectors(int k, F &&f) {
    if (k <= 1) f(std::integral_constant<int, 1>{});
    else if (k <= 2) f(std::integral_constant<int, 2>{});
    else if (k <= 4) f(std::integral_constant<int, 4>{});
    else if (k <= 6) f(std::integral_constant<int, 6>{});
    else if (k <= 8) f(std::integral_constant<int, 8>{});
    else if (k <= 10) f(std::integral_constant<int, 10>{});
    else if (k <= 12) f(std::integral_constant<int, 12>{});
    else f(std::integral_constant<int, kMaxLaneK>{});
}

// Rows from which on a wave takes 64 of them: below, four lanes a row fill more of
// the device (27,000 rows of Anderson, 16 vectors 7.2 us against 8.9; 64,000 rows
// 12.9 against 9.8, ten vectors 7.9 against 7.5).  More than 16 vectors take four
// lanes a row, too (20 vectors, L = 100: 144 us against 214 in steps of 16).
constexpr int kLaneRows = 32768;

}  // namespace jdhip

extern "C" {

int jdhip_adjoint_csr(void *stream, int n, const int *ia_dev, const int *ja_dev,
                      const double *x_dev, long ldx, int k, const double *w, double *g_dev) {
    if (k <= 0 || k > jdhip::kMaxK || n <= 0) return -1;
    jdhip::Weights W{};
    for (int c = 0; c < k; ++c) W.w[c] = w[c];
    const hipStream_t s = (hipStream_t)stream;
    if (n < jdhip::kLaneRows || k > jdhip::kMaxLaneK) {
        const int blocks = (int)(((long)n + 63) / 64);
        jdhip::k_adjoint_rows<<<blocks, jdhip::kAB, 0, s>>>(n, ia_dev, ja_dev, x_dev, ldx, k, W,
                                                            g_dev);
    } else {
        const int blocks = (int)(((long)n + jdhip::kAB - 1) / jdhip::kAB);
        jdhip::by_vectors(k, [&](auto nc) {
            jdhip::k_adjoint_csr<nc.value><<<blocks, jdhip::kAB, 0, s>>>(n, ia_dev, ja_dev, x_dev,
                                                                         ldx, k, W, g_dev);
        });
    }
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
