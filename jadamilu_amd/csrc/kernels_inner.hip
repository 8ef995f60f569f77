// kernels_inner.hip -- inner correction-equation solver (LSOLREVCOM,
// src/jd/JDaux.F:2989-3268) as fused gfx950 kernels, templated on the vector
// type T: double for the FP64 path, float for the mixed path (FP32 vectors,
// FP32 SpMV and preconditioner; every dot product and norm accumulates in
// double).  All scalars live in device memory (InnerScalars), so a step is a
// chain of launches with no host round trip; breakdown tests set a flag
// that turns the rest of the step into no-ops (the reference's early exits).
#include "kernels.hpp"
#include "reduce.hpp"
#include "rowsum.hpp"
#include "xcd.hpp"

#include <algorithm>

namespace jdhip {

// ---------------------------------------------------------------------------
// out[c] = sum_i V[c*ldv+i] * w[i].  Bound by memory; eight columns' loads are
// in flight at a time, without a branch between them (columns past jv load the
// last one and are not added).  The scheduling barrier keeps them so: without
// it the FP64 form was compiled to one load and one wait after another.
// 3,000,000 rows, 512 blocks, with and without it: 4 columns 22.3 / 45.3 us, 8
// columns 37.8 / 88.9, 16 columns 72.7 / 111.5; 230,000 rows: 4.6 / 5.2, 7.1 /
// 9.5, 11.9 / 14.3.
template <typename T, int NC>
__global__ __launch_bounds__(kBlock) void k_multidot(const T *__restrict__ V, long ldv, int jv,
                                                     const T *__restrict__ w, long n,
                                                     double *partials) {
    double acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.0;
    constexpr int CH = NC < 8 ? NC : 8;
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        const double wi = (double)w[i];
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += CH) {
            if (c0 >= jv) break;
            T v[CH];
#pragma unroll
            for (int c = 0; c < CH; ++c) v[c] = V[(long)min(c0 + c, jv - 1) * ldv + i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < CH; ++c) acc[c0 + c] += (double)v[c] * wi;
        }
    }
    grid_reduce<NC>(acc, jv, partials, 0, nullptr);
}

// finish of a multi-column reduction: block c sums column c of the partials
// (columns are independent, so they are summed in parallel)
__global__ __launch_bounds__(kBlock) void k_finish_columns(const double *__restrict__ partials,
                                                          int nparts, double *out) {
    __shared__ double red[kBlock / 64];
    const int c = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const double s = wave_sum(thread_partials(partials + (long)c * nparts, nparts));
    if (lane == 0) red[wid] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) t += red[w];
        out[c] = t;
    }
}

void finish_sum(hipStream_t s, const double *partials, int np, double *out) {
    k_finish_columns<<<1, kBlock, 0, s>>>(partials, np, out);
}

template <typename T>
void multidot(hipStream_t s, const RedBuf &rb, const T *V, long ldv, int jv, const T *w, long n,
              double *out) {
    if (jv <= 0) return;
    // a row per thread up to 512 blocks, then a few, to amortise the reduction
    const int g = grid_for(n, kBlock, std::max(512, grid_for(n, 4 * kBlock, 1024)));
    double *P = rb.partials;
#define JDHIP_MD(NC)                                                                    \
    do {                                                                                \
        k_multidot<T, NC><<<g, kBlock, 0, s>>>(V, ldv, jv, w, n, P);                    \
        k_finish_columns<<<jv, kBlock, 0, s>>>(P, g, out);                               \
    } while (0)
    if (jv <= 1) JDHIP_MD(1);
    else if (jv <= 2) JDHIP_MD(2);
    else if (jv <= 4) JDHIP_MD(4);
    else if (jv <= 8) JDHIP_MD(8);
    else if (jv <= 16) JDHIP_MD(16);
    else if (jv <= 32) JDHIP_MD(32);
    else JDHIP_MD(64);
#undef JDHIP_MD
}

// ---------------------------------------------------------------------------
// SpMV on the device-built full CSR; LPR lanes per row; optional epilogue
//   y_i -= eta x_i   and   udot += u_i y_i   (u.y in double).
// Rows are accumulated in double also for FP32 storage: near an eigenvalue
// of A - eta I the row sums cancel to a tiny fraction of their terms, and a
// float accumulator would leave errors of the size of that result.
template <typename T, typename TA, int LPR, bool ETA, bool UDOT>
__global__ __launch_bounds__(kBlock) void k_spmv(int n, const int *__restrict__ rowptr,
                                                 const int *__restrict__ col,
                                                 const TA *__restrict__ val,
                                                 const T *__restrict__ x, T *__restrict__ y,
                                                 double eta_host, const T *__restrict__ u,
                                                 double *partials) {
    constexpr int GPB = kBlock / LPR;
    const int g = threadIdx.x / LPR, l = threadIdx.x % LPR;
    double acc[1] = {0.0};
    for (long row = logical_block(1) * GPB + g; row < n; row += (long)gridDim.x * GPB) {
        const int b = rowptr[row], e = rowptr[row + 1];
        double s = csr_lane_sum<LPR>(col, val, x, b, e, l);
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, LPR);
        if (l == 0) {
            if (ETA) s -= eta_host * (double)x[row];
            const T yi = (T)s;
            y[row] = yi;
            if (UDOT) acc[0] += (double)u[row] * (double)yi;
        }
    }
    if (UDOT) grid_reduce<1>(acc, 1, partials, 0, nullptr);
}

template <typename T, typename TA, int LPR>
static int spmv_lpr(hipStream_t s, const RedBuf &rb, int n, const int *rp, const int *ci,
                     const TA *val, const T *x, T *y, double eta, const T *u, double *udot) {
    constexpr int GPB = kBlock / LPR;
    const long rows_blocks = ((long)n + GPB - 1) / GPB;
    if (u) {
        const int g = (int)std::min<long>(rows_blocks, kMaxRedBlocks);
        double *P = g <= kInnerBlocks ? rb.inner_u() : rb.partials;
        if (eta != 0.0)
            k_spmv<T, TA, LPR, true, true><<<g, kBlock, 0, s>>>(n, rp, ci, val, x, y, eta, u, P);
        else
            k_spmv<T, TA, LPR, false, true><<<g, kBlock, 0, s>>>(n, rp, ci, val, x, y, eta, u, P);
        if (g <= kInnerBlocks) return g;
        k_finish_columns<<<1, kBlock, 0, s>>>(P, g, udot);
        return 0;
    }
    const int g = (int)std::min<long>(rows_blocks, 8192);
    if (eta != 0.0)
        k_spmv<T, TA, LPR, true, false><<<g, kBlock, 0, s>>>(n, rp, ci, val, x, y, eta, u, nullptr);
    else
        k_spmv<T, TA, LPR, false, false><<<g, kBlock, 0, s>>>(n, rp, ci, val, x, y, eta, u,
                                                              nullptr);
    return 0;
}

// Sliced ELL: one wave64 per slice of 64 rows, lane = row within the slice.
template <typename T, typename TA, bool ETA, bool UDOT>
__global__ __launch_bounds__(kBlock) void k_spmv_sell(
    int n, int nslices, const long *__restrict__ vptr, const long *__restrict__ iptr,
    const int *__restrict__ wm, const TA *__restrict__ val, const char *__restrict__ idx,
    const T *__restrict__ x, T *__restrict__ y, double eta_host, const T *__restrict__ u,
    double *partials) {
    constexpr int WPB = kBlock / 64;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double acc[1] = {0.0};
    // XCD-contiguous slice ranges: a slice's x gathers overlap its
    // neighbours', so they are served from one L2
    for (long sl = logical_block(1) * WPB + wv; sl < nslices; sl += (long)gridDim.x * WPB) {
        const long row = sl * 64 + lane;
        if (row >= n) continue;
        const int code = wm[sl];
        const int w = code >> 1;
        const TA *v = val + vptr[sl] + lane;
        double s0 = 0.0, s1 = 0.0;
        if (code & 1) {
            const short *ci = (const short *)(idx + iptr[sl]) + lane;
            int k = 0;
            for (; k + 1 < w; k += 2) {
                s0 += (double)v[k * 64] * (double)x[row + ci[k * 64]];
                s1 += (double)v[(k + 1) * 64] * (double)x[row + ci[(k + 1) * 64]];
            }
            if (k < w) s0 += (double)v[k * 64] * (double)x[row + ci[k * 64]];
        } else {
            const int *ci = (const int *)(idx + iptr[sl]) + lane;
            int k = 0;
            for (; k + 1 < w; k += 2) {
                s0 += (double)v[k * 64] * (double)x[ci[k * 64]];
                s1 += (double)v[(k + 1) * 64] * (double)x[ci[(k + 1) * 64]];
            }
            if (k < w) s0 += (double)v[k * 64] * (double)x[ci[k * 64]];
        }
        double ys = s0 + s1;
        if (ETA) ys -= eta_host * (double)x[row];
        const T yi = (T)ys;
        y[row] = yi;
        if (UDOT) acc[0] += (double)u[row] * (double)yi;
    }
    if (UDOT) grid_reduce<1>(acc, 1, partials, 0, nullptr);
}

template <typename T, typename TA>
static int spmv_sell(hipStream_t s, const RedBuf &rb, const CsrDev &A, const TA *val,
                      const T *x, T *y, double eta, const T *u, double *udot) {
    constexpr int WPB = kBlock / 64;
    const long blocks = ((long)A.nslices + WPB - 1) / WPB;
#define JDHIP_SELL(E, U, P)                                                                  \
    k_spmv_sell<T, TA, E, U><<<g, kBlock, 0, s>>>(A.n, A.nslices, A.s_vptr, A.s_iptr, A.s_wm, \
                                                  val, A.s_idx, x, y, eta, u, P)
    if (u) {
        // one partial sum per block: the full grid fits the scratch
        const int g = (int)std::min<long>(blocks, kMaxPartials);
        double *P = g <= kInnerBlocks ? rb.inner_u() : rb.partials;
        if (eta != 0.0) JDHIP_SELL(true, true, P);
        else JDHIP_SELL(false, true, P);
        if (g <= kInnerBlocks) return g;
        k_finish_columns<<<1, kBlock, 0, s>>>(P, g, udot);
        return 0;
    }
    const int g = (int)std::min<long>(blocks, 1L << 20);
    if (eta != 0.0) JDHIP_SELL(true, false, nullptr);
    else JDHIP_SELL(false, false, nullptr);
#undef JDHIP_SELL
    return 0;
}

template <typename T, typename TA>
static int spmv_vals(hipStream_t s, const RedBuf &rb, const CsrDev &A, const TA *val,
                      const TA *sv, const T *x, T *y, double eta, const T *u,
                      double *udot_out) {
    if (A.lpr == 0 && A.nslices > 0)
        return spmv_sell<T, TA>(s, rb, A, sv, x, y, eta, u, udot_out);
#define JDHIP_LPR(L) spmv_lpr<T, TA, L>(s, rb, A.n, A.rowptr, A.col, val, x, y, eta, u, udot_out)
    switch (A.lpr) {
    case 1: return JDHIP_LPR(1);
    case 2: return JDHIP_LPR(2);
    case 4: return JDHIP_LPR(4);
    case 16: return JDHIP_LPR(16);
    case 32: return JDHIP_LPR(32);
    default: return JDHIP_LPR(8);
    }
#undef JDHIP_LPR
}

template <typename T>
int spmv(hipStream_t s, const RedBuf &rb, const CsrDev &A, const T *x, T *y, double eta,
         const T *u, double *udot_out) {
    if (A.lpr == kLprDia && A.dia.nd > 0)
        return spmv_dia<T>(s, rb, A.dia, A.f_vals64, x, y, eta, u, udot_out);
    if constexpr (sizeof(T) == 8)
        return spmv_vals<T, double>(s, rb, A, A.val, A.s_val, x, y, eta, u, udot_out);
    else if (A.f_vals64)
        return spmv_vals<T, double>(s, rb, A, A.val, A.s_val, x, y, eta, u, udot_out);
    else
        return spmv_vals<T, float>(s, rb, A, A.valf, A.s_valf, x, y, eta, u, udot_out);
}

// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_diag(T *z, const T *d, const T *r, long n) {
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock)
        z[i] = d[i] * r[i];
}
template <typename T>
void diag_apply(hipStream_t s, T *z, const T *d, const T *r, long n) {
    k_diag<T><<<grid_for(n, kBlock, 4096), kBlock, 0, s>>>(z, d, r, n);
}

template <typename TD, typename TS>
__global__ __launch_bounds__(kBlock) void k_convert(TD *dst, const TS *src, long n) {
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock)
        dst[i] = (TD)src[i];
}
void convert(hipStream_t s, float *dst, const double *src, long n) {
    if (n > 0) k_convert<float, double><<<grid_for(n, kBlock, 4096), kBlock, 0, s>>>(dst, src, n);
}
void convert(hipStream_t s, double *dst, const float *src, long n) {
    if (n > 0) k_convert<double, float><<<grid_for(n, kBlock, 4096), kBlock, 0, s>>>(dst, src, n);
}

// ---------------------------------------------------------------------------
// One step of the inner solver.  Its kernels are short (a few us up to some
// 100k rows), so what counts is how many there are: a sum over all rows ends
// in one partial sum per block, and every block of the next kernel adds those
// up again (at most kInnerBlocks, in a fixed order: the same total in every
// block) instead of waiting for a launch of its own.  A kernel reads scalars
// that earlier kernels wrote; block 0 writes new ones that no block of the
// same kernel reads.  12 launches and a copy to the host before, 7 now
// (PCG): a diagonally preconditioned run of 1,000 rows 18.7 -> 12.1 ms.  Up to
// 131,072 rows the sums are grouped as one block per 256 rows and one finishing
// block would, to the bit.

// The total of np partial sums, in every thread.
__device__ __forceinline__ double block_total(const double *__restrict__ p, int np) {
    __shared__ double red[kBlock / 64];
    const double s = wave_sum(thread_partials(p, np));
    __syncthreads();  // red may still be read from the total before
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += red[w];
    return t;
}

// ys[c] = -(total of column c's np <= kInnerBlocks partial sums), a wave per
// column, added in k_finish_columns' order
__device__ __forceinline__ void column_totals(const double *__restrict__ py, int np, int jq,
                                              double *ys) {
    static_assert(kInnerBlocks <= 2 * kBlock, "two partial sums per thread of k_finish_columns");
    const int lane = threadIdx.x & 63;
    for (int c = threadIdx.x >> 6; c < jq; c += kBlock / 64) {
        const double *p = py + (long)c * np;
        double v[kBlock / 64];
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) {
            const int b = w * 64 + lane;
            v[w] = b < np ? p[b] : 0.0;
            if (b + kBlock < np) v[w] += p[b + kBlock];
        }
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) t += wave_sum(v[w]);
        if (lane == 0) ys[c] = -t;
    }
    __syncthreads();
}

__device__ __forceinline__ bool broke(const InnerScalars *sc, double v) {
    return (sc->posdef && v <= 0.0) || v == 0.0;
}

// z -= Q ycoef ; partial sums of rho = r.z (JDaux.F:1916-1922 projection, then
// LSOLREVCOM label 3)
template <typename T, int NC>
__global__ __launch_bounds__(kBlock) void k_project_rho(T *__restrict__ z,
                                                        const T *__restrict__ Q, int jq,
                                                        const T *__restrict__ r, long n,
                                                        const double *__restrict__ py,
                                                        double *prho) {
    // the projection cancels the large components of z along the basis:
    // summed in double also for FP32 vectors
    __shared__ double ys[NC];
    column_totals(py, gridDim.x, jq, ys);
    constexpr int CH = NC < 8 ? NC : 8;
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        double zd = (double)z[i];
        const double ri = (double)r[i];
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += CH) {
            if (c0 >= jq) break;
            T v[CH];
#pragma unroll
            for (int c = 0; c < CH; ++c) v[c] = Q[(long)min(c0 + c, jq - 1) * n + i];
#pragma unroll
            for (int c = 0; c < CH; ++c)
                if (c0 + c < jq) zd += ys[c0 + c] * (double)v[c];
        }
        const T zi = (T)zd;
        z[i] = zi;
        acc[0] += ri * (double)zi;
    }
    grid_reduce<1>(acc, 1, prho, 0, nullptr);
}

// direction (LSOLREVCOM label 3): z += (rho/rho1) p ; p = z
template <typename T>
__global__ __launch_bounds__(kBlock) void k_direction(T *__restrict__ z, T *__restrict__ p,
                                                      long n, InnerScalars *sc, int iter,
                                                      const double *__restrict__ prho) {
    const double rho = block_total(prho, gridDim.x);
    const bool bad = broke(sc, rho);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->rho = rho;
        sc->flag = bad ? 1 : 0;
    }
    if (bad) return;
    const bool first = iter <= 1;
    const T beta = first ? T(0) : (T)(rho / sc->rho1);
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        T zi = z[i];
        if (!first && beta != T(0)) zi += beta * p[i];
        z[i] = zi;
        p[i] = zi;
    }
}

// after the matvec (JDaux.F:1898-1909 and LSOLREVCOM label 4): q -= u alprho,
// partial sums of pq = p.q
template <typename T>
__global__ __launch_bounds__(kBlock) void k_project_alpha(T *__restrict__ q,
                                                          const T *__restrict__ u,
                                                          const T *__restrict__ p, long n,
                                                          InnerScalars *sc,
                                                          const double *__restrict__ pu, int np,
                                                          double *ppq) {
    if (sc->flag) return;
    const double alprho = np > 0 ? block_total(pu, np) : sc->alprho;
    if (np > 0 && blockIdx.x == 0 && threadIdx.x == 0) sc->alprho = alprho;
    const T a = (T)(-alprho);
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        T qi = q[i] + a * u[i];
        q[i] = qi;
        acc[0] += (double)p[i] * (double)qi;
    }
    grid_reduce<1>(acc, 1, ppq, 0, nullptr);
}

// alpha = rho / pq in every thread; false on breakdown
__device__ __forceinline__ bool step_length(InnerScalars *sc, const double *__restrict__ ppq,
                                            double &alpha) {
    const double pq = block_total(ppq, gridDim.x);
    const bool ok = !broke(sc, pq);
    alpha = ok ? sc->rho / pq : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->pq = pq;
        if (ok) sc->alpha = alpha;
    }
    return ok;
}

// PCG update: r -= alpha q ; x += alpha p ; ||r||^2, ||x||^2
template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg_update(T *__restrict__ r, const T *__restrict__ q,
                                                      T *__restrict__ x, const T *__restrict__ p,
                                                      long n, InnerScalars *sc,
                                                      const double *__restrict__ ppq,
                                                      double *pout) {
    if (sc->flag) return;
    double alpha;
    if (!step_length(sc, ppq, alpha)) return;
    const T al = (T)alpha;
    double acc[2] = {0.0, 0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        T ri = r[i] + (-al) * q[i];
        r[i] = ri;
        acc[0] += (double)ri * (double)ri;
        T xi = x[i] + al * p[i];
        x[i] = xi;
        acc[1] += (double)xi * (double)xi;
    }
    grid_reduce<2>(acc, 2, pout, 0, nullptr);
}

// sQMR (LSOLREVCOM, JDaux.F:3167-3190): r -= alpha q, ||r||^2
template <typename T>
__global__ __launch_bounds__(kBlock) void k_qmr_r(T *__restrict__ r, const T *__restrict__ q,
                                                  long n, InnerScalars *sc,
                                                  const double *__restrict__ ppq, double *pout) {
    if (sc->flag) return;
    double alpha;
    if (!step_length(sc, ppq, alpha)) return;
    const T al = (T)alpha;
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        T ri = r[i] + (-al) * q[i];
        r[i] = ri;
        acc[0] += (double)ri * (double)ri;
    }
    grid_reduce<1>(acc, 1, pout, 0, nullptr);
}

// the smoothing scalars that ||r||^2 gives
struct Smooth {
    double ttk2m, ttk2, ck2, ggk2;
    __device__ Smooth(const InnerScalars *sc, double rr) {
        const double gk = sqrt(rr), gk2 = gk * gk;
        ttk2m = sc->ttk2;
        ttk2 = gk2 / sc->ggk2;
        ck2 = 1.0 / (1.0 + ttk2);
        ggk2 = sc->ggk2 * ttk2 * ck2;
    }
};

template <typename T>
__global__ __launch_bounds__(kBlock) void k_qmr_x(T *__restrict__ x, T *__restrict__ x2,
                                                  const T *__restrict__ p, long n,
                                                  const InnerScalars *sc, int iter,
                                                  const double *__restrict__ prr, double *pout) {
    if (sc->flag || broke(sc, sc->pq)) return;
    const Smooth m(sc, block_total(prr, gridDim.x));
    const double al = sc->alpha;
    const bool first = iter <= 1;
    const T c1 = first ? T(0) : (T)(al / m.ttk2m);
    const T c2 = first ? (T)(al * m.ck2) : (T)(m.ttk2m * m.ck2);
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        T xi;
        if (first) {
            T t = p[i] * c2;
            x2[i] = t;
            xi = t;
        } else {
            T t = (x2[i] + c1 * p[i]) * c2;
            x2[i] = t;
            xi = x[i] + t;
        }
        x[i] = xi;
        acc[0] += (double)xi * (double)xi;
    }
    grid_reduce<1>(acc, 1, pout, 0, nullptr);
}

// The end of a step (one block): the norms and, for sQMR, the smoothing
// scalars; then all scalars into the host's copy.  pout: the partial sums of
// ||r||^2, then those of ||x||^2.
__global__ __launch_bounds__(kBlock) void k_inner_end(InnerScalars *sc, bool posdef,
                                                      const double *__restrict__ pout, int np,
                                                      InnerScalars *host, Done done) {
    const bool on = !sc->flag;
    const bool bad = on && broke(sc, sc->pq);
    double rr = 0.0, xx = 0.0;
    if (on && !bad) {
        rr = block_total(pout, np);
        xx = block_total(pout + np, np);
    }
    if (threadIdx.x != 0) return;
    InnerScalars h = *sc;
    if (bad) {
        h.flag = 2;
    } else if (on) {
        if (!posdef) {
            const Smooth m(sc, rr);
            h.ttk2m = m.ttk2m;
            h.ttk2 = m.ttk2;
            h.ck2 = m.ck2;
            h.ggk2 = m.ggk2;
        }
        h.gk2 = rr;
        h.xn2 = xx;
        h.rho1 = h.rho;
    }
    *sc = h;
    *host = h;
    __hip_atomic_store(done.seq, done.v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

static inline int inner_grid(long n) { return grid_for(n, kBlock, kInnerBlocks); }

template <typename T>
void inner_direction(hipStream_t s, const RedBuf &rb, T *z, const T *Q, int jq, const T *r, T *p,
                     long n, InnerScalars *sc, int iter) {
    const int g = inner_grid(n);
    double *py = rb.inner(8), *prho = rb.inner(1);
#define JDHIP_PR(NC)                                                                    \
    do {                                                                                \
        k_multidot<T, NC><<<g, kBlock, 0, s>>>(Q, n, jq, z, n, py);                     \
        k_project_rho<T, NC><<<g, kBlock, 0, s>>>(z, Q, jq, r, n, py, prho);            \
    } while (0)
    if (jq <= 1) JDHIP_PR(1);
    else if (jq <= 2) JDHIP_PR(2);
    else if (jq <= 4) JDHIP_PR(4);
    else if (jq <= 8) JDHIP_PR(8);
    else if (jq <= 16) JDHIP_PR(16);
    else if (jq <= 32) JDHIP_PR(32);
    else JDHIP_PR(64);
#undef JDHIP_PR
    k_direction<T><<<g, kBlock, 0, s>>>(z, p, n, sc, iter, prho);
}

__global__ void k_inner_flag(const InnerScalars *sc, InnerScalars *host, Done done) {
    host->flag = sc->flag;
    __hip_atomic_store(done.seq, done.v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
void inner_flag(hipStream_t s, const InnerScalars *sc, InnerScalars *host, Done done) {
    k_inner_flag<<<1, 1, 0, s>>>(sc, host, done);
}

template <typename T>
void inner_update(hipStream_t s, const RedBuf &rb, bool posdef, T *r, T *q, const T *u, T *x,
                  T *x2, const T *p, long n, InnerScalars *sc, int iter, int np,
                  InnerScalars *host, Done done) {
    const int g = inner_grid(n);
    double *ppq = rb.inner(1), *pout = rb.inner(2);
    k_project_alpha<T><<<g, kBlock, 0, s>>>(q, u, p, n, sc, rb.inner_u(), np, ppq);
    if (posdef) {
        k_cg_update<T><<<g, kBlock, 0, s>>>(r, q, x, p, n, sc, ppq, pout);
    } else {
        k_qmr_r<T><<<g, kBlock, 0, s>>>(r, q, n, sc, ppq, pout);
        k_qmr_x<T><<<g, kBlock, 0, s>>>(x, x2, p, n, sc, iter, pout, pout + g);
    }
    k_inner_end<<<1, kBlock, 0, s>>>(sc, posdef, pout, g, host, done);
}

__global__ __launch_bounds__(kBlock) void k_inner_shift(double *__restrict__ q, double eta,
                                                        const double *__restrict__ p,
                                                        const double *__restrict__ u, long n,
                                                        double *pu) {
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) {
        double qi = q[i];
        if (eta != 0.0) qi += -eta * p[i];
        q[i] = qi;
        acc[0] += u[i] * qi;
    }
    grid_reduce<1>(acc, 1, pu, 0, nullptr);
}
int inner_shift(hipStream_t s, const RedBuf &rb, double *q, double eta, const double *p,
                const double *u, long n) {
    const int g = inner_grid(n);
    k_inner_shift<<<g, kBlock, 0, s>>>(q, eta, p, u, n, rb.inner_u());
    return g;
}

__global__ void k_inner_init(InnerScalars *sc, InnerScalars h) { *sc = h; }
void inner_init(hipStream_t s, InnerScalars *sc, const InnerScalars &h) {
    k_inner_init<<<1, 1, 0, s>>>(sc, h);
}

struct Small {
    double v[kMaxCols];
};
__global__ __launch_bounds__(kMaxCols) void k_put(double *dev, Small h, int cnt) {
    if ((int)threadIdx.x < cnt) dev[threadIdx.x] = h.v[threadIdx.x];
}
void put_small(hipStream_t s, double *dev, const double *host, int cnt) {
    Small h{};
    for (int i = 0; i < cnt; ++i) h.v[i] = host[i];
    k_put<<<1, kMaxCols, 0, s>>>(dev, h, cnt);
}
__global__ __launch_bounds__(kBlock) void k_get(double *host, const double *__restrict__ dev,
                                                int cnt, Done done) {
    for (int i = threadIdx.x; i < cnt; i += kBlock) host[i] = dev[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(done.seq, done.v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
void get_small(hipStream_t s, double *host, const double *dev, int cnt, Done done) {
    k_get<<<1, kBlock, 0, s>>>(host, dev, cnt, done);
}

#define JDHIP_INST(T)                                                                          \
    template void multidot<T>(hipStream_t, const RedBuf &, const T *, long, int, const T *,    \
                              long, double *);                                                 \
    template int spmv<T>(hipStream_t, const RedBuf &, const CsrDev &, const T *, T *, double,  \
                         const T *, double *);                                                 \
    template void diag_apply<T>(hipStream_t, T *, const T *, const T *, long);                 \
    template void inner_direction<T>(hipStream_t, const RedBuf &, T *, const T *, int,         \
                                     const T *, T *, long, InnerScalars *, int);                                          \
    template void inner_update<T>(hipStream_t, const RedBuf &, bool, T *, T *, const T *, T *, \
                                  T *, const T *, long, InnerScalars *, int, int,              \
                                  InnerScalars *, Done);
JDHIP_INST(double)
JDHIP_INST(float)

}  // namespace jdhip
