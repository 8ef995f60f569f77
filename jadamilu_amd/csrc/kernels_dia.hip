// kernels_dia.hip -- SpMV and SpMM for matrices whose entries lie on a few
// diagonals (the stencils on a box, with or without periodic sides).
//
// MATVECA (src/jd/JDaux.F:3397-3418).  The symmetric product is bound by HBM,
// and the general formats store both triangles with a column index an entry.
// Here only the upper triangle is stored, one array per diagonal, and no
// indices: row i's entry left of the diagonal, A(i, i-d) = A(i-d, i), is read
// where row i-d keeps it.  That read and the one of x(i-d) repeat loads that
// the same XCD made d rows earlier, so with every XCD on one contiguous range
// of rows (xcd.hpp) they are served by its L2 while d rows of values and
// vectors fit there.
//
// One wave64 takes a slice of 64 rows, a lane a row.  For each diagonal two
// 64-bit masks say which of the slice's rows have an entry there, above and
// below: a slice without any skips the loads (periodic sides touch few), and
// an absent entry is never multiplied (an infinite or NaN x must not reach
// rows that do not refer to it).
//
// Against the general formats (three matrices in turn, so that the Infinity
// Cache does not hold them): 128^3 Laplacian 35.9 -> 22.1 us (107 MB of HBM
// traffic instead of 182 MB), and with two in turn 35.0 -> 14.5 us; Anderson
// L = 100 with two in turn 11.6 -> 8.3 us; ten vectors of it 79.2 -> 72.7 us
// (239 MB of HBM traffic for 192 MB needed, and 26.8 million L1 accesses, 44 us
// of the L1's time: neither alone is the whole).
#include "kernels.hpp"
#include "reduce.hpp"
#include "xcd.hpp"

namespace jdhip {

namespace {

typedef unsigned long long u64;

// Whether this lane's bit of a mask that is the same in the whole wave is set:
// the mask itself is the condition (testing the bit by shifts made the kernels
// bound by integer instructions).
__device__ __forceinline__ bool has(u64 m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// p[i] with a byte offset of 32 bits (kDiaRows rows at most), so that the
// array's address stays in scalar registers.
template <typename T>
__device__ __forceinline__ T at(const T *p, unsigned i) {
    return *(const T *)((const char *)p + i * (unsigned)sizeof(T));
}

// A wave's slices: XCD-contiguous blocks, one slice a wave.
#define JDHIP_SLICES(sl, row)                                                                  \
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;  \
    const long sl = logical_block(1) * (kBlock / 64) + wv;                                     \
    const unsigned row = (unsigned)(sl * 64 + lane)

// Entries below the diagonal in ascending column order, then the diagonal and
// above: the order of a row's entries in the CSR copy.  ND: the number of
// diagonals, all loads issued before the first use (FP32 values are therefore
// kept as they are until then: converted beside their loads they were compiled
// to three loads in flight; FP32 SpMV, 80^3 Laplacian 6.6 -> 5.4 us, Anderson L =
// 52 6.4 -> 4.8).
template <typename T, typename TA, int ND, bool ETA, bool UDOT>
__global__ __launch_bounds__(kBlock) void k_spmv_dia(DiaDev A, const TA *__restrict__ val,
                                                     const T *__restrict__ x,
                                                     T *__restrict__ y, double eta,
                                                     const T *__restrict__ u, double *partials) {
    double acc[1] = {0.0};
    JDHIP_SLICES(sl, row);
    if (sl < A.nslices && row < (unsigned)A.n) {
        const u64 *m = A.mask + sl * 2 * A.nd;
        double s = 0.0;
        TA vu[ND], vl[ND];
        T xu[ND], xl[ND];
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const u64 mu = m[2 * k], ml = m[2 * k + 1];
            const unsigned d = (unsigned)A.off[k];
            vu[k] = vl[k] = TA(0);
            xu[k] = xl[k] = T(0);
            if (mu) {
                vu[k] = at(val + k * A.stride, row);
                xu[k] = at(x, has(mu) ? row + d : row);
            }
            if (k > 0 && ml) {
                const unsigned j = has(ml) ? row - d : row;
                vl[k] = at(val + k * A.stride, j);
                xl[k] = at(x, j);
            }
        }
#pragma unroll
        for (int k = ND - 1; k > 0; --k) s = has(m[2 * k + 1]) ? s + (double)vl[k] * (double)xl[k] : s;
#pragma unroll
        for (int k = 0; k < ND; ++k) s = has(m[2 * k]) ? s + (double)vu[k] * (double)xu[k] : s;
        if (ETA) s -= eta * (double)x[row];
        const T yi = (T)s;
        y[row] = yi;
        if (UDOT) acc[0] += (double)u[row] * (double)yi;
    }
    if (UDOT) grid_reduce<1>(acc, 1, partials, 0, nullptr);
}

// kv vectors, per of them a block.  A row's values are loaded once and stay in
// registers for these; the vectors go by one at a time (two or four at a time,
// whose loads would all be in flight, leave too few waves: 78 and 88 us against
// 70 for 5 vectors of the 128^3 Laplacian).  A small matrix is bound by that
// chain of loads, so its vectors go to different blocks.  Us for 3 / 10 vectors,
// all in one block, spread, and the CSR form: 64^2 Laplacian 2.99, 2.38, 2.40 /
// 5.22, 2.42, 5.10; 250^2 3.19, 2.90, 4.11 / 6.13, 4.75, 10.7; Anderson L = 17
// (7 diagonals) 3.81, 2.91, 2.61 / 7.29, 2.96, 5.60.  Spread to 1,024 blocks, L =
// 50 takes 5.36 instead of 4.94 us for 3 vectors, to 4,096 6.22.
constexpr int kSpread = 512;
template <int ND>
__global__ __launch_bounds__(kBlock) void k_spmm_dia(DiaDev A, int kv, int per,
                                                     const double *__restrict__ x, long ldx,
                                                     double *__restrict__ y, long ldy) {
    JDHIP_SLICES(sl, row);
    if (sl >= A.nslices || row >= (unsigned)A.n) return;
    const u64 *m = A.mask + sl * 2 * A.nd;
    double vu[ND], vl[ND];
    unsigned ju[ND], jl[ND];
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        const unsigned d = (unsigned)A.off[k];
        vu[k] = vl[k] = 0.0;
        ju[k] = has(m[2 * k]) ? row + d : row;
        jl[k] = has(m[2 * k + 1]) ? row - d : row;
        if (m[2 * k]) vu[k] = at(A.val + k * A.stride, row);
        if (k > 0 && m[2 * k + 1]) vl[k] = at(A.val + k * A.stride, jl[k]);
    }
#pragma unroll 1
    for (int c = blockIdx.y * per; c < min(kv, (int)(blockIdx.y + 1) * per); ++c) {
        const double *xc = x + c * ldx;
        double xu[ND], xl[ND];
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            xu[k] = xl[k] = 0.0;
            if (m[2 * k]) xu[k] = at(xc, ju[k]);
            if (k > 0 && m[2 * k + 1]) xl[k] = at(xc, jl[k]);
        }
        double s = 0.0;
#pragma unroll
        for (int k = ND - 1; k > 0; --k) s = has(m[2 * k + 1]) ? s + vl[k] * xl[k] : s;
#pragma unroll
        for (int k = 0; k < ND; ++k) s = has(m[2 * k]) ? s + vu[k] * xu[k] : s;
        y[row + c * ldy] = s;
    }
}
#undef JDHIP_SLICES

template <typename T, typename TA, int ND>
void launch(hipStream_t s, int g, const DiaDev &A, const TA *val, const T *x, T *y, double eta,
            const T *u, double *P) {
#define JDHIP_D(E, U) k_spmv_dia<T, TA, ND, E, U><<<g, kBlock, 0, s>>>(A, val, x, y, eta, u, P)
    if (u) {
        if (eta != 0.0) JDHIP_D(true, true);
        else JDHIP_D(false, true);
    } else {
        if (eta != 0.0) JDHIP_D(true, false);
        else JDHIP_D(false, false);
    }
#undef JDHIP_D
}

template <typename T, typename TA>
int product(hipStream_t s, const RedBuf &rb, const DiaDev &A, const TA *val, const T *x, T *y,
            double eta, const T *u, double *udot_out) {
    const long blocks = ((long)A.nslices + kBlock / 64 - 1) / (kBlock / 64);
    const int g = (int)blocks;  // at most kDiaRows / 256, which fits the partial sums' scratch
    double *P = g <= kInnerBlocks ? rb.inner_u() : rb.partials;
#define JDHIP_ND(D) launch<T, TA, D>(s, g, A, val, x, y, eta, u, P)
    switch (A.nd) {
        case 1: JDHIP_ND(1); break;
        case 2: JDHIP_ND(2); break;
        case 3: JDHIP_ND(3); break;
        case 4: JDHIP_ND(4); break;
        case 5: JDHIP_ND(5); break;
        case 6: JDHIP_ND(6); break;
        default: JDHIP_ND(7); break;
    }
#undef JDHIP_ND
    if (!u) return 0;
    if (g <= kInnerBlocks) return g;
    finish_sum(s, P, g, udot_out);
    return 0;
}

}  // namespace

template <>
int spmv_dia<double>(hipStream_t s, const RedBuf &rb, const DiaDev &A, bool, const double *x,
                     double *y, double eta, const double *u, double *udot_out) {
    return product<double, double>(s, rb, A, A.val, x, y, eta, u, udot_out);
}
template <>
int spmv_dia<float>(hipStream_t s, const RedBuf &rb, const DiaDev &A, bool vals64,
                    const float *x, float *y, double eta, const float *u, double *udot_out) {
    if (vals64) return product<float, double>(s, rb, A, A.val, x, y, eta, u, udot_out);
    return product<float, float>(s, rb, A, A.valf, x, y, eta, u, udot_out);
}

void spmm_dia(hipStream_t s, const DiaDev &A, int k, const double *x, long ldx, double *y,
              long ldy) {
    const long blocks = ((long)A.nslices + kBlock / 64 - 1) / (kBlock / 64);
    const int g = (int)blocks;
    // vectors a block takes: all of them, or so many that there are kSpread blocks
    const int groups = std::max(1, std::min(k, kSpread / g)), per = (k + groups - 1) / groups;
    switch (A.nd) {
#define JDHIP_ND(D) \
    k_spmm_dia<D><<<dim3(g, (k + per - 1) / per), kBlock, 0, s>>>(A, k, per, x, ldx, y, ldy)
        case 1: JDHIP_ND(1); break;
        case 2: JDHIP_ND(2); break;
        case 3: JDHIP_ND(3); break;
        case 4: JDHIP_ND(4); break;
        case 5: JDHIP_ND(5); break;
        case 6: JDHIP_ND(6); break;
        default: JDHIP_ND(7); break;
#undef JDHIP_ND
    }
}

// The layout of an upper CSR (1-based): false if it has an entry below the
// diagonal or one twice, more than kDiaMax diagonals, or slices so empty that a
// pass would load more than twice its entries (there the general formats, at
// 1.6 times the bytes an entry, are as good).
bool build_dia(int n, const int *ia, const int *ja, const double *a, DiaHost &h) {
    h = DiaHost{};
    if (n > kDiaRows) return false;
    // the diagonals in order of appearance; an entry's is mostly the one after
    // the entry's before it
    int d[kDiaMax], nd = 0, guess = 0;
    auto find = [&](int o) {
        for (int t = 0; t < nd; ++t) {
            guess = guess + 1 < nd ? guess + 1 : 0;
            if (d[guess] == o) return guess;
        }
        return -1;
    };
    for (int i = 0; i < n; ++i)
        for (int e = ia[i] - 1; e < ia[i + 1] - 1; ++e) {
            const int o = ja[e] - 1 - i;
            if (o < 0) return false;  // not the upper triangle
            if (find(o) < 0) {
                if (nd == kDiaMax) return false;
                d[nd++] = o;
            }
        }
    if (find(0) < 0) {
        if (nd == kDiaMax) return false;
        d[nd++] = 0;
    }
    h.nd = nd;
    h.nslices = (n + 63) / 64;
    h.stride = 64L * h.nslices;
    // the arrays hold every row of every diagonal; at most four times the entries
    if ((double)nd * h.stride > 4.0 * (ia[n] - 1) + 4096.0) return false;
    h.off.assign(d, d + nd);
    std::sort(h.off.begin(), h.off.end());
    int rank[kDiaMax];
    for (int k = 0; k < nd; ++k)
        rank[k] = (int)(std::lower_bound(h.off.begin(), h.off.end(), d[k]) - h.off.begin());
    h.val.assign((size_t)nd * h.stride, 0.0);
    h.mask.assign((size_t)h.nslices * 2 * nd, 0);
    for (int i = 0; i < n; ++i)
        for (int e = ia[i] - 1; e < ia[i + 1] - 1; ++e) {
            const int j = ja[e] - 1, k = rank[find(j - i)];
            u64 &mu = h.mask[(size_t)(i >> 6) * 2 * nd + 2 * k];
            if (mu >> (i & 63) & 1) return false;  // the entry is there twice
            mu |= 1ull << (i & 63);
            if (k > 0) h.mask[(size_t)(j >> 6) * 2 * nd + 2 * k + 1] |= 1ull << (j & 63);
            h.val[(size_t)k * h.stride + i] = a[e];
        }
    // what a pass loads: 64 values for every diagonal present in a slice,
    // above; a matrix whose present slices are mostly empty stays general
    long loaded = 0;
    for (int s = 0; s < h.nslices; ++s)
        for (int k = 0; k < h.nd; ++k) loaded += h.mask[(size_t)s * 2 * h.nd + 2 * k] ? 64 : 0;
    return loaded <= 2L * (ia[n] - 1);
}

}  // namespace jdhip
