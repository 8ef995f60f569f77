// ildl_kernels.hip -- gfx950 kernels of the multilevel ILDL apply
// (see ildl_kernels.hpp).  Products with short rows run one lane per row
// on SELL-C-sigma copies (every load of a wave contiguous); long rows run
// on CSR with lane groups of 4 to 64 lanes and a butterfly reduction; the exact
// level-scheduled solve uses 4-lane groups per row of a level.  Every loop
// is grid-stride; vector entries are gathered through the column index.
// The factor's values are stored and streamed as T (double, or float on
// the mixed path), the apply's work vectors as W; every sum is double.  On
// indefinite matrices the mixed path keeps W = double: the substitutions
// cancel large terms, and float intermediates measurably slow the outer
// iteration there, while the vector traffic is small next to the
// factor's and the extra arithmetic is free in these HBM-bound loops.
#include "ildl_kernels.hpp"
#include "rowsum.hpp"
#include "xcd.hpp"

#include <algorithm>
#include <climits>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

namespace jdhip {

static constexpr int kB = 256;
static constexpr int kLpr = 4;

// With xcd != 0 the kernels below take their block id from logical_block()
// (xcd.hpp): every XCD works on one contiguous range of rows or slices.

// Launch k on q's stream, or add it to q's graph behind the last node.
template <typename... P, typename... A>
static void put(const Put &q, void (*k)(P...), int grid, A... args) {
    if (!q.graph) {
        k<<<grid, kB, 0, q.stream>>>(args...);
        return;
    }
    std::tuple<P...> held(static_cast<P>(args)...);
    std::apply(
        [&](auto &...x) {
            void *ptrs[] = {(void *)&x...};
            hipKernelNodeParams np{};
            np.func = (void *)k;
            np.gridDim = dim3(grid);
            np.blockDim = dim3(kB);
            np.kernelParams = ptrs;
            hipGraphNode_t node;
            const hipError_t e =
                hipGraphAddKernelNode(&node, q.graph, q.last ? &q.last : nullptr,
                                      q.last ? 1 : 0, &np);
            if (e != hipSuccess)
                throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e) +
                                         " adding a graph node");
            q.last = node;
            ++q.nodes;
        },
        held);
}

static inline int blocks_for(long n, int per_block, int cap = 8192) {
    long b = (n + per_block - 1) / per_block;
    return (int)std::max<long>(1, std::min<long>(b, cap));
}

template <typename TI, typename W>
__global__ __launch_bounds__(kB) void k_gather(int n, const int *__restrict__ perm,
                                               const double *__restrict__ scal,
                                               const TI *__restrict__ in,
                                               W *__restrict__ buf) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB) {
        int p = perm[i];
        buf[i] = (W)(scal[p] * (double)in[p]);
    }
}

template <typename W, typename TO>
__global__ __launch_bounds__(kB) void k_scatter(int n, int nB, const int *__restrict__ perm,
                                                const double *__restrict__ scal,
                                                const W *__restrict__ buf,
                                                const W *__restrict__ zc,
                                                TO *__restrict__ out) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB) {
        int p = perm[i];
        double v = (i < nB) ? (double)buf[i] : (double)zc[i - nB];
        out[p] = (TO)(scal[p] * v);
    }
}

template <typename T, typename W>
__global__ __launch_bounds__(kB) void k_trsv_level(const int *__restrict__ rows, int count,
                                                   const int *__restrict__ ptr,
                                                   const int *__restrict__ idx,
                                                   const T *__restrict__ val, W *x) {
    const int g = threadIdx.x / kLpr, l = threadIdx.x % kLpr;
    for (long t = (long)blockIdx.x * (kB / kLpr) + g; t < count;
         t += (long)gridDim.x * (kB / kLpr)) {
        const int r = rows[t];
        double s = 0.0;
        for (int k = ptr[r] + l; k < ptr[r + 1]; k += kLpr) s += (double)val[k] * (double)x[idx[k]];
#pragma unroll
        for (int o = kLpr / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kLpr);
        if (l == 0) x[r] = (W)((double)x[r] - s);
    }
}

// Loads of the matrix stream; NT = nontemporal, so the single-use values and
// columns do not push the reused x entries out of L2.
template <bool NT, typename X>
__device__ __forceinline__ X ld(const X *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Dot product of one SELL lane's row with x: w entries, column-major with
// stride 64; columns as int32 (CI = int, base 0) or as 16-bit offsets from
// the slice's base column (CI = unsigned short).  Four independent chains
// keep four gathers of x in flight per lane.
template <bool NT, typename T, typename W, typename CI>
__device__ __forceinline__ double sell_row(const T *v, const CI *c, int base, int w,
                                           const W *x) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int k = 0;
    for (; k + 3 < w; k += 4) {
        s0 += (double)ld<NT>(v + k * 64) * (double)x[base + (int)ld<NT>(c + k * 64)];
        s1 += (double)ld<NT>(v + (k + 1) * 64) * (double)x[base + (int)ld<NT>(c + (k + 1) * 64)];
        s2 += (double)ld<NT>(v + (k + 2) * 64) * (double)x[base + (int)ld<NT>(c + (k + 2) * 64)];
        s3 += (double)ld<NT>(v + (k + 3) * 64) * (double)x[base + (int)ld<NT>(c + (k + 3) * 64)];
    }
    for (; k < w; ++k) s0 += (double)ld<NT>(v + k * 64) * (double)x[base + (int)ld<NT>(c + k * 64)];
    return (s0 + s1) + (s2 + s3);
}

template <bool NT, typename T, typename W>
__device__ __forceinline__ double sell_slice_row(const SellView &M, const T *__restrict__ val,
                                                 long sl, int lane, const W *x) {
    const int code = M.code[sl];
    const T *v = val + M.vptr[sl] + lane;
    if (code & 1)
        return sell_row<NT>(v, (const unsigned short *)(M.idx + M.iptr[sl]) + lane, M.cbase[sl],
                            code >> 1, x);
    return sell_row<NT>(v, (const int *)(M.idx + M.iptr[sl]) + lane, 0, code >> 1, x);
}

// One row of a RowOp: its inputs, loaded ahead of the row's sum, and the write.
template <typename W>
struct RowIn {
    double src = 0.0, dinv = 1.0, add = 0.0;
    __device__ __forceinline__ void load(const RowOp<W> &op, long r) {
        if (op.src) src = (double)op.src[r];
        if (op.dinv) dinv = op.dinv[r];
        if (op.add) add = (double)op.add[r];
    }
    __device__ __forceinline__ void store(const RowOp<W> &op, long r, double sum) const {
        W v = (W)(src - sum);
        if (op.dinv) v = (W)((double)v * dinv);
        if (op.add) v = (W)(add + (double)v);
        op.out[r] = v;
    }
};

template <typename T, typename W, bool NT>
__global__ __launch_bounds__(kB) void k_sell(SellView M, const T *__restrict__ val, const W *x,
                                             RowOp<W> op, int xcd) {
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (long sl = logical_block(xcd) * (kB / 64) + wv; sl < M.nslices;
         sl += (long)gridDim.x * (kB / 64)) {
        const int r = M.rowid[sl * 64 + lane];
        if (r < 0) continue;
        RowIn<W> in;
        in.load(op, r);
        in.store(op, r, sell_slice_row<NT>(M, val, sl, lane, x));
    }
}

// CSR forms for matrices with long rows (LPR lanes per row, xor-butterfly
// reduction inside the lane group): with one lane per row such levels keep
// too few waves in flight and each lane walks its row serially.
template <typename T, typename W, int LPR>
__global__ __launch_bounds__(kB) void k_csr(int nrows, const int *__restrict__ ptr,
                                            const int *__restrict__ idx,
                                            const T *__restrict__ val, const W *x, RowOp<W> op,
                                            int xcd) {
    const int g = threadIdx.x / LPR, l = threadIdx.x % LPR;
    for (long r = logical_block(xcd) * (kB / LPR) + g; r < nrows; r += (long)gridDim.x * (kB / LPR)) {
        RowIn<W> in;
        if (l == 0) in.load(op, r);
        double s = csr_lane_sum<LPR>(idx, val, x, ptr[r], ptr[r + 1], l);
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, LPR);
        if (l == 0) in.store(op, r, s);
    }
}

// CSR-stream form: a block owns a run of consecutive rows with at most CAP
// entries (and at most kB rows), or a single longer row.  It streams the entries
// of its rows with coalesced, independent loads, parks the products in LDS, then
// sums each row with a group of t lanes (t = the power of two that spreads the
// block's rows over its 256 threads, at most 64) and a butterfly.  Every row is
// written.
//
// Bound by memory on large levels and by the chain of dependent loads on small
// ones, so the chain is kept to two: columns and values (at places that follow
// from the block's number) together with the block's descriptor; then the
// gathers of x together with the row's entry range and its RowOp inputs.  A
// thread takes entries in pairs (16 bytes of values, 4 or 8 of columns a load).
// From 2048 entries a block, one entry a load and row pointers in two dependent
// steps to entries in pairs behind one descriptor: sweeps of the 128^3 Laplacian
// (7.5M and 10.0M entries) 26.4 -> 24.7 and 27.4 -> 27.0 us, of 64^3 (1.0M and
// 1.2M) 7.2 -> 6.0 and 6.9 -> 5.4 us, of Anderson L = 32 (609k) 8.1 -> 5.4 us; to
// places that need no descriptor: a 64^3 apply 250 -> 244 us, a 73x61x51 solve
// 72.6 -> 70.3 ms, a 128^3 solve 951 -> 925 ms.
template <int CAP, bool NARROW, typename T, typename W>
__global__ __launch_bounds__(kB) void k_stream(StreamView<T> M, const int *__restrict__ idx,
                                               const T *__restrict__ val, const W *x,
                                               RowOp<W> op, int xcd) {
    typedef T T2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double prod[CAP];
    __shared__ double red[kB / 64];
    constexpr int kPairs = CAP / kB / 2;  // pairs per thread
    static_assert(kPairs * kB * 2 == CAP, "a block holds kPairs pairs per thread");
    const long blk = logical_block(xcd);
    const int tid = threadIdx.x;
    int c0[kPairs], c1[kPairs];
    T2 v[kPairs];
#pragma unroll
    for (int u = 0; u < kPairs; ++u) {
        const long k = blk * (CAP / 2) + tid + u * kB;
        if (NARROW) {
            const ushort2 q = ((const ushort2 *)M.c16)[k];
            c0[u] = q.x;
            c1[u] = q.y;
        } else {
            const int2 q = ((const int2 *)M.c32)[k];
            c0[u] = q.x;
            c1[u] = q.y;
        }
        v[u] = ((const T2 *)M.val)[k];
    }
    const int4 d = M.desc[blk];
    int cb = NARROW ? M.cbase[blk] : 0;
    if (NARROW && cb < 0) {  // a wide block
#pragma unroll
        for (int u = 0; u < kPairs; ++u) {
            const int2 q = ((const int2 *)M.c32)[(long)~cb * (CAP / 2) + tid + u * kB];
            c0[u] = q.x;
            c1[u] = q.y;
        }
        cb = 0;
    }
    const int r0 = d.x, nr = d.y, e0 = d.z, ne = d.w;
    if (ne > CAP) {  // one long row
        double s0 = 0.0, s1 = 0.0;
        int k = e0 + tid;
        for (; k + kB < e0 + ne; k += 2 * kB) {
            s0 += (double)val[k] * (double)x[idx[k]];
            s1 += (double)val[k + kB] * (double)x[idx[k + kB]];
        }
        if (k < e0 + ne) s0 += (double)val[k] * (double)x[idx[k]];
        double s = s0 + s1;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if ((tid & 63) == 0) red[tid >> 6] = s;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < kB / 64; ++w) t += red[w];
            RowIn<W> in;
            in.load(op, r0);
            in.store(op, r0, t);
        }
        return;
    }
    int t = 64;
    while (t > 1 && t * nr > kB) t >>= 1;
    const int g = tid / t, l = tid % t;
    const bool mine = g < nr;
    int a = 0, b = 0;
    RowIn<W> in;
    if (mine) {
        const unsigned short *o = M.off + (r0 + blk + g);
        a = o[0];
        b = o[1];
        if (l == 0) in.load(op, r0 + g);
    }
    // padding has column 0 of the block (a valid place) and is not summed
#pragma unroll
    for (int u = 0; u < kPairs; ++u) {
        const int k = 2 * (tid + u * kB);
        if (k < ne) {
            double2 p;
            p.x = (double)v[u].x * (double)x[cb + c0[u]];
            p.y = (double)v[u].y * (double)x[cb + c1[u]];
            *(double2 *)(prod + k) = p;
        }
    }
    __syncthreads();
    double s = 0.0;
    if (mine)
        for (int k = a + l; k < b; k += t) s += prod[k];
    for (int o = t / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, t);
    if (mine && l == 0) in.store(op, r0 + g, s);
}

template <typename W>
__global__ __launch_bounds__(kB) void k_dscale(int n, const double *__restrict__ dinv, W *x) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB)
        x[i] = (W)((double)x[i] * dinv[i]);
}

template <typename W>
__global__ __launch_bounds__(kB) void k_dscale2(int n, const double *__restrict__ dinv,
                                                const double *__restrict__ doff,
                                                const int *__restrict__ pair, W *x) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB) {
        const int p = pair[i];
        if (p < 0) {
            x[i] = (W)((double)x[i] * dinv[i]);
        } else if (i < p) {
            const double xi = (double)x[i], xp = (double)x[p];
            x[i] = (W)(dinv[i] * xi + doff[i] * xp);
            x[p] = (W)(doff[p] * xi + dinv[p] * xp);
        }
    }
}

template <typename W>
__global__ __launch_bounds__(kB) void k_zero(int n, W *x) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB)
        x[i] = W(0);
}
template <typename W>
__global__ __launch_bounds__(kB) void k_copy(int n, const W *__restrict__ t, W *__restrict__ y) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB)
        y[i] = t[i];
}
template <typename W>
__global__ __launch_bounds__(kB) void k_add(int n, const W *__restrict__ t, W *__restrict__ y) {
    for (long i = blockIdx.x * (long)kB + threadIdx.x; i < n; i += (long)gridDim.x * kB)
        y[i] = (W)((double)y[i] + (double)t[i]);
}

// one wave per row of the dense inverse
template <typename T, typename W>
__global__ __launch_bounds__(kB) void k_dense_gemv(int m, const T *__restrict__ Minv,
                                                   const W *__restrict__ x, W *__restrict__ y) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (long r = (long)blockIdx.x * (kB / 64) + w; r < m; r += (long)gridDim.x * (kB / 64)) {
        const T *row = Minv + r * (long)m;
        double s = 0.0;
        for (int j = lane; j < m; j += 64) s += (double)row[j] * (double)x[j];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) y[r] = (W)s;
    }
}

template <typename TI, typename W>
void ildl_gather(const Put &s, int n, const int *perm, const double *scal, const TI *in,
                 W *buf) {
    if (n <= 0) return;
    put(s, k_gather<TI, W>, blocks_for(n, kB), n, perm, scal, in, buf);
}
template <typename W, typename TO>
void ildl_scatter(const Put &s, int n, int nB, const int *perm, const double *scal,
                  const W *buf, const W *zc, TO *out) {
    if (n <= 0) return;
    put(s, k_scatter<W, TO>, blocks_for(n, kB), n, nB, perm, scal, buf, zc, out);
}
template <typename T, typename W>
void ildl_trsv_level(const Put &s, const int *rows, int count, const int *ptr, const int *idx,
                     const T *val, W *x) {
    if (count <= 0) return;
    put(s, k_trsv_level<T, W>, blocks_for(count, kB / kLpr), rows, count, ptr, idx, val,
                                                                   x);
}
template <typename T, typename W>
void ildl_sell(const Put &s, const SellView &M, const T *val, const W *x, const RowOp<W> &op,
               int xcd) {
    if (M.nslices <= 0) return;
    const int g = blocks_for(M.nslices, kB / 64, 1 << 20);
    if (xcd & 2) put(s, k_sell<T, W, true>, g, M, val, x, op, xcd & 1);
    else put(s, k_sell<T, W, false>, g, M, val, x, op, xcd & 1);
}
template <typename T, typename W>
void ildl_csr(const Put &s, int lpr, int nrows, const int *ptr, const int *idx, const T *val,
              const W *x, const RowOp<W> &op, int xcd) {
    if (nrows <= 0) return;
#define JDHIP_C(L) \
    put(s, k_csr<T, W, L>, blocks_for(nrows, kB / L, 1 << 20), nrows, ptr, idx, val, x, op, xcd)
    if (lpr >= 64) JDHIP_C(64);
    else if (lpr >= 32) JDHIP_C(32);
    else if (lpr >= 16) JDHIP_C(16);
    else if (lpr >= 8) JDHIP_C(8);
    else JDHIP_C(4);
#undef JDHIP_C
}
template <typename T, typename W>
void ildl_stream(const Put &s, const StreamView<T> &M, const int *idx, const T *val, const W *x,
                 const RowOp<W> &op, int xcd) {
    if (M.nblk <= 0) return;
#define JDHIP_ST(C, N) put(s, k_stream<C, N, T, W>, M.nblk, M, idx, val, x, op, xcd)
    if (M.c16) {
        if (M.cap == 512) JDHIP_ST(512, true);
        else JDHIP_ST(1024, true);
    } else {
        if (M.cap == 512) JDHIP_ST(512, false);
        else JDHIP_ST(1024, false);
    }
#undef JDHIP_ST
}

// Entries a block holds: 1024 where that leaves enough blocks for the 256 CUs,
// else 512.  Measured (us a sweep, 512 against 1024): 354k entries 3.8 / 4.1,
// 609k 5.4 / 5.8, 988k 6.3 / 6.0, 1.2M 5.8 / 5.4, 7.5M 28.7 / 24.7.
static constexpr long kStreamWide = 800000;

// Columns take 16 bits where at most one block in this many is wide (spans
// 65,536 columns or more): a wide block loads its columns again, in 32 bits, once
// it knows its descriptor.  100^3 Laplacian, 17 wide blocks of 3,623: sweep 14.7
// -> 14.1 us, apply 569 -> 560 us, with FP32 values 11.6 -> 10.5 and 453 -> 434.
// With a quarter of wide blocks it is no gain: Anderson L = 100, level 2 (10.2M
// entries), 34.1 and 33.3 us all in 32 bits, 34.2 and 34.0 in both widths.
static constexpr size_t kFewWide = 8;

template <typename T>
StreamHost<T> build_stream(int nrows, const std::vector<int> &ptr, const std::vector<int> &idx,
                           const std::vector<T> &val) {
    StreamHost<T> h;
    const int nnz = ptr[nrows];
    h.cap = nnz >= kStreamWide ? 1024 : 512;
    int wide = 0;
    int r = 0;
    while (r < nrows) {
        const int r0 = r, e0 = ptr[r];
        while (r < nrows && r - r0 < kB && ptr[r + 1] - e0 <= h.cap) ++r;
        if (r == r0) ++r;  // a long row alone
        const int ne = ptr[r] - e0;
        int cmin = INT_MAX, cmax = INT_MIN;
        if (ne <= h.cap)
            for (int k = e0; k < e0 + ne; ++k) {
                cmin = std::min(cmin, idx[k]);
                cmax = std::max(cmax, idx[k]);
            }
        if (cmin > cmax) cmin = cmax = 0;
        h.desc.push_back(make_int4(r0, r - r0, e0, ne));
        h.cbase.push_back((long)cmax - cmin < 65536 ? cmin : ~wide++);
        // entry range of each row, from the block's first entry (a long row's
        // range is not read)
        for (int i = r0; i <= r; ++i) h.off.push_back((unsigned short)(ptr[i] - e0));
    }
    const size_t slots = h.desc.size() * h.cap;
    const bool narrow = wide * kFewWide <= h.desc.size();
    h.val.assign(slots, T(0));
    if (narrow) h.c16.assign(slots, 0);
    h.c32.assign(narrow ? (size_t)wide * h.cap : slots, 0);
    for (size_t b = 0; b < h.desc.size(); ++b) {
        const int e0 = h.desc[b].z, ne = h.desc[b].w, cb = h.cbase[b];
        const bool n16 = narrow && cb >= 0 && ne <= h.cap;
        (n16 ? h.nnz16 : h.nnz32) += ne;
        if (ne > h.cap) continue;
        std::copy(val.begin() + e0, val.begin() + e0 + ne, h.val.begin() + b * h.cap);
        if (n16)
            for (int k = 0; k < ne; ++k) h.c16[b * h.cap + k] = (unsigned short)(idx[e0 + k] - cb);
        else
            std::copy(idx.begin() + e0, idx.begin() + e0 + ne,
                      h.c32.begin() + (narrow ? (size_t)~cb : b) * h.cap);
    }
    return h;
}
template StreamHost<double> build_stream(int, const std::vector<int> &, const std::vector<int> &,
                                         const std::vector<double> &);
template StreamHost<float> build_stream(int, const std::vector<int> &, const std::vector<int> &,
                                        const std::vector<float> &);

template <typename W>
void ildl_dscale(const Put &s, int n, const double *dinv, W *x) {
    if (n <= 0) return;
    put(s, k_dscale<W>, blocks_for(n, kB), n, dinv, x);
}
template <typename W>
void ildl_dscale2(const Put &s, int n, const double *dinv, const double *doff, const int *pair,
                  W *x) {
    if (n <= 0) return;
    put(s, k_dscale2<W>, blocks_for(n, kB), n, dinv, doff, pair, x);
}
template void ildl_dscale2<double>(const Put &, int, const double *, const double *, const int *,
                                   double *);
template void ildl_dscale2<float>(const Put &, int, const double *, const double *, const int *,
                                  float *);
template <typename W>
void ildl_zero(const Put &s, int n, W *x) {
    if (n <= 0) return;
    put(s, k_zero<W>, blocks_for(n, kB), n, x);
}
template <typename W>
void ildl_copy(const Put &s, int n, const W *t, W *y) {
    if (n <= 0) return;
    put(s, k_copy<W>, blocks_for(n, kB), n, t, y);
}
template void ildl_copy<double>(const Put &, int, const double *, double *);
template void ildl_copy<float>(const Put &, int, const float *, float *);
template <typename W>
void ildl_add(const Put &s, int n, const W *t, W *y) {
    if (n <= 0) return;
    put(s, k_add<W>, blocks_for(n, kB), n, t, y);
}
template void ildl_zero<double>(const Put &, int, double *);
template void ildl_zero<float>(const Put &, int, float *);
template void ildl_add<double>(const Put &, int, const double *, double *);
template void ildl_add<float>(const Put &, int, const float *, float *);
template <typename T, typename W>
void ildl_dense_gemv(const Put &s, int m, const T *Minv, const W *x, W *y) {
    if (m <= 0) return;
    put(s, k_dense_gemv<T, W>, blocks_for(m, kB / 64, 4096), m, Minv, x, y);
}

#define INST(T, W)                                                                           \
    template void ildl_trsv_level<T, W>(const Put &, const int *, int, const int *,          \
                                        const int *, const T *, W *);                        \
    template void ildl_sell<T, W>(const Put &, const SellView &, const T *, const W *,        \
                                  const RowOp<W> &, int);                                     \
    template void ildl_csr<T, W>(const Put &, int, int, const int *, const int *, const T *,  \
                                 const W *, const RowOp<W> &, int);                           \
    template void ildl_dense_gemv<T, W>(const Put &, int, const T *, const W *, W *);         \
    template void ildl_stream<T, W>(const Put &, const StreamView<T> &, const int *, const T *,  \
                                    const W *, const RowOp<W> &, int);
INST(double, double)
INST(float, double)
INST(float, float)
template void ildl_dscale<double>(const Put &, int, const double *, double *);
template void ildl_dscale<float>(const Put &, int, const double *, float *);
#define INST_IO(A, B)                                                                        \
    template void ildl_gather<A, B>(const Put &, int, const int *, const double *, const A *, \
                                    B *);                                                    \
    template void ildl_scatter<B, A>(const Put &, int, int, const int *, const double *,      \
                                     const B *, const B *, A *);
INST_IO(double, double)
INST_IO(double, float)
INST_IO(float, double)
INST_IO(float, float)

}  // namespace jdhip
