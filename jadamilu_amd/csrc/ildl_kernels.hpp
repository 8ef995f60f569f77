// ildl_kernels.hpp -- gfx950 kernels of the multilevel ILDL apply.
//
// Per level (src/ilupack/symAMGsol.c:173-628 restated), with the coupling
// block F^T = A_CB (the reference's structure):
//   gather+scale -> y_B = B^-1 b_B (forward L_B sweep, D^-1, backward L_B^T
//   sweep) -> coarse rhs b_C - F^T y_B -> [next level] -> x_B = y_B -
//   B^-1 F x_C (a second solve with B) -> scatter+scale;
// with the factor's own coupling rows L_CB instead:
//   gather+scale -> forward L_B sweep -> coarse rhs (C rows) -> D^-1 ->
//   [next level] -> B rows minus L_CB^T z_C -> backward L_B^T sweep ->
//   scatter+scale.
// The triangular sweeps are level-scheduled (one launch per dependency
// level, rows of a level in parallel) or, in sweep mode, a fixed number of
// Jacobi iterations x <- b - N x on the strictly triangular part.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

namespace jdhip {

// Where the launches below go: onto a stream or, when graph is set, behind the
// last node of a graph that is being built.  The graph is built node by node
// and not by capture: a capture would make other threads' work on the legacy
// null stream fail while it lasts.
struct Put {
    hipStream_t stream = nullptr;
    hipGraph_t graph = nullptr;
    mutable hipGraphNode_t last = nullptr;
    mutable int nodes = 0;  // in the graph so far
    Put(hipStream_t s) : stream(s) {}
    Put(hipGraph_t g) : graph(g) {}
};

// Factor values are T (double or float), work vectors W (double or float);
// sums are double.
template <typename TI, typename W>
void ildl_gather(const Put &s, int n, const int *perm, const double *scal, const TI *in,
                 W *buf);
template <typename W, typename TO>
void ildl_scatter(const Put &s, int n, int nB, const int *perm, const double *scal,
                  const W *buf, const W *zc, TO *out);
// x[rows of one level] -= sum_j M(row, j) x[j]   (unit-diagonal triangular)
template <typename T, typename W>
void ildl_trsv_level(const Put &s, const int *rows, int count, const int *ptr, const int *idx,
                     const T *val, W *x);
// Device view of a SELL-C-sigma matrix: slices of 64 rows (one wave64, one
// lane per row) taken from windows of rows sorted by length; entries of a
// slice stored column-major (value at val[vptr[s] + k*64 + lane], k <
// width); the slice's column indices start at byte iptr[s] of idx, as
// 16-bit offsets from cbase[s] when code[s] is odd, else as int32 columns;
// width = code[s] >> 1; rowid[s*64 + lane] is the row a lane owns (-1 for
// padding lanes).
struct SellView {
    int nslices = 0;
    const long *vptr = nullptr;
    const long *iptr = nullptr;
    const int *code = nullptr;
    const int *rowid = nullptr;
    const int *cbase = nullptr;
    const char *idx = nullptr;
};
// What a product M x becomes, row by row: v = src - (M x) (src null: 0), then
// v = dinv v (dinv null: as it is), then v = add + v (add null: as it is),
// rounded to the work vectors' type after each step, into out.  src, add and
// out may be one array (a row is read and written by the same thread); out is
// never x.  So a sweep is src = b, the last sweep before D^-1 carries dinv, the
// last one of the second solve adds into y_B, and F x_C needs no zeroed vector.
template <typename W>
struct RowOp {
    const W *src = nullptr;
    const double *dinv = nullptr;
    const W *add = nullptr;
    W *out = nullptr;
};
// SELL-C-sigma form, one lane per row.  xcd bit 0: XCD-contiguous block order;
// bit 1: nontemporal loads of the matrix stream.
template <typename T, typename W>
void ildl_sell(const Put &s, const SellView &M, const T *val, const W *x, const RowOp<W> &op,
               int xcd);
// CSR form with lpr (4, 8, 16, 32 or 64) lanes per row, for small matrices and
// long rows; xcd != 0: XCD-contiguous block order
template <typename T, typename W>
void ildl_csr(const Put &s, int lpr, int nrows, const int *ptr, const int *idx, const T *val,
              const W *x, const RowOp<W> &op, int xcd);
// CSR-stream form: blocks of consecutive rows with at most cap entries (and 256
// rows) each, or one longer row, streamed through LDS with coalesced loads.
// Block b's entries are laid out again from entry b*cap on (padded with zeros),
// so that a block finds them without looking anything up: values val, and
// columns c16 (offsets from cbase[b] >= 0) if most blocks' span less than 2^16,
// else c32.  Beside c16, c32 holds only the blocks whose columns span more, block
// b from entry ~cbase[b]*cap on.  desc[b] = {first row, rows, first entry in the CSR, entries} (a longer
// row is read from there); off[row + b] and the next are a row's entry range
// from the block's first entry.
template <typename T>
struct StreamView {
    int nblk = 0;
    int cap = 1024;
    const int4 *desc = nullptr;
    const int *cbase = nullptr;
    const unsigned short *off = nullptr;
    const unsigned short *c16 = nullptr;
    const int *c32 = nullptr;
    const T *val = nullptr;
};
template <typename T>
struct StreamHost {
    int cap = 1024;
    std::vector<int4> desc;
    std::vector<int> cbase, c32;
    std::vector<unsigned short> off, c16;
    std::vector<T> val;
    long nnz16 = 0, nnz32 = 0;  // entries (no padding) by the column width they are read with
};
template <typename T>
StreamHost<T> build_stream(int nrows, const std::vector<int> &ptr, const std::vector<int> &idx,
                           const std::vector<T> &val);
// xcd != 0: every XCD takes one contiguous range of row blocks.
template <typename T, typename W>
void ildl_stream(const Put &s, const StreamView<T> &M, const int *idx, const T *val, const W *x,
                 const RowOp<W> &op, int xcd);
template <typename W>
void ildl_dscale(const Put &s, int n, const double *dinv, W *x);
// x = D^-1 x with 2x2 blocks: row i pairs with pair[i] (-1: 1x1 pivot,
// x_i *= dinv_i); a pair is updated by its lower index,
// (x_i, x_p) <- (dinv_i x_i + doff_i x_p, doff_p x_i + dinv_p x_p)
template <typename W>
void ildl_dscale2(const Put &s, int n, const double *dinv, const double *doff, const int *pair,
                  W *x);
// x = 0 (a kernel, not a memset: the apply may be captured in a HIP graph)
template <typename W>
void ildl_zero(const Put &s, int n, W *x);
// y = t
template <typename W>
void ildl_copy(const Put &s, int n, const W *t, W *y);
// y += t
template <typename W>
void ildl_add(const Put &s, int n, const W *t, W *y);
// y = Minv x, Minv m x m row-major
template <typename T, typename W>
void ildl_dense_gemv(const Put &s, int m, const T *Minv, const W *x, W *y);

}  // namespace jdhip
