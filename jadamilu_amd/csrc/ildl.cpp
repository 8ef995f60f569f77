// ildl.cpp -- multilevel ILDL preconditioner: device upload and apply.
//
// apply(z, r) restates DSYMAMGsol (src/ilupack/symAMGsol.c:110-631) and the
// wrappers SYMILUPACKSOL / sdsymamgsol (symilupacksol.c:60-128,
// singlesymilupacksol.c:69-104): FP64 in/out, the factor applied in T
// (double, or float for the mixed path with conversion at the first gather
// and the last scatter).
#include "ildl.hpp"

#include <algorithm>
#include <climits>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <thread>

#include "ildl_kernels.hpp"

namespace jdhip {

namespace {

// Copies run on the context's stream and are waited for (the source is a
// temporary): the legacy null stream would wait for every other context's
// stream in the process and break another thread's graph capture.
template <typename X>
X *dev_upload(hipStream_t s, const std::vector<X> &h) {
    X *p = nullptr;
    size_t bytes = sizeof(X) * std::max<size_t>(h.size(), 1);
    JDHIP_CHECK(hipMalloc(&p, bytes));
    if (!h.empty()) {
        JDHIP_CHECK(hipMemcpyAsync(p, h.data(), sizeof(X) * h.size(), hipMemcpyHostToDevice, s));
        JDHIP_CHECK(hipStreamSynchronize(s));
    }
    return p;
}

template <typename X>
X *dev_alloc(size_t cnt) {
    X *p = nullptr;
    JDHIP_CHECK(hipMalloc(&p, sizeof(X) * std::max<size_t>(cnt, 1)));
    return p;
}

// Sort the entries of every CSR row by column.
template <typename T>
void sort_rows(int nrows, const std::vector<int> &ptr, std::vector<int> &idx,
               std::vector<T> &val) {
    std::vector<std::pair<int, T>> row;
    for (int r = 0; r < nrows; ++r) {
        const int b = ptr[r], e = ptr[r + 1];
        if (e - b < 2) continue;
        row.clear();
        for (int k = b; k < e; ++k) row.emplace_back(idx[k], val[k]);
        std::sort(row.begin(), row.end(),
                  [](const auto &x, const auto &y) { return x.first < y.first; });
        for (int k = b; k < e; ++k) {
            idx[k] = row[k - b].first;
            val[k] = row[k - b].second;
        }
    }
}

// CSR transpose (rows x cols) -> (cols x rows)
template <typename T>
void transpose(int rows, int cols, const std::vector<int> &ptr, const std::vector<int> &idx,
               const std::vector<T> &val, std::vector<int> &tp, std::vector<int> &ti,
               std::vector<T> &tv) {
    tp.assign(cols + 1, 0);
    for (int c : idx) tp[c + 1]++;
    for (int c = 0; c < cols; ++c) tp[c + 1] += tp[c];
    ti.assign(idx.size(), 0);
    tv.assign(idx.size(), T(0));
    std::vector<int> f(tp.begin(), tp.end() - 1);
    for (int r = 0; r < rows; ++r)
        for (int k = ptr[r]; k < ptr[r + 1]; ++k) {
            int c = idx[k];
            ti[f[c]] = r;
            tv[f[c]++] = val[k];
        }
}

// Level schedule of a unit triangular CSR: forward (entries j < row) in
// increasing order, backward (entries j > row) in decreasing order.
void schedule(int n, const std::vector<int> &ptr, const std::vector<int> &idx, bool forward,
              std::vector<int> &lvl_ptr, std::vector<int> &rows) {
    std::vector<int> lvl(n, 0);
    int nlev = 0;
    if (forward) {
        for (int i = 0; i < n; ++i) {
            int l = 0;
            for (int k = ptr[i]; k < ptr[i + 1]; ++k) l = std::max(l, lvl[idx[k]] + 1);
            lvl[i] = l;
            nlev = std::max(nlev, l + 1);
        }
    } else {
        for (int i = n - 1; i >= 0; --i) {
            int l = 0;
            for (int k = ptr[i]; k < ptr[i + 1]; ++k) l = std::max(l, lvl[idx[k]] + 1);
            lvl[i] = l;
            nlev = std::max(nlev, l + 1);
        }
    }
    lvl_ptr.assign(nlev + 1, 0);
    for (int i = 0; i < n; ++i) lvl_ptr[lvl[i] + 1]++;
    for (int l = 0; l < nlev; ++l) lvl_ptr[l + 1] += lvl_ptr[l];
    rows.assign(n, 0);
    std::vector<int> f(lvl_ptr.begin(), lvl_ptr.end() - 1);
    for (int i = 0; i < n; ++i) rows[f[lvl[i]]++] = i;
}

// SELL-C-sigma copy of a CSR (C = 64 rows per slice, rows sorted by length
// inside windows of sigma rows; sigma <= 64 keeps the row order) for the
// Jacobi sweeps.

template <typename T>
struct SellHost {
    std::vector<long> vptr, iptr;
    std::vector<int> code, rowid, cbase;
    std::vector<char> idx;
    std::vector<T> val;
    long nnz16 = 0, nnz32 = 0;  // stored (non-padding) entries by index width
};

// skip_empty: rows without entries get no lane (products y -= M x, where such
// rows are no-ops; a sweep must still copy b into them, so it keeps them).
// A slice stores its columns as 16-bit offsets from its smallest column when
// they span less than 65536, else as int32; padding entries point at that
// smallest column (a valid index) with value 0.
template <typename T>
SellHost<T> build_sell(int nrows, const std::vector<int> &ptr, const std::vector<int> &idx,
                       const std::vector<T> &val, int sigma, bool skip_empty = false) {
    SellHost<T> h;
    std::vector<int> order(nrows);
    std::vector<int> cols;
    sigma = std::max(sigma, 64);
    for (int r0 = 0; r0 < nrows; r0 += sigma) {
        const int r1 = std::min(nrows, r0 + sigma);
        const int w0 = r0;
        int w1 = r0;
        for (int r = r0; r < r1; ++r)
            if (!skip_empty || ptr[r + 1] > ptr[r]) order[w1++] = r;
        if (sigma > 64)
            std::stable_sort(order.begin() + w0, order.begin() + w1, [&](int a, int b) {
                return ptr[a + 1] - ptr[a] > ptr[b + 1] - ptr[b];
            });
        for (int s0 = w0; s0 < w1; s0 += 64) {
            int w = 0, cmin = INT_MAX, cmax = INT_MIN;
            for (int r = s0; r < std::min(w1, s0 + 64); ++r) {
                const int row = order[r];
                w = std::max(w, ptr[row + 1] - ptr[row]);
                for (int k = ptr[row]; k < ptr[row + 1]; ++k) {
                    cmin = std::min(cmin, idx[k]);
                    cmax = std::max(cmax, idx[k]);
                }
            }
            if (cmin > cmax) cmin = cmax = 0;  // no entries in the slice
            const bool narrow = (long)cmax - cmin < 65536;
            long real = 0;
            for (int r = s0; r < std::min(w1, s0 + 64); ++r) real += ptr[order[r] + 1] - ptr[order[r]];
            (narrow ? h.nnz16 : h.nnz32) += real;
            const long base = h.val.size();
            h.vptr.push_back(base);
            h.code.push_back(2 * w + (narrow ? 1 : 0));
            h.cbase.push_back(narrow ? cmin : 0);
            h.val.resize(base + 64L * w, T(0));
            cols.assign(64L * w, cmin);
            for (int lane = 0; lane < 64; ++lane) {
                const int t = s0 + lane;
                const int row = (t < w1) ? order[t] : -1;
                h.rowid.push_back(row);
                if (row < 0) continue;
                for (int k = 0; k < ptr[row + 1] - ptr[row]; ++k) {
                    h.val[base + (long)k * 64 + lane] = val[ptr[row] + k];
                    cols[(long)k * 64 + lane] = idx[ptr[row] + k];
                }
            }
            // index bytes of the slice, 4-byte aligned
            long at = (long)h.idx.size();
            at = (at + 3) & ~3L;
            h.iptr.push_back(at);
            if (narrow) {
                h.idx.resize(at + 2L * cols.size());
                auto *o = reinterpret_cast<unsigned short *>(h.idx.data() + at);
                for (size_t e = 0; e < cols.size(); ++e) o[e] = (unsigned short)(cols[e] - cmin);
            } else {
                h.idx.resize(at + 4L * cols.size());
                std::memcpy(h.idx.data() + at, cols.data(), 4 * cols.size());
            }
        }
    }
    h.vptr.push_back((long)h.val.size());
    if (h.idx.empty()) h.idx.resize(4);
    return h;
}

template <typename T>
struct SellDev {
    SellView v;  // device arrays of the layout (see SellView)
    T *val = nullptr;
    long idx_bytes = 0;
    long nnz16 = 0, nnz32 = 0;
};

template <typename T>
struct StreamDev {
    StreamView<T> v;  // device arrays of the layout
    long nnz16 = 0, nnz32 = 0;
};

// Kernel form of a product (CSR row pointers ptr) before any timing:
// CSR-stream for large products, whose entries it balances, else CSR lane
// groups of about the average row length.  Measured (us a launch in a graph,
// stream / the rule's lanes): 609k entries of 22 a row 5.4 / 6.2, 354k of 98
// 3.8 / 3.9, 186k of 16 3.5 / 3.3, 107k of 134 3.8 / 3.1, 22k of 2.8 3.2 / 2.6; an
// apply of 50,000 rows of one entry, 21.8 us in stream, 31.5 with 8 lanes.
// Where the average meets the next power of two matters little: with factors of
// 0.5 to 1.6 in place of 0.8 eight applies differ by 3 % at most, without an order
// (0.25: up to 6 % slower).
// A row much longer than its lanes is a chain of its own (0.3 us for every four
// entries a lane), which stream spreads over a block: an apply with rows of up
// to 9,706 entries among short ones (30,001 rows, four levels) 427 us by the
// average alone, 166 with the last line, which lies between 8 and 64 times the
// lanes without a difference.
constexpr long kTimed = 200000;
inline int pick_form(const std::vector<int> &ptr) {
    const int rows = (int)ptr.size() - 1;
    if (rows <= 0) return 0;
    const long nnz = ptr[rows];
    if (nnz >= kTimed || rows >= 32768) return 1;
    const double avg = 0.8 * (double)nnz / rows;
    int lanes = 8, longest = 0;
    while (lanes < 64 && lanes < avg) lanes *= 2;
    for (int r = 0; r < rows; ++r) longest = std::max(longest, ptr[r + 1] - ptr[r]);
    return longest > 16 * lanes ? 1 : lanes;
}

template <typename T, typename W>
struct DevLevel {
    int n = 0, nB = 0, nC = 0;
    int *perm = nullptr;
    double *scal = nullptr, *dinv = nullptr;  // per row, double on both paths
    // 2x2 pivots (null if the level has none): off-diagonal entry of each
    // row's block of D^-1 and the partner row (storage numbering, -1: 1x1)
    double *doinv = nullptr;
    int *dpair = nullptr;
    int *lb_ptr = nullptr, *lb_idx = nullptr;
    T *lb_val = nullptr;
    int *lt_ptr = nullptr, *lt_idx = nullptr;
    T *lt_val = nullptr;
    int *lc_ptr = nullptr, *lc_idx = nullptr;
    T *lc_val = nullptr;
    int *lct_ptr = nullptr, *lct_idx = nullptr;
    T *lct_val = nullptr;
    // row blocks of the CSR-stream form for L_B, L_B^T, L_CB, L_CB^T
    StreamDev<T> st_b, st_t, st_c, st_ct;
    std::vector<int> fwd_ptr, bwd_ptr;  // host level pointers
    int *fwd_rows = nullptr, *bwd_rows = nullptr;
    W *buf = nullptr, *out = nullptr, *t1 = nullptr, *t2 = nullptr;  // work vectors
    long nnz_lb = 0, nnz_lc = 0;
    SellDev<T> sf, sb;  // sweep copies of L_B (forward) and L_B^T (backward)
    int k = 0;          // this level's triangular solves: 0 exact, k Jacobi sweeps
    // kernel form of each product: 0 SELL (one lane per row), else CSR with
    // that many lanes per row (long rows)
    int wf = 0, wb = 0, wc = 0, wct = 0;
    SellDev<T> sc, sct; // L_CB and L_CB^T
};

// T: type of the stored factor values, W: type of the apply's work vectors
template <typename T, typename W>
class IldlImpl : public IldlImplBase {
  public:
    IldlImpl(DevCtx *ctx, IldlMultilevel<T> &&f, int sweeps, int storage_order, int xcd,
             int sigma)
        : ctx_(ctx), f_(std::move(f)), sweeps_(sweeps), storage_(storage_order), xcd_(xcd),
          sigma_(sigma) {}
    ~IldlImpl() override {
        hipStreamSynchronize(ctx_->stream);
        clear_graph();
        for (void *p : allocs_) hipFree(p);
    }

    // Upload with a storage renumbering per level: the B and the C positions
    // are each stored in the order of the original matrix index they stand
    // for, so gathers, scatters and the sweeps' x reads follow the locality
    // of the input (the factor's own order is the fill-reducing one, which
    // scatters neighbours).  Dependency levels are computed in the factor's
    // triangular order and relabelled; the host copy f_ keeps the factor's
    // numbering for export.
    void upload(IldlResult &res) {
        const int nlev = (int)f_.levels.size();
        std::vector<long> orig;  // original index of each (relabelled) input index
        std::vector<int> cnew;   // previous level: old C index -> new C index
        std::vector<int> qC_last;
        for (int l = 0; l < nlev; ++l) {
            const IldlLevel<T> &L = f_.levels[l];
            const int n = L.n, nB = L.nB, nC = n - nB;
            if (l == 0) {
                orig.resize(n);
                for (int i = 0; i < n; ++i) orig[i] = i;
            }
            std::vector<int> perm(n);
            std::vector<double> scal(n);
            for (int i = 0; i < n; ++i) perm[i] = cnew.empty() ? L.perm[i] : cnew[L.perm[i]];
            for (int j = 0; j < n; ++j) scal[cnew.empty() ? j : cnew[j]] = L.scal[j];
            std::vector<int> q(n), qinv(n);
            for (int i = 0; i < n; ++i) q[i] = i;
            if (storage_ == 1) {
                auto by_orig = [&](int a, int b) { return orig[perm[a]] < orig[perm[b]]; };
                std::stable_sort(q.begin(), q.begin() + nB, by_orig);
                std::stable_sort(q.begin() + nB, q.end(), by_orig);
            }
            for (int t = 0; t < n; ++t) qinv[q[t]] = t;

            DevLevel<T, W> D;
            D.n = n;
            D.nB = nB;
            D.nC = nC;
            std::vector<int> permN(n);
            for (int t = 0; t < n; ++t) permN[t] = perm[q[t]];
            D.perm = track(dev_upload(ctx_->stream, permN));
            D.scal = track(dev_upload(ctx_->stream, scal));
            // D^-1 per stored row: 1 / d for a 1x1 pivot; for a 2x2 block
            // [a o; o c] the row's entries of [c -o; -o a] / (ac - o^2) and the
            // partner's storage index
            std::vector<double> dinv(nB), doinv(nB, 0.0);
            std::vector<int> dpair_s(nB, -1);
            bool any_pair = false;
            for (int t = 0; t < nB; ++t) {
                const int b = q[t];
                const int pb = L.dpair.empty() ? -1 : L.dpair[b];
                if (pb < 0) {
                    dinv[t] = 1.0 / (double)L.d[b];
                } else {
                    any_pair = true;
                    const double a = (double)L.d[b], o = (double)L.doff[b], c = (double)L.d[pb];
                    const double det = a * c - o * o;
                    dinv[t] = c / det;
                    doinv[t] = -o / det;
                    dpair_s[t] = qinv[pb];
                }
            }
            D.dinv = track(dev_upload(ctx_->stream, dinv));
            if (any_pair) {
                D.doinv = track(dev_upload(ctx_->stream, doinv));
                D.dpair = track(dev_upload(ctx_->stream, dpair_s));
            }
            // L_B and L_CB in the storage numbering
            std::vector<int> bp(nB + 1, 0), bi, cp(nC + 1, 0), ci;
            std::vector<T> bv, cv;
            bi.reserve(L.lb_idx.size());
            bv.reserve(L.lb_idx.size());
            for (int t = 0; t < nB; ++t) {
                const int i = q[t];
                for (int k = L.lb_ptr[i]; k < L.lb_ptr[i + 1]; ++k) {
                    bi.push_back(qinv[L.lb_idx[k]]);
                    bv.push_back(L.lb_val[k]);
                }
                bp[t + 1] = (int)bi.size();
            }
            ci.reserve(L.lc_idx.size());
            cv.reserve(L.lc_idx.size());
            for (int c = 0; c < nC; ++c) {
                const int oc = q[nB + c] - nB;
                for (int k = L.lc_ptr[oc]; k < L.lc_ptr[oc + 1]; ++k) {
                    ci.push_back(qinv[L.lc_idx[k]]);
                    cv.push_back(L.lc_val[k]);
                }
                cp[c + 1] = (int)ci.size();
            }
            // columns ascending inside every row: neighbouring lanes of the
            // stream and lane-group kernels then gather from the same cache
            // lines (the transposes built below inherit the order)
            sort_rows(nB, bp, bi, bv);
            sort_rows(nC, cp, ci, cv);
            D.lb_ptr = track(dev_upload(ctx_->stream, bp));
            D.lb_idx = track(dev_upload(ctx_->stream, bi));
            D.lb_val = track(dev_upload(ctx_->stream, bv));
            std::vector<int> tp, ti;
            std::vector<T> tv;
            transpose(nB, nB, bp, bi, bv, tp, ti, tv);
            D.lt_ptr = track(dev_upload(ctx_->stream, tp));
            D.lt_idx = track(dev_upload(ctx_->stream, ti));
            D.lt_val = track(dev_upload(ctx_->stream, tv));
            D.st_b = upload_stream(nB, bp, bi, bv);
            D.st_t = upload_stream(nB, tp, ti, tv);
            D.wf = pick_form(bp);
            D.wb = pick_form(tp);
            D.sf = upload_sell(build_sell(nB, bp, bi, bv, sigma_));
            D.sb = upload_sell(build_sell(nB, tp, ti, tv, sigma_));
            // dependency levels from the triangular (factor) numbering
            {
                std::vector<int> rows, otp, oti;
                std::vector<T> otv;
                schedule(nB, L.lb_ptr, L.lb_idx, true, D.fwd_ptr, rows);
                for (int &r : rows) r = qinv[r];
                D.fwd_rows = track(dev_upload(ctx_->stream, rows));
                transpose(nB, nB, L.lb_ptr, L.lb_idx, L.lb_val, otp, oti, otv);
                schedule(nB, otp, oti, false, D.bwd_ptr, rows);
                for (int &r : rows) r = qinv[r];
                D.bwd_rows = track(dev_upload(ctx_->stream, rows));
            }
            D.sc = upload_sell(build_sell(nC, cp, ci, cv, sigma_, true));
            D.lc_ptr = track(dev_upload(ctx_->stream, cp));
            D.lc_idx = track(dev_upload(ctx_->stream, ci));
            D.lc_val = track(dev_upload(ctx_->stream, cv));
            D.st_c = upload_stream(nC, cp, ci, cv);
            D.wc = pick_form(cp);
            transpose(nC, nB, cp, ci, cv, tp, ti, tv);
            D.sct = upload_sell(build_sell(nB, tp, ti, tv, sigma_, true));
            D.lct_ptr = track(dev_upload(ctx_->stream, tp));
            D.lct_idx = track(dev_upload(ctx_->stream, ti));
            D.lct_val = track(dev_upload(ctx_->stream, tv));
            D.st_ct = upload_stream(nB, tp, ti, tv);
            D.wct = pick_form(tp);
            D.buf = track(dev_alloc<W>(n));
            D.out = track(dev_alloc<W>(n));
            D.t1 = track(dev_alloc<W>(std::max(nB, 1)));
            D.t2 = track(dev_alloc<W>(std::max(nB, 1)));
            D.nnz_lb = (long)L.lb_idx.size();
            D.nnz_lc = (long)L.lc_idx.size();
            res.fwd_levels.push_back((int)D.fwd_ptr.size() - 1);
            res.bwd_levels.push_back((int)D.bwd_ptr.size() - 1);
            lv_.push_back(std::move(D));
            // relabelling of the next level's input (this level's C part)
            std::vector<long> norig(nC);
            for (int c = 0; c < nC; ++c) norig[c] = orig[permN[nB + c]];
            orig.swap(norig);
            cnew.assign(nC, 0);
            qC_last.assign(nC, 0);
            for (int c = 0; c < nC; ++c) {
                cnew[q[nB + c] - nB] = c;
                qC_last[c] = q[nB + c] - nB;
            }
        }
        if (f_.m > 0) {
            const int m = f_.m;
            std::vector<T> mv((size_t)m * m);
            for (int a = 0; a < m; ++a)
                for (int b = 0; b < m; ++b) {
                    const int oa = nlev ? qC_last[a] : a, ob = nlev ? qC_last[b] : b;
                    mv[(size_t)a * m + b] = (T)f_.dinv[(size_t)oa * m + ob];
                }
            dmat_ = track(dev_upload(ctx_->stream, mv));
            dx_ = track(dev_alloc<W>(m));
            dy_ = track(dev_alloc<W>(m));
        }
        for (auto &D : lv_) D.k = sweeps_;
        JDHIP_CHECK(hipStreamSynchronize(ctx_->stream));
    }

    // Triangular solve with L_B (fwd) or L_B^T on x (nB entries), then times
    // dinv and added to add (both may be null, see RowOp), into out (which may
    // be x, and add).
    void tri_solve(const Put &s, const DevLevel<T, W> &D, bool fwd, W *x, const double *dinv,
                   const W *add, W *out) {
        const int nsw = D.k;
        if (nsw <= 0) {
            const int *ptr = fwd ? D.lb_ptr : D.lt_ptr;
            const int *idx = fwd ? D.lb_idx : D.lt_idx;
            const T *val = fwd ? D.lb_val : D.lt_val;
            const std::vector<int> &lp = fwd ? D.fwd_ptr : D.bwd_ptr;
            const int *rows = fwd ? D.fwd_rows : D.bwd_rows;
            for (size_t l = 1; l + 1 < lp.size(); ++l)  // level 0 rows have no entries
                ildl_trsv_level<T, W>(s, rows + lp[l], lp[l + 1] - lp[l], ptr, idx, val, x);
            if (dinv) ildl_dscale<W>(s, D.nB, dinv, x);
            if (add) ildl_add<W>(s, D.nB, x, out);
            return;
        }
        // Jacobi sweeps y <- b - N y from y = b (b = x).  The first sweep
        // reads b itself; the last writes out, which may be x: every row
        // reads only its own b entry and all y entries come from the other
        // buffer (a single sweep into x goes via t1).
        W *bufs[2] = {D.t1, D.t2};
        const W *xin = x;
        for (int k = 0; k < nsw; ++k) {
            RowOp<W> op;
            op.src = x;
            op.out = bufs[k & 1];
            if (k == nsw - 1) {
                op.dinv = dinv;
                op.add = add;
                if (out != xin) op.out = out;
            }
            sweep_launch(s, D, fwd, fwd ? D.wf : D.wb, xin, op);
            xin = op.out;
        }
        if (xin != out) ildl_copy<W>(s, D.nB, xin, out);
    }

    // One product with the level's L_B (fwd) or L_B^T in the given kernel
    // form: 0 one lane per row on the SELL-C-sigma copy, 1 CSR-stream, else
    // CSR with that many lanes per row.
    void sweep_launch(const Put &s, const DevLevel<T, W> &D, bool fwd, int form, const W *x,
                      const RowOp<W> &op) {
        const int *idx = fwd ? D.lb_idx : D.lt_idx;
        const T *val = fwd ? D.lb_val : D.lt_val;
        if (form == 1) {
            ildl_stream<T, W>(s, fwd ? D.st_b.v : D.st_t.v, idx, val, x, op, xcd_ & 1);
        } else if (form > 0) {
            ildl_csr<T, W>(s, form, D.nB, fwd ? D.lb_ptr : D.lt_ptr, idx, val, x, op, xcd_ & 1);
        } else {
            const SellDev<T> &M = fwd ? D.sf : D.sb;
            ildl_sell<T, W>(s, M.v, M.val, x, op, xcd_);
        }
    }
    // y -= L_CB x (C rows; trans = false) or y -= L_CB^T x (B rows); with
    // fresh, y = -(the product)
    void sub_launch(const Put &s, const DevLevel<T, W> &D, bool trans, int form, const W *x,
                    W *y, bool fresh = false) {
        const int rows = trans ? D.nB : D.nC;
        const int *idx = trans ? D.lct_idx : D.lc_idx;
        const T *val = trans ? D.lct_val : D.lc_val;
        RowOp<W> op;
        op.src = fresh ? nullptr : y;
        op.out = y;
        if (form == 1) {
            ildl_stream<T, W>(s, trans ? D.st_ct.v : D.st_c.v, idx, val, x, op, xcd_ & 1);
        } else if (form > 0) {
            ildl_csr<T, W>(s, form, rows, trans ? D.lct_ptr : D.lc_ptr, idx, val, x, op,
                           xcd_ & 1);
        } else {
            // this copy has no lanes for empty rows
            if (fresh) ildl_zero<W>(s, rows, y);
            op.src = y;
            const SellDev<T> &M = trans ? D.sct : D.sc;
            ildl_sell<T, W>(s, M.v, M.val, x, op, xcd_ & 1);
        }
    }

    // Kernel form of every product of every level (both sweeps, L_CB and
    // L_CB^T).  Products of at least kTimed entries by measurement: the fastest
    // of one lane per row on the SELL-C-sigma copy, the CSR-stream form (form
    // 1) and CSR with 4 to 64 lanes per row, each timed over six launches of a
    // graph on zeroed vectors (launched one by one they would be timed at the
    // host's rate).  Smaller ones differ by less than a timing is worth and
    // keep the lanes of the upload's rule.
    void autotune_forms() override {
        hipStream_t s = ctx_->stream;
        hipEvent_t e0, e1;
        JDHIP_CHECK(hipEventCreate(&e0));
        JDHIP_CHECK(hipEventCreate(&e1));
        auto timed = [&](auto &&launch) {
            hipGraph_t g = nullptr;
            hipGraphExec_t x = nullptr;
            JDHIP_CHECK(hipGraphCreate(&g, 0));
            const Put q(g);
            for (int i = 0; i < 6; ++i) launch(q);
            JDHIP_CHECK(hipGraphInstantiate(&x, g, nullptr, nullptr, 0));
            JDHIP_CHECK(hipGraphDestroy(g));
            float best = 0.f;
            for (int i = 0; i < 3; ++i) {
                JDHIP_CHECK(hipEventRecord(e0, s));
                JDHIP_CHECK(hipGraphLaunch(x, s));
                JDHIP_CHECK(hipEventRecord(e1, s));
                JDHIP_CHECK(hipEventSynchronize(e1));
                float ms = 0.f;
                JDHIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
                if (i == 1 || ms < best) best = ms;  // the first one warms up
            }
            JDHIP_CHECK(hipGraphExecDestroy(x));
            return best;
        };
        auto best = [&](auto &&launch_form) {
            int bf = 1;
            float bt = 0.f;
            for (int f : {1, 0, 4, 8, 16, 32, 64}) {
                const float t = timed([&](const Put &q) { launch_form(q, f); });
                if (f == 1 || t < bt) {
                    bt = t;
                    bf = f;
                }
            }
            return bf;
        };
        for (auto &D : lv_) {
            if (D.nnz_lb < kTimed && D.nnz_lc < kTimed) continue;
            ildl_zero<W>(s, D.n, D.buf);
            ildl_zero<W>(s, D.n, D.out);
            ildl_zero<W>(s, D.nB, D.t1);
            ildl_zero<W>(s, D.nB, D.t2);
            RowOp<W> op;
            op.src = D.buf;
            op.out = D.t2;
            if (D.nB > 0 && D.nnz_lb >= kTimed) {
                D.wf = best([&](const Put &q, int f) { sweep_launch(q, D, true, f, D.t1, op); });
                D.wb = best([&](const Put &q, int f) { sweep_launch(q, D, false, f, D.t1, op); });
            }
            if (D.nC > 0 && D.nnz_lc >= kTimed) {
                D.wc = best([&](const Put &q, int f) {
                    sub_launch(q, D, false, f, D.buf, D.buf + D.nB);
                });
                D.wct = best([&](const Put &q, int f) {
                    sub_launch(q, D, true, f, D.out, D.buf, fform());
                });
            }
        }
        JDHIP_CHECK(hipStreamSynchronize(s));
        hipEventDestroy(e0);
        hipEventDestroy(e1);
        clear_graph();
    }
    void set_forms(int form) override {
        for (auto &D : lv_) D.wf = D.wb = D.wc = D.wct = form;
        clear_graph();
    }
    std::vector<int> level_forms() const override {
        std::vector<int> v;
        for (const auto &D : lv_) {
            v.push_back(D.wf);
            v.push_back(D.wb);
            v.push_back(D.wc);
            v.push_back(D.wct);
        }
        return v;
    }

    StreamDev<T> upload_stream(int nrows, const std::vector<int> &ptr,
                               const std::vector<int> &idx, const std::vector<T> &val) {
        const StreamHost<T> h = build_stream(nrows, ptr, idx, val);
        StreamDev<T> d;
        StreamView<T> &v = d.v;
        v.nblk = (int)h.desc.size();
        v.cap = h.cap;
        v.desc = track(dev_upload(ctx_->stream, h.desc));
        v.cbase = track(dev_upload(ctx_->stream, h.cbase));
        v.off = track(dev_upload(ctx_->stream, h.off));
        if (!h.c16.empty()) v.c16 = track(dev_upload(ctx_->stream, h.c16));
        if (!h.c32.empty()) v.c32 = track(dev_upload(ctx_->stream, h.c32));
        v.val = track(dev_upload(ctx_->stream, h.val));
        d.nnz16 = h.nnz16;
        d.nnz32 = h.nnz32;
        return d;
    }

    SellDev<T> upload_sell(const SellHost<T> &h) {
        SellDev<T> d;
        d.v.nslices = (int)h.code.size();
        d.v.vptr = track(dev_upload(ctx_->stream, h.vptr));
        d.v.iptr = track(dev_upload(ctx_->stream, h.iptr));
        d.v.code = track(dev_upload(ctx_->stream, h.code));
        d.v.rowid = track(dev_upload(ctx_->stream, h.rowid));
        d.v.cbase = track(dev_upload(ctx_->stream, h.cbase));
        d.v.idx = track(dev_upload(ctx_->stream, h.idx));
        d.val = track(dev_upload(ctx_->stream, h.val));
        d.idx_bytes = (long)h.idx.size();
        d.nnz16 = h.nnz16;
        d.nnz32 = h.nnz32;
        return d;
    }

    int sweeps() const override { return sweeps_; }

    void set_all(int k) {
        sweeps_ = k;
        for (auto &D : lv_) D.k = k;
        clear_graph();
    }

    int tune_sweeps(double tol, bool by_time) override {
        set_all(0);
        if (lv_.empty()) return 0;
        tuning_ = true;  // per-level counts change between applies
        const int n = lv_[0].n;
        hipStream_t s = ctx_->stream;
        std::vector<double> hr(n), h0(n), hk(n);
        uint64_t st = 0x9e3779b97f4a7c15ULL;
        for (int i = 0; i < n; ++i) {  // splitmix64 -> uniform(-1, 1)
            uint64_t z = (st += 0x9e3779b97f4a7c15ULL);
            z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
            z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
            z ^= z >> 31;
            hr[i] = 2.0 * ((double)(z >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
        }
        double *r = dev_alloc<double>(n), *z = dev_alloc<double>(n);
        JDHIP_CHECK(hipMemcpyAsync(r, hr.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        hipEvent_t e0, e1;
        JDHIP_CHECK(hipEventCreate(&e0));
        JDHIP_CHECK(hipEventCreate(&e1));
        auto timed = [&](int reps) {
            apply(z, r);
            JDHIP_CHECK(hipEventRecord(e0, s));
            for (int i = 0; i < reps; ++i) apply(z, r);
            JDHIP_CHECK(hipEventRecord(e1, s));
            JDHIP_CHECK(hipEventSynchronize(e1));
            float ms = 0.f;
            JDHIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
            return ms / reps;
        };
        // the exact apply is the reference of the accuracy test; it is timed
        // only when the sweeps must also beat it, and then once after the
        // first (warm-up) run (a level-scheduled apply of a large factor is
        // ~10^5 launches, about 1.5 s for Anderson L=100)
        float t_exact = 0.f;
        apply(z, r);
        if (by_time) {
            JDHIP_CHECK(hipEventRecord(e0, s));
            apply(z, r);
            JDHIP_CHECK(hipEventRecord(e1, s));
            JDHIP_CHECK(hipEventSynchronize(e1));
            JDHIP_CHECK(hipEventElapsedTime(&t_exact, e0, e1));
        }
        JDHIP_CHECK(hipMemcpyAsync(h0.data(), z, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        JDHIP_CHECK(hipStreamSynchronize(s));
        double n0 = 0.0;
        for (double v : h0) n0 += v * v;
        n0 = std::sqrt(n0);
        auto close = [&]() {  // apply of the current setting within tol of exact?
            apply(z, r);
            JDHIP_CHECK(hipMemcpyAsync(hk.data(), z, sizeof(double) * n, hipMemcpyDeviceToHost, s));
            JDHIP_CHECK(hipStreamSynchronize(s));
            double e = 0.0;
            for (int i = 0; i < n; ++i) e += (hk[i] - h0[i]) * (hk[i] - h0[i]);
            return std::sqrt(e) <= tol * n0;
        };
        // 1) one sweep count for all levels: the smallest that is accurate
        int kg = 0;
        for (int k : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64}) {
            set_all(k);
            if (close()) {
                kg = k;
                break;
            }
        }
        if (kg > 0) {
            // 2) per level (largest first), lower the count one by one while
            //    the whole apply stays within tol
            std::vector<int> order(lv_.size());
            for (size_t l = 0; l < lv_.size(); ++l) order[l] = (int)l;
            std::stable_sort(order.begin(), order.end(),
                             [&](int a, int b) { return lv_[a].nB > lv_[b].nB; });
            for (int l : order) {
                while (lv_[l].k > 1) {
                    const int keep = lv_[l].k;
                    lv_[l].k = keep > 8 ? keep * 3 / 4 : keep - 1;
                    if (!close()) {
                        lv_[l].k = keep;
                        break;
                    }
                }
            }
            sweeps_ = 0;
            for (auto &D : lv_) sweeps_ = std::max(sweeps_, D.k);
            // 3) keep the sweeps only if they beat the exact solve
            if (by_time && timed(2) >= t_exact) set_all(0);
        } else {
            // no uniform count reproduces the exact apply: keep exact solves
            set_all(0);
        }
        tuning_ = false;
        clear_graph();
        hipEventDestroy(e0);
        hipEventDestroy(e1);
        hipFree(r);
        hipFree(z);
        return sweeps_;
    }

    std::vector<int> level_sweeps() const override {
        std::vector<int> v;
        for (const auto &D : lv_) v.push_back(D.k);
        return v;
    }

    void apply(double *z, const double *r) override { apply_any<double>(z, r); }
    void apply_f(float *z, const float *r) override { apply_any<float>(z, r); }

    // The apply is a fixed sequence of some tens to hundreds of launches, most
    // of them shorter than the 2.5-4.5 us that the host takes to enqueue one
    // (a graph's node takes 1.6-1.9 us).  Everything between the first gather
    // and the last scatter works on the factor's own vectors, so it is built
    // once per factor into a HIP graph and replayed for any input and output.
    // Exact solves (a launch per dependency level) can have 10^5 launches and
    // keep to the stream, as does everything on a stream under capture, which
    // cannot take a graph launch.
    template <typename TV>
    void apply_any(TV *z, const TV *r) {
        const Put q(ctx_->stream);
        const bool replay = graph_ && !tuning_ && !capturing();
        head<TV>(q, r);
        if (replay) JDHIP_CHECK(hipGraphLaunch(graph_, ctx_->stream));
        else body(q);
        tail<TV>(q, z);
    }
    bool capturing() const {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        JDHIP_CHECK(hipStreamIsCapturing(ctx_->stream, &st));
        return st != hipStreamCaptureStatusNone;
    }
    // launches of body() with sweeps (exact solves: one per dependency level)
    long body_launches() const {
        long c = 0;
        for (const auto &D : lv_) {
            const long half = D.k > 0 ? 2 * (D.k + 1)
                                      : (long)D.fwd_ptr.size() + (long)D.bwd_ptr.size();
            c += 8 + half * ((fform() && D.nC > 0) ? 2 : 1);
        }
        return c;
    }
    void clear_graph() {
        if (!graph_) return;
        hipStreamSynchronize(ctx_->stream);
        hipGraphExecDestroy(graph_);
        graph_ = nullptr;
    }
    void set_graphs(int mode) override {
        clear_graph();
        if (mode == 0 || lv_.empty() || body_launches() > kGraphMax) return;
        hipGraph_t g = nullptr;
        JDHIP_CHECK(hipGraphCreate(&g, 0));
        try {
            const Put q(g);
            body(q);
            if (q.nodes >= kGraphMin)
                JDHIP_CHECK(hipGraphInstantiate(&graph_, g, nullptr, nullptr, 0));
        } catch (...) {
            hipGraphDestroy(g);
            throw;
        }
        JDHIP_CHECK(hipGraphDestroy(g));
    }

    template <typename TV>
    void head(const Put &s, const TV *r) {
        if (lv_.empty()) ildl_gather<TV, W>(s, f_.m, ident_(), ones_(), r, dx_);
        else ildl_gather<TV, W>(s, lv_[0].n, lv_[0].perm, lv_[0].scal, r, lv_[0].buf);
    }
    template <typename TV>
    void tail(const Put &s, TV *z) {
        if (lv_.empty()) {
            ildl_scatter<W, TV>(s, f_.m, f_.m, ident_(), ones_(), dy_, dy_, z);
            return;
        }
        const DevLevel<T, W> &D = lv_[0];
        ildl_scatter<W, TV>(s, D.n, D.nB, D.perm, D.scal, D.buf, coarse_of(0), z);
    }
    // x_C of level l: the next level's result, or the dense level's
    const W *coarse_of(int l) const {
        return l + 1 < (int)lv_.size() ? lv_[l + 1].out : dy_;
    }
    void body(const Put &s) {
        const int L = (int)lv_.size();
        if (L == 0) {  // only a dense level: z = Minv r
            ildl_dense_gemv<T, W>(s, f_.m, dmat_, dx_, dy_);
            return;
        }
        for (int l = 0; l < L; ++l) {
            DevLevel<T, W> &D = lv_[l];
            if (l > 0) {
                const DevLevel<T, W> &P = lv_[l - 1];
                ildl_gather<W, W>(s, D.n, D.perm, D.scal, P.buf + P.nB, D.buf);
            }
            if (fform()) {
                // y_B = B^-1 b_B, then b_C -= F^T y_B
                block_solve(s, D, D.buf, nullptr, D.buf);
                if (D.nC > 0) sub_launch(s, D, false, D.wc, D.buf, D.buf + D.nB);
            } else {
                tri_solve(s, D, true, D.buf, nullptr, nullptr, D.buf);
                if (D.nC > 0) sub_launch(s, D, false, D.wc, D.buf, D.buf + D.nB);
                if (!D.dpair) ildl_dscale<W>(s, D.nB, D.dinv, D.buf);
                else ildl_dscale2<W>(s, D.nB, D.dinv, D.doinv, D.dpair, D.buf);
            }
        }
        if (f_.m > 0) {
            const DevLevel<T, W> &P = lv_[L - 1];
            ildl_dense_gemv<T, W>(s, f_.m, dmat_, P.buf + P.nB, dy_);
        }
        for (int l = L - 1; l >= 0; --l) {
            DevLevel<T, W> &D = lv_[l];
            const W *zc = coarse_of(l);
            if (fform()) {
                if (D.nC > 0) {
                    // x_B = y_B - B^-1 F x_C; D.out is free until the scatter
                    W *t = D.out;
                    sub_launch(s, D, true, D.wct, zc, t, true);
                    block_solve(s, D, t, D.buf, D.buf);
                }
            } else {
                if (D.nC > 0) sub_launch(s, D, true, D.wct, zc, D.buf);
                tri_solve(s, D, false, D.buf, nullptr, nullptr, D.buf);
            }
            if (l > 0) ildl_scatter<W, W>(s, D.n, D.nB, D.perm, D.scal, D.buf, zc, D.out);
        }
    }

    bool fform() const { return f_.coupling == 0; }
    // out = add + B^-1 x (add may be null): forward solve, D^-1 (1x1 pivots in
    // the last forward sweep, 2x2 pivots by a launch of their own), backward
    // solve; x is overwritten
    void block_solve(const Put &s, const DevLevel<T, W> &D, W *x, const W *add, W *out) {
        tri_solve(s, D, true, x, D.dpair ? nullptr : D.dinv, nullptr, x);
        if (D.dpair) ildl_dscale2<W>(s, D.nB, D.dinv, D.doinv, D.dpair, x);
        tri_solve(s, D, false, x, nullptr, add, out);
    }
    int nlevels() const override { return (int)f_.levels.size(); }
    int dense_m() const override { return f_.m; }
    void level_sizes(int lev, int *n, int *nB, long *nnz_lb, long *nnz_lc) const override {
        const auto &L = f_.levels[lev];
        *n = L.n;
        *nB = L.nB;
        *nnz_lb = (long)L.lb_idx.size();
        *nnz_lc = (long)L.lc_idx.size();
    }
    void level_data(int lev, int *perm, double *scal, int *lb_ptr, int *lb_idx, double *lb_val,
                    int *lc_ptr, int *lc_idx, double *lc_val, double *d) const override {
        const auto &L = f_.levels[lev];
        std::copy(L.perm.begin(), L.perm.end(), perm);
        for (int i = 0; i < L.n; ++i) scal[i] = (double)L.scal[i];
        std::copy(L.lb_ptr.begin(), L.lb_ptr.end(), lb_ptr);
        std::copy(L.lb_idx.begin(), L.lb_idx.end(), lb_idx);
        for (size_t i = 0; i < L.lb_val.size(); ++i) lb_val[i] = (double)L.lb_val[i];
        std::copy(L.lc_ptr.begin(), L.lc_ptr.end(), lc_ptr);
        std::copy(L.lc_idx.begin(), L.lc_idx.end(), lc_idx);
        for (size_t i = 0; i < L.lc_val.size(); ++i) lc_val[i] = (double)L.lc_val[i];
        for (int i = 0; i < L.nB; ++i) d[i] = (double)L.d[i];
    }
    void dense_data(double *minv) const override {
        for (size_t i = 0; i < f_.dinv.size(); ++i) minv[i] = (double)(T)f_.dinv[i];
    }
    // What one product with a matrix of nnz entries and rows rows streams in the
    // given form, without padding: values, columns in the width they are read
    // with, and what finds a row's entries.
    static long mat_bytes(const SellDev<T> &M, const StreamDev<T> &S, int form, long nnz,
                          long rows) {
        const long values = (long)sizeof(T) * nnz;
        if (form == 1)
            return values + 2 * S.nnz16 + 4 * S.nnz32 + 2 * (rows + S.v.nblk) + 20L * S.v.nblk;
        if (form > 0) return values + 4 * nnz + 4 * (rows + 1);
        return values + 2 * M.nnz16 + 4 * M.nnz32 + 4 * rows;
    }
    long sweep_bytes(const DevLevel<T, W> &D, bool fwd) const {
        return (fwd ? mat_bytes(D.sf, D.st_b, D.wf, D.nnz_lb, D.nB)
                    : mat_bytes(D.sb, D.st_t, D.wb, D.nnz_lb, D.nB)) +
               3L * (long)sizeof(W) * D.nB;
    }
    long apply_bytes() const override {
        // per level: one pass over L_B per sweep and direction (matrix, b, x,
        // result), L_CB and L_CB^T once, gather/scatter (perm + scal + in/out),
        // D^-1, dense inverse.  Factor values are sizeof(T) bytes, vectors
        // sizeof(W); matrix bytes follow each product's chosen form.
        const long s = sizeof(T), v = sizeof(W);
        long b = 0;
        for (const auto &D : lv_) {
            const long k = D.k > 0 ? D.k : 1;
            // F blocks: a level with a coarse part solves with B twice
            const long solves = (fform() && D.nC > 0) ? 2 : 1;
            b += solves * k * (sweep_bytes(D, true) + sweep_bytes(D, false));
            if (solves == 2) b += v * D.nB;  // y_B, added to
            b += mat_bytes(D.sc, D.st_c, D.wc, D.nnz_lc, D.nC) +
                 mat_bytes(D.sct, D.st_ct, D.wct, D.nnz_lc, D.nB) + 2 * v * (D.nB + D.nC);
            b += 2 * (4L + v) * D.n + 2 * v * D.n + 2 * v * D.nB;
        }
        b += s * (long)f_.m * f_.m + 2 * v * f_.m;
        return b;
    }
    bool single() const override { return sizeof(T) == 4; }

    int time_sweep(int reps, double *avg_ms, long *alg_bytes) override {
        if (lv_.empty() || reps <= 0) return -1;
        const DevLevel<T, W> &D = lv_[0];
        hipStream_t s = ctx_->stream;
        JDHIP_CHECK(hipMemsetAsync(D.buf, 0, sizeof(W) * D.n, s));
        JDHIP_CHECK(hipMemsetAsync(D.t1, 0, sizeof(W) * std::max(D.nB, 1), s));
        hipEvent_t e0, e1;
        JDHIP_CHECK(hipEventCreate(&e0));
        JDHIP_CHECK(hipEventCreate(&e1));
        RowOp<W> op;
        op.src = D.buf;
        op.out = D.t2;
        auto one = [&]() { sweep_launch(s, D, true, D.wf, D.t1, op); };
        one();
        JDHIP_CHECK(hipEventRecord(e0, s));
        for (int i = 0; i < reps; ++i) one();
        JDHIP_CHECK(hipEventRecord(e1, s));
        JDHIP_CHECK(hipEventSynchronize(e1));
        float ms = 0.f;
        JDHIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
        hipEventDestroy(e0);
        hipEventDestroy(e1);
        *avg_ms = ms / reps;
        *alg_bytes = sweep_bytes(D, true);
        return 0;
    }

  private:
    template <typename X>
    X *track(X *p) {
        allocs_.push_back((void *)p);
        return p;
    }
    const int *ident_() {
        if (!idp_) {
            std::vector<int> id(f_.m);
            for (int i = 0; i < f_.m; ++i) id[i] = i;
            idp_ = track(dev_upload(ctx_->stream, id));
            std::vector<double> one(f_.m, 1.0);
            onep_ = track(dev_upload(ctx_->stream, one));
        }
        return idp_;
    }
    const double *ones_() {
        ident_();
        return onep_;
    }

    DevCtx *ctx_;
    IldlMultilevel<T> f_;
    // Launches that a graph holds.  At least: a graph launch takes the host 32 us,
    // however few its nodes, a kernel launch 2.5-4.5 us, so short applies are
    // enqueued one by one: a solve of 50,000 rows with 6 launches an apply takes
    // 7.33 ms so and 8.53 ms with graphs, with 8 7.98 and 8.86, with 12 9.05 and
    // 8.83.  (Applies alone in the stream, on two machines: of 6 launches 21.8
    // and 33.7 us, as graphs 32.8 and 32.2; of 12 37.8 and 52.8, 39.5 and 39.7;
    // of 24 69 and 96, 67 and 67.)  At most (exact solves, a launch per dependency
    // level): the gain is the same for each launch (760 of them 2.72 -> 1.73 ms),
    // but a factor of some thousand levels would hold a graph of 10^5 nodes.
    static constexpr int kGraphMin = 12;
    static constexpr long kGraphMax = 1024;
    hipGraphExec_t graph_ = nullptr;
    bool tuning_ = false;
    int sweeps_;
    int storage_;  // 0: factor order, 1: original-index order per level
    int xcd_;      // XCD-contiguous block order in the SELL kernels
    int sigma_;    // SELL-C-sigma sorting window
    std::vector<DevLevel<T, W>> lv_;
    std::vector<void *> allocs_;
    T *dmat_ = nullptr;
    W *dx_ = nullptr, *dy_ = nullptr;
    int *idp_ = nullptr;
    double *onep_ = nullptr;
};

}  // namespace

// Copy of a double factor with every stored value rounded to float.
static IldlMultilevel<float> round_to_float(const IldlMultilevel<double> &d) {
    IldlMultilevel<float> f;
    f.coupling = d.coupling;
    for (const auto &L : d.levels) {
        IldlLevel<float> F;
        F.n = L.n;
        F.nB = L.nB;
        F.perm = L.perm;
        F.scal.assign(L.scal.begin(), L.scal.end());
        F.lb_ptr = L.lb_ptr;
        F.lb_idx = L.lb_idx;
        F.lb_val.assign(L.lb_val.begin(), L.lb_val.end());
        F.lc_ptr = L.lc_ptr;
        F.lc_idx = L.lc_idx;
        F.lc_val.assign(L.lc_val.begin(), L.lc_val.end());
        F.d.assign(L.d.begin(), L.d.end());
        F.doff.assign(L.doff.begin(), L.doff.end());
        F.dpair = L.dpair;
        f.levels.push_back(std::move(F));
    }
    f.m = d.m;
    f.dinv = d.dinv;
    f.nnz_factor = d.nnz_factor;
    f.nneg = d.nneg;
    return f;
}

void ildl_factor_host(int n, const int *ia, const int *ja, const double *a, double shift,
                      const IldlOptions &opt, IldlHost &out) {
    auto t0 = std::chrono::steady_clock::now();
    IldlResult &res = out.res;
    res = IldlResult();
    SymCsr A = sym_from_upper(n, ia, ja, a, shift);
    long nnzu = ia[n] - 1;
    out.nnz_upper = nnzu;
    IldlParams prm;
    prm.droptol = opt.droptol;
    prm.condest = opt.condest;
    prm.mem = opt.mem;
    prm.spd = opt.spd;
    prm.ordering = opt.ordering;
    prm.dense_max = opt.dense_max;
    prm.coupling = opt.coupling;
    prm.threads = opt.threads > 0
                      ? opt.threads
                      : (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
    IldlStats st;
    out.single = opt.single;
    out.spd = opt.spd;
    // The factor is always computed in double; the mixed path stores and
    // applies it in float.  (A float factorisation of the strongly indefinite
    // Anderson matrices loses the Schur complements: at L=100 its
    // preconditioner no longer lets the iteration converge.)
    st = ildl_factor<double>(A, prm, out.fd, nnzu);
    if (opt.single && st.ierr == 0) {
        out.ff = round_to_float(out.fd);
        out.fd = IldlMultilevel<double>();
    }
    res.ierr = st.ierr;
    res.nlev = st.nlev;
    res.nnz = st.nnz;
    res.nneg = st.nneg;
    res.condest = st.condest_used;
    // fill-in factor as the reference prints it (JDaux.F:1221-1228): the
    // count of symilupacknnz.c:80-125 over nnzU = the strict triangular
    // factor entries and the coupling block entries of every sparse level;
    // a dense final level of order j is weighted as sparse storage of its
    // indices and values would be, nnzU - j(j+1)/2 + 2n - j + j(j+1)/3
    // (j(j-1)/2 of its entries counted first); divided by nnz(A_upper)
    {
        long nnz_lev = 0;
        int m = 0;
        auto count = [&](const auto &ml) {
            for (const auto &L : ml.levels)
                nnz_lev += (long)L.lb_idx.size() + (long)L.lc_idx.size();
            m = ml.m;
        };
        if (opt.single) count(out.ff);
        else count(out.fd);
        double tot;
        if (m > 0) {
            const long j = m;
            const long a1 = nnz_lev + (j * (j - 1)) / 2 - (j * (j + 1)) / 2 + 2L * n - j;
            tot = std::floor((double)a1 + (double)(j * (j + 1)) / 3.0);
        } else {
            tot = (double)(nnz_lev + 2L * n);
        }
        res.fill = tot / (double)std::max(nnzu, 1L);
    }
    res.level_n = st.level_n;
    res.level_nB = st.level_nB;
    res.seconds =
        std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

void IldlPrecond::attach(const IldlHost &h, int sweeps) {
    impl_.reset();
    result = h.res;
    result.fwd_levels.clear();
    result.bwd_levels.clear();
    const int k0 = sweeps < 0 ? 0 : sweeps;
    // An FP32 factor streams float values; its work vectors stay FP64 on
    // indefinite problems (float intermediates cost the Anderson L=100
    // interior solve more than 4000 MATVECs instead of 2186 in the oracle
    // with exact solves) and are FP32 on definite ones, where they cost
    // nothing measurable and save a tenth of the apply's time (128^3
    // Laplacian).
    const bool w32 = vec32 > 0 || (vec32 < 0 && h.spd);
    if (h.single && w32) {
        IldlMultilevel<float> f = h.ff;
        auto *p = new IldlImpl<float, float>(ctx_, std::move(f), k0, storage_order, xcd_remap,
                                             sell_sigma);
        impl_.reset(p);
        p->upload(result);
    } else if (h.single) {
        IldlMultilevel<float> f = h.ff;
        auto *p = new IldlImpl<float, double>(ctx_, std::move(f), k0, storage_order, xcd_remap,
                                              sell_sigma);
        impl_.reset(p);
        p->upload(result);
    } else {
        IldlMultilevel<double> f = h.fd;
        auto *p = new IldlImpl<double, double>(ctx_, std::move(f), k0, storage_order, xcd_remap,
                                               sell_sigma);
        impl_.reset(p);
        p->upload(result);
    }
    // tuned mode: Jacobi sweeps only where they reproduce the exact apply
    // closely enough and are faster than the level-scheduled solve.  3 % is
    // enough for definite problems (128^3 Laplacian: 849 MATVECs against 842
    // with uniform sweeps); interior eigenvalues of an indefinite matrix need
    // the preconditioner closer to exact along the near-null space of
    // A - sigma I (Anderson L=100: per-level counts accurate to 3 % on a
    // random vector stalled the iteration), so there the bound is 1 %.
    // Anderson L=100, 10 eigenvalues nearest 0: 1e-4 takes 13-18 sweeps per
    // solve and 1317 MATVECs, 1e-3 12-16 sweeps and 1217, 1e-2 9-12 sweeps
    // and 1202 MATVECs (10.3 s, 7.8 s, 6.0 s), the same eigenvalues.
    if (force_form >= 0) impl_->set_forms(force_form);
    else if (autotune) impl_->autotune_forms();
    if (sweeps < 0)
        impl_->tune_sweeps(tune_tol > 0.0 ? tune_tol : (h.spd ? 0.03 : 1e-2), tune_time);
    result.sweeps = impl_->sweeps();
    impl_->set_graphs(graphs);
}

IldlResult IldlPrecond::setup(int n, const int *ia, const int *ja, const double *a,
                              double shift, const IldlOptions &opt) {
    IldlHost h;
    ildl_factor_host(n, ia, ja, a, shift, opt, h);
    impl_.reset();
    result = h.res;
    if (h.res.ierr != 0) return result;
    attach(h, opt.sweeps);
    return result;
}

}  // namespace jdhip
