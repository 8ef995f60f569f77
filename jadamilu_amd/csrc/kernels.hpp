// kernels.hpp -- launch wrappers for the gfx950 kernels of the JD hot path.
//
// All kernels run on the caller's HIP stream.  Reductions are deterministic:
// every block writes its partial sums, the last block to finish (ticket from
// a device counter) sums the partials in a fixed order and writes the result
// into device memory, so a dependent kernel can consume it without a host
// round trip.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <vector>

namespace jdhip {

constexpr int kBlock = 256;      // threads per block (4 wave64)
constexpr int kMaxCols = 64;     // max columns of a tall-skinny product
constexpr int kMaxRedBlocks = 4096;  // enough waves in flight to cover HBM latency
constexpr int kMaxPartials = kMaxRedBlocks * 64;  // reduction scratch (doubles)
// Blocks of an inner-step kernel: every block of the next kernel sums their
// partial sums again, so there are few of them.  Two a CU are enough where a
// thread's loads are all in flight: k_multidot of 8 columns takes 37.8 us with
// 512 blocks, 38.5 with 1,024 and 40.4 with 4,096 (3,000,000 rows; 14.5 / 14.9 /
// 21.2 for 1,000,000), of one column 11.3 / 9.2 / 9.7; against 4,096 blocks and
// finishing launches of their own, k_cg_update 24.0 against 22.8 + 4.7 us,
// k_project_rho of 4 columns 26.5 against 24.9 + 4.3.
constexpr int kInnerBlocks = 512;
constexpr int kInnerPartials = kInnerBlocks * (kMaxCols + 8);

// Device-resident scalars of the inner solver (one per engine).
struct InnerScalars {
    double rho, rho1, alpha, pq, alprho, gk2, xn2, eta;
    double ggk2, ttk2, ttk2m, ck2;
    int iter;    // unused on device (the host passes the iteration number)
    int posdef;  // 1: PCG, 0: sQMR
    int flag;    // 0 ok, 1: rho breakdown (before matvec), 2: alpha breakdown
    int pad;
};

// Reduction scratch owned by an engine.
struct RedBuf {
    double *partials;   // kMaxPartials
    // the inner step's partial sums (at most kInnerBlocks of each): they follow
    // those of the products, which begin at partials
    double *inner(int k) const { return partials + kMaxPartials + (long)k * kInnerBlocks; }
    double *inner_u() const { return inner(0); }
    unsigned *counter;  // 8 counters
    double *out;        // kMaxCols results
};

int red_blocks(long n);

// ---- BLAS-1 / tall-skinny building blocks (double) ----
void fill(hipStream_t s, double *x, double v, long n);
void scal(hipStream_t s, double *x, double a, long n);
void axpy(hipStream_t s, double *y, double a, const double *x, long n);
// out[c] = sum_i V[c*ldv+i] * w[i], c < jv (device, accumulated in double)
template <typename T>
void multidot(hipStream_t s, const RedBuf &rb, const T *V, long ldv, int jv, const T *w, long n,
              double *out);
// w = beta*w + alpha * V * y (y device, jv entries); if nrm2out, also
// nrm2out[0] = ||w||^2 after the update.
void gemv_n(hipStream_t s, const RedBuf &rb, double *w, const double *V, long ldv,
            int jv, const double *y, double alpha, double beta, long n,
            double *nrm2out);
// y += a x ; out[0] = ||y||^2
void axpy_nrm2(hipStream_t s, const RedBuf &rb, double *y, double a, const double *x, long n,
               double *out);
// out[0] = x.y
void dot(hipStream_t s, const RedBuf &rb, const double *x, const double *y, long n,
         double *out);
// out[j*ldo+i] = sum_k V[k*ldv+i] Q[k+j*ldq]   (n x K times K x J)
void tall_gemm(hipStream_t s, const double *V, long ldv, int K, const double *Q,
               int ldq, int J, double *out, long ldo, long n);
// ---- FP64 matrix-core (MFMA) contractions, kernels_mfma.hip ----
// Partial sums of gram() hold at most this many doubles (4 MiB).
constexpr long kGramScratch = 524288;
// Workgroups of gram() for these sizes: at most 1024, at most one per 64 rows,
// and nblk * K * M <= kGramScratch.
int gram_blocks(long n, int K, int M);
// C(i + j*ldc) = sum_r V[i*ldv + r] W[j*ldw + r]  (C = V^T W, K, M <= 64),
// with gram_blocks(n, K, M) * K * M doubles of partial sums in scratch
// (device).  Deterministic (the same summation order on every call).  0 on success,
// -1 if K or M exceeds 64.
int gram(hipStream_t s, long n, int K, int M, const double *V, long ldv, const double *W,
         long ldw, double *C, int ldc, double *scratch);
// Y = V Q on the matrix cores (K, J <= 64); same result layout as tall_gemm.
int tall_gemm_mfma(hipStream_t s, const double *V, long ldv, int K, const double *Q, int ldq,
                   int J, double *Y, long ldy, long n);
// out = {index of max |x_i| (first), x_idx} as doubles
void argmax_abs(hipStream_t s, const RedBuf &rb, const double *x, long n, double *out);

// ---- sparse ----
// Diagonal form (kernels_dia.hip): the upper triangle as one array per
// diagonal, val[k*stride + i] = A(i, i + off[k]), off ascending from 0; for
// slice s of 64 rows and diagonal k, mask[2*(s*nd + k)] has the rows with an
// entry A(i, i + off[k]) and the next word those with A(i, i - off[k]).
// Most diagonals of the upper triangle: the kernels have a row's entries all in
// flight at once, in registers, up to this many.  A loop over more (8 to 16) was
// slower than the general formats up to 250,000 rows (27-point stencil of 40^3:
// SpMV 4.5 -> 7.2 us; 5,000 rows on 16 diagonals 2.3 -> 7.6) and with several
// vectors beyond (three on 80^3 36.8 -> 60.2), and took longer to set up.
constexpr int kDiaMax = 7;
// most rows: byte offsets of 32 bits, and a partial sum of u.y per 256 rows
constexpr int kDiaRows = kMaxPartials * 256;
struct DiaDev {
    int nd = 0, n = 0, nslices = 0;
    long stride = 0;
    double *val = nullptr;
    float *valf = nullptr;  // FP32 copy
    unsigned long long *mask = nullptr;
    int off[kDiaMax] = {};
};
struct DiaHost {
    int nd = 0, nslices = 0;
    long stride = 0;
    std::vector<int> off;
    std::vector<double> val;
    std::vector<unsigned long long> mask;
};
// false: the matrix does not have that form
bool build_dia(int n, const int *ia, const int *ja, const double *a, DiaHost &h);
// (vals64: FP32 vectors with the FP64 values)
template <typename T>
int spmv_dia(hipStream_t s, const RedBuf &rb, const DiaDev &A, bool vals64, const T *x, T *y,
             double eta, const T *u, double *udot_out);
void spmm_dia(hipStream_t s, const DiaDev &A, int k, const double *x, long ldx, double *y,
              long ldy);
// out[0] = the sum of np partial sums
void finish_sum(hipStream_t s, const double *partials, int np, double *out);

constexpr int kLprDia = -2;
struct CsrDev {
    int n = 0;
    long nnz = 0;
    int *rowptr = nullptr;  // 0-based, n+1
    int *col = nullptr;
    double *val = nullptr;
    float *valf = nullptr;  // optional FP32 copy
    int lpr = 8;            // lanes per row (CSR kernel); 0: sliced-ELL kernel, kLprDia: dia
    DiaDev dia;             // nd = 0: none
    // Sliced ELL (slices of 64 consecutive rows, one wave64 per slice, one
    // lane per row, entries of a slice stored column-major so every load of
    // the wave is contiguous).  Column indices are 16-bit offsets from the
    // row when the whole slice allows it, otherwise 32-bit columns.
    int nslices = 0;
    long *s_vptr = nullptr;   // element offset of each slice's values
    long *s_iptr = nullptr;   // byte offset of each slice's indices
    int *s_wm = nullptr;      // 2*width + (1 if 16-bit offsets)
    double *s_val = nullptr;
    float *s_valf = nullptr;
    char *s_idx = nullptr;
    long s_entries = 0;       // padded entries
    long s_idx_bytes = 0;
    bool f_vals64 = false;    // FP32 vectors read the double values
};
// y = A x (T = double: A.val, T = float: A.valf); if eta != 0: y -= eta x;
// if u: u.y (double), in *udot_out, or as partial sums at rb.inner_u() where
// there are at most kInnerBlocks of them: their number is returned, else 0
template <typename T>
int spmv(hipStream_t s, const RedBuf &rb, const CsrDev &A, const T *x, T *y, double eta,
         const T *u, double *udot_out);

// Y = A X for k vectors (column-major, leading dimensions ldx, ldy), FP64,
// in passes of up to 8 vectors over the matrix (kernels_spmm.hip)
void spmm(hipStream_t s, const CsrDev &A, int k, const double *x, long ldx, double *y,
          long ldy);

// ---- preconditioners / conversion ----
template <typename T>
void diag_apply(hipStream_t s, T *z, const T *d, const T *r, long n);
void convert(hipStream_t s, float *dst, const double *src, long n);
void convert(hipStream_t s, double *dst, const float *src, long n);

// Where a kernel tells the host that it has finished writing to pinned memory:
// it stores v at seq (see DevCtx::wait).
struct Done {
    unsigned *seq;
    unsigned v;
};

// ---- inner solver (LSOLREVCOM) fused steps, T = double or float ----
// A step is project_direction, the product Q = (A - eta) P, update; the
// scalars stay in sc, and update leaves a copy of them in host, which is
// pinned memory that the caller reads after it has waited for the stream.
//
// z = P^-1 r is already in z: z -= Q Q^T z (jq columns); rho = r.z, breakdown
// test (flag 1); z += (rho/rho1) p; p = z.  iter: the iteration number.
template <typename T>
void inner_direction(hipStream_t s, const RedBuf &rb, T *z, const T *Q, int jq, const T *r, T *p,
                     long n, InnerScalars *sc, int iter);
// sc's flag into host, behind everything on the stream
void inner_flag(hipStream_t s, const InnerScalars *sc, InnerScalars *host, Done done);
// q = (A - eta) p; np = 0: sc->alprho = u.q is known, np > 0: as np partial
// sums at rb.inner_u().  Then q -= u alprho, pq = p.q, alpha (breakdown: flag
// 2), and PCG's r -= alpha q, x += alpha p, |r|^2, |x|^2, or (posdef = false)
// sQMR's smoothed update of x and x2.
template <typename T>
void inner_update(hipStream_t s, const RedBuf &rb, bool posdef, T *r, T *q, const T *u, T *x,
                  T *x2, const T *p, long n, InnerScalars *sc, int iter, int np,
                  InnerScalars *host, Done done);
// q -= eta p and the partial sums of u.q at rb.inner_u(), after a product that
// the caller made; returns their number
int inner_shift(hipStream_t s, const RedBuf &rb, double *q, double eta, const double *p,
                const double *u, long n);
// sc = *h (by value: no copy, no wait)
void inner_init(hipStream_t s, InnerScalars *sc, const InnerScalars &h);
// dst[0..cnt) = src[0..cnt) by a kernel: into pinned memory, or (put_small, cnt
// <= kMaxCols) from the host's values by value
void get_small(hipStream_t s, double *host, const double *dev, int cnt, Done done);
void put_small(hipStream_t s, double *dev, const double *host, int cnt);

}  // namespace jdhip
