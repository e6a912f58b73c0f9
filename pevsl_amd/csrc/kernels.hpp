// kernels.hpp -- launchers of the HIP kernels (kernels.hip) used by the host
// side of the library.  All launchers enqueue on the given stream and never
// synchronize; shapes are validated by the callers (see check_* in dev.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace pevsl {

// Diagonal layout of a matrix whose nonzeros lie on at most kMaxDiags
// diagonals, each holding one value wherever it holds an entry -- except the
// main diagonal, whose values may differ from row to row: the constant-
// coefficient stencils of structured grids, with or without a potential.
// Per row it stores a bit mask of the diagonals present (1 byte up to 8
// diagonals, else 4) and, where they differ, the main diagonal's value,
// against 8-12 bytes per nonzero in CSR.  Diagonals ascend, as the columns of
// every row do, so a row's sum has the same terms in the same order.
constexpr int kMaxDiags = 32;
struct DevDia {
  int ndiag = 0;         // 0: the matrix has no such layout
  int off[kMaxDiags] = {};     // column - row, ascending
  double c[kMaxDiags] = {};    // the diagonal's value
  int qd = -1;           // index of the main diagonal if it varies, else -1
  const void *mask = nullptr;  // per row: bit q set = entry on diagonal q
  const double *dg64 = nullptr;  // main diagonal per row (qd >= 0)
  const float *dg32 = nullptr;
};
// Diagonals of the kernel that runs a layout of ndiag: the counts of the usual
// stencils (chains, 5- and 9-point, 7-, 13-, 19- and 27-point), so that from two
// diagonals on at most a third of the slots are spare: one costs its load and its
// arithmetic as a real one does.  Microseconds with more slots -> with these:
//   8 -> 5, 250^2 filter 1.8 -> 1.65 a degree     8 -> 7, 20^3 1.95 -> 1.89
//   32 -> 9, 9-point 1000^2: filter FP64 19.6 -> 9.4, FP32 9.9 -> 5.5; width 8
//     FP64 77 -> 34, FP32 36.8 -> 17.9 (CSR 34.4: 32 slots lost to it)
//   32 -> 13, 19, 27, 100^3: width 8 FP32 38 -> 23, 27, 33; FP64 73 -> 47, 51, 70
inline int dia_slots(int ndiag) {
  constexpr int kSlots[] = {3, 5, 7, 8, 9, 13, 19, 27, kMaxDiags};
  for (int s : kSlots)
    if (ndiag <= s) return s;
  return 0;
}
inline int dia_mask_bytes(const DevDia &D) { return D.ndiag <= 8 ? 1 : 4; }

// Device CSR: int32 row pointers / column indices, values in FP64 and FP32.
struct DevCsr {
  int n = 0;       // rows == cols
  int nnz = 0;
  int *ia = nullptr;
  int *ja = nullptr;
  double *a64 = nullptr;
  float *a32 = nullptr;
  int max_row = 0;  // longest row
  // row blocks of the CSR-stream kernels: consecutive rows with at most
  // kStreamRows rows and kStreamNnz nonzeros (a longer row is a block alone)
  int *rowblk = nullptr;
  int *blknz = nullptr;  // first nonzero of each row block, ia[rowblk[b]]
  int nrowblk = 0;
  // row blocks of the nnz-balanced block kernels, one partition per number
  // Q = 2^i of 16-byte pieces in a B-wide row: at most kStreamRows/Q rows and
  // kStreamNnz/Q nonzeros per block (rowblk_q[0] == rowblk)
  int *rowblk_q[5] = {};
  int nrowblk_q[5] = {};
  // ja as 16-bit offsets from the first row of each nonzero's block in
  // `rowblk` (null when an offset does not fit in a short): the CSR-stream
  // and row-per-thread block kernels then read 2 index bytes per nonzero
  short *jo16 = nullptr;
  // every entry has its mirror, equal to a few roundings (square, columns
  // ascending within rows): pEVSL_Kpmdos then forms two moments per product
  bool sym = false;
  // diagonal layout, where the matrix has one (dia.ndiag > 0): the one-column
  // step, the row-per-thread block steps and the products then read it
  DevDia dia;
  // on == 0: the plain CSR form (32-bit indices), without the layouts that
  // replace the column indices
  void use_offsets(int on) {
    if (on) return;
    jo16 = nullptr;
    dia.ndiag = 0;
  }
};

// index bytes per nonzero read by the CSR-stream and row-block kernels
inline int index_bytes(const DevCsr &A) { return A.jo16 ? 2 : 4; }

// bytes of the matrix that a step reads: its diagonal layout, or the CSR form
// with `idx` index bytes per nonzero
inline double matrix_bytes(const DevCsr &A, int elem, int idx, bool dia) {
  if (dia) return (double)A.n * (dia_mask_bytes(A.dia) + (A.dia.qd >= 0 ? elem : 0));
  return (double)A.nnz * (elem + idx) + 4.0 * (A.n + 1);
}

// Rows longer than this are uneven: the CSR-stream kernels sum them by a wave,
// and the batched filter defaults to the nnz-balanced block kernels.
constexpr int kUnevenRow = 64;

constexpr int kStreamRows = 256;
constexpr int kStreamNnz = 2048;

// host: row-block partition with at most max_rows rows and max_nnz nonzeros
// per block, a longer row being a block alone (returns nrowblk+1 offsets);
// the CSR-stream kernels use (kStreamRows, kStreamNnz)
void build_row_blocks(int n, const int *ia, std::vector<int> &blk,
                      int max_rows = kStreamRows, int max_nnz = kStreamNnz);

// jo[j] = ja[j] - (first row of nonzero j's row block); *over set to 1 if one
// does not fit in 16 bits
void offsets16(const DevCsr &A, short *jo, int *over, hipStream_t s);
// *bad set to 1 unless every entry (i, j) has a mirror (j, i) of its value and
// columns ascend strictly within rows (A square)
void check_symmetric(const DevCsr &A, int *bad, hipStream_t s);

// ---- sparse products -------------------------------------------------------
// y = A x, one column.  lanes = lanes per row in {1,2,4,8,16,32,64}, or 0 for
// the kernel that suits the matrix: its diagonal layout, else the CSR-stream
// or vector-CSR form by size.
void spmv_f64(const DevCsr &A, const double *x, double *y, int lanes,
              hipStream_t s);
// Y(:,c) = A X(:,c) for ncol column-major columns with leading dim ld.
void spmv_cols_f64(const DevCsr &A, const double *X, double *Y, int ncol,
                   size_t ld, int lanes, hipStream_t s);

// One Chebyshev degree step of the filter for one column (T = float/double):
//   first:  vkp1 = t (A vk - cc vk);        y = mu0 vk + muk vkp1
//   else:   vkp1 = t (A vk - cc vk) - vkm1; y = y + muk vkp1
template <typename T>
void cheb_step_vec(const DevCsr &A, const T *vk, const T *vkm1, T *vkp1, T *y,
                   double cc, double t, double mu0, double muk, bool first,
                   int lanes, hipStream_t s);

// How a three-term step of degree d updates the accumulator y, whose term of
// degree d is mu_d v_d (vk = v_{d-1}, vkm1 = v_{d-2}, vkp1 = v_d):
//   kYSkip       y is neither read nor written: its term waits
//   1, 2, 3      y += the terms of the last 1, 2 or 3 degrees, in order
//   kYInit | 1   y = mu_0 v_0 + mu_1 v_1              (d == 1)
//   kYInit | 2   y = mu_0 v_0 + mu_1 v_1 + mu_2 v_2   (d == 2, v_0 = vkm1)
// A step holds v_{d-2}, v_{d-1} and v_d anyway, so y need pass through memory
// only every third degree, with the results of one update per degree bit for
// bit.  YPlan gives the modes of a run of degrees 1..m.
constexpr int kYSkip = 0, kYInit = 4;
struct YPlan {
  int pend = 0;          // degrees whose terms wait
  bool started = false;  // y holds the terms of the degrees before them
  int next(int d, int m) {
    pend++;
    const bool flush = d == m || pend == (started ? 3 : 2);
    if (!flush) return kYSkip;
    const int mode = (started ? 0 : kYInit) | pend;
    started = true;
    pend = 0;
    return mode;
  }
};
// passes over y of a step: none, a write, or a read and a write
inline int y_passes(int mode) { return mode == kYSkip ? 0 : (mode & kYInit) ? 1 : 2; }

// Same step, y updated as `ymode` says (mu0, mu3, mu2, mu1: the coefficients
// of degrees 0, d-2, d-1, d; vkm1 null at d == 1), with the kernel that suits
// the matrix: its diagonal layout, or the CSR-stream kernel (one block per row
// block: coalesced products staged in LDS, then one sequential sum per row).
template <typename T>
void cheb_step_stream(const DevCsr &A, const T *vk, const T *vkm1, T *vkp1,
                      T *y, double cc, double t, double mu0, double mu3, double mu2, double mu1,
                      int ymode, hipStream_t s);
// whether cheb_step_stream and the row-per-thread block steps of width B read
// the diagonal layout (32-bit byte offsets into a block of B columns)
inline bool use_dia(const DevCsr &A, int elem, int B) {
  return A.dia.ndiag > 0 && (double)A.n * elem * B < 4294967296.0;
}
// kernels of the diagonal layout (dia.hip)
void dia_spmv_f64(const DevCsr &A, const double *X, double *Y, int ncol, size_t ld,
                  hipStream_t s);
template <typename T>
void dia_cheb_step(const DevCsr &A, const T *vk, const T *vkm1, T *vkp1, T *y, double cc,
                   double t, double mu0, double mu3, double mu2, double mu1, int ymode,
                   hipStream_t s);

template <typename T>
void dia_cheb_blk(const DevCsr &A, int B, const T *vk, const T *vkm1, T *vkp1, T *y, double cc,
                  double t, const double *mus, int k, int nact, hipStream_t s, int ymode);
template <typename T>
void dia_clen_blk(const DevCsr &A, int B, const T *b1, const T *b2, const T *v, T *out, double cc,
                  double t, const double *mus, int k, hipStream_t s);

// launches of several degrees: degrees per launch (1: none), rows per
// workgroup, widest diagonal
struct MultiPlan {
  int s = 1, R = 0, bw = 0;
};
// The degrees 1..m >= 1 of the filter y = sum mu_k T_k((A - cc)/dd) x for one
// column in the stream form: a launch per degree, or on the diagonal layout of
// a small or narrow matrix several degrees per launch (k_cheb_multi), with the
// same bits.  p = dia_multi_plan(A, sizeof(T), m).  w: 4 n elements (3 n if n >
// 2^20).  Returns the launches and the bytes of their passes over memory.
struct ChebRun {
  long long launches = 0;
  double bytes = 0.0;
};
template <typename T>
ChebRun cheb_run(const DevCsr &A, const MultiPlan &p, const double *mu, int m, double cc, double dd,
                 const T *x, T *y, T *w, hipStream_t s);
constexpr int kMultiMax = 32;      // degrees per launch at most
// rows of a workgroup's window at most: its two FP64 vectors fill 64 KiB of LDS
constexpr int kMultiRows = 4080;
MultiPlan dia_multi_plan(const DevCsr &A, int elem, int m);
template <typename T>
void dia_cheb_multi(const DevCsr &A, const MultiPlan &p, const T *v, const T *vm, T *vout,
                    T *vmout, T *y, double cc, double dd, const double *mu, int d0, int s,
                    bool last, hipStream_t st);

// Same for B interleaved columns (row-major n x B block, column fastest).
// mus: device array [(deg_max+1) x B] of per-column coefficients; k = degree
// index of this step (1..); columns c >= nact are left untouched.
template <typename T>
void cheb_step_blk(const DevCsr &A, int B, const T *vk, const T *vkm1, T *vkp1,
                   T *y, double cc, double t, const double *mus, int k,
                   int nact, hipStream_t s);

// Same with one thread per row (row blocks of the CSR-stream partition,
// a/ja staged in LDS, B-wide 16-byte row gathers), or on the diagonal layout
// with one thread per (row, 16-byte piece); B <= 32.  y is updated as
// `ymode` says, for columns c < nact (active at the lowest degree whose term
// is added; mus is zero past each column's degree).
template <typename T>
void cheb_step_blkrow(const DevCsr &A, int B, const T *vk, const T *vkm1, T *vkp1,
                      T *y, double cc, double t, const double *mus, int k,
                      int nact, hipStream_t s, int ymode);

// Clenshaw step on B interleaved columns (same kernels, B <= 32):
//   out = mu_k v + t (A b1 - cc b1) - b2,  mu_k per column = mus[k*B + c];
// b2 == nullptr reads as zero; b1 == nullptr gives the top term out = mu_k v.
template <typename T>
void clen_step_blkrow(const DevCsr &A, int B, const T *b1, const T *b2, const T *v, T *out,
                      double cc, double t, const double *mus, int k, hipStream_t s);

// Clenshaw step on the active 16-byte pieces (SEG = 16/sizeof(T) columns
// each) of an interleaved block of Bp columns (Bp a multiple of SEG, at most
// kMaxSegs pieces), one thread per (row, piece): pieces 0..nseg-1 are active
// (sorted by top degree, descending); piece s writes the top term mu_d v at
// d == tops.top[s], reads b2 as zero at d == top - 1, and otherwise computes
// out = mu_d v + t (A b1 - cc b1) - b2 with mus[d*Bp + c], as
// clen_step_blkrow does per column.  Pieces >= nseg are not touched.
constexpr int kMaxSegs = 16;
struct SegTops {
  int top[kMaxSegs];
};
template <typename T>
void clen_step_seg(const DevCsr &A, int Bp, const T *b1, const T *b2, const T *v, T *out,
                   double cc, double t, const double *mus, int d, int nseg, const SegTops &tops,
                   hipStream_t s);

// nnz-balanced forms of cheb_step_blkrow and clen_step_blkrow (same
// arguments and results; products formed in parallel over nonzeros and
// staged in LDS, long rows reduced by a whole workgroup); B <= 32.
template <typename T>
void cheb_step_bal(const DevCsr &A, int B, const T *vk, const T *vkm1, T *vkp1,
                   T *y, double cc, double t, const double *mus, int k,
                   int nact, hipStream_t s, int ymode);
template <typename T>
void clen_step_bal(const DevCsr &A, int B, const T *b1, const T *b2, const T *v, T *out,
                   double cc, double t, const double *mus, int k, hipStream_t s);
// partition index of the balanced kernels for element size elem, width B
int bal_level(int elem, int B);

// One KPM step v -> w = scal (A v - ctr v) - vm of ng groups of B interleaved
// columns (group g at v + g n B; B a power of two <= 32), w written over vm
// (vw); vm is zero, and not read, if `first`.  Per column c = g B + b the block
// partials of w.w, w.v and (first) v.v, or of w.v0 alone where v0 is given:
// part[(i ng B + c) nblk + blk] for sum i and blk < nblk = kpm_blocks(A, dia,
// sizeof(T), B).  On the diagonal layout (dia: row sums and recurrence in FP64
// whatever T is, without v0) or with the nnz-balanced products (in T); `dia`
// is the caller's KpmPlan::dia, since the two forms differ in their sums.
template <typename T>
void kpm_step(const DevCsr &A, bool dia, int B, int ng, const T *v, T *vw, const T *v0, double ctr,
              double scal, bool first, double *part, hipStream_t s);
int kpm_blocks(const DevCsr &A, bool dia, int elem, int B);
// How pEVSL_Kpmdos forms the moments of nvec vectors of `elem` bytes an element.
struct KpmPlan {
  bool dia;     // steps on the diagonal layout
  bool direct;  // one product per moment and <w, v0>; else two moments a product
  int B, ng;    // vectors in a group, groups in a run
};
KpmPlan kpm_plan(const DevCsr &A, int elem, int nvec);
int dia_kpm_blocks(int n, int elem, int B);
template <typename T>
void dia_kpm_step(const DevCsr &A, int B, int ng, const T *v, T *vw, double ctr, double scal,
                  bool first, double *part, hipStream_t s);
// raw: ncol column-major n-vectors; group g of blk gets columns g B .. as
// x / sqrt(nrm2[c]), zero past ncol
template <typename T>
void kpm_pack(int n, int B, int ng, int ncol, const double *raw, const double *nrm2, T *blk,
              hipStream_t s);
// out[i] = sum of part[i*nblk .. (i+1)*nblk), i < nrows
void row_sums(const double *part, int nrows, int nblk, double *out, hipStream_t s);

// ---- dense / vector kernels (FP64 unless stated) --------------------------
// out[c] = sum_b part[b*ncol + c], b < nblk (fixed order); out may be strided.
void reduce_partials(const double *part, int nblk, int ncol, double *out,
                     hipStream_t s);
// y = x for n doubles: plain copy kernel (16-byte pairs where n and the
// alignment allow)
void copy_f64(size_t n, const double *x, double *y, hipStream_t s);
// part[p] (m1 x m2, column-major) = X(rows p*chunk .. , :)^T Y(same rows, :)
// for p < nparts (the last part ends at row n), FP64 MFMA (hand-written
// v_mfma_f64_16x16x4 tiles); X and Y column-major with leading dims ldx, ldy.
// upper (m1 == m2): only the 64 x 64 tiles on and above the diagonal.
void gram_tn_mfma(int n, int m1, const double *X, size_t ldx, int m2, const double *Y,
                  size_t ldy, int chunk, int nparts, bool upper, double *part, hipStream_t s);
// C (m x m) = sum over p < nparts of the upper triangles of part[p], in part
// order, stored in both triangles (a symmetric C)
void sum_parts_upper(const double *part, int nparts, int m, double *C, hipStream_t s);
// out[e] = sum_p part[p*nel + e] over p = 0..nparts-1 in order
void sum_parts(const double *part, int nparts, size_t nel, double *out, hipStream_t s);
// part[blk] = sum x_i*y_i over the block's rows; returns nblk
int dot_partials(int n, const double *x, const double *y, double *part,
                 hipStream_t s);
int dot_part_blocks(int n);
void scale_vec(int n, double *x, const double *inv_scale_dev, double hostscale,
               hipStream_t s);
void axpy_vec(int n, double a, const double *x, double *y, hipStream_t s);
// vkp1 = t (vkp1 - cc vk) - vkm1 (vkm1 may be null);  y += mu vkp1 (y may be
// null): the vector part of a Chebyshev step with a separately formed product
void cheb_update(int n, const double *vk, const double *vkm1, double *vkp1, double *y,
                 double cc, double t, double mu, hipStream_t s);
void copy_f64_to_f32(size_t n, const double *x, float *y, hipStream_t s);
void copy_f32_to_f64(size_t n, const float *x, double *y, hipStream_t s);
void fill_zero_f64(size_t n, double *x, hipStream_t s);

// Pack/unpack between one column-major vector of type TV per slice and an
// interleaved n x B block of type T.  cols[c] points to the n-vector of
// column c (device array of pointers), c < ncol.
template <typename T, typename TV = double>
void pack_cols(int n, int B, int ncol, const TV *const *cols, T *blk,
               hipStream_t s);
template <typename T, typename TV = double>
void unpack_cols(int n, int B, int ncol, const T *blk, TV *const *cols,
                 hipStream_t s);
// FP32 vector helpers (FP64 accumulation)
int dot_partials_f32(int n, const float *x, const float *y, double *part,
                     hipStream_t s);
void scale_vec_f32(int n, float *x, double hostscale, hipStream_t s);

// ---- Lanczos on a batch of slices ----------------------------------------
// Slices are independent; slice s owns V_s (chunked columns, leading dim ld
// a multiple of 64, chunks of 2^chunk_shift >= 32 columns whose rows
// [n, ld) are zero) and per-step scalars.  Column j of slice s is
//   vtab[s*maxchunks + (j >> chunk_shift)] + (size_t)(j & chunk_mask)*ld
// elements of vbytes bytes: FP64 (8) or FP32 (4) storage.  All arithmetic
// (dots, updates, norms) is FP64 either way.
struct LanBatch {
  int n = 0;
  size_t ld = 0;
  int nslice = 0;
  int chunk_shift = 9;
  int maxchunks = 0;
  int vbytes = 8;           // basis element size: 8 (double) or 4 (float)
  void **vtab = nullptr;    // device [nslice*maxchunks]
  // device scalars per slice
  double *alpha = nullptr;  // [nslice]
  double *beta = nullptr;   // [nslice] (beta of the previous step)
  double *nrm2a = nullptr;  // [nslice] |v|^2 before reorth pass
  double *nrm2b = nullptr;  // [nslice] |v|^2 after a reorth pass
  int *pass2 = nullptr;     // [nslice] 1 if the 2nd DGKS pass is needed
  int *active = nullptr;    // [nslice] 1 if the slice takes part
  double *h = nullptr;      // [nslice * hcap]
  int hcap = 0;
  double *part = nullptr;   // partial sums workspace
  size_t part_cap = 0;      // doubles
};

// doubles of LanBatch::part needed for n rows, nslice slices and hcap
// reorthogonalization coefficients per slice
size_t lan_part_doubles(int n, int nslice, int hcap);

// Three-term update: znew_s -= beta_s zold_s (k > 0), alpha_s = <z_s, znew_s>,
// znew_s -= alpha_s z_s, and partials of |znew_s|^2.  norm_only: only these.
void lan_update(const LanBatch &L, int k, bool norm_only, hipStream_t s);
// One classical Gram-Schmidt pass against V_s(:,0:k): h = V^T znew,
// znew -= V h, and partials of |znew|^2.  pass = 0 runs for active slices;
// pass = 1 only for those among them whose pass2 flag is set.
void lan_cgs_pass(const LanBatch &L, int k, int pass, hipStream_t s);
// nrm2b = |znew|^2 from the partials of a pass, pass2 = the DGKS test against
// nrm2a (a Gram-Schmidt pass outside a Lanczos step)
void lan_cgs_norm(const LanBatch &L, hipStream_t s);
// End of a Lanczos step after lan_update and lan_cgs_pass(pass): nrm2b and beta
// = |znew|; with pass 0 also nrm2a and pass2 (DGKS test); znew /= beta unless a
// second pass is due.  host[3s ..] = alpha, nrm2b, pass2 of slice s, in memory
// that the device writes and the host reads once the stream has drained.  With
// a second pass due: lan_cgs_pass(1), lan_finish(1).
void lan_finish(const LanBatch &L, int k, int pass, double *host, hipStream_t s);

// ---- tridiagonal (FP64) ---------------------------------------------------
// Restricted trace of T (diag d[0..m-1], sub-diag e[0..m-2]): eigenvalues
// >= thr by Sturm bisection.  out[0] = sum, out[1] = count (as double).
// Workspace: lam (m doubles).
void tridiag_trace_above(int m, const double *d, const double *e, double thr,
                         double *lam, double *out, hipStream_t s);
// The same for np matrices of equal order m at once: T_p in d/e + p*ld,
// thresholds thr[p] (device), eigenvalues in lam + p*ld, 4 workspace values
// per problem in ws, out[2p] = sum and out[2p+1] = count.
void tridiag_trace_above_batch(int np, int m, size_t ld, const double *d, const double *e,
                               const double *thr, double *lam, double *ws, double *out,
                               hipStream_t s);
// All eigenvalues of T by bisection (ascending), for tests and small m.
void tridiag_eigvals(int m, const double *d, const double *e, double *lam,
                     hipStream_t s);

// ---- column-major multi-vectors (Ritz stage) ------------------------------
// part must hold ncol * col_part_blocks(n) doubles.
int col_part_blocks(int n);
// out[c] = <X(:,c), Y(:,c)>
void col_dots(int n, int ncol, const double *X, size_t ldx, const double *Y,
              size_t ldy, double *part, double *out, hipStream_t s);
// X(:,c) *= f[c]
void col_scale(int n, int ncol, double *X, size_t ld, const double *f,
               hipStream_t s);
// Y(:,c) += a[c] X(:,c)
void col_axpy(int n, int ncol, const double *a, const double *X, size_t ldx,
              double *Y, size_t ldy, hipStream_t s);

// ---- misc -----------------------------------------------------------------
// y[j] = integral of the KPM DOS at x[j] (closed form, per-point sequential
// sum over degrees as the reference does).
void kpm_intchx(int Mdeg, const double *mu, int npts, const double *th,
                double th0, double *yi, hipStream_t s);
// Elements i0 .. i0 + cnt - 1 of the columns X (n rows, column stride ld) from
// outputs r of the rand() stream: ((r >> 1) - t) / t, t = RAND_MAX / 2.
void rand_convert(int n, size_t i0, size_t cnt, const uint32_t *r, double *X, size_t ld,
                  hipStream_t s);
// Rademacher (+-1) or uniform [-1,1] counter-based random numbers.
void rand_fill(size_t n, double *x, uint64_t seed, uint64_t offset,
               int rademacher, hipStream_t s);

}  // namespace pevsl
