// dia.hip -- kernels on the diagonal layout (DevDia): the matrix is a list of
// diagonals, each with one value, and a bit mask per row of the diagonals
// present (constant-coefficient grid stencils, optionally with a main
// diagonal that varies).
//
// The CSR kernels of these steps move 8-12 bytes per nonzero, more than all
// vectors of a one-column step together (100^3 Laplacian, FP64: 69 of 113 MB),
// and walk a chain of dependent loads (row block, row pointers, indices,
// gathered values, LDS).  Here the matrix costs 1 byte per row, every load of
// x is coalesced (neighbouring threads read neighbouring rows at one offset),
// and all loads of a row are independent of each other.  What remains is the
// vectors.
//
// A row's terms are the CSR row's, in column order, each product rounded
// before it is added; absent diagonals add nothing (not a zero times x), so
// results equal the CSR kernels' bit for bit.
#include "dev.hpp"

#include <algorithm>
#include <type_traits>

namespace pevsl {

namespace {

// Diagonals as kernel arguments (scalar registers); entries past ndiag have
// no mask bit.
template <typename T, int UC, typename C = T>
struct DiaArg {
  int off[UC];
  C c[UC];
  int qd;
  const T *dg;
};

template <int UC>
using DiaMask = std::conditional_t<UC <= 8, uint8_t, uint32_t>;

// loads of a row in flight together
constexpr int dia_chunk(int uc) { return uc <= 9 ? uc : 8; }

// x[i] with a 32-bit byte offset from a uniform base (use_dia bounds it)
template <typename T>
__device__ __forceinline__ T ld32(const T *x, uint32_t i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(x) + i * (uint32_t)sizeof(T));
}

// sum of row r times x: all loads first (absent diagonals read x[0]), then
// the terms in column order
template <typename T, int UC>
__device__ __forceinline__ T dia_row(const DiaArg<T, UC> &d, uint32_t m, T dgv, int r,
                                     const T *__restrict__ x) {
#pragma clang fp contract(off)
  T acc = 0;
  constexpr int CH = dia_chunk(UC);
#pragma unroll
  for (int q0 = 0; q0 < UC; q0 += CH) {
    T xv[CH];
#pragma unroll
    for (int q = 0; q < CH && q0 + q < UC; q++)
      xv[q] = ld32(x, (m >> (q0 + q)) & 1 ? (uint32_t)(r + d.off[q0 + q]) : 0u);
#pragma unroll
    for (int q = 0; q < CH && q0 + q < UC; q++) {
      const T a = q0 + q == d.qd ? dgv : d.c[q0 + q];
      const T s = acc + a * xv[q];
      acc = (m >> (q0 + q)) & 1 ? s : acc;
    }
  }
  return acc;
}

template <int UC>
__global__ void __launch_bounds__(kThreads)
k_dia_spmv(int n, DiaArg<double, UC> d, const DiaMask<UC> *__restrict__ mask,
           const double *__restrict__ x, double *__restrict__ y, size_t ld) {
  x += (size_t)blockIdx.y * ld;
  y += (size_t)blockIdx.y * ld;
  const int r = xcd_block(blockIdx.x, gridDim.x) * kThreads + threadIdx.x;
  if (r >= n) return;
  const double dgv = d.qd >= 0 ? d.dg[r] : 0.0;
  y[r] = dia_row<double, UC>(d, mask[r], dgv, r, x);
}

// One degree of the filter for one column, one row per thread.  Bound by the
// vector passes (vk, vkm1, vkp1, and y every third degree) and, below about
// 1e5 rows, by the launch and one trip of independent loads.  Microseconds per
// degree of a whole filter call, CSR-stream kernel -> this kernel:
//   100^3 Laplacian, FP64  19.96 -> 7.85 (30 MB: 3.8 TB/s)   FP32 15.8 -> 5.3
//   113x97x83 with a potential, FP64 7.7   FP32  15.3 -> 5.3
//   60^3, FP64  6.6 -> 4.5
// of which a launch of its own (HIP events, back to back) takes FP64 7.8 and
// FP32 4.7 at 100^3, 3.7 and 2.75 at 60^3, 2.6-3.0 below.  With 8 slots for the
// 7 diagonals, 100^3 FP64: one, two and four rows per thread 8.36, 8.29 and
// 8.93, 60^3 3.8, 4.1 and 4.6: one row gives the most waves.
template <typename T, int UC>
__global__ void __launch_bounds__(kThreads)
k_cheb_dia(int n, DiaArg<T, UC> d, const DiaMask<UC> *__restrict__ mask,
           const T *__restrict__ vk, const T *__restrict__ vkm1, T *__restrict__ vkp1,
           T *__restrict__ y, T cc, T t, T m0, T m3, T m2, T m1, int ymode) {
#pragma clang fp contract(off)
  const int r = xcd_block(blockIdx.x, gridDim.x) * kThreads + threadIdx.x;
  if (r >= n) return;
  const uint32_t m = mask[r];
  const T v = ld32(vk, (uint32_t)r);
  const T dgv = d.qd >= 0 ? ld32(d.dg, (uint32_t)r) : (T)0;
  const T vm = vkm1 ? ld32(vkm1, (uint32_t)r) : (T)0;
  const T yv = ymode != kYSkip && !(ymode & kYInit) ? y[r] : (T)0;
  T w = dia_row<T, UC>(d, m, dgv, r, vk) + (-cc) * v;
  w = w * t;
  if (vkm1) w = w + (T)(-1) * vm;
  vkp1[r] = w;
  if (ymode != kYSkip) y[r] = y_next<T>(ymode, yv, vm, v, w, m0, m3, m2, m1);
}

// Coefficients of the degrees of one k_cheb_multi launch.
template <typename T>
struct MuArg {
  T m0, mu[kMultiMax];
};

// Degrees d0 .. d0+s-1 of the filter for one column in one launch: a workgroup
// owns R rows and keeps them, with the s*bw rows on either side that they
// depend on (bw: the widest diagonal), in LDS; it steps the window, which
// shrinks by bw at both ends per degree, with one barrier per degree, and
// writes its own rows' last two vectors and y.  Each row goes through the
// operations of k_cheb_dia in their order, hence the same bits; rows in the
// overlap of two windows are computed by both.
//
// For grids and chains whose degree takes less than the launch around it:
// k_cheb_dia needs 2.6-3.0 us a degree at any size below 1e5 rows (launch, one
// trip to memory), up to 4 where the host launches no faster.  Bound by LDS
// reads and barriers inside, by the overlap of the windows where the band is
// wide.  FP64, microseconds per degree, launches of one degree back to back ->
// this kernel in a whole filter call at the plan's s:
//   chain 64,000 rows 2.9 -> 0.34 (s = 32)   1e6 rows 5.8 -> 1.15 (s = 32)
//   12^3 2.8 -> 0.96 (s = 10)   20^3 2.9 -> 1.72 (s = 5), FP32 1.60
//   60^2 2.9 -> 0.62 (s = 16)   250^2 2.8 -> 1.48 (s = 7)  400^2 2.9 -> 2.55 (4)
// (with a select per absent diagonal instead of the zeros below, and 8 slots:
// 20^3 2.4 against 1.95, 250^2 2.1 against 1.8)
// K rows of the window per thread, blockDim.x apart.
template <typename T, int UC, int K, bool DV>
__global__ void __launch_bounds__(1024)
k_cheb_multi(int n, DiaArg<T, UC> d, const DiaMask<UC> *__restrict__ mask, int bw, int R, int d0,
             int s, int last, const T *__restrict__ vin, const T *__restrict__ vmin,
             T *__restrict__ vout, T *__restrict__ vmout, T *__restrict__ y, T cc, T t1, T t2,
             MuArg<T> mus) {
#pragma clang fp contract(off)
  // the window's two vectors, each with a zero at its end that absent
  // diagonals read: adding c times zero leaves the sum as it is, bit for bit (a
  // sum that starts at +0 never becomes -0), and an entry costs no selects
  constexpr int kSlot = kMultiRows + 8;
  extern __shared__ char multi_lds[];
  const int r0 = blockIdx.x * R, r1 = min(n, r0 + R);
  const int w0 = max(0, r0 - s * bw), w1 = min(n, r1 + s * bw), L = w1 - w0;
  T *const va = reinterpret_cast<T *>(multi_lds), *const vb = va + kSlot;
  // byte offsets of each row's neighbours in a vector, two to a register
  uint32_t at[K][(UC + 1) / 2];
  T dg[K], yv[K];
#pragma unroll
  for (int i = 0; i < K; i++) {
    const int x = threadIdx.x + i * (int)blockDim.x, r = w0 + x;
    dg[i] = yv[i] = 0;
    uint32_t m = 0;
    if (x < L) {
      m = mask[r];
      if (DV) dg[i] = d.dg[r];
      const T v = vin[r];
      va[x] = v;
      vb[x] = d0 > 1 ? vmin[r] : (T)0;
      if (r >= r0 && r < r1) yv[i] = d0 > 1 ? y[r] : v * mus.m0;
    }
#pragma unroll
    for (int q = 0; q < UC; q++) {
      const int c = x + d.off[q];
      // rows near the window's ends have neighbours outside it, in steps that
      // do not compute them
      const bool on = ((m >> q) & 1) && c >= 0 && c < L;
      const uint32_t o = (uint32_t)(on ? c : L) * (uint32_t)sizeof(T);
      at[i][q / 2] = q % 2 ? at[i][q / 2] | (o << 16) : o;
    }
  }
  if (threadIdx.x == 0) va[L] = vb[L] = 0;
  __syncthreads();
  // degree d0 + j from `from` (v_{d-1}) over `to` (v_{d-2} -> v_d)
  auto step = [&](int j, const T *from, T *to) {
    const int h = (s - 1 - j) * bw;
    const int lo = max(0, r0 - h), hi = min(n, r1 + h);
    const T t = d0 + j == 1 ? t1 : t2;
#pragma unroll
    for (int i = 0; i < K; i++) {
      const int x = threadIdx.x + i * (int)blockDim.x, r = w0 + x;
      if (r < lo || r >= hi) continue;
      T xv[UC];
#pragma unroll
      for (int q = 0; q < UC; q++) {
        const uint32_t o = q % 2 ? at[i][q / 2] >> 16 : at[i][q / 2] & 0xffffu;
        xv[q] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(from) + o);
      }
      T acc = 0;
#pragma unroll
      for (int q = 0; q < UC; q++) acc = acc + (DV && q == d.qd ? dg[i] : d.c[q]) * xv[q];
      T w = acc + (-cc) * from[x];
      w = w * t;
      if (d0 + j > 1) w = w + (T)(-1) * to[x];
      to[x] = w;
      if (r >= r0 && r < r1) yv[i] = yv[i] + mus.mu[j] * w;
    }
    __syncthreads();
  };
  int j = 0;
  for (; j + 1 < s; j += 2) {
    step(j, va, vb);
    step(j + 1, vb, va);
  }
  const T *fin = va, *prev = vb;
  if (j < s) {
    step(j, va, vb);
    fin = vb;
    prev = va;
  }
#pragma unroll
  for (int i = 0; i < K; i++) {
    const int x = threadIdx.x + i * (int)blockDim.x, r = w0 + x;
    if (r < r0 || r >= r1) continue;
    y[r] = yv[i];
    if (!last) {
      vout[r] = fin[x];
      vmout[r] = prev[x];
    }
  }
}

// sum of row r times piece pc (columns pc*P ..) of the interleaved block x of
// n rows, in type C.  Absent diagonals read a row inside the block, so that the
// loads need not wait for the mask (100^3 FP32: B=4 11.4 -> 10.4 us, B=8 20.7
// -> 20.1).  FMA: with fused multiply-adds and their operand selected before
// the conversion, for sums in FP64 that need not repeat the scalar loop's bits.
template <typename T, int B, int UC, bool FMA = false, typename C = T>
__device__ __forceinline__ void dia_row_piece(const DiaArg<T, UC, C> &d, uint32_t m, T dgv, int r,
                                              int pc, int n, const T *__restrict__ x,
                                              C (&acc)[Pieces<T, B>::P]) {
#pragma clang fp contract(off)
  constexpr int P = Pieces<T, B>::P;
  constexpr int CH = dia_chunk(UC);
#pragma unroll
  for (int e = 0; e < P; e++) acc[e] = 0;
#pragma unroll
  for (int q0 = 0; q0 < UC; q0 += CH) {
    T xv[CH][P];
#pragma unroll
    for (int q = 0; q < CH && q0 + q < UC; q++) {
      const uint32_t row = (uint32_t)min(max(r + d.off[q0 + q], 0), n - 1);
      const uint32_t at = (row * (uint32_t)B + (uint32_t)(pc * P)) * (uint32_t)sizeof(T);
      ld_piece<T, P>(reinterpret_cast<const T *>(reinterpret_cast<const char *>(x) + at), xv[q]);
    }
#pragma unroll
    for (int q = 0; q < CH && q0 + q < UC; q++) {
      const C a = q0 + q == d.qd ? (C)dgv : d.c[q0 + q];
      const bool on = (m >> (q0 + q)) & 1;
#pragma unroll
      for (int e = 0; e < P; e++) {
        if constexpr (FMA) {
          acc[e] = __builtin_elementwise_fma(a, (C)(on ? xv[q][e] : (T)0), acc[e]);
        } else {
          const C s = acc[e] + a * (C)xv[q][e];
          acc[e] = on ? s : acc[e];
        }
      }
    }
  }
}

// One degree of the filter on B interleaved columns, one thread per (row,
// 16-byte piece): every load is contiguous over the wave.  Bound by the vector
// passes (four of n B values) once they exceed the latency of one trip; the
// row-per-thread CSR kernels gather whole rows with one thread each, wait for
// their LDS staging, and have Q times fewer threads.  Microseconds per launch,
// row kernels -> this kernel:
//   100^3, FP32 Clenshaw    B=4 19.1 -> 10.0  8: 28.9 -> 17.4  16: 77.7 -> 33-40
//   100^3, FP64 three-term  B=4 38.0 -> 17.6  8: 91.3 -> 32.6
//   48x40x44, FP32 Clenshaw B=8 5.9 -> 3.6    20^3, FP32 B=8 5.2 -> 2.9
// (100^3, B=8 FP32: 129 MB, 7.4 TB/s, served by the Infinity Cache.)
template <typename T, int B, int UC, class Epi>
__global__ void __launch_bounds__(kThreads)
k_dia_blk(int n, DiaArg<T, UC> d, const DiaMask<UC> *__restrict__ mask, const T *__restrict__ x,
          Epi epi) {
  constexpr uint32_t Q = Pieces<T, B>::Q;
  const uint32_t g = (uint32_t)xcd_block(blockIdx.x, gridDim.x) * kThreads + threadIdx.x;
  const int r = (int)(g / Q), pc = (int)(g % Q);
  if (r >= n) return;
  const uint32_t m = mask[r];
  const T dgv = d.qd >= 0 ? d.dg[r] : (T)0;
  typename Epi::Ops ops;
  epi.load(r, pc, ops);
  T acc[Pieces<T, B>::P];
  dia_row_piece<T, B, UC>(d, m, dgv, r, pc, n, x, acc);
  epi.finish(r, pc, ops, acc);
}

// One KPM step on B interleaved columns, group blockIdx.y: the workgroups of
// an XCD sweep its contiguous range of (row, piece) items together, kThreads
// each at a time, `iters` times, so that the rows in use at one moment are few
// and stay in its L2, and a workgroup's sums end in one reduction and one set of
// partials.  Bound by the three vector passes (u_j, u_j-1 read, u_j+1 over it)
// in FP64, by the FP64 arithmetic on FP32 vectors.  Whole
// pEVSL_Kpmdos, one thread per (row, column) and one product per moment -> this:
// 100^3, Mdeg 300, 64 FP32 vectors 263 -> 24.0 ms (600 launches of 192 MB: 4.8
// TB/s); 20^3, 60 FP64 vectors 8.8 -> 1.5 ms (150 launches of 5.7 us).  Each workgroup a contiguous range of its own, and
// products, sums and selections of absent entries in separate FP64
// instructions: 33.3 ms at 100^3.
template <typename T, int B, int UC, bool FIRST>
__global__ void __launch_bounds__(kThreads)
k_dia_kpm(int n, DiaArg<T, UC, double> d, const DiaMask<UC> *__restrict__ mask,
          EpiKpm<T, B, double> epi, size_t gstride, int iters, int ncol,
          double *__restrict__ part) {
  constexpr uint32_t Q = Pieces<T, B>::Q;
  constexpr int P = Pieces<T, B>::P;
  // this XCD's workgroups lo .. lo + cnt - 1, this one number j of them
  const int x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
  const int lo = xcd_block(x, gridDim.x), cnt = xcd_count(x, gridDim.x);
  epi.group(blockIdx.y, gstride);
  epi.v0 = nullptr;
  epi.first = FIRST;
  KpmSums<P> sums;
  for (int it = 0; it < iters; it++) {
    const uint32_t g = ((uint32_t)lo * iters + (uint32_t)it * cnt + j) * kThreads + threadIdx.x;
    const int r = (int)(g / Q), pc = (int)(g % Q);
    if (r >= n) break;
    const uint32_t m = mask[r];
    const T dgv = d.qd >= 0 ? d.dg[r] : (T)0;
    typename EpiKpm<T, B, double>::Ops ops;
    epi.load(r, pc, ops);
    double acc[P];
    dia_row_piece<T, B, UC, true>(d, m, dgv, r, pc, n, epi.v, acc);
    epi.finish(r, pc, ops, acc, sums);
  }
  kpm_block_sums<T, B>(sums, epi.nsum(), ncol, gridDim.x, lo + j,
                       part + (size_t)blockIdx.y * B * gridDim.x);
}

template <typename T, int UC, typename C = T>
DiaArg<T, UC, C> dia_arg(const DevDia &D) {
  DiaArg<T, UC, C> d;
  for (int q = 0; q < UC; q++) {
    d.off[q] = q < D.ndiag ? D.off[q] : 0;
    d.c[q] = q < D.ndiag ? (C)D.c[q] : (C)0;
  }
  d.qd = D.qd;
  d.dg = std::is_same<T, double>::value ? (const T *)D.dg64 : (const T *)D.dg32;
  return d;
}

// f(std::integral_constant<int, UC>) for the diagonal count's kernel
// (dia_slots).
template <class F>
void dia_dispatch(const DevDia &D, F &&f) {
  switch (dia_slots(D.ndiag)) {
#define CASE(UC)                           \
  case UC:                                 \
    f(std::integral_constant<int, UC>{});  \
    break;
    CASE(3) CASE(5) CASE(7) CASE(8) CASE(9) CASE(13) CASE(19) CASE(27) CASE(kMaxDiags)
#undef CASE
  }
}

}  // namespace

void dia_spmv_f64(const DevCsr &A, const double *X, double *Y, int ncol, size_t ld,
                  hipStream_t s) {
  dia_dispatch(A.dia, [&](auto uc) {
    constexpr int UC = decltype(uc)::value;
    hipLaunchKernelGGL((k_dia_spmv<UC>), dim3(grid_for((size_t)A.n), ncol), dim3(kThreads), 0, s,
                       A.n, dia_arg<double, UC>(A.dia), (const DiaMask<UC> *)A.dia.mask, X, Y, ld);
  });
}

template <typename T>
void dia_cheb_step(const DevCsr &A, const T *vk, const T *vkm1, T *vkp1, T *y, double cc,
                   double t, double mu0, double mu3, double mu2, double mu1, int ymode,
                   hipStream_t s) {
  dia_dispatch(A.dia, [&](auto uc) {
    constexpr int UC = decltype(uc)::value;
    hipLaunchKernelGGL((k_cheb_dia<T, UC>), dim3(grid_for((size_t)A.n)), dim3(kThreads), 0, s,
                       A.n, dia_arg<T, UC>(A.dia), (const DiaMask<UC> *)A.dia.mask, vk, vkm1,
                       vkp1, y, (T)cc, (T)t, (T)mu0, (T)mu3, (T)mu2, (T)mu1, ymode);
  });
}
template void dia_cheb_step<double>(const DevCsr &, const double *, const double *, double *,
                                    double *, double, double, double, double, double, double,
                                    int, hipStream_t);
template void dia_cheb_step<float>(const DevCsr &, const float *, const float *, float *, float *,
                                   double, double, double, double, double, double, int,
                                   hipStream_t);

namespace {
// k_dia_blk of width B with epilogue `epi`
template <typename T, int B, class Epi>
void dia_blk_launch(const DevCsr &A, const T *x, const Epi &epi, hipStream_t s) {
  dia_dispatch(A.dia, [&](auto uc) {
    constexpr int UC = decltype(uc)::value;
    hipLaunchKernelGGL((k_dia_blk<T, B, UC, Epi>),
                       dim3(grid_for((size_t)A.n * Pieces<T, B>::Q)), dim3(kThreads), 0, s, A.n,
                       dia_arg<T, UC>(A.dia), (const DiaMask<UC> *)A.dia.mask, x, epi);
  });
}

// f(std::integral_constant<int, B>) for the block width
template <class F>
void width_dispatch(int B, F &&f) {
  switch (B) {
#define CASE(BB)                              \
  case BB:                                    \
    f(std::integral_constant<int, BB>{});     \
    break;
    CASE(1) CASE(2) CASE(4) CASE(8) CASE(16) CASE(32)
#undef CASE
    default:
      break;
  }
}
}  // namespace

template <typename T>
void dia_cheb_blk(const DevCsr &A, int B, const T *vk, const T *vkm1, T *vkp1, T *y, double cc,
                  double t, const double *mus, int k, int nact, hipStream_t s, int ymode) {
  width_dispatch(B, [&](auto b) {
    constexpr int BB = decltype(b)::value;
    dia_blk_launch<T, BB>(
        A, vk, EpiCheb<T, BB>{vk, vkm1, vkp1, y, (T)cc, (T)t, mus, k, nact, ymode}, s);
  });
}
template <typename T>
void dia_clen_blk(const DevCsr &A, int B, const T *b1, const T *b2, const T *v, T *out, double cc,
                  double t, const double *mus, int k, hipStream_t s) {
  width_dispatch(B, [&](auto b) {
    constexpr int BB = decltype(b)::value;
    dia_blk_launch<T, BB>(A, b1, EpiClen<T, BB>{b1, b2, v, out, (T)cc, (T)t, mus, k}, s);
  });
}
template void dia_cheb_blk<double>(const DevCsr &, int, const double *, const double *, double *,
                                   double *, double, double, const double *, int, int, hipStream_t,
                                   int);
template void dia_cheb_blk<float>(const DevCsr &, int, const float *, const float *, float *,
                                  float *, double, double, const double *, int, int, hipStream_t,
                                  int);
template void dia_clen_blk<double>(const DevCsr &, int, const double *, const double *,
                                   const double *, double *, double, double, const double *, int,
                                   hipStream_t);
template void dia_clen_blk<float>(const DevCsr &, int, const float *, const float *,
                                  const float *, float *, double, double, const double *, int,
                                  hipStream_t);

// Degrees per launch s and rows per workgroup R of k_cheb_multi for a filter of
// degree m; s = 1 where one launch per degree is at least as good.  Model in
// microseconds, fitted to the times of s = 2 .. 32 on the grids at
// k_cheb_multi: a launch costs 4.5 and 0.8e-3 per row of the window it loads; a
// degree inside it 0.2, and 0.35e-3 (U + 3)/10 per row it steps for U diagonals,
// for each round of workgroups over the CUs; one launch per degree costs 3.0 +
// 5.6e-6 n.  The window must fit kMultiRows, 64 KiB of LDS (of the CU's 160:
// the kernel packs its neighbours' byte offsets in 16 bits), and as one of
// contiguous rows it grows by the whole band per degree, which ends the gain
// where the band is wide (30^3: 900 rows either side per degree) or the grid
// large.
MultiPlan dia_multi_plan(const DevCsr &A, int elem, int m) {
  MultiPlan best;
  if (!use_dia(A, elem, 1) || m < 2 || A.n > (1 << 20) || A.dia.ndiag > 8) return best;
  int bw = 0;
  for (int q = 0; q < A.dia.ndiag; q++) bw = std::max(bw, std::abs(A.dia.off[q]));
  const double row = 0.35e-3 * (A.dia.ndiag + 3) / 10.0;
  double tbest = 3.0 + 5.6e-6 * A.n;
  for (int per = 1; per <= 8; per *= 2) {
    const int R = std::max(64, (A.n + 256 * per - 1) / (256 * per));
    const int wgs = (A.n + R - 1) / R;
    for (int s = 2; s <= std::min(m, kMultiMax); s++) {
      const long long L = (long long)R + 2LL * s * bw;
      if (L > kMultiRows) break;
      const double t = (4.5 + 0.8e-3 * (double)L) / s +
                       ((wgs + 255) / 256) * (0.2 + row * (R + (double)bw * (s - 1)));
      if (t < tbest) {
        tbest = t;
        best.s = s;
        best.R = R;
        best.bw = bw;
      }
    }
  }
  // equal launches
  if (best.s > 1) best.s = (m + (m + best.s - 1) / best.s - 1) / ((m + best.s - 1) / best.s);
  return best;
}

template <typename T>
void dia_cheb_multi(const DevCsr &A, const MultiPlan &p, const T *v, const T *vm, T *vout,
                    T *vmout, T *y, double cc, double dd, const double *mu, int d0, int s,
                    bool last, hipStream_t st) {
  MuArg<T> ma;
  ma.m0 = (T)mu[0];
  for (int j = 0; j < kMultiMax; j++) ma.mu[j] = j < s ? (T)mu[d0 + j] : (T)0;
  const int L = p.R + 2 * s * p.bw;
  const int nt = std::min(1024, (L + 63) / 64 * 64);
  const int K = (L + nt - 1) / nt;
  auto go = [&](auto uc, auto k) {
    constexpr int UC = decltype(uc)::value, KK = decltype(k)::value;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((A.n + p.R - 1) / p.R), dim3(nt),
                         (size_t)(kMultiRows + 8 + L + 1) * sizeof(T), st, A.n,
                         dia_arg<T, UC>(A.dia), (const DiaMask<UC> *)A.dia.mask, p.bw, p.R, d0, s,
                         last ? 1 : 0, v, vm, vout, vmout, y, (T)cc, (T)(1.0 / dd), (T)(2.0 / dd),
                         ma);
    };
    if (A.dia.qd >= 0)
      launch(k_cheb_multi<T, UC, KK, true>);
    else
      launch(k_cheb_multi<T, UC, KK, false>);
  };
  auto width = [&](auto uc) {
    if (K <= 1)
      go(uc, std::integral_constant<int, 1>{});
    else if (K <= 2)
      go(uc, std::integral_constant<int, 2>{});
    else
      go(uc, std::integral_constant<int, 4>{});
  };
  dia_dispatch(A.dia, [&](auto uc) {
    if constexpr (decltype(uc)::value <= 8) width(uc);
  });
}
template void dia_cheb_multi<double>(const DevCsr &, const MultiPlan &, const double *,
                                     const double *, double *, double *, double *, double, double,
                                     const double *, int, int, bool, hipStream_t);
template void dia_cheb_multi<float>(const DevCsr &, const MultiPlan &, const float *,
                                    const float *, float *, float *, float *, double, double,
                                    const double *, int, int, bool, hipStream_t);

template <typename T>
ChebRun cheb_run(const DevCsr &A, const MultiPlan &p, const double *mu, int m, double cc, double dd,
                 const T *x, T *y, T *w, hipStream_t st) {
  const int n = A.n;
  const double vec = (double)n * sizeof(T);
  const double mat = matrix_bytes(A, sizeof(T), index_bytes(A), use_dia(A, sizeof(T), 1));
  const T *vk = x, *vkm1 = nullptr;
  ChebRun run;
  if (p.s > 1) {
    int set = 0;
    for (int d = 1; d <= m; d += p.s, set ^= 1) {
      const int s = std::min(p.s, m + 1 - d);
      T *vo = w + (size_t)2 * set * n, *vmo = vo + n;
      dia_cheb_multi<T>(A, p, vk, vkm1, vo, vmo, y, cc, dd, mu, d, s, d + s > m, st);
      vk = vo;
      vkm1 = vmo;
      run.bytes += mat + (d == 1 ? 2.0 : 4.0) * vec + (d + s > m ? 0.0 : 2.0) * vec;
      run.launches++;
    }
    return run;
  }
  T *b[3] = {w, w + n, w + 2 * (size_t)n};
  YPlan yp;
  for (int k = 1; k <= m; k++) {
    T *vkp1 = b[(k - 1) % 3];
    const int ymode = yp.next(k, m);
    cheb_step_stream<T>(A, vk, vkm1, vkp1, y, cc, k == 1 ? 1.0 / dd : 2.0 / dd, mu[0],
                        k > 2 ? mu[k - 2] : 0.0, mu[k - 1], mu[k], ymode, st);
    vkm1 = vk;
    vk = vkp1;
    run.bytes += mat + ((k == 1 ? 2 : 3) + y_passes(ymode)) * vec;
    run.launches++;
  }
  return run;
}
template ChebRun cheb_run<double>(const DevCsr &, const MultiPlan &, const double *, int, double,
                                  double, const double *, double *, double *, hipStream_t);
template ChebRun cheb_run<float>(const DevCsr &, const MultiPlan &, const double *, int, double,
                                 double, const float *, float *, float *, hipStream_t);

// runs of kThreads (row, piece) items per workgroup: as many as leave about
// kKpmBlocks workgroups (four per CU).  100^3 FP32, 64 vectors: 512 29.5 ms,
// 768 26.0, 1024 25.3, 2048 28.3, 4096 29.2; FP64, 32 vectors: 21.0, 20.5, 23.6,
// 27.4, 27.7; 48x40x44 and 300^2: 1024 the best or within 3%
constexpr int kKpmBlocks = 1024;
static int dia_kpm_iters(int n, int elem, int B) {
  const long long items = (long long)n * std::max(1, B * elem / 16);
  return (int)((items + (long long)kThreads * kKpmBlocks - 1) / ((long long)kThreads * kKpmBlocks));
}
int dia_kpm_blocks(int n, int elem, int B) {
  const long long items = (long long)n * std::max(1, B * elem / 16);
  const long long per = (long long)kThreads * dia_kpm_iters(n, elem, B);
  return (int)((items + per - 1) / per);
}

template <typename T>
void dia_kpm_step(const DevCsr &A, int B, int ng, const T *v, T *vw, double ctr, double scal,
                  bool first, double *part, hipStream_t s) {
  width_dispatch(B, [&](auto b) {
    constexpr int BB = decltype(b)::value;
    dia_dispatch(A.dia, [&](auto uc) {
      constexpr int UC = decltype(uc)::value;
      auto go = [&](auto fi) {
        hipLaunchKernelGGL((k_dia_kpm<T, BB, UC, decltype(fi)::value>),
                           dim3(dia_kpm_blocks(A.n, sizeof(T), BB), ng), dim3(kThreads), 0, s, A.n,
                           dia_arg<T, UC, double>(A.dia), (const DiaMask<UC> *)A.dia.mask,
                           EpiKpm<T, BB, double>{v, vw, nullptr, ctr, scal, 0},
                           (size_t)A.n * BB, dia_kpm_iters(A.n, sizeof(T), BB), ng * BB, part);
      };
      if (first)
        go(std::true_type{});
      else
        go(std::false_type{});
    });
  });
}
template void dia_kpm_step<double>(const DevCsr &, int, int, const double *, double *, double,
                                   double, bool, double *, hipStream_t);
template void dia_kpm_step<float>(const DevCsr &, int, int, const float *, float *, double, double,
                                  bool, double *, hipStream_t);

}  // namespace pevsl
