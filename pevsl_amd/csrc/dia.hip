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
  constexpr int CH = UC < 8 ? UC : 8;
#pragma unroll
  for (int q0 = 0; q0 < UC; q0 += CH) {
    T xv[CH];
#pragma unroll
    for (int q = 0; q < CH; q++)
      xv[q] = ld32(x, (m >> (q0 + q)) & 1 ? (uint32_t)(r + d.off[q0 + q]) : 0u);
#pragma unroll
    for (int q = 0; q < CH; q++) {
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
//   100^3 Laplacian, FP64  19.96 -> 8.36 (30 MB: 3.6 TB/s)   FP32 15.8 -> 5.1
//   113x97x83 with a potential, FP32  15.3 -> 5.0
//   60^3, FP64  6.6 -> 3.8      20^3, FP64  5.4 -> 2.7
// Two and four rows per thread were no faster at 1e6 rows (8.29 and 8.93) and
// slower below (60^3: 4.1 and 4.6): one row gives the most waves.
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

// sum of row r times piece pc (columns pc*P ..) of the interleaved block x,
// in type C
template <typename T, int B, int UC, typename C = T>
__device__ __forceinline__ void dia_row_piece(const DiaArg<T, UC, C> &d, uint32_t m, T dgv, int r,
                                              int pc, const T *__restrict__ x,
                                              C (&acc)[Pieces<T, B>::P]) {
#pragma clang fp contract(off)
  constexpr int P = Pieces<T, B>::P;
  constexpr int CH = UC < 8 ? UC : 8;
#pragma unroll
  for (int e = 0; e < P; e++) acc[e] = 0;
#pragma unroll
  for (int q0 = 0; q0 < UC; q0 += CH) {
    T xv[CH][P];
#pragma unroll
    for (int q = 0; q < CH; q++) {
      const uint32_t row = (m >> (q0 + q)) & 1 ? (uint32_t)(r + d.off[q0 + q]) : 0u;
      const uint32_t at = (row * (uint32_t)B + (uint32_t)(pc * P)) * (uint32_t)sizeof(T);
      ld_piece<T, P>(reinterpret_cast<const T *>(reinterpret_cast<const char *>(x) + at), xv[q]);
    }
#pragma unroll
    for (int q = 0; q < CH; q++) {
      const C a = q0 + q == d.qd ? (C)dgv : d.c[q0 + q];
      const bool on = (m >> (q0 + q)) & 1;
#pragma unroll
      for (int e = 0; e < P; e++) {
        const C s = acc[e] + a * (C)xv[q][e];
        acc[e] = on ? s : acc[e];
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
//   100^3, FP32 Clenshaw    B=4 19.1 -> 11.0  8: 28.9 -> 19.0  16: 77.7 -> 33.8
//   100^3, FP64 three-term  B=4 38.0 -> 18.4  8: 91.3 -> 32.8
//   48x40x44, FP32 Clenshaw B=8 5.9 -> 3.7    20^3, FP32 B=8 5.2 -> 2.9
// (100^3, B=8 FP32: 129 MB, 6.8 TB/s, served by the Infinity Cache.)
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
  dia_row_piece<T, B, UC>(d, m, dgv, r, pc, x, acc);
  epi.finish(r, pc, ops, acc);
}

// One KPM step on B interleaved columns, group blockIdx.y: each workgroup
// takes `iters` runs of kThreads (row, piece) items, so that its sums end in
// one reduction and one set of partials.  Bound by the three vector passes
// (u_j, u_j-1 read, u_j+1 over it).  Whole pEVSL_Kpmdos, against one thread per
// (row, column) and one product per moment: 100^3, Mdeg 300, 64 FP32 vectors
// 263 -> 33.6 ms (600 launches of 192 MB: 3.4 TB/s); 20^3, 60 FP64 vectors 8.8
// -> 3.5 ms, of which 2.5 ms are the rand() stream on the host.
template <typename T, int B, int UC>
__global__ void __launch_bounds__(kThreads)
k_dia_kpm(int n, DiaArg<T, UC, double> d, const DiaMask<UC> *__restrict__ mask,
          EpiKpm<T, B, double> epi, size_t gstride, int iters, int ncol,
          double *__restrict__ part) {
  constexpr uint32_t Q = Pieces<T, B>::Q;
  constexpr int P = Pieces<T, B>::P;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  epi.group(blockIdx.y, gstride);
  KpmSums<P> sums;
  for (int it = 0; it < iters; it++) {
    const uint32_t g = ((uint32_t)blk * iters + it) * kThreads + threadIdx.x;
    const int r = (int)(g / Q), pc = (int)(g % Q);
    if (r >= n) break;
    const uint32_t m = mask[r];
    const T dgv = d.qd >= 0 ? d.dg[r] : (T)0;
    typename EpiKpm<T, B, double>::Ops ops;
    epi.load(r, pc, ops);
    double acc[P];
    dia_row_piece<T, B, UC, double>(d, m, dgv, r, pc, epi.v, acc);
    epi.finish(r, pc, ops, acc, sums);
  }
  kpm_block_sums<T, B>(sums, epi.nsum(), ncol, gridDim.x, blk,
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
template <class F>
void dia_dispatch(const DevDia &D, F &&f) {
  if (D.ndiag <= 4)
    f(std::integral_constant<int, 4>{});
  else if (D.ndiag <= 8)
    f(std::integral_constant<int, 8>{});
  else
    f(std::integral_constant<int, kMaxDiags>{});
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

// runs of kThreads (row, piece) items per workgroup: as many as leave about
// kKpmBlocks workgroups (eight per CU)
constexpr int kKpmBlocks = 2048;
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
void dia_kpm_step(const DevCsr &A, int B, int ng, const T *v, T *vw, const T *v0, double ctr,
                  double scal, bool first, double *part, hipStream_t s) {
  width_dispatch(B, [&](auto b) {
    constexpr int BB = decltype(b)::value;
    dia_dispatch(A.dia, [&](auto uc) {
      constexpr int UC = decltype(uc)::value;
      hipLaunchKernelGGL((k_dia_kpm<T, BB, UC>),
                         dim3(dia_kpm_blocks(A.n, sizeof(T), BB), ng), dim3(kThreads), 0, s, A.n,
                         dia_arg<T, UC, double>(A.dia), (const DiaMask<UC> *)A.dia.mask,
                         EpiKpm<T, BB, double>{v, vw, v0, ctr, scal, first ? 1 : 0},
                         (size_t)A.n * BB, dia_kpm_iters(A.n, sizeof(T), BB), ng * BB, part);
    });
  });
}
template void dia_kpm_step<double>(const DevCsr &, int, int, const double *, double *,
                                   const double *, double, double, bool, double *, hipStream_t);
template void dia_kpm_step<float>(const DevCsr &, int, int, const float *, float *, const float *,
                                  double, double, bool, double *, hipStream_t);

}  // namespace pevsl
