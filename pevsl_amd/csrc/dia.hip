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

#include <type_traits>

namespace pevsl {

namespace {

// Diagonals as kernel arguments (scalar registers); entries past ndiag have
// no mask bit.
template <typename T, int UC>
struct DiaArg {
  int off[UC];
  T c[UC];
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

template <typename T, int UC>
DiaArg<T, UC> dia_arg(const DevDia &D) {
  DiaArg<T, UC> d;
  for (int q = 0; q < UC; q++) {
    d.off[q] = q < D.ndiag ? D.off[q] : 0;
    d.c[q] = q < D.ndiag ? (T)D.c[q] : (T)0;
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

}  // namespace pevsl
