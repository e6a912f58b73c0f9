// dev.hpp -- device-side helpers shared by the kernel files (kernels.hip,
// dia.hip): launch constants, the XCD-aware block order, 16-byte pieces of
// interleaved rows and the update of the filter's accumulator.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "kernels.hpp"

namespace pevsl {

constexpr int kThreads = 256;

inline int grid_for(size_t work, int threads = kThreads) {
  return (int)((work + threads - 1) / threads);
}

// Row-block index of this workgroup such that each XCD works on one
// contiguous range of row blocks.  Workgroups are dispatched to the 8 XCDs
// round-robin (workgroup i to XCD i mod 8), and each XCD has its own L2: with
// contiguous ranges the neighbour rows that a stencil-like matrix gathers
// (+-1, +-nx, +-nx*ny) mostly sit in the same L2.  A bijection of [0, nb).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int bid, int nb) {
  const int q = nb / kXcds, r = nb % kXcds;
  const int x = bid % kXcds, j = bid / kXcds;
  return x * q + min(x, r) + j;
}

// number of row blocks of XCD x; its first is xcd_block(x, nb)
__device__ __forceinline__ int xcd_count(int x, int nb) {
  return nb / kXcds + (x < nb % kXcds ? 1 : 0);
}

// B-wide rows of an interleaved block cut into Q pieces of P columns (16
// bytes where the row has that much).
//
// Budget of the balanced kernels: NZ = kStreamNnz / Q staged products of B
// values (32 KiB of LDS when a piece is 16 bytes) and at most kStreamRows / Q
// rows per block; the host builds one row partition per Q (DevCsr::rowblk_q).
template <typename T, int B>
struct Pieces {
  static constexpr int P = (B * (int)sizeof(T) >= 16) ? 16 / (int)sizeof(T) : B;
  static constexpr int Q = B / P;
  static constexpr int NZ = kStreamNnz / Q;
};

template <typename T, int P>
__device__ __forceinline__ void ld_piece(const T *p, T (&x)[P]) {
  if constexpr (P * sizeof(T) == 16) {
    *reinterpret_cast<float4 *>(x) = *reinterpret_cast<const float4 *>(p);
  } else if constexpr (P * sizeof(T) == 8) {
    *reinterpret_cast<float2 *>(x) = *reinterpret_cast<const float2 *>(p);
  } else {
#pragma unroll
    for (int e = 0; e < P; e++) x[e] = p[e];
  }
}
template <typename T, int P>
__device__ __forceinline__ void st_piece(T *p, const T (&x)[P]) {
  if constexpr (P * sizeof(T) == 16) {
    *reinterpret_cast<float4 *>(p) = *reinterpret_cast<const float4 *>(x);
  } else if constexpr (P * sizeof(T) == 8) {
    *reinterpret_cast<float2 *>(p) = *reinterpret_cast<const float2 *>(x);
  } else {
#pragma unroll
    for (int e = 0; e < P; e++) p[e] = x[e];
  }
}

// y after a degree step with update mode `mode` (kernels.hpp): yv its old
// value (not read with kYInit), vm, v, w the vectors of degrees d-2, d-1, d
// and m3, m2, m1 their coefficients, m0 that of degree 0.  Each term is
// rounded and added on its own, in degree order, as one update per degree
// adds them.
template <typename T>
__device__ __forceinline__ T y_next(int mode, T yv, T vm, T v, T w, T m0, T m3, T m2, T m1) {
#pragma clang fp contract(off)
  const int terms = mode & 3;
  if (mode & kYInit) yv = (terms == 1 ? v : vm) * m0;
  if (terms == 3) yv = yv + m3 * vm;
  if (terms >= 2) yv = yv + m2 * v;
  return yv + m1 * w;
}

// y_next of column c of an interleaved block: coefficients mus[d*B + c]
template <typename T>
__device__ __forceinline__ T y_col(int ymode, const double *mus, int k, int B, int c, T yv, T vm,
                                   T v, T w) {
  const int terms = ymode & 3;
  const T m0 = (ymode & kYInit) ? (T)mus[c] : (T)0;
  const T m3 = terms == 3 ? (T)mus[(size_t)(k - 2) * B + c] : (T)0;
  const T m2 = terms >= 2 ? (T)mus[(size_t)(k - 1) * B + c] : (T)0;
  return y_next<T>(ymode, yv, vm, v, w, m0, m3, m2, (T)mus[(size_t)k * B + c]);
}

// Epilogues of the block steps on piece `piece` (columns piece*P ..) of row r:
// load() reads the row's own operands (before the row sum where the kernel can,
// so that their latency overlaps its loads), finish() applies the recurrence
// to the row sum acc and stores.

// three-term step (same operations as k_cheb_blkrow)
template <typename T, int B>
struct EpiCheb {
  const T *vk, *vkm1;
  T *vkp1, *y;
  T cc, t;
  const double *mus;
  int k, nact, ymode;
  static constexpr int P = Pieces<T, B>::P;
  struct Ops {
    T v[P], vm[P], yy[P];
  };
  __device__ __forceinline__ void load(int r, int piece, Ops &o) const {
    const size_t at = (size_t)r * B + piece * P;
    ld_piece<T, P>(vk + at, o.v);
    // with kYInit, columns >= nact still keep y
    if (ymode != kYSkip) ld_piece<T, P>(y + at, o.yy);
    if (vkm1) {
      ld_piece<T, P>(vkm1 + at, o.vm);
    } else {
#pragma unroll
      for (int e = 0; e < P; e++) o.vm[e] = 0;
    }
  }
  __device__ __forceinline__ void finish(int r, int piece, Ops &o, const T (&acc)[P]) const {
#pragma clang fp contract(off)
    const size_t at = (size_t)r * B + piece * P;
    T w[P];
#pragma unroll
    for (int e = 0; e < P; e++) {
      w[e] = acc[e] + (-cc) * o.v[e];
      w[e] = w[e] * t;
      if (vkm1) w[e] = w[e] + (T)(-1) * o.vm[e];
    }
    if (ymode != kYSkip) {
#pragma unroll
      for (int e = 0; e < P; e++) {
        const int c = piece * P + e;
        if (c < nact) o.yy[e] = y_col<T>(ymode, mus, k, B, c, o.yy[e], o.vm[e], o.v[e], w[e]);
      }
      st_piece<T, P>(y + at, o.yy);
    }
    st_piece<T, P>(vkp1 + at, w);
  }
};

// Clenshaw step (same operations as k_clen_blkrow); b1 is the gathered block
template <typename T, int B>
struct EpiClen {
  const T *b1, *b2, *v;
  T *out;
  T cc, t;
  const double *mus;
  int k;
  static constexpr int P = Pieces<T, B>::P;
  struct Ops {
    T bb[P], vv[P], b2r[P], mu[P];
  };
  __device__ __forceinline__ void load(int r, int piece, Ops &o) const {
    const size_t at = (size_t)r * B + piece * P;
    ld_piece<T, P>(b1 + at, o.bb);
    ld_piece<T, P>(v + at, o.vv);
    if (b2) {
      ld_piece<T, P>(b2 + at, o.b2r);
    } else {
#pragma unroll
      for (int e = 0; e < P; e++) o.b2r[e] = 0;
    }
#pragma unroll
    for (int e = 0; e < P; e++) o.mu[e] = (T)mus[(size_t)k * B + piece * P + e];
  }
  __device__ __forceinline__ void finish(int r, int piece, Ops &o, const T (&acc)[P]) const {
#pragma clang fp contract(off)
    T w[P];
#pragma unroll
    for (int e = 0; e < P; e++) {
      T z = acc[e] + (-cc) * o.bb[e];
      z = z * t;
      z = z + o.mu[e] * o.vv[e];
      w[e] = z + (T)(-1) * o.b2r[e];
    }
    st_piece<T, P>(out + (size_t)r * B + piece * P, w);
  }
};

// ---- KPM step --------------------------------------------------------------
// Sums of one thread over its rows' piece of P columns, in FP64: s[0] = w.w,
// s[1] = w.v and (first step) s[2] = v.v for the step v -> w; or, with the
// start vectors v0 given, s[0] = w.v0 alone.
template <int P>
struct KpmSums {
  double s[3][P];
  __device__ __forceinline__ KpmSums() {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int e = 0; e < P; e++) s[i][e] = 0.0;
  }
};

// The step on piece pc of row r: w = scal (acc - ctr v) - vm, written over vm
// (vw; vm is zero, and not read, on the first step), and its sums.  acc, ctr
// and scal are of type AT: with AT = double on FP32 vectors the step rounds to
// FP32 once, where it stores w.
template <typename T, int B, typename AT>
struct EpiKpm {
  const T *v;
  T *vw;
  const T *v0;
  AT ctr, scal;
  int first;
  static constexpr int P = Pieces<T, B>::P;
  struct Ops {
    T v[P], vm[P], z[P];
  };
  __device__ __forceinline__ void load(int r, int pc, Ops &o) const {
    const size_t at = (size_t)r * B + pc * P;
    ld_piece<T, P>(v + at, o.v);
    if (v0) ld_piece<T, P>(v0 + at, o.z);
    if (!first) {
      ld_piece<T, P>(vw + at, o.vm);
    } else {
#pragma unroll
      for (int e = 0; e < P; e++) o.vm[e] = 0;
    }
  }
  __device__ __forceinline__ void finish(int r, int pc, const Ops &o, const AT (&acc)[P],
                                         KpmSums<P> &s) const {
    T w[P];
#pragma unroll
    for (int e = 0; e < P; e++) {
      const AT x = __builtin_elementwise_fma(-ctr, (AT)o.v[e], acc[e]);
      w[e] = (T)__builtin_elementwise_fma(scal, x, -(AT)o.vm[e]);
      const double we = w[e], ve = o.v[e];
      if (v0) {
        s.s[0][e] = __builtin_fma(we, (double)o.z[e], s.s[0][e]);
      } else {
        s.s[0][e] = __builtin_fma(we, we, s.s[0][e]);
        s.s[1][e] = __builtin_fma(we, ve, s.s[1][e]);
        if (first) s.s[2][e] = __builtin_fma(ve, ve, s.s[2][e]);
      }
    }
    st_piece<T, P>(vw + (size_t)r * B + pc * P, w);
  }
  // sums a launch writes per column
  __device__ __forceinline__ int nsum() const { return v0 ? 1 : first ? 3 : 2; }
  // group `g` of vectors, gstride elements apart
  __device__ __forceinline__ void group(int g, size_t gstride) {
    v += g * gstride;
    vw += g * gstride;
    if (v0) v0 += g * gstride;
  }
};

// Block sums of the threads' KpmSums (thread t holds piece t % Q) in a fixed
// order: lanes of a wave that hold the same piece, then the waves.  Sum i <
// nsum of column c goes to part[(i*ncol + c) * nblk + blk].
template <typename T, int B>
__device__ __forceinline__ void kpm_block_sums(const KpmSums<Pieces<T, B>::P> &s, int nsum,
                                               int ncol, int nblk, int blk, double *part) {
  constexpr int P = Pieces<T, B>::P, Q = Pieces<T, B>::Q, W = kThreads / 64;
  __shared__ double red[3][W][B];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, pc = threadIdx.x % Q;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    if (i >= nsum) break;
#pragma unroll
    for (int e = 0; e < P; e++) {
      double x = s.s[i][e];
#pragma unroll
      for (int off = 32; off >= Q; off >>= 1) x += __shfl_xor(x, off, 64);
      if (lane < Q) red[i][wave][pc * P + e] = x;
    }
  }
  __syncthreads();
  for (int u = threadIdx.x; u < nsum * B; u += kThreads) {
    const int i = u / B, c = u % B;
    double x = 0.0;
#pragma unroll
    for (int w = 0; w < W; w++) x += red[i][w][c];
    part[((size_t)i * ncol + c) * nblk + blk] = x;
  }
}

}  // namespace pevsl
