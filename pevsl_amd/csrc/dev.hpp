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

}  // namespace pevsl
