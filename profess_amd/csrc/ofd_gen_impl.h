// Register-resident two-stage FFT passes in FP64 for every grid length that
// PadFFTdims can pad to: the products of 2, 3, 5 and 7 from 16 to 256 along y
// and z, and n1/2 from 9 to 128, and 256, along x (SetupFFT.f90:275-380). Rows of 16
// points stay on the staged passes, which serve the 16^3 grids of the
// reference's sample runs: the solves compared with those runs follow
// recurrences of some 200 steps that carry a last-bit difference along, and
// at 16^3 an evaluation is launches, not transforms.
//
// A line of N = R1*R2 points belongs to T threads. Thread t holds the stage-1
// columns c = t + T j (j < J1, c < R2), the points c + R2 m, and after the
// forward transform the stage-2 rows k1 = t + T q (q < J2, k1 < R1), the
// outputs k1 + R1 k2. Forward is decimation in time (columns to rows), the
// inverse decimation in frequency (rows to columns), so what stands between
// them works on registers and nothing is reordered.
//
// Against the staged LDS transform these passes replace for such lengths
// (ping-pong buffers, one radix per stage, run-time divisions): each element
// crosses LDS once per transform instead of once per radix plus a staging
// copy on either side, and half to a quarter of the LDS per line leaves more
// workgroups per CU. A Wang-Teter evaluation, staged passes / these: 72^3
// 75.7 / 47.3 us, 100^3 145 / 74, 144^3 368 / 157, 200^3 951 / 463, 240^3
// 1701 / 906; second-order WGC 100^3 284 / 153, 160^3 1171 / 672.
#pragma once
#include "ofd_fast_impl.h"

namespace ofd {
namespace gen {

using fast::kPi;
constexpr int kPlain = 9;   // one real field, no functional (per-geometry tables)

// X(N, R1, R2, T): R1 and R2 as even as the factors allow and T dividing what
// it can, so that few lanes idle in either stage; at most 16 points a thread
// where a split allows it (64 VGPRs of data). Short lines take more threads
// than they need for that: a small grid has few lines.
#define OFD_GEN_SHORT(X) X(9, 3, 3, 3) X(10, 2, 5, 2) X(12, 3, 4, 3) X(14, 2, 7, 2) X(15, 3, 5, 3)
#define OFD_GEN_A(X)                                                                                             \
  X(16, 4, 4, 4) X(18, 3, 6, 3) X(20, 4, 5, 5) X(21, 3, 7, 3) X(24, 4, 6, 6) X(25, 5, 5, 5) X(27, 3, 9, 3)        \
  X(28, 4, 7, 4) X(30, 5, 6, 6) X(32, 4, 8, 4) X(35, 5, 7, 7) X(36, 6, 6, 6) X(40, 5, 8, 5) X(42, 6, 7, 7)        \
  X(45, 5, 9, 5) X(48, 6, 8, 8) X(49, 7, 7, 7) X(50, 5, 10, 5)
#define OFD_GEN_B(X)                                                                                             \
  X(54, 6, 9, 9) X(56, 7, 8, 8) X(60, 4, 15, 4) X(63, 7, 9, 9) X(64, 8, 8, 8) X(70, 7, 10, 7) X(72, 8, 9, 9)      \
  X(75, 5, 15, 5) X(80, 8, 10, 10) X(81, 9, 9, 9) X(84, 7, 12, 7) X(90, 9, 10, 10) X(96, 8, 12, 8)                \
  X(98, 7, 14, 7) X(100, 10, 10, 10)
#define OFD_GEN_C(X)                                                                                             \
  X(105, 7, 15, 8) X(108, 9, 12, 12) X(112, 8, 14, 8) X(120, 8, 15, 8) X(125, 5, 25, 5) X(126, 9, 14, 14)         \
  X(128, 8, 16, 8)
#define OFD_GEN_D(X)                                                                                             \
  X(135, 9, 15, 15) X(140, 10, 14, 14) X(144, 12, 12, 12) X(147, 7, 21, 7) X(150, 10, 15, 15) X(160, 10, 16, 16)  \
  X(162, 9, 18, 9) X(168, 12, 14, 14) X(175, 7, 25, 7) X(180, 12, 15, 15) X(189, 7, 27, 7) X(192, 12, 16, 16)
#define OFD_GEN_E(X)                                                                                             \
  X(196, 14, 14, 14) X(200, 10, 20, 10) X(210, 14, 15, 15) X(216, 12, 18, 18) X(224, 14, 16, 16)                  \
  X(225, 15, 15, 15) X(240, 15, 16, 16) X(243, 9, 27, 9) X(245, 7, 35, 7) X(250, 10, 25, 13) X(252, 14, 18, 18)   \
  X(256, 16, 16, 16)
#define OFD_GEN_COLS(X) OFD_GEN_A(X) OFD_GEN_B(X) OFD_GEN_C(X) OFD_GEN_D(X) OFD_GEN_E(X)
#define OFD_GEN_ROWS_LO(X) OFD_GEN_SHORT(X) OFD_GEN_A(X)
#define OFD_GEN_ROWS_HI(X) OFD_GEN_B(X) OFD_GEN_C(X) X(256, 16, 16, 16)
#define OFD_GEN_ROWS(X) OFD_GEN_ROWS_LO(X) OFD_GEN_ROWS_HI(X)

template <int N> struct Split;
#define X(N, A, B, T_) \
  template <> struct Split<N> { static constexpr int R1 = A, R2 = B, T = T_; };
OFD_GEN_SHORT(X)
OFD_GEN_COLS(X)
#undef X

template <int N> struct L {
  static constexpr int R1 = Split<N>::R1, R2 = Split<N>::R2, T = Split<N>::T;
  static constexpr int J1 = (R2 + T - 1) / T, J2 = (R1 + T - 1) / T;
  static constexpr int LDR = R1 | 1;
  static constexpr int LINE = (R2 * LDR > N ? R2 * LDR : N + 1) | 1;   // elements per line block (>= N + 1), odd
  static constexpr int NC = J1 * R1, NS = J2 * R2;
  static constexpr bool allc = J1 * T == R2, allr = J2 * T == R1;
  static_assert(R1 * R2 == N, "two factors");
  __device__ static bool col_ok(int t, int j) { return allc || t + T * j < R2; }
  __device__ static bool row_ok(int t, int q) { return allr || t + T * q < R1; }
};

// Forward, columns xc to rows xs, through a complex line block: two barriers.
template <int N, typename C>
__device__ __forceinline__ void fwd_c(C (&xc)[L<N>::NC], C (&xs)[L<N>::NS], C* __restrict__ lds, int t,
                                      const C* __restrict__ tw, bool active) {
  using G = L<N>;
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
      const int c = t + G::T * j;
      Bfly<G::R1, -1, C>::run(&xc[j * G::R1]);
#pragma unroll
      for (int m = 0; m < G::R1; ++m) lds[c * G::LDR + m] = xc[j * G::R1 + m];
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
      const int k1 = t + G::T * q;
      C* y = &xs[q * G::R2];
#pragma unroll
      for (int c = 0; c < G::R2; ++c) y[c] = lds[c * G::LDR + k1];
#pragma unroll
      for (int c = 1; c < G::R2; ++c) y[c] = cmul(y[c], tw[c * k1]);
      Bfly<G::R2, -1, C>::run(y);
    }
  }
  __syncthreads();
}

// Inverse, rows xs to columns xc.
template <int N, typename C>
__device__ __forceinline__ void inv_c(C (&xs)[L<N>::NS], C (&xc)[L<N>::NC], C* __restrict__ lds, int t,
                                      const C* __restrict__ tw, bool active) {
  using G = L<N>;
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
      const int k1 = t + G::T * q;
      C* y = &xs[q * G::R2];
      Bfly<G::R2, +1, C>::run(y);
      lds[k1] = y[0];
#pragma unroll
      for (int c = 1; c < G::R2; ++c) {
        C w = tw[c * k1];
        w.y = -w.y;
        lds[c * G::LDR + k1] = cmul(y[c], w);
      }
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
      const int c = t + G::T * j;
#pragma unroll
      for (int k1 = 0; k1 < G::R1; ++k1) xc[j * G::R1 + k1] = lds[c * G::LDR + k1];
      Bfly<G::R1, +1, C>::run(&xc[j * G::R1]);
    }
  }
  __syncthreads();
}

// The same two transforms with the exchange done one real component at a time
// through a line of LINE reals (half the LDS, two more barriers): the column
// passes, whose workgroups per CU are bound by LDS.
template <int N>
__device__ __forceinline__ void fwd_s(double2 (&xc)[L<N>::NC], double2 (&xs)[L<N>::NS], double* __restrict__ lds,
                                      int t, const double2* __restrict__ tw, bool active) {
  using G = L<N>;
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
      Bfly<G::R1, -1, double2>::run(&xc[j * G::R1]);
#pragma unroll
      for (int m = 0; m < G::R1; ++m) lds[(t + G::T * j) * G::LDR + m] = xc[j * G::R1 + m].x;
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
#pragma unroll
      for (int c = 0; c < G::R2; ++c) xs[q * G::R2 + c].x = lds[c * G::LDR + t + G::T * q];
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
#pragma unroll
      for (int m = 0; m < G::R1; ++m) lds[(t + G::T * j) * G::LDR + m] = xc[j * G::R1 + m].y;
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
      const int k1 = t + G::T * q;
      double2* y = &xs[q * G::R2];
#pragma unroll
      for (int c = 0; c < G::R2; ++c) y[c].y = lds[c * G::LDR + k1];
#pragma unroll
      for (int c = 1; c < G::R2; ++c) y[c] = cmul(y[c], tw[c * k1]);
      Bfly<G::R2, -1, double2>::run(y);
    }
  }
  __syncthreads();
}

template <int N>
__device__ __forceinline__ void inv_s(double2 (&xs)[L<N>::NS], double2 (&xc)[L<N>::NC], double* __restrict__ lds,
                                      int t, const double2* __restrict__ tw, bool active) {
  using G = L<N>;
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
      const int k1 = t + G::T * q;
      double2* y = &xs[q * G::R2];
      Bfly<G::R2, +1, double2>::run(y);
#pragma unroll
      for (int c = 1; c < G::R2; ++c) {
        double2 w = tw[c * k1];
        w.y = -w.y;
        y[c] = cmul(y[c], w);
      }
#pragma unroll
      for (int c = 0; c < G::R2; ++c) lds[c * G::LDR + k1] = y[c].x;
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
#pragma unroll
      for (int k1 = 0; k1 < G::R1; ++k1) xc[j * G::R1 + k1].x = lds[(t + G::T * j) * G::LDR + k1];
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
#pragma unroll
      for (int c = 0; c < G::R2; ++c) lds[c * G::LDR + t + G::T * q] = xs[q * G::R2 + c].y;
    }
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
#pragma unroll
      for (int k1 = 0; k1 < G::R1; ++k1) xc[j * G::R1 + k1].y = lds[(t + G::T * j) * G::LDR + k1];
      Bfly<G::R1, +1, double2>::run(&xc[j * G::R1]);
    }
  }
  __syncthreads();
}

// The twiddle pointer, hidden from the optimizer and tied to a thread's last
// result so far: the loads of the transform that follows are issued after it.
// Left alone they are hoisted over the G-space operator, up to 4 (R2 - 1)
// more VGPRs alive with the line's data (k_zgop<128>: 218 VGPRs, two waves per
// SIMD).
__device__ __forceinline__ const double2* again(const double2* p, double done) {
  asm volatile("" : "+s"(p) : "v"(done));
  return p;
}

// ------------------------------------------------------------ columns
// A set of equal columns of one field: column e starts at
// (e / inner) * outer + e % inner and its points are `es` apart. y: inner =
// K1, outer = n2 K1, es = K1; z: inner = n2 K1 (one group), es = n2 K1.
struct Cols {
  unsigned ncol, inner, outer, es;
};

// Element access by 32-bit byte offset from a workgroup-uniform base (the
// largest field served here, 512 x 256 x 256, takes 2^28 bytes and a plane):
// scalar base and one offset register per element. offs() hides an offset from the optimizer
// where a kernel uses it again, so that the elements' offsets are formed anew
// (one add each) instead of staying alive through the transforms.
static_assert((256ull + 1) * 256 * 256 * sizeof(double2) < 1ull << 32, "offsets within a field");
__device__ __forceinline__ double2 ld16(gptr<const double2> b, unsigned off) {
  return ldc((gptr<const double2>)((gptr<const char>)b + off));
}
__device__ __forceinline__ double ld8(gptr<const double> b, unsigned off) {
  return *(gptr<const double>)((gptr<const char>)b + off);
}
__device__ __forceinline__ void st16(gptr<double2> b, unsigned off, const double2& v) {
  stc((gptr<double2>)((gptr<char>)b + off), v);
}
__device__ __forceinline__ unsigned offs(unsigned o) {
  asm volatile("" : "+v"(o));
  return o;
}

// Elements c + R2 m of a thread's stage-1 columns, or k1 + R1 k2 of its
// stage-2 rows; o: byte offset of the line, es: bytes between its points.
template <int N> __device__ __forceinline__ void load_cols(double2 (&xc)[L<N>::NC], gptr<const double2> b, unsigned o,
                                                           unsigned es, int t) {
  using G = L<N>;
#pragma unroll
  for (int j = 0; j < G::J1; ++j)
    if (G::col_ok(t, j)) {
#pragma unroll
      for (int m = 0; m < G::R1; ++m) xc[j * G::R1 + m] = ld16(b, o + (unsigned)t * es + (unsigned)(G::T * j + G::R2 * m) * es);
    }
}
template <int N> __device__ __forceinline__ void store_cols(const double2 (&xc)[L<N>::NC], gptr<double2> b, unsigned o,
                                                            unsigned es, int t) {
  using G = L<N>;
#pragma unroll
  for (int j = 0; j < G::J1; ++j)
    if (G::col_ok(t, j)) {
#pragma unroll
      for (int m = 0; m < G::R1; ++m) st16(b, o + (unsigned)t * es + (unsigned)(G::T * j + G::R2 * m) * es, xc[j * G::R1 + m]);
    }
}
template <int N> __device__ __forceinline__ void load_rows(double2 (&xs)[L<N>::NS], gptr<const double2> b, unsigned o,
                                                           unsigned es, int t) {
  using G = L<N>;
#pragma unroll
  for (int q = 0; q < G::J2; ++q)
    if (G::row_ok(t, q)) {
#pragma unroll
      for (int k = 0; k < G::R2; ++k) xs[q * G::R2 + k] = ld16(b, o + (unsigned)t * es + (unsigned)(G::T * q + G::R1 * k) * es);
    }
}
template <int N> __device__ __forceinline__ void store_rows(const double2 (&xs)[L<N>::NS], gptr<double2> b, unsigned o,
                                                            unsigned es, int t) {
  using G = L<N>;
#pragma unroll
  for (int q = 0; q < G::J2; ++q)
    if (G::row_ok(t, q)) {
#pragma unroll
      for (int k = 0; k < G::R2; ++k) st16(b, o + (unsigned)t * es + (unsigned)(G::T * q + G::R1 * k) * es, xs[q * G::R2 + k]);
    }
}

// In-place transform of the columns of field blockIdx.y.
template <int N, int S>
__global__ void __launch_bounds__(256) k_cols(const ReqDesc* __restrict__ descs, long long nc, Cols cs,
                                              const double2* __restrict__ tw, int kb) {
  using G = L<N>;
  extern __shared__ __align__(16) unsigned char smem[];
  const ReqDesc& D = descs[blockIdx.z];
  const int c = threadIdx.x % kb, t = threadIdx.x / kb;
  const unsigned col = (unsigned)xcd_block(blockIdx.x, gridDim.x) * kb + c;
  const bool active = t < G::T && col < cs.ncol;
  const unsigned grp = active ? col / cs.inner : 0;
  const unsigned o = active ? (grp * cs.outer + (col - grp * cs.inner)) * 16u : 0, es = cs.es * 16u;
  gptr<double2> base = glb(reinterpret_cast<double2*>(D.work)) + (size_t)blockIdx.y * nc;
  double* line = reinterpret_cast<double*>(smem) + (size_t)c * G::LINE;
  double2 xc[G::NC], xs[G::NS];
  if constexpr (S < 0) {
    if (active) load_cols<N>(xc, base, o, es, t);
    fwd_s<N>(xc, xs, line, t, tw, active);
    if (active) store_rows<N>(xs, base, o, es, t);
  } else {
    if (active) load_rows<N>(xs, base, o, es, t);
    inv_s<N>(xs, xc, line, t, tw, active);
    if (active) store_cols<N>(xc, base, o, es, t);
  }
}

// |G|^2 along a z column at (m1, m2): a0 + m3 (a1 + m3 a2)
struct G2Col {
  double a0, a1, a2;
  __device__ __forceinline__ G2Col(const ReqDesc& D, int m1, int m2) {
    const double gx = D.rb[0] * m1 + D.rb[1] * m2, gy = D.rb[3] * m1 + D.rb[4] * m2, gz = D.rb[6] * m1 + D.rb[7] * m2;
    a0 = gx * gx + gy * gy + gz * gz;
    a1 = 2.0 * (gx * D.rb[2] + gy * D.rb[5] + gz * D.rb[8]);
    a2 = D.rb[2] * D.rb[2] + D.rb[5] * D.rb[5] + D.rb[8] * D.rb[8];
  }
  __device__ __forceinline__ double at(int m3) const {
    const double m = (double)m3;
    return fma(m, fma(m, a2, a1), a0);
  }
};

// z columns with the diagonal G-space operator: field 0 Hartree 4 pi / G^2,
// fields from fvw on G^2 (vW), the others the Wang-Teter kernel table.
template <int N>
__global__ void __launch_bounds__(256) k_zgop(const ReqDesc* __restrict__ descs, GridDims d,
                                              const double2* __restrict__ tw, int kb, int fvw) {
  using G = L<N>;
  extern __shared__ __align__(16) unsigned char smem[];
  const ReqDesc& D = descs[blockIdx.z];
  const int f = blockIdx.y;
  const int c = threadIdx.x % kb, t = threadIdx.x / kb;
  const unsigned col = (unsigned)xcd_block(blockIdx.x, gridDim.x) * kb + c;
  const unsigned es = (unsigned)(d.n2 * d.K1);
  const bool active = t < G::T && col < es;
  const int i2 = active ? (int)(col / d.K1) : 0, m1 = active ? (int)col - i2 * d.K1 : 0;
  const int m2 = i2 > d.n2 / 2 ? i2 - d.n2 : i2;
  const double invn = 1.0 / (double)d.nr;
  gptr<double2> base = glb(reinterpret_cast<double2*>(D.work)) + (size_t)f * d.nc;
  double* line = reinterpret_cast<double*>(smem) + (size_t)c * G::LINE;
  // the inverse writes an array of its own: lanes that skip the branches would
  // keep xc's old contents alive through the whole pass otherwise
  double2 xc[G::NC], xs[G::NS], yc[G::NC];
  if (active) load_cols<N>(xc, base, col * 16u, es * 16u, t);
  fwd_s<N>(xc, xs, line, t, tw, active);
  if (active) {
    if (f != 0 && f < fvw) {
      gptr<const double> wk = glb(D.wtk);
      const unsigned ow = (col + (unsigned)t * es) * 8u;
#pragma unroll
      for (int q = 0; q < G::J2; ++q)
        if (G::row_ok(t, q)) {
#pragma unroll
          for (int k = 0; k < G::R2; ++k) {
            const double s = ld8(wk, ow + (unsigned)(G::T * q + G::R1 * k) * (es * 8u));
            xs[q * G::R2 + k].x *= s;
            xs[q * G::R2 + k].y *= s;
          }
        }
    } else {
      const G2Col g2(D, m1, m2);
      const double ch = 4.0 * kPi * invn;
#pragma unroll
      for (int q = 0; q < G::J2; ++q)
        if (G::row_ok(t, q)) {
#pragma unroll
          for (int k = 0; k < G::R2; ++k) {
            const int i3 = t + G::T * q + G::R1 * k;
            const double q2 = g2.at(i3 > N / 2 ? i3 - N : i3);
            const double s = f == 0 ? (q2 > 0.0 ? ch / q2 : 0.0) : q2 * invn;
            xs[q * G::R2 + k].x *= s;
            xs[q * G::R2 + k].y *= s;
          }
        }
    }
  }
  inv_s<N>(xs, yc, line, t, again(tw, xs[G::NS - 1].y), active);
  if (active) store_cols<N>(yc, base, offs(col * 16u), es * 16u, t);
}

// z columns of the WGC fields with the coupled operator, as fast::k_fz_wgc:
// blockIdx.y = 0 Hartree and vW, 1 and 2 the rho^alpha and rho^beta blocks
// (A, B, C), which leave (c', b', a') = (K3 A, K2 A + K4 B, K1 A + K2 B +
// K3 C) in the slots of (A, B, C). Bound by the line's three arrays in
// registers: 170 to 252 VGPRs and two waves per SIMD from 84 points on. At 128,
// 160, 162, 192, 224, 240, 252 and 256 points it takes 2 to 10 registers more,
// at 200 and with radices of 21 and more 36 to 234, and runs one wave. So it
// does at 256^3, in 755 us; the two-column form before it took 825 with two.
template <int N>
__global__ void __launch_bounds__(256) k_zwgc(const ReqDesc* __restrict__ descs, GridDims d,
                                              const double2* __restrict__ tw, int kb) {
  using G = L<N>;
  extern __shared__ __align__(16) unsigned char smem[];
  const ReqDesc& D = descs[blockIdx.z];
  const int g = blockIdx.y;
  const int f0 = g == 0 ? 0 : 3 * g - 1;
  const int c = threadIdx.x % kb, t = threadIdx.x / kb;
  const unsigned col = (unsigned)xcd_block(blockIdx.x, gridDim.x) * kb + c;
  const unsigned es = (unsigned)(d.n2 * d.K1);
  const bool active = t < G::T && col < es;
  const double invn = 1.0 / (double)d.nr;
  gptr<double2> base = glb(reinterpret_cast<double2*>(D.work)) + (size_t)f0 * d.nc;
  double* line = reinterpret_cast<double*>(smem) + (size_t)c * G::LINE;
  // every transform between arrays of its own (see k_zgop)
  auto get = [&](int j, double2 (&xs)[G::NS]) {
    double2 xc[G::NC];
    if (active) load_cols<N>(xc, base + (size_t)j * d.nc, offs(col * 16u), es * 16u, t);
    fwd_s<N>(xc, xs, line, t, again(tw, xc[G::NC - 1].y), active);
  };
  auto put = [&](int j, double2 (&xs)[G::NS]) {
    double2 xc[G::NC];
    inv_s<N>(xs, xc, line, t, again(tw, xs[G::NS - 1].y), active);
    if (active) store_cols<N>(xc, base + (size_t)j * d.nc, offs(col * 16u), es * 16u, t);
  };
  // each(fn): fn(slot, i3) for every point the thread holds
  auto each = [&](auto&& fn) {
    if (!active) return;
#pragma unroll
    for (int q = 0; q < G::J2; ++q)
      if (G::row_ok(t, q)) {
#pragma unroll
        for (int k = 0; k < G::R2; ++k) fn(q * G::R2 + k, t + G::T * q + G::R1 * k);
      }
  };
  if (g == 0) {
    const int i2 = active ? (int)(col / d.K1) : 0, m1 = active ? (int)col - i2 * d.K1 : 0;
    const G2Col g2(D, m1, i2 > d.n2 / 2 ? i2 - d.n2 : i2);
    for (int j = 0; j < 2; ++j) {
      double2 xs[G::NS];
      get(j, xs);
      each([&](int s, int i3) {
        const double q2 = g2.at(i3 > N / 2 ? i3 - N : i3);
        const double sc = j == 0 ? (q2 > 0.0 ? 4.0 * kPi / q2 * invn : 0.0) : q2 * invn;
        xs[s].x *= sc;
        xs[s].y *= sc;
      });
      put(j, xs);
    }
    return;
  }
  gptr<const double> wk = glb(D.wgck);
  double2 xa[G::NS], xb[G::NS];
  get(0, xa);
  {
    double2 xs[G::NS];
    each([&](int s, int i3) {
      const double k3 = ld8(wk + 2 * d.nc, (col + (unsigned)i3 * es) * 8u) * invn;
      xs[s].x = k3 * xa[s].x;
      xs[s].y = k3 * xa[s].y;
    });
    put(0, xs);
  }
  {
    double2 xs[G::NS];
    get(1, xs);
    each([&](int s, int i3) {
      const unsigned gi = (col + (unsigned)i3 * es) * 8u;
      const double k1 = ld8(wk, gi) * invn, k2 = ld8(wk + d.nc, gi) * invn, k4 = ld8(wk + 3 * d.nc, gi) * invn;
      const double2 a = xa[s], b = xs[s];
      xb[s].x = k1 * a.x + k2 * b.x;
      xb[s].y = k1 * a.y + k2 * b.y;
      xs[s].x = k2 * a.x + k4 * b.x;
      xs[s].y = k2 * a.y + k4 * b.y;
    });
    put(1, xs);
  }
  double2 xs[G::NS];
  get(2, xs);
  each([&](int s, int i3) {
    const double k3 = ld8(wk + 2 * d.nc, (col + (unsigned)i3 * es) * 8u) * invn;
    xs[s].x = xb[s].x + k3 * xs[s].x;
    xs[s].y = xb[s].y + k3 * xs[s].y;
  });
  put(2, xs);
}

// ------------------------------------------------------------ x rows
template <int KIND> struct NFg { static constexpr int v = fast::NF_<KIND>::v; };
template <> struct NFg<kPlain> { static constexpr int v = 1; };

// Rows per workgroup: whole rows of NF lines, at most 48 KB of lines (`bytes`
// each), the count that leaves the fewest lanes idle within 128 threads (64 for
// the short rows of small grids, which have few workgroups to fill the chip
// with), or within 256 where 128 would leave one lane in eight idle. (256
// throughout: 200^3 WT inverse 92 against 83 us, 100^3 15.8 against 14.2.)
constexpr int row_rpb(int m, int nf, int t, int bytes) {
  int best = 1;
  double eff = 0.0;
  for (int cap = m <= 24 ? 64 : 128; cap <= 256 && eff < 0.875; cap *= 2)
    for (int r = 1; r == 1 || r * nf * t <= cap; ++r) {
      if (r > 1 && (long long)r * nf * bytes > 49152) break;
      const int th = r * nf * t, up = (th + 63) / 64 * 64;
      const double e = (double)th / up;
      if (e >= eff) {
        eff = e;
        best = r;
      }
    }
  return best;
}
// The inverse pass. Rows with 15 points and more per thread (60, 112, 120, 128)
// exchange one real component at a time and run their epilogue over the two
// halves of each row in turn (columns m < R1/2 of every thread are the row's
// first M reals): at 16 points a thread complex lines leave 9 waves per CU
// (256^3 WT 263 -> 244 us for the pass, 120 x 125 x 240 54.3 -> 53.8). With
// fewer points a thread the complex lines are faster (200^3 92 against 99 us).
// The power-of-two form that this pass replaced at 256^3 took 232 us for WT
// with eight rows on 192 lanes (here five on 120 of 128) and 453 for WGC (here
// 437); the call gained more before it than it lost there (1055 -> 980 us).
template <int M> struct InvLine {
  static constexpr bool SC = L<M>::R1 % 2 == 0 && std::max(L<M>::NC, L<M>::NS) >= 15;
  static constexpr int LINE = L<M>::LINE;   // reals (SC) or complex
  static constexpr int BYTES = LINE * (SC ? 8 : 16);
};
template <int M, int KIND> struct RowGeo {
  static constexpr int NF = NFg<KIND>::v, T = L<M>::T;
  static constexpr int RPB = row_rpb(M, NF, T, InvLine<M>::BYTES);
  static constexpr int NL = RPB * NF;                          // lines per workgroup, field-major
  static constexpr int NT = (NL * T + 63) / 64 * 64;           // threads
  static constexpr size_t LDS = (size_t)NL * InvLine<M>::BYTES;
};
// The forward pass: one wave per field with as many rows as it has lanes for,
// so that no wave forms two kinds of field (a divergent wave pays for each);
// the short rows of small grids pack their lines densely instead, for more
// workgroups. Rows of 60 points and more (WGC 36) exchange one real component
// at a time (half the LDS, twice the waves per CU: 256^3 WT 294 -> 212 us for
// the pass, 200^3 89 -> 75, 108^3 WGC 36.4 -> 32.0); below that the complex
// exchange is 5 % faster.
template <int M, int KIND> struct RowGeoF {
  static constexpr int NF = NFg<KIND>::v, T = L<M>::T, LINE = L<M>::LINE;
  static constexpr bool SC = M >= (KIND == kWGC8 ? 36 : 60), WF = M > 24;
  static constexpr int RPB = WF ? 64 / T : row_rpb(M, NF, T, 16 * LINE);
  static constexpr int NL = RPB * NF;
  static constexpr int NT = WF ? NF * 64 : (NL * T + 63) / 64 * 64;
  static constexpr size_t LDS = std::max((size_t)NL * LINE * (SC ? 1 : 2), KIND == kWGC8 ? (size_t)RPB * 4 * M : (size_t)0) *
                                sizeof(double);   // the lines; before them WGC's two powers of each point
};

// Rows along x, forward: every line forms its field from rho, transforms it
// and leaves it in LDS; then the workgroup's threads write the R2C split of
// all lines, consecutive threads on consecutive k (whole cache lines, where a
// line's own T threads would write T elements at a time).
template <int M, int KIND>
__global__ void __launch_bounds__((RowGeoF<M, KIND>::NT)) k_rows_fwd(const ReqDesc* __restrict__ descs, GridDims d,
                                                  const double2* __restrict__ tw, const double2* __restrict__ tws,
                                                  int inmode) {
  using G = L<M>;
  using W = RowGeoF<M, KIND>;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = reinterpret_cast<double*>(smem);
  const ReqDesc& D = descs[blockIdx.y];
  const int lane = W::WF ? threadIdx.x % 64 : threadIdx.x;
  const int t = lane % G::T;
  int f, r;
  if constexpr (W::WF) {
    f = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    r = lane / G::T;
  } else {
    f = lane / G::T / W::RPB;
    r = lane / G::T - f * W::RPB;
  }
  const int line = f * W::RPB + r;
  const long long nrows = (long long)d.n2 * d.n3;
  const long long row0 = (long long)xcd_block(blockIdx.x, gridDim.x) * W::RPB;
  const bool active = f < W::NF && r < W::RPB && row0 + r < nrows;
  double2 xc[G::NC], xs[G::NS];
  if constexpr (KIND == kWGC8) {
    // each point's two powers once per row, shared through LDS
    double* pw = lds;
    const int nrow = (int)min((long long)W::RPB, nrows - row0);
    for (int e = threadIdx.x; e < nrow * 2 * M; e += W::NT) {
      const size_t g = (size_t)row0 * (2 * M) + e;
      double rho = glb(D.u)[g];
      if (inmode == kInPhi) {
        double tp = D.ca * rho;
        if (D.cb != 0.0) tp = fma(D.cb, (double)glb(D.v)[g], tp);
        rho = tp * tp;
      }
      const double l2 = log2(rho);
      pw[e] = exp2(D.alpha * l2);
      pw[W::RPB * 2 * M + e] = exp2(D.beta * l2);
    }
    __syncthreads();
    if (active) {
      const double* mypw = pw + (f < 5 ? 0 : W::RPB * 2 * M) + r * 2 * M;
      const int kk = (f - 2) % 3;
      const size_t base = (size_t)(row0 + r) * (2 * M);
#pragma unroll
      for (int j = 0; j < G::J1; ++j) {
        if (!G::col_ok(t, j)) continue;
#pragma unroll
        for (int m = 0; m < G::R1; ++m) {
          const int i = 2 * (t + G::T * j + G::R2 * m);
          double rho[2], v[2];
          if (inmode == kInRho) fast::rho_pair<kInRho>(D.u, D.v, D.ca, D.cb, base + i, rho[0], rho[1]);
          else fast::rho_pair<kInPhi>(D.u, D.v, D.ca, D.cb, base + i, rho[0], rho[1]);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (f == 0) {
              v[h] = rho[h];
            } else if (f == 1) {
              v[h] = sqrt(rho[h]);
            } else {
              const double p = mypw[i + h], th = rho[h] - D.rhoS;
              v[h] = kk == 0 ? p : (kk == 1 ? th * p : th * th * p / 2.0);
            }
          }
          xc[j * G::R1 + m] = make_double2(v[0], v[1]);
        }
      }
    }
    __syncthreads();
  } else if (active) {
    const size_t base = (size_t)(row0 + r) * (2 * M);
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
#pragma unroll
      for (int m = 0; m < G::R1; ++m) {
        const size_t g = base + 2 * (t + G::T * j + G::R2 * m);
        double2 z;
        if constexpr (KIND == kPlain) z = ldc(glb(reinterpret_cast<const double2*>(D.u + g)));
        else if (inmode == kInRho) z = fast::field_pair<KIND, kInRho, double>(D, f, g);
        else z = fast::field_pair<KIND, kInPhi, double>(D, f, g);
        xc[j * G::R1 + m] = z;
      }
    }
  }
  // The split X[k] = E[k] + W^k O[k] of Z reads Z[k] and Z[M-k]; an element's
  // place and factor are the same for every field.
  constexpr int PER = (W::RPB * (M + 1) + W::NT - 1) / W::NT;
  const int nel = (int)min((long long)W::RPB, nrows - row0) * (M + 1);
  gptr<double2> work = glb(reinterpret_cast<double2*>(D.work));
  auto natural = [&](auto* mine, auto&& part) {
    if (active) {
#pragma unroll
      for (int q = 0; q < G::J2; ++q)
        if (G::row_ok(t, q)) {
#pragma unroll
          for (int k2 = 0; k2 < G::R2; ++k2) mine[t + G::T * q + G::R1 * k2] = part(xs[q * G::R2 + k2]);
        }
    }
    __syncthreads();
  };
  if constexpr (W::SC) {
    // real parts through LDS first (giving Re E and Im O), then the imaginary parts
    double* mine = lds + (size_t)line * G::LINE;
    fwd_s<M>(xc, xs, mine, t, tw, active);
    double er[PER][W::NF], oi[PER][W::NF];
    natural(mine, [](const double2& z) { return z.x; });
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = min((int)threadIdx.x + q * W::NT, nel - 1);
      const int rr = e / (M + 1), k = e - rr * (M + 1);
      const double* z = lds + (size_t)rr * G::LINE;
#pragma unroll
      for (int ff = 0; ff < W::NF; ++ff) {
        const double zk = z[ff * W::RPB * G::LINE + (k == M ? 0 : k)],
                     zm = z[ff * W::RPB * G::LINE + (k == 0 ? 0 : M - k)];
        er[q][ff] = 0.5 * (zk + zm);
        oi[q][ff] = -0.5 * (zk - zm);
      }
    }
    __syncthreads();
    natural(mine, [](const double2& z) { return z.y; });
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = threadIdx.x + q * W::NT;
      if (e >= nel) break;
      const int rr = e / (M + 1), k = e - rr * (M + 1);
      const double2 w = tws[k];
      const double* z = lds + (size_t)rr * G::LINE;
      gptr<double2> out = work + ((size_t)row0 * (M + 1) + e);
#pragma unroll
      for (int ff = 0; ff < W::NF; ++ff) {
        const double zk = z[ff * W::RPB * G::LINE + (k == M ? 0 : k)],
                     zm = z[ff * W::RPB * G::LINE + (k == 0 ? 0 : M - k)];
        const double ei = 0.5 * (zk - zm), orr = 0.5 * (zk + zm);
        double2 x;
        x.x = er[q][ff] + (w.x * orr - w.y * oi[q][ff]);
        x.y = ei + (w.x * oi[q][ff] + w.y * orr);
        stc(out + (size_t)ff * d.nc, x);
      }
    }
  } else {
    double2* all = reinterpret_cast<double2*>(smem);
    double2* mine = all + (size_t)line * G::LINE;
    fwd_c<M>(xc, xs, mine, t, tw, active);
    natural(mine, [](const double2& z) { return z; });
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = threadIdx.x + q * W::NT;
      if (e >= nel) break;
      const int rr = e / (M + 1), k = e - rr * (M + 1);
      const double2 w = tws[k];
      const double2* z = all + (size_t)rr * G::LINE;
      gptr<double2> out = work + ((size_t)row0 * (M + 1) + e);
#pragma unroll
      for (int ff = 0; ff < W::NF; ++ff) {
        const double2 zk = z[ff * W::RPB * G::LINE + (k == M ? 0 : k)], zm = z[ff * W::RPB * G::LINE + (k == 0 ? 0 : M - k)];
        const double er = 0.5 * (zk.x + zm.x), ei = 0.5 * (zk.y - zm.y);
        const double orr = 0.5 * (zk.y + zm.y), oi = -0.5 * (zk.x - zm.x);
        double2 x;
        x.x = er + (w.x * orr - w.y * oi);
        x.y = ei + (w.x * oi + w.y * orr);
        stc(out + (size_t)ff * d.nc, x);
      }
    }
  }
}

// Rows along x, inverse: the workgroup's half rows are read with consecutive
// threads on consecutive k into LDS, merged (C2R) and transformed line by
// line, and the epilogue runs over the rows' points. INMODE / OUTMODE as
// fast::x_epi_points; OUTMODE = -1 takes the form from `outmode` (phi inputs).
template <int M, int KIND, int INMODE, int OUTMODE>
__global__ void __launch_bounds__(256) k_rows_inv(const ReqDesc* __restrict__ descs, GridDims d,
                                                  const double2* __restrict__ tw, const double2* __restrict__ tws,
                                                  int outmode) {
  using G = L<M>;
  using W = RowGeo<M, KIND>;
  using Q = InvLine<M>;
  extern __shared__ __align__(16) unsigned char smem[];
  const ReqDesc& D = descs[blockIdx.y];
  const int line = threadIdx.x / G::T, t = threadIdx.x % G::T;
  const int f = line / W::RPB, r = line - f * W::RPB;
  const long long nrows = (long long)d.n2 * d.n3;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const long long row0 = (long long)blk * W::RPB;
  const int nrow = (int)min((long long)W::RPB, nrows - row0);
  const bool active = line < W::NL && r < nrow;
  gptr<const double2> work = glb(reinterpret_cast<const double2*>(D.work));
  // all of a thread's loads in flight together (past the workgroup's last
  // element it reads that one again), then the LDS writes
  constexpr int PER = (W::RPB * (M + 1) + W::NT - 1) / W::NT;
  const int nel = nrow * (M + 1);
  double2 v[W::NF][PER];
#pragma unroll
  for (int ff = 0; ff < W::NF; ++ff) {
    gptr<const double2> in = work + (size_t)ff * d.nc + (size_t)row0 * (M + 1);
#pragma unroll
    for (int q = 0; q < PER; ++q) v[ff][q] = ldc(in + min((int)threadIdx.x + q * W::NT, nel - 1));
  }
  // merge of X[k] and X[M-k] (C2R; the imaginary parts of X[0] and X[M] drop)
  auto merge = [&](int k, double er, double dr, double ei, double di) {
    const double2 w = tws[k];
    const double orr = w.x * dr + w.y * di, oi = w.x * di - w.y * dr;
    return make_double2(er - oi, ei + orr);
  };
  double2 xc[G::NC], xs[G::NS];
  // natural(part): the loaded element's part to its place in its line
  auto natural = [&](auto* all, auto&& part) {
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = threadIdx.x + q * W::NT;
      if (e < nel) {
        const int rr = e / (M + 1), k = e - rr * (M + 1);
#pragma unroll
        for (int ff = 0; ff < W::NF; ++ff) all[(size_t)(ff * W::RPB + rr) * Q::LINE + k] = part(v[ff][q]);
      }
    }
    __syncthreads();
  };
  // each(fn): fn(slot, k) for the elements of the thread's rows
  auto each = [&](auto&& fn) {
    if (!active) return;
#pragma unroll
    for (int q = 0; q < G::J2; ++q)
      if (G::row_ok(t, q)) {
#pragma unroll
        for (int k2 = 0; k2 < G::R2; ++k2) fn(q * G::R2 + k2, t + G::T * q + G::R1 * k2);
      }
  };
  double acc[kNSum];
#pragma unroll
  for (int k = 0; k < kNSum; ++k) acc[k] = 0.0;
  if constexpr (Q::SC) {
    double* all = reinterpret_cast<double*>(smem);
    double* mine = all + (size_t)line * Q::LINE;
    double er[G::NS], dr[G::NS];
    natural(all, [](const double2& z) { return z.x; });
    each([&](int s, int k) {
      const double a = mine[k], b = mine[M - k];
      er[s] = a + b;
      dr[s] = a - b;
    });
    __syncthreads();
    natural(all, [](const double2& z) { return z.y; });
    each([&](int s, int k) {
      const double a = k == 0 ? 0.0 : mine[k], b = k == 0 ? 0.0 : mine[M - k];
      xs[s] = merge(k, er[s], dr[s], a - b, a + b);
    });
    __syncthreads();
    inv_s<M>(xs, xc, mine, t, tw, active);
    constexpr int H1 = G::R1 / 2;
    auto half = [&](auto h) {
      constexpr int H = decltype(h)::value;
      if (H) __syncthreads();   // the first half's points are read
      if (active) {
#pragma unroll
        for (int j = 0; j < G::J1; ++j)
          if (G::col_ok(t, j)) {
#pragma unroll
            for (int m = 0; m < H1; ++m) {
              const int i = 2 * (t + G::T * j + G::R2 * m);
              mine[i] = xc[j * G::R1 + m + H * H1].x;
              mine[i + 1] = xc[j * G::R1 + m + H * H1].y;
            }
          }
      }
      if constexpr (KIND == kPlain) {
        __syncthreads();
        for (int e = threadIdx.x; e < nrow * M; e += W::NT) {
          const int rr = e / M, i = e - rr * M;
          glb(D.out)[(size_t)(row0 + rr) * (2 * M) + H * M + i] = all[(size_t)rr * Q::LINE + i];
        }
      } else {
        fast::x_epi_points<M, KIND, INMODE, OUTMODE, W::RPB, W::NT, Q::LINE, M, true>(D, all, row0, nrows, H * M, acc,
                                                                                      outmode);
      }
    };
    half(std::integral_constant<int, 0>());
    half(std::integral_constant<int, 1>());
  } else {
    double2* all = reinterpret_cast<double2*>(smem);
    double2* mine = all + (size_t)line * Q::LINE;
    natural(all, [](const double2& z) { return z; });
    each([&](int s, int k) {
      double2 xk = mine[k], xm = mine[M - k];
      if (k == 0) { xk.y = 0.0; xm.y = 0.0; }
      xs[s] = merge(k, xk.x + xm.x, xk.x - xm.x, xk.y - xm.y, xk.y + xm.y);
    });
    __syncthreads();
    inv_c<M>(xs, xc, mine, t, tw, active);
    if (active) {
#pragma unroll
      for (int j = 0; j < G::J1; ++j)
        if (G::col_ok(t, j)) {
#pragma unroll
          for (int m = 0; m < G::R1; ++m) mine[t + G::T * j + G::R2 * m] = xc[j * G::R1 + m];
        }
    }
    if constexpr (KIND == kPlain) {
      __syncthreads();
      gptr<double2> out = glb(reinterpret_cast<double2*>(D.out)) + (size_t)row0 * M;
      for (int e = threadIdx.x; e < nrow * M; e += W::NT) {
        const int rr = e / M, k = e - rr * M;
        stc(out + e, all[(size_t)rr * Q::LINE + k]);
      }
    } else {
      fast::x_epi_points<M, KIND, INMODE, OUTMODE, W::RPB, W::NT, 2 * Q::LINE, 2 * M, true>(
          D, reinterpret_cast<const double*>(all), row0, nrows, 0, acc, outmode);
    }
  }
  if constexpr (KIND != kPlain) fast::x_epi_sums<OUTMODE>(D, acc, blk);
}

// ------------------------------------------------------------ launchers (one translation unit per group)
// Columns per workgroup: up to 256 threads and 40 KB of scalar lines (four
// workgroups per CU), fewer where the launch would otherwise have under 1024
// workgroups, never below one wave.
template <int N> static int cols_kb(int tuned, long long ncol, int nf_nb) {
  constexpr int T = L<N>::T, lb = L<N>::LINE * 8;
  const int most = std::min(256 / T, std::max(1, 65536 / lb)), least = std::min(most, std::max(1, 64 / T));
  if (tuned > 0) return std::max(least, std::min(tuned, most));
  const int kb = std::min(most, std::max(least, 40960 / lb));
  return (int)std::max<long long>(least, std::min<long long>(kb, ncol * nf_nb / 1024));
}
static inline unsigned cdiv(long long a, int b) { return (unsigned)((a + b - 1) / b); }

template <int N>
static void launch_cols(int S, const ReqDesc* dd, long long nc, const Cols& cs, int nf, int nb, int tuned,
                        const double2* tw, hipStream_t st) {
  const int kb = cols_kb<N>(tuned, cs.ncol, nf * nb);
  const dim3 grid(cdiv(cs.ncol, kb), nf, nb), block((kb * L<N>::T + 63) / 64 * 64);
  const size_t lds = (size_t)kb * L<N>::LINE * sizeof(double);
  if (S < 0) hipLaunchKernelGGL((k_cols<N, -1>), grid, block, lds, st, dd, nc, cs, tw, kb);
  else hipLaunchKernelGGL((k_cols<N, +1>), grid, block, lds, st, dd, nc, cs, tw, kb);
}
template <int N>
static void launch_z(int kind, const ReqDesc* dd, const GridDims& d, int nb, int tuned, const double2* tw,
                     hipStream_t st) {
  const long long ncol = (long long)d.K1 * d.n2;
  const int nf = kind == kWGC8 ? 3 : func_nf(kind);
  const int kb = cols_kb<N>(tuned, ncol, nf * nb);
  const dim3 grid(cdiv(ncol, kb), nf, nb), block((kb * L<N>::T + 63) / 64 * 64);
  const size_t lds = (size_t)kb * L<N>::LINE * sizeof(double);
  if (kind == kWGC8) hipLaunchKernelGGL((k_zwgc<N>), grid, block, lds, st, dd, d, tw, kb);
  else
    hipLaunchKernelGGL((k_zgop<N>), grid, block, lds, st, dd, d, tw, kb, is_spin_kind(kind) ? nf - 2 : nf - 1);
}

template <int M, int KIND>
static void launch_rows(bool fwd, int inmode, int outmode, const ReqDesc* dd, const GridDims& d, int nb,
                        const double2* tw, const double2* tws, hipStream_t st) {
  using W = RowGeo<M, KIND>;
  using F = RowGeoF<M, KIND>;
  const dim3 grid(cdiv((long long)d.n2 * d.n3, W::RPB), nb), block(W::NT);
  if (fwd) {
    allow_lds<k_rows_fwd<M, KIND>>(F::LDS);
    hipLaunchKernelGGL((k_rows_fwd<M, KIND>), dim3(cdiv((long long)d.n2 * d.n3, F::RPB), nb), dim3(F::NT), F::LDS, st, dd, d, tw, tws, inmode);
  } else if (inmode == kInRho) {
    hipLaunchKernelGGL((k_rows_inv<M, KIND, kInRho, kOutPot>), grid, block, W::LDS, st, dd, d, tw, tws, kOutPot);
  } else if constexpr (KIND != kPlain) {
    hipLaunchKernelGGL((k_rows_inv<M, KIND, kInPhi, -1>), grid, block, W::LDS, st, dd, d, tw, tws, outmode);
  }
}

// The launchers of each group of lengths; null for a length of another group.
using ColsFn = void (*)(int S, const ReqDesc* dd, long long nc, const Cols& cs, int nf, int nb, int tuned,
                        const double2* tw, hipStream_t st);
using ZFn = void (*)(int kind, const ReqDesc* dd, const GridDims& d, int nb, int tuned, const double2* tw,
                     hipStream_t st);
using RowsFn = void (*)(bool fwd, int inmode, int outmode, const ReqDesc* dd, const GridDims& d, int nb,
                        const double2* tw, const double2* tws, hipStream_t st);
struct ColFns {
  ColsFn cols;
  ZFn z;
};
ColFns cols_a(int n);
ColFns cols_b(int n);
ColFns cols_c(int n);
ColFns cols_d(int n);
ColFns cols_e(int n);
template <int KIND> RowsFn rows_lo(int m);
template <int KIND> RowsFn rows_hi(int m);

}  // namespace gen
}  // namespace ofd
