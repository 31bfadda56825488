// FP64 evaluations in three passes: the y transform divided between the x
// passes and the z pass, n2 = A B.
//
// With y = a + A b and k2 = kb + B ka,
//   Y[k2] = sum_a w_A^(a ka) [ w^(a kb) sum_b w_B^(b kb) x[a + A b] ],  w = exp(-2 pi i / n2).
// A workgroup of the x-forward pass holds the B rows a, a + A, ... of one
// plane, so after its row transforms it takes the inner sum (radix B, one
// thread per k1) and the twiddle; a workgroup of the z pass holds, for one kb
// and W neighbouring k1, the A rows' columns, takes the outer sum (radix A),
// the z transform, the G-space operator and both back; the x-inverse pass
// undoes its part as it reads. The two y passes, a read and a write of every
// spectrum each, are gone, and two launches with them.
//
// Layout of a field between the passes: element (z, kb, k1, a) at
//   (z B + kb) K1 A + kt W A + a w + (k1 - kt W),  kt = k1 / W, w = min(W, K1 - kt W):
// W neighbouring k1 stay together (64 bytes at W = 4), so neither side moves
// single elements: the x side's writes / reads of three fields alone took, at
// 128^3, 18.9 / 16.1 us with W = 1, 11.7 / 10.9 with 2, 9.8 / 9.0 with 4 and
// 9.7 / 8.7 with 8 (whole rows: 9.1 / 8.7), and the z side's read and write
// 27.6, 21.4, 16.7 and 16.8. Same size as the rows they replace.
//
// Kernel times of the three passes against the general five, Wang-Teter with
// alpha = beta, us (x, y + z, x against x, y, z, y, x):
//    32^3  4.5   5.4  5.2 = 15.1   4.5  3.1  3.8  3.1  4.7 =  19.2
//    72^3  8.1  10.6  9.7 = 28.4   7.0  5.8  7.1  5.8  7.7 =  33.5
//   100^3 14.4  20.5 17.5 = 52.2  12.8  9.2 13.2  8.8 14.3 =  58.3
//   128^3 23.0  34.3 26.5 = 83.8  17.3 18.0 22.8 19.9 25.2 = 103.2
// The y + z pass moves 2.5 to 3 TB/s: sixteen barriers (four exchanges, one
// real component at a time) at three or four waves per SIMD bound it, not HBM;
// the x passes' radix-B steps keep fewer lanes busy than the row transforms.
#pragma once
#include "ofd_gen_impl.h"

namespace ofd {
namespace yz {

using namespace gen;

struct YZ {
  int A, B;
  int W;        // tile of the layout
  int w, nkt;   // tile of a z workgroup (a power of two up to W) and their number, ceil(K1 / w)
  int fw;       // fields of an x-forward workgroup: 1 or all
};

// f(integral_constant) for the run-time radix r of a list
#define OFD_YZ_A(X) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16)
#define OFD_YZ_B(X) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
#define OFD_YZ_CASE(R) case R: f(std::integral_constant<int, R>()); break;
template <typename F> __device__ __forceinline__ void with_a(int r, F&& f) {
  switch (r) { OFD_YZ_A(OFD_YZ_CASE) }
}
template <typename F> __device__ __forceinline__ void with_b(int r, F&& f) {
  switch (r) { OFD_YZ_B(OFD_YZ_CASE) }
}
#undef OFD_YZ_CASE

// byte offset of (kb = 0, k1, a) within plane z, and of one kb
__device__ __forceinline__ unsigned col_off(const YZ& g, int K1, int k1, int a) {
  const int kt = k1 / g.W, w = min(g.W, K1 - kt * g.W);
  return (unsigned)(kt * g.W * g.A + a * w + (k1 - kt * g.W)) * 16u;
}

// ------------------------------------------------------------ x forward
// One workgroup: the B rows of residue a in plane z, of one field or of all.
// Numbered (z, a, field), so that the fields of a row find its values in the
// XCD's L2 and the workgroups that fill a line of the layout run next to each
// other.
template <int M, int KIND>
__global__ void __launch_bounds__(512) k_rows_fwd(const ReqDesc* __restrict__ descs, GridDims d, YZ g,
                                                  const double2* __restrict__ tw, const double2* __restrict__ tws,
                                                  const double2* __restrict__ twy, int inmode) {
  using G = L<M>;
  extern __shared__ __align__(16) unsigned char smem[];
  double2* lds = reinterpret_cast<double2*>(smem);
  const ReqDesc& D = descs[blockIdx.y];
  constexpr int NF = fast::NF_<KIND>::v;
  const int nfw = NF / g.fw, blk = xcd_block(blockIdx.x, gridDim.x), za = blk / nfw, f0 = blk - za * nfw;
  const int z = za / g.A, a = za - z * g.A;
  const int line = threadIdx.x / G::T, t = threadIdx.x % G::T, fl = line / g.B, r = line - fl * g.B, f = f0 + fl;
  const bool active = fl < g.fw;
  double2 xc[G::NC], xs[G::NS];
  double2* mine = lds + (size_t)line * G::LINE;
  auto field = [&](int ff, size_t i) {
    return inmode == kInRho ? fast::field_pair<KIND, kInRho, double>(D, ff, i)
                            : fast::field_pair<KIND, kInPhi, double>(D, ff, i);
  };
  if constexpr (KIND == kWT4) {
    // a point's two powers (fields 1 and 2) once, by all threads of the
    // workgroup, which holds all fields: the lines of these two fields would
    // each take both, on two of the four SIMDs (120 x 63 x 120: 35 us against
    // 23.7, 128 x 48 x 128: 25.7 against 21.2)
    for (int e = threadIdx.x; e < g.B * M; e += blockDim.x) {
      const int rr = e / M, i = e - rr * M;
      const size_t p = ((size_t)z * d.n2 + a + (size_t)g.A * rr) * (2 * M) + 2 * i;
      double r0, r1;
      if (inmode == kInRho) fast::rho_pair<kInRho>(D.u, D.v, D.ca, D.cb, p, r0, r1);
      else fast::rho_pair<kInPhi>(D.u, D.v, D.ca, D.cb, p, r0, r1);
      double2 pa, pb;
      fwd_pows(r0, D.alpha, D.beta, pa.x, pb.x);
      fwd_pows(r1, D.alpha, D.beta, pa.y, pb.y);
      lds[(size_t)(g.B + rr) * G::LINE + i] = pb;
      lds[(size_t)(2 * g.B + rr) * G::LINE + i] = pa;
    }
    __syncthreads();
  }
  if (active) {
    const size_t base = ((size_t)z * d.n2 + a + (size_t)g.A * r) * (2 * M);
#pragma unroll
    for (int j = 0; j < G::J1; ++j) {
      if (!G::col_ok(t, j)) continue;
#pragma unroll
      for (int m = 0; m < G::R1; ++m) {
        const int i = t + G::T * j + G::R2 * m;
        xc[j * G::R1 + m] = KIND == kWT4 && (f == 1 || f == 2) ? mine[i] : field(KIND == kWT4 ? f & 2 ? 3 : 0 : f, base + 2 * i);
      }
    }
  }
  if constexpr (KIND == kWT4) __syncthreads();
  fwd_c<M>(xc, xs, mine, t, tw, active);
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q)
      if (G::row_ok(t, q)) {
#pragma unroll
        for (int k2 = 0; k2 < G::R2; ++k2) mine[t + G::T * q + G::R1 * k2] = xs[q * G::R2 + k2];
      }
  }
  __syncthreads();
  gptr<double2> out = glb(reinterpret_cast<double2*>(D.work)) + (size_t)z * g.B * d.K1 * g.A;
  const unsigned kbs = (unsigned)(d.K1 * g.A) * 16u;
  with_b(g.B, [&](auto bb) {
    constexpr int B = decltype(bb)::value;
    for (int e = threadIdx.x; e < g.fw * (M + 1); e += blockDim.x) {
      const int ff = e / (M + 1), k = e - ff * (M + 1);
      const double2* lf = lds + ff * B * G::LINE;
      gptr<double2> of = out + (size_t)(f0 + ff) * d.nc;
      const double2 w = tws[k];
      double2 x[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const double2 zk = lf[b * G::LINE + (k == M ? 0 : k)], zm = lf[b * G::LINE + (k == 0 ? 0 : M - k)];
        const double er = 0.5 * (zk.x + zm.x), ei = 0.5 * (zk.y - zm.y);
        const double orr = 0.5 * (zk.y + zm.y), oi = -0.5 * (zk.x - zm.x);
        x[b].x = er + (w.x * orr - w.y * oi);
        x[b].y = ei + (w.x * oi + w.y * orr);
      }
      Bfly<B, -1, double2>::run(x);
      const unsigned o = col_off(g, d.K1, k, a);
      st16(of, o, x[0]);
#pragma unroll
      for (int kb = 1; kb < B; ++kb) st16(of, o + kb * kbs, cmul(x[kb], twy[a * kb]));
    }
  });
}

// ------------------------------------------------------------ y + z
// One workgroup: the w A columns (ka, k1) of one kb and one tile of k1, of
// field blockIdx.y. Thread (z, k1) moves the A values of its place between
// memory, the radix-A step and the columns in LDS; thread (column, t) runs the
// column's z transform as gen::k_zgop does. All exchanges go one real
// component at a time.
template <int N>
__global__ void __launch_bounds__(256, 3) k_yz(const ReqDesc* __restrict__ descs, GridDims d, YZ g,
                                            const double2* __restrict__ tw, int fvw) {
  using G = L<N>;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = reinterpret_cast<double*>(smem);
  const ReqDesc& D = descs[blockIdx.z];
  const int f = blockIdx.y;
  const int blk = xcd_block(blockIdx.x, gridDim.x), kb = blk / g.nkt, kt = blk - kb * g.nkt;
  const int k0 = kt * g.w, w = min(g.w, d.K1 - k0), nc = w * g.A;
  const int l0 = k0 / g.W * g.W, wl = min(g.W, d.K1 - l0);   // the layout's tile
  // place (z, wi)
  const int pz = threadIdx.x / w, wi = threadIdx.x - pz * w;
  const bool place = pz < N;
  gptr<double2> base = glb(reinterpret_cast<double2*>(D.work)) + (size_t)f * d.nc;
  const unsigned po = ((((unsigned)pz * g.B + kb) * (unsigned)d.K1 + (unsigned)l0) * (unsigned)g.A +
                       (unsigned)(k0 - l0 + wi)) * 16u;
  const unsigned as = (unsigned)wl * 16u;
  // column (ka, ci) and its lane t
  const int c = threadIdx.x % nc, t = threadIdx.x / nc;
  const bool active = t < G::T;
  double* line = lds + (size_t)c * G::LINE;
  double* spot = lds + (size_t)wi * G::LINE + pz;   // column (a, wi) at + a w LINE
  const int ss = w * G::LINE;
  double2 xc[G::NC], xs[G::NS], yc[G::NC];
  auto cols = [&](auto&& fn) {   // fn(slot, point) over the thread's stage-1 points
    if (!active) return;
#pragma unroll
    for (int j = 0; j < G::J1; ++j)
      if (G::col_ok(t, j)) {
#pragma unroll
        for (int m = 0; m < G::R1; ++m) fn(j * G::R1 + m, t + G::T * j + G::R2 * m);
      }
  };
  with_a(g.A, [&](auto aa) {
    constexpr int A = decltype(aa)::value;
    double2 v[A];
    if (place) {
#pragma unroll
      for (int a = 0; a < A; ++a) v[a] = ld16(base, po + a * as);
      Bfly<A, -1, double2>::run(v);
#pragma unroll
      for (int a = 0; a < A; ++a) spot[a * ss] = v[a].x;
    }
    __syncthreads();
    cols([&](int s, int i) { xc[s].x = line[i]; });
    __syncthreads();
    if (place) {
#pragma unroll
      for (int a = 0; a < A; ++a) spot[a * ss] = v[a].y;
    }
    __syncthreads();
    cols([&](int s, int i) { xc[s].y = line[i]; });
    __syncthreads();
  });
  fwd_s<N>(xc, xs, line, t, tw, active);
  if (active) {
    const int ka = c / w, m1 = k0 + (c - ka * w), i2 = kb + g.B * ka;
    const unsigned es = (unsigned)(d.n2 * d.K1), col = (unsigned)(i2 * d.K1 + m1);
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
      const double invn = 1.0 / (double)d.nr;
      const G2Col g2(D, m1, i2 > d.n2 / 2 ? i2 - d.n2 : i2);
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
  with_a(g.A, [&](auto aa) {
    constexpr int A = decltype(aa)::value;
    double2 u[A];
    cols([&](int s, int i) { line[i] = yc[s].x; });
    __syncthreads();
    if (place) {
#pragma unroll
      for (int a = 0; a < A; ++a) u[a].x = spot[a * ss];
    }
    __syncthreads();
    cols([&](int s, int i) { line[i] = yc[s].y; });
    __syncthreads();
    if (place) {
#pragma unroll
      for (int a = 0; a < A; ++a) u[a].y = spot[a * ss];
      Bfly<A, +1, double2>::run(u);
      const unsigned o = offs(po);
#pragma unroll
      for (int a = 0; a < A; ++a) st16(base, o + a * as, u[a]);
    }
  });
}

// ------------------------------------------------------------ x inverse
// One workgroup: the B rows of residue a in plane z, all fields (lines field
// by field). Thread (field, k1) reads its B values, undoes the twiddle and the
// radix-B step and leaves the rows' half spectra in LDS; the rest is
// gen::k_rows_inv on rows that are A apart.
template <int M, int KIND, int INMODE, int OUTMODE>
__global__ void __launch_bounds__(512) k_rows_inv(const ReqDesc* __restrict__ descs, GridDims d, YZ g,
                                                  const double2* __restrict__ tw, const double2* __restrict__ tws,
                                                  const double2* __restrict__ twy, int outmode) {
  using G = L<M>;
  constexpr int NF = fast::NF_<KIND>::v;
  extern __shared__ __align__(16) unsigned char smem[];
  double2* lds = reinterpret_cast<double2*>(smem);
  const ReqDesc& D = descs[blockIdx.y];
  const int blk = xcd_block(blockIdx.x, gridDim.x), z = blk / g.A, a = blk - z * g.A;
  const int line = threadIdx.x / G::T, t = threadIdx.x % G::T;
  const bool active = line < g.B * NF;
  gptr<const double2> in = glb(reinterpret_cast<const double2*>(D.work)) + (size_t)z * g.B * d.K1 * g.A;
  const unsigned kbs = (unsigned)(d.K1 * g.A) * 16u;
  with_b(g.B, [&](auto bb) {
    constexpr int B = decltype(bb)::value;
    for (int e = threadIdx.x; e < NF * (M + 1); e += blockDim.x) {
      const int ff = e / (M + 1), k = e - ff * (M + 1);
      const unsigned o = col_off(g, d.K1, k, a);
      double2 x[B];
#pragma unroll
      for (int kb = 0; kb < B; ++kb) x[kb] = ld16(in + (size_t)ff * d.nc, o + kb * kbs);
#pragma unroll
      for (int kb = 1; kb < B; ++kb) {
        double2 w = twy[a * kb];
        w.y = -w.y;
        x[kb] = cmul(x[kb], w);
      }
      Bfly<B, +1, double2>::run(x);
#pragma unroll
      for (int b = 0; b < B; ++b) lds[(ff * B + b) * G::LINE + k] = x[b];
    }
  });
  __syncthreads();
  double2* mine = lds + (size_t)line * G::LINE;
  double2 xc[G::NC], xs[G::NS];
  if (active) {
#pragma unroll
    for (int q = 0; q < G::J2; ++q) {
      if (!G::row_ok(t, q)) continue;
#pragma unroll
      for (int k2 = 0; k2 < G::R2; ++k2) {
        const int k = t + G::T * q + G::R1 * k2;
        double2 xk = mine[k], xm = mine[M - k];
        if (k == 0) { xk.y = 0.0; xm.y = 0.0; }
        const double er = xk.x + xm.x, ei = xk.y - xm.y;
        const double dr = xk.x - xm.x, di = xk.y + xm.y;
        const double2 w = tws[k];
        const double orr = w.x * dr + w.y * di, oi = w.x * di - w.y * dr;
        xs[q * G::R2 + k2] = make_double2(er - oi, ei + orr);
      }
    }
  }
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
  double acc[kNSum];
#pragma unroll
  for (int k = 0; k < kNSum; ++k) acc[k] = 0.0;
  const long long row0 = (long long)z * d.n2 + a;
  fast::x_epi_points<M, KIND, INMODE, OUTMODE, 0, 0, 2 * G::LINE, 2 * M, true>(
      D, reinterpret_cast<const double*>(lds), row0, 0, 0, acc, outmode, fast::DynRows{g.B, (int)blockDim.x, g.A});
  fast::x_epi_sums<OUTMODE>(D, acc, blk);
}

// ------------------------------------------------------------ launchers
// Half row lengths M and z lengths. Left out, with what they took against the
// general passes: rows of 168, 196 and 200 points (168 x 84 x 72, alpha != beta:
// 112 / 106 us; 196 x 70 x 70: 90 / 88; 200 x 80 x 80: 93 / 86; a workgroup's
// NF (M + 1) elements need a fifth and sixth wave), columns of 125 (its 25-point
// radix beside the y radix spills 360 bytes; 128 x 128 x 125: 133 / 120).
#define OFD_YZ_ROWS_LO(X) OFD_GEN_SHORT(X) OFD_GEN_A(X)
#define OFD_YZ_ROWS_HI(X)                                                                                         \
  X(54, 6, 9, 9) X(56, 7, 8, 8) X(60, 4, 15, 4) X(63, 7, 9, 9) X(64, 8, 8, 8) X(70, 7, 10, 7) X(72, 8, 9, 9)      \
  X(75, 5, 15, 5) X(80, 8, 10, 10) X(81, 9, 9, 9) X(96, 8, 12, 8)
#define OFD_YZ_ROWS(X) OFD_YZ_ROWS_LO(X) OFD_YZ_ROWS_HI(X)
#define OFD_YZ_COLS_A(X) OFD_GEN_A(X)
#define OFD_YZ_COLS_B(X)                                                                                         \
  OFD_GEN_B(X) X(105, 7, 15, 8) X(108, 9, 12, 12) X(112, 8, 14, 8) X(120, 8, 15, 8) X(126, 9, 14, 14)             \
  X(128, 8, 16, 8) X(135, 9, 15, 15) X(140, 10, 14, 14) X(144, 12, 12, 12) X(150, 10, 15, 15) X(160, 10, 16, 16)

constexpr int up64(int n) { return (n + 63) / 64 * 64; }

template <int N>
static void launch_yz(int kind, const ReqDesc* dd, const GridDims& d, const YZ& g, int nb, const double2* tw,
                      hipStream_t st) {
  const int nf = func_nf(kind);
  const int threads = up64(g.w * std::max(g.A * L<N>::T, N));
  const size_t lds = (size_t)g.w * g.A * L<N>::LINE * sizeof(double);
  allow_lds<k_yz<N>>(lds);
  hipLaunchKernelGGL((k_yz<N>), dim3(g.B * g.nkt, nf, nb), dim3(threads), lds, st, dd, d, g, tw,
                     is_spin_kind(kind) ? nf - 2 : nf - 1);
}
template <int M, int KIND>
static void launch_rows(bool fwd, int inmode, int outmode, const ReqDesc* dd, const GridDims& d, const YZ& g, int nb,
                        const double2* tw, const double2* tws, const double2* twy, hipStream_t st) {
  constexpr int NF = fast::NF_<KIND>::v, T = L<M>::T;
  const size_t line = L<M>::LINE * sizeof(double2);
  if (fwd) {
    allow_lds<k_rows_fwd<M, KIND>>(g.B * g.fw * line);
    hipLaunchKernelGGL((k_rows_fwd<M, KIND>), dim3(d.n3 * g.A * (NF / g.fw), nb),
                       dim3(up64(g.fw * std::max(g.B * T, M + 1))), g.B * g.fw * line, st, dd, d, g, tw, tws, twy, inmode);
    return;
  }
  const dim3 grid(d.n3 * g.A, nb), block(up64(std::max(g.B * NF * T, NF * (M + 1))));
  const size_t lds = g.B * NF * line;
  if (inmode == kInRho) {
    allow_lds<k_rows_inv<M, KIND, kInRho, kOutPot>>(lds);
    hipLaunchKernelGGL((k_rows_inv<M, KIND, kInRho, kOutPot>), grid, block, lds, st, dd, d, g, tw, tws, twy, kOutPot);
  } else {
    allow_lds<k_rows_inv<M, KIND, kInPhi, -1>>(lds);
    hipLaunchKernelGGL((k_rows_inv<M, KIND, kInPhi, -1>), grid, block, lds, st, dd, d, g, tw, tws, twy, outmode);
  }
}

using YzFn = void (*)(int kind, const ReqDesc* dd, const GridDims& d, const YZ& g, int nb, const double2* tw,
                      hipStream_t st);
using YzRowsFn = void (*)(bool fwd, int inmode, int outmode, const ReqDesc* dd, const GridDims& d, const YZ& g, int nb,
                          const double2* tw, const double2* tws, const double2* twy, hipStream_t st);
YzFn yz_a(int n);
YzFn yz_b(int n);
template <int KIND> YzRowsFn yz_rows_lo(int m);
template <int KIND> YzRowsFn yz_rows_hi(int m);

}  // namespace yz
}  // namespace ofd
