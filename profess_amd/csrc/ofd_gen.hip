// Dispatch of the general register-resident FP64 passes (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
static ColFns cols_of(int n) {
  if (n < 54) return cols_a(n);
  if (n < 105) return cols_b(n);
  if (n < 135) return cols_c(n);
  return n < 196 ? cols_d(n) : cols_e(n);
}
template <int KIND> static RowsFn rows_k(int m) { return m < 54 ? rows_lo<KIND>(m) : rows_hi<KIND>(m); }
template <> RowsFn rows_lo<kWT3>(int);
template <> RowsFn rows_hi<kWT3>(int);
template <> RowsFn rows_lo<kWT4>(int);
template <> RowsFn rows_hi<kWT4>(int);
template <> RowsFn rows_lo<kWGC8>(int);
template <> RowsFn rows_hi<kWGC8>(int);
template <> RowsFn rows_lo<kWT3S>(int);
template <> RowsFn rows_hi<kWT3S>(int);
template <> RowsFn rows_lo<kWT4S>(int);
template <> RowsFn rows_hi<kWT4S>(int);
template <> RowsFn rows_lo<kPlain>(int);
template <> RowsFn rows_hi<kPlain>(int);
static RowsFn rows_of(int kind, int m) {
  switch (kind) {
    case kWT3: return rows_k<kWT3>(m);
    case kWT4: return rows_k<kWT4>(m);
    case kWGC8: return rows_k<kWGC8>(m);
    case kWT3S: return rows_k<kWT3S>(m);
    case kWT4S: return rows_k<kWT4S>(m);
    default: return rows_k<kPlain>(m);
  }
}
static int rpb_of(int kind, int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return row_rpb(N, kind == kPlain ? 1 : func_nf(kind), T_, InvLine<N>::BYTES);
    OFD_GEN_ROWS(X)
#undef X
    default: return 1;
  }
}
static Cols y_cols(const GridDims& d) {
  return {(unsigned)(d.K1 * d.n3), (unsigned)d.K1, (unsigned)(d.n2 * d.K1), (unsigned)d.K1};
}
static Cols z_cols(const GridDims& d) {
  const unsigned p = (unsigned)(d.n2 * d.K1);
  return {p, p, 0u, p};
}
}  // namespace gen

bool gen_path_ok(const ShapePlan& sp) {
  return gen::rows_of(gen::kPlain, sp.d.M) != nullptr && gen::cols_of(sp.d.n2).cols != nullptr &&
         gen::cols_of(sp.d.n3).cols != nullptr;
}

int gen_eval(const ShapePlan& sp, int kind, int inmode, int outmode, const ReqDesc* dd, int nb, hipStream_t st) {
  using namespace gen;
  const GridDims& d = sp.d;
  const RowsFn rows = rows_of(kind, d.M);
  const ColFns cy = cols_of(d.n2), cz = cols_of(d.n3);
  const int nf = func_nf(kind);
  rows(true, inmode, outmode, dd, d, nb, sp.tw_x, sp.tw_s, st);
  cy.cols(-1, dd, d.nc, y_cols(d), nf, nb, sp.kb_y[0], sp.tw_y, st);
  cz.z(kind, dd, d, nb, sp.kb_z[0], sp.tw_z, st);
  cy.cols(+1, dd, d.nc, y_cols(d), nf, nb, sp.kb_y[0], sp.tw_y, st);
  rows(false, inmode, outmode, dd, d, nb, sp.tw_x, sp.tw_s, st);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int gen_rows_inv(const ShapePlan& sp, int kind, int inmode, int outmode, const ReqDesc* dd, int nb, hipStream_t st) {
  gen::rows_of(kind, sp.d.M)(false, inmode, outmode, dd, sp.d, nb, sp.tw_x, sp.tw_s, st);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int gen_partials(const ShapePlan& sp, int kind) {
  const int rpb = gen::rpb_of(kind, sp.d.M);
  return (int)(((long long)sp.d.n2 * sp.d.n3 + rpb - 1) / rpb);
}

int gen_fft3d_plain(const ShapePlan& sp, int forward, const ReqDesc* dd, int nb, hipStream_t st) {
  using namespace gen;
  const GridDims& d = sp.d;
  const RowsFn rows = rows_of(kPlain, d.M);
  const ColFns cy = cols_of(d.n2), cz = cols_of(d.n3);
  if (forward) {
    rows(true, kInRho, kOutPot, dd, d, nb, sp.tw_x, sp.tw_s, st);
    cy.cols(-1, dd, d.nc, y_cols(d), 1, nb, 0, sp.tw_y, st);
    cz.cols(-1, dd, d.nc, z_cols(d), 1, nb, 0, sp.tw_z, st);
  } else {
    cz.cols(+1, dd, d.nc, z_cols(d), 1, nb, 0, sp.tw_z, st);
    cy.cols(+1, dd, d.nc, y_cols(d), 1, nb, 0, sp.tw_y, st);
    rows(false, kInRho, kOutPot, dd, d, nb, sp.tw_x, sp.tw_s, st);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ofd
