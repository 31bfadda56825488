// Dispatch of the three-pass FP64 evaluations (ofd_yz_impl.h).
#include "ofd_yz_impl.h"

namespace ofd {
namespace yz {
template <> YzRowsFn yz_rows_lo<kWT3>(int);
template <> YzRowsFn yz_rows_hi<kWT3>(int);
template <> YzRowsFn yz_rows_lo<kWT4>(int);
template <> YzRowsFn yz_rows_hi<kWT4>(int);
template <> YzRowsFn yz_rows_lo<kWT3S>(int);
template <> YzRowsFn yz_rows_hi<kWT3S>(int);

static YzFn z_of(int n) { return n < 54 ? yz_a(n) : yz_b(n); }
template <int KIND> static YzRowsFn rows_k(int m) { return m < 54 ? yz_rows_lo<KIND>(m) : yz_rows_hi<KIND>(m); }
static YzRowsFn rows_of(int kind, int m) {
  switch (kind) {
    case kWT3: return rows_k<kWT3>(m);
    case kWT4: return rows_k<kWT4>(m);
    case kWT3S: return rows_k<kWT3S>(m);
    default: return nullptr;
  }
}
// lanes per row of a half length M and per column of a z length
static int row_lanes(int m) {
  switch (m) {
#define X(N, A, B, T_) case N: return T_;
    OFD_YZ_ROWS(X)
#undef X
    default: return 0;
  }
}
static int col_lanes(int n) {
  switch (n) {
#define X(N, A, B, T_) case N: return T_;
    OFD_YZ_COLS_A(X) OFD_YZ_COLS_B(X)
#undef X
    default: return 0;
  }
}
#define OFD_YZ_IS(R) || r == R
static bool is_a(int r) { return false OFD_YZ_A(OFD_YZ_IS); }
#undef OFD_YZ_IS

// The split of the shape's y length and the tiles, or A = 0 where the five
// passes stay: WGC (its z pass couples the fields), FP32, two spin channels on
// the 32 x 32 planes (which keep the plane passes' bits) or with alpha != beta
// (7 fields: 80 x 75 x 63 115 / 90 us, 90 x 75 x 96 150 / 129); an x workgroup of more than 256 lanes (five
// waves share a CU badly: 108 x 72 x 108 with four fields and 288 lanes
// 94.5 / 89.4 us a call; at 240 to 256 lanes 96 x 64 x 96 56 / 82, 128^3
// 147 / 161), z columns of more than 256 lanes, and y lengths without two
// factors A, B of 4..16 and 3..10 within a factor of three. Synchronous calls
// against the five passes (for 32^3, 64^3 and 128^3 the plane passes), alpha =
// beta / alpha != beta: 32^3 26.3 / 28.4 and 29.7 / 32.5, 72^3 44.1 / 52.7 and
// 60.7 / 70.9, 100^3 66.6 / 79.2 and 82.6 / 99.4, 128^3 96.4 / 103.2 and
// 147 / 161, 150^3 172 / 197 and 264 / 275, 100 x 75 x 81 62 / 77 and 73 / 87;
// two channels 90^3 89 / 97; over 230 random shapes of 18 to 160 points an axis
// none lost more than the runs differ.
// A z workgroup takes the widest tile of at most four waves. An x-forward
// workgroup takes one field (100^3 14.4 us, all three 17.5) unless its M + 1
// elements then leave a second wave nearly empty (128^3 28.7, all three 22.9)
// or the fields share powers (alpha != beta).
static YZ plan(const ShapePlan& sp, int kind) {
  const GridDims& d = sp.d;
  YZ g{};
  if (kind == kWGC8 || kind == kWT4S || (kind == kWT3S && fast_path_ok(sp, kind, 0))) return g;
  const int nf = func_nf(kind), tx = row_lanes(d.M), tz = col_lanes(d.n3);
  if (tx == 0 || tz == 0 || nf * (d.M + 1) > 512) return g;
  for (int b = 10; b >= 3; --b) {
    const int a = d.n2 / b;
    if (a * b != d.n2 || a < b || a > 3 * b || !is_a(a)) continue;
    if (b * nf * tx > 256 || std::max(a * tz, d.n3) > 256) return g;
    g.A = a;
    g.B = b;
    g.W = g.w = 4;
    // a tuned tile only groups columns: results keep their bits
    while (sp.kb_z[0] > 0 && g.w > sp.kb_z[0]) g.w /= 2;
    while (g.w * std::max(a * tz, d.n3) > 256) g.w /= 2;
    g.nkt = (d.K1 + g.w - 1) / g.w;
    g.fw = kind == kWT4 || d.M >= 64 ? nf : 1;
    return g;
  }
  return g;
}
}  // namespace yz

bool yz_path_ok(const ShapePlan& sp, int kind, int fp32) {
  return !fp32 && !sp.force_generic && yz::plan(sp, kind).A != 0;
}

int yz_partials(const ShapePlan& sp, int kind) { return sp.d.n3 * yz::plan(sp, kind).A; }

int yz_eval(const ShapePlan& sp, int kind, int inmode, int outmode, const ReqDesc* dd, int nb, hipStream_t st) {
  const GridDims& d = sp.d;
  const yz::YZ g = yz::plan(sp, kind);
  const yz::YzRowsFn rows = yz::rows_of(kind, d.M);
  rows(true, inmode, outmode, dd, d, g, nb, sp.tw_x, sp.tw_s, sp.tw_y, st);
  yz::z_of(d.n3)(kind, dd, d, g, nb, sp.tw_z, st);
  rows(false, inmode, outmode, dd, d, g, nb, sp.tw_x, sp.tw_s, sp.tw_y, st);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ofd
