// Dispatch of the register-resident fast path (two-stage line lengths,
// Wang-Teter and WGC functionals). The kernels live in ofd_fast_impl.h; each
// (precision, functional) pair is instantiated in its own translation unit
// (ofd_fast_{d,f}{3,4,5,7,8}.hip: the number is the kind's field count).
#include "ofd_fast_impl.h"

namespace ofd {

// instantiated in their own translation units (not again here)
extern template int fast_eval_k<double, kWT3>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<double, kWT4>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<float, kWT3>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<float, kWT4>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<double, kWGC8>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<float, kWGC8>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<double, kWT3S>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<float, kWT3S>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<double, kWT4S>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);
extern template int fast_eval_k<float, kWT4S>(const ShapePlan&, int, int, const ReqDesc*, int, hipStream_t);

namespace fast {
// One workgroup per (slot, request): fin[slot] = sum over the workgroups'
// partials, fixed order.
__global__ void __launch_bounds__(256) k_fin(const ReqDesc* __restrict__ descs, int nwg) {
  const ReqDesc& D = descs[blockIdx.y];
  const int k = blockIdx.x;
  gptr<const double> src = glb(D.sums) + (size_t)k * nwg;
  double acc = 0.0;
  // eight independent loads in flight per thread, summed in a fixed order
  for (int base = 0; base < nwg; base += 8 * 256) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int w = base + threadIdx.x + 256 * j;
      v[j] = w < nwg ? src[w] : 0.0;
    }
    acc += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  __shared__ double red[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) put_fin(D, k, ((red[0] + red[1]) + red[2]) + red[3]);
}

}  // namespace fast

// FP32: every shape of the line lengths below. FP64, of what the three-pass
// evaluations (ofd_yz.hip, asked first) leave: shapes of the power-of-two plane
// passes, where two fused passes beat the general form's three. These are
// Wang-Teter with the z lengths 192 and 256 that the three passes lack, WGC on
// 128 x 128 planes and two spin channels on 32 x 32 (which keep their bits: the
// three passes would be faster there, 32^3 28 us). A call, plane / general
// passes: 32 x 32 x 192 39.8 / 41.1 us, 64 x 64 x 256 65 / 73, 128 x 128 x 192
// 144 / 159, alpha != beta 64 x 64 x 192 76 / 81 and 128 x 128 x 256 288 / 282;
// WGC 128 x 128 x 24 83 / 81, x 64 148 / 151, x 128 266 / 283, x 256 563 / 600;
// left to the general passes, WGC 64^3 70 / 70, two channels 64 x 64 x 192 92 / 92.
bool fast_path_ok(const ShapePlan& sp, int kind, int fp32) {
  if (!fast_path_ok_impl(sp, kind)) return false;
  if (fp32) return true;
  // the FP64 chain has no forward passes but the plane's, so it takes a shape
  // only where the plane fits in LDS
  const int M = sp.d.M;
  if ((M != 16 && M != 32 && M != 64) || is_gp_len(sp.d.n3) || !plane_for<double>(sp)) return false;
  return kind == kWGC8 ? M == 64 : (is_spin_kind(kind) ? M == 16 : sp.d.n3 >= 192);
}


int fast_eval(const ShapePlan& sp, int kind, int inmode, int outmode, int fp32, const ReqDesc* dd, int nb,
              hipStream_t st) {
  if (kind == kWT3)
    return fp32 ? fast_eval_k<float, kWT3>(sp, inmode, outmode, dd, nb, st)
                : fast_eval_k<double, kWT3>(sp, inmode, outmode, dd, nb, st);
  if (kind == kWGC8)
    return fp32 ? fast_eval_k<float, kWGC8>(sp, inmode, outmode, dd, nb, st)
                : fast_eval_k<double, kWGC8>(sp, inmode, outmode, dd, nb, st);
  if (kind == kWT3S)
    return fp32 ? fast_eval_k<float, kWT3S>(sp, inmode, outmode, dd, nb, st)
                : fast_eval_k<double, kWT3S>(sp, inmode, outmode, dd, nb, st);
  if (kind == kWT4S)
    return fp32 ? fast_eval_k<float, kWT4S>(sp, inmode, outmode, dd, nb, st)
                : fast_eval_k<double, kWT4S>(sp, inmode, outmode, dd, nb, st);
  return fp32 ? fast_eval_k<float, kWT4>(sp, inmode, outmode, dd, nb, st)
              : fast_eval_k<double, kWT4>(sp, inmode, outmode, dd, nb, st);
}

std::vector<int> fast_tile_candidates(const ShapePlan& sp, int kind, int fp32, int which) {
  const int n = which == 1 ? sp.d.n2 : sp.d.n3;
  const int T = len_T(n), w = 64 / T;
  const int cb = fp32 ? (int)sizeof(float2) : (int)sizeof(double2);
  std::vector<int> out;
  for (int kb = w; kb * T <= 256; kb += w)
    if (kb * col_line_bytes(n, cb, which) <= sp.lds_cap) out.push_back(kb);
  (void)kind;
  return out;
}

bool fast_plane_available(const ShapePlan& sp, int fp32) { return fp32 ? plane_for<float>(sp) : plane_for<double>(sp); }

// Sums the x-inverse pass's per-workgroup partials into each request's fin.
int fast_finalize(const ShapePlan& sp, int kind, int fp32, const ReqDesc* dd, int nb, double*, hipStream_t st) {
  const int rpb = fast::inv_rpb(func_nf(kind), len_T(sp.d.M));
  const long long nrows = (long long)sp.d.n2 * sp.d.n3;
  const int nwg = gen_inverse(sp, fp32) ? gen_partials(sp, kind) : (int)((nrows + rpb - 1) / rpb);
  hipLaunchKernelGGL(fast::k_fin, dim3(kNSum, nb), dim3(256), 0, st, dd, nwg);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ofd
