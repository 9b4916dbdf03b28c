// pdr_spec.hip -- the pass kernels of pdr_passes.hpp for one line length and precision:
// compiled once per PDR_SPEC_N and PDR_SPEC_FP32 (build_lib.py), each a code object of
// its own (pdr_spec.hpp).
#include "pdr_passes.hpp"
#include "pdr_plane.hpp"
#include "pdr_spec.hpp"
#include "pdr_zall.hpp"

#ifndef PDR_SPEC_N
#define PDR_SPEC_N 32
#define PDR_SPEC_FP32 0
#endif
#define PDR_CAT2(a, b) a##b
#define PDR_CAT(a, b) PDR_CAT2(a, b)

namespace pdr {

namespace {

template <typename T, int N>
SpecOps ops_of() {
  SpecOps o;
  o.prec = sizeof(T) == 4 ? 1 : 0;
  o.n = N;
  o.yinv = yinv_n<T, N, false>;
  o.yinv5 = yinv5_n<T, N>;
  o.y_planes = y_planes<T>(N);
  o.yinv_conv = yinv_n<T, N, true>;
  o.xpass_conv = xpass_conv_n<T, N>;
  o.xpass = xpass_n<T, N>;
  o.yfwd = yfwd_n<T, N>;
  o.zfwd = zfwd_n<T, N>;
  o.zinv = zinv_n<T, N>;
  o.zfwd_formf = zfwd_formf_n<T, N>;
  o.zall_inv = nullptr;
  o.zall_fwd = nullptr;
  if constexpr (zall_lines<T>(N) > 0) {
    o.zall_inv = zall_inv_n<T, N>;
    o.zall_fwd = zall_fwd_n<T, N>;
  }
  o.zall_most = zall_most<T>(N);
  o.zall_lines = zall_lines<T>(N);
  constexpr int parts = plane_parts_box<T>(N);
  o.plane = parts ? plane_n<T, N> : nullptr;
  o.plane_parts = parts;
  o.plane_most = parts ? plane_most<T>(N, parts) : 0;
  o.lds_plane = parts ? size_t(plane_lds_bytes<T>(N, parts) + plane_static_bytes<T>(N, parts)) : 0;
  o.lds_z = lds_lines<T, N>() > lds_fwd<T, N>() ? lds_lines<T, N>() : lds_fwd<T, N>();
  o.lds_y = lds_y<T, N>();
  o.lds_x = lds_x<T, N>() > lds_x<T, N, true>() ? lds_x<T, N>() : lds_x<T, N, true>();
  o.lds_xc = size_t(lds_xc_bytes<T>(N));
  o.xrows = xrows<T>(N);
  o.xrows_rs = xrows<T, true>(N);
  o.xrows_conv = xrows_conv<T>(N);
  o.x_tw_global = x_tw_global<T>(N) ? 1 : 0;
  constexpr bool reg = PDR_ZINV_REG && N <= 512;
  o.zinv_register = reg ? 1 : 0;
  o.zinv_lines = reg ? zinv_lines_t<T, PDR_ZINV_THREADS>(N) : tile_lines<T>(N);
  return o;
}

}  // namespace

#if PDR_SPEC_FP32
const SpecOps* PDR_CAT(spec_ops_f32_, PDR_SPEC_N)() {
  static const SpecOps o = ops_of<float, PDR_SPEC_N>();
#else
const SpecOps* PDR_CAT(spec_ops_f64_, PDR_SPEC_N)() {
  static const SpecOps o = ops_of<double, PDR_SPEC_N>();
#endif
  return &o;
}

}  // namespace pdr
