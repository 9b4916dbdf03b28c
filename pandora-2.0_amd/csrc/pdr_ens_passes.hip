// pdr_ens_passes.hip -- the batched ensemble passes: one launch of a pass over the
// members of one line length, on the compile-time bodies of the single-box kernels
// (pdr_passes.hpp, pdr_plane.hpp, pdr_zall.hpp).  The members of a launch have the same
// tiles, so a workgroup's member and tile follow from its index; each member computes
// what its own launches would (up to the order of the plane's parts and the rounding of
// multiply-adds that the compiler contracts differently in another kernel).
#include "pdr_ens_ops.hpp"
#include "pdr_plane.hpp"
#include "pdr_zall.hpp"

namespace pdr {

namespace {

// Lengths whose planes run as one kernel and whose z passes take all fields at once.
// us per step of 16 members (FP32-mixed, FP64), one launch over all lengths with the
// separate passes -> here: 32 points 109 -> 62, 174 -> 82; 48 points 297 -> 173, 470 -> 288;
// 64 points 448 -> 299, 777 -> 543; 96 points 1368 -> 1289, 2564 -> 2357 (planes as one
// kernel 1881 FP32-mixed, joined z passes 1412 and 2702); 128 points 2945 -> 2684,
// 5975 -> 5109.  16 members each of 32, 48, 64 and 96 points 2194 -> 1646, 4221 -> 3130.
#ifndef PDR_ENS_PLANE_MAX
#define PDR_ENS_PLANE_MAX 64
#endif
#ifndef PDR_ENS_ZALL_MAX
#define PDR_ENS_ZALL_MAX 64
#endif
// Parts of a member's plane, all of one workgroup: the fewest that fit (the ensemble
// fills the chip with planes, and a part more is one more reading of the plane's modes:
// 64 points FP32-mixed 314 us a step with one part, 378 with two, 509 with four).
template <typename T>
constexpr int plane_parts_ens(int n) {
  return n <= PDR_ENS_PLANE_MAX ? plane_parts<T, true>(n, 1) : 0;
}

template <typename T, int N>
__global__ void __launch_bounds__((plane_threads(N, plane_parts_ens<T>(N))))
    k_ens_plane(const EnsMember* __restrict__ mem) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[b / unsigned(N)];
  plane_body<T, N, plane_parts_ens<T>(N), false>(int(b % unsigned(N)), 0, 1, e.g, e.cf, (const cx<T>*)e.w1,
                                                 (cx<T>*)e.w1, (T*)nullptr, 0, 0, nullptr, (const cx<T>*)e.twx,
                                                 nullptr);
}

template <typename T, int N>
__global__ void __launch_bounds__(kBlock2) k_ens_zinv(const EnsMember* __restrict__ mem, int nt) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x), per = unsigned(nt) * (N / 3 + 1);
  const EnsMember& e = mem[b / per];
  k2_zinv_r_body<T, N>(b % per, e.g, e.cf, (const cx<T>*)e.u[0], (const cx<T>*)e.u[1], (const cx<T>*)e.u[2],
                       (cx<T>*)e.w1, (const cx<T>*)e.twz, nt);
}

template <typename T, int N>
__global__ void __launch_bounds__(kBlock2) k_ens_yinv(const EnsMember* __restrict__ mem, int nt, unsigned per,
                                                    int fpb) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[b / per];
  k2_yinv_body<T, N, true, false>(b % per, e.g, (const cx<T>*)e.w1, (cx<T>*)e.w2, (const cx<T>*)e.twy, nt, 0, N, fpb);
}

template <typename T, int N>
__global__ void __launch_bounds__(kBlock2) k_ens_xpass(const EnsMember* __restrict__ mem, int nt) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x), per = unsigned(nt) * N;
  const EnsMember& e = mem[b / per];
  k2_xpass_body<T, N, 0>(b % per, e.g, e.cf, (cx<T>*)e.w2, (T*)nullptr, 0, 0, e.umax, (const cx<T>*)e.twx, nt, 0,
                         nullptr);
}

template <typename T, int N>
__global__ void __launch_bounds__(kBlock2) k_ens_yfwd(const EnsMember* __restrict__ mem, int nt, unsigned per,
                                                    int fpb) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[b / per];
  k2_yfwd_body<T, N, true>(b % per, e.g, (const cx<T>*)e.w2, (cx<T>*)e.w1, (const cx<T>*)e.twy, nt, 0, N, fpb);
}

template <typename T, int N>
__global__ void __launch_bounds__(kBlock2) k_ens_zfwd_formf(const EnsMember* __restrict__ mem, int nt, double beta,
                                                          double gamma) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x), per = unsigned(nt) * (N / 3 + 1);
  const EnsMember& e = mem[b / per];
  k2_zfwd_formf_body<T, N, kBlock2, 0, zff_fresh<T>(N, 0)>(b % per, e.g, e.cf, (const cx<T>*)e.w1, (cx<T>*)e.u[0], (cx<T>*)e.u[1],
                                       (cx<T>*)e.u[2], (cx<T>*)e.rk[0], (cx<T>*)e.rk[1], (cx<T>*)e.rk[2], nullptr, 0,
                                       0.0, beta, gamma * e.dt, (const cx<T>*)e.twz, nt, T(e.norm));
}

template <typename T, int N, bool FWD, bool INV>
__global__ void __launch_bounds__((zall_threads<T>(N))) k_ens_zall(const EnsMember* __restrict__ mem, int nt,
                                                                  double beta, double gamma) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x), per = unsigned(nt) * (N / 3 + 1);
  const EnsMember& e = mem[b / per];
  zall_body<T, N, FWD, INV, 0>(b % per, e.g, e.cf, e.cf, (const cx<T>*)e.w1, 1, (cx<T>*)e.w1, (cx<T>*)e.u[0],
                               (cx<T>*)e.u[1], (cx<T>*)e.u[2], (cx<T>*)e.rk[0], (cx<T>*)e.rk[1], (cx<T>*)e.rk[2],
                               nullptr, 0, 0.0, beta, gamma * e.dt, (const cx<T>*)e.twz, nt, T(e.norm));
}

template <typename T, int N>
struct Ens {
  static constexpr int NKI = N / 3 + 1, NKJ = 2 * (N / 3) + 1;
  static constexpr bool zall = N <= PDR_ENS_ZALL_MAX;
  static constexpr int parts = plane_parts_ens<T>(N);
  static constexpr int PP = y_planes<T>(N);
  static constexpr int tiles(int lines, int per) { return (lines + per - 1) / per; }

  static hipError_t prepare() {
    hipError_t e = hipSuccess;
    auto set = [&](auto* fn, size_t lds) {
      if (e == hipSuccess) e = big_lds((const void*)fn, lds);
    };
    if constexpr (zall) {
      const size_t l = size_t(zall_lds_bytes<T>(N));
      set(k_ens_zall<T, N, false, true>, l);
      set(k_ens_zall<T, N, true, true>, l);
      set(k_ens_zall<T, N, true, false>, l);
    } else {
      set(k_ens_zinv<T, N>, size_t(lds_zinv_bytes<T>(N)));
      set(k_ens_zfwd_formf<T, N>, lds_fwd<T, N>());
    }
    if constexpr (parts > 0) {
      set(k_ens_plane<T, N>, size_t(plane_lds_bytes<T>(N, parts)));
    } else {
      set(k_ens_yinv<T, N>, size_t(lds_y_bytes<T>(N)));
      set(k_ens_xpass<T, N>, lds_x<T, N>());
      set(k_ens_yfwd<T, N>, size_t(lds_yf_bytes<T>(N)));
    }
    return e;
  }
  static hipError_t zinv(const EnsMember* mem, int nm, hipStream_t s) {
    if constexpr (zall) {
      const int nt = tiles(NKJ, zall_lines<T>(N));
      k_ens_zall<T, N, false, true>
          <<<unsigned(nm * nt * NKI), zall_threads<T>(N), size_t(zall_lds_bytes<T>(N)), s>>>(mem, nt, 0.0, 0.0);
    } else {
      const int nt = tiles(NKJ, zinv_lines<T>(N));
      k_ens_zinv<T, N><<<unsigned(nm * nt * NKI), kBlock2, size_t(lds_zinv_bytes<T>(N)), s>>>(mem, nt);
    }
    return hipGetLastError();
  }
  static hipError_t mid(const EnsMember* mem, int nm, int fpb_y, int fpb_yf, hipStream_t s) {
    if constexpr (parts > 0) {
      k_ens_plane<T, N><<<unsigned(nm * N), plane_threads(N, parts), size_t(plane_lds_bytes<T>(N, parts)), s>>>(mem);
    } else {
      const int ny = PP ? tiles(N, PP) : tiles(NKI, y_lines<T>(N));
      const unsigned py = unsigned(ny * (PP ? 1 : N) * (6 / fpb_y));
      k_ens_yinv<T, N><<<unsigned(nm) * py, kBlock2, size_t(lds_y_bytes<T>(N)), s>>>(mem, ny, py, fpb_y);
      const int nx = tiles(N, xrows<T>(N));
      k_ens_xpass<T, N><<<unsigned(nm * nx * N), kBlock2, lds_x<T, N>(), s>>>(mem, nx);
      const int nf = PP ? tiles(N, PP) : tiles(NKI, y_lines_fwd<T>(N));
      const unsigned pf = unsigned(nf * (PP ? 1 : N) * (3 / fpb_yf));
      k_ens_yfwd<T, N><<<unsigned(nm) * pf, kBlock2, size_t(lds_yf_bytes<T>(N)), s>>>(mem, nf, pf, fpb_yf);
    }
    return hipGetLastError();
  }
  static hipError_t zend(const EnsMember* mem, int nm, double beta, double gamma, bool join, hipStream_t s) {
    if constexpr (zall) {
      const int nt = tiles(NKJ, zall_lines<T>(N));
      const size_t l = size_t(zall_lds_bytes<T>(N));
      const unsigned grid = unsigned(nm * nt * NKI);
      if (join)
        k_ens_zall<T, N, true, true><<<grid, zall_threads<T>(N), l, s>>>(mem, nt, beta, gamma);
      else
        k_ens_zall<T, N, true, false><<<grid, zall_threads<T>(N), l, s>>>(mem, nt, beta, gamma);
    } else {
      if (join) return hipErrorNotSupported;
      const int nt = tiles(NKJ, tile_lines_fwd<T>(N));
      k_ens_zfwd_formf<T, N><<<unsigned(nm * nt * NKI), kBlock2, lds_fwd<T, N>(), s>>>(mem, nt, beta, gamma);
    }
    return hipGetLastError();
  }
  static EnsOps ops() { return {sizeof(T) == 4 ? 1 : 0, N, zall, parts == 0, prepare, zinv, mid, zend}; }
};

}  // namespace

const EnsOps* ens_ops(int prec, int n) {
#define PDR_ENS_SIZES(X) X(32) X(48) X(64) X(96) X(128) X(192) X(256)
  static const EnsOps t[] = {
#define PDR_ROW(n) Ens<float, n>::ops(), Ens<double, n>::ops(),
      PDR_ENS_SIZES(PDR_ROW)
#undef PDR_ROW
  };
  for (const EnsOps& o : t)
    if (o.prec == prec && o.n == n) return &o;
  return nullptr;
}

}  // namespace pdr
