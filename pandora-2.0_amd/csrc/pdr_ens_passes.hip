// pdr_ens_passes.hip -- the batched ensemble passes: one launch of a pass over the
// tiles of every member, on the compile-time bodies of pdr_passes.hpp.
#include "pdr_passes.hpp"

namespace pdr {

namespace {

// ---------------------------------------------------------------------------
// Batched ensemble passes: one launch runs a pass for every member.  Block b
// (after the XCD remap, so that a member's tiles share one XCD's L2) belongs to
// the last member whose start is <= b; the member's descriptor supplies the
// geometry, coefficients, buffers and tile counts, and a switch on its line
// length selects the compile-time body that the single-box kernel also uses,
// so each member computes what its own launches would (up to the rounding of
// multiply-adds that the compiler contracts differently in another kernel).
// ---------------------------------------------------------------------------
#define PDR_ENS_SIZES(X) X(32) X(48) X(64) X(96) X(128) X(192) X(256)

// member of block b of a pass: binary search of the members' first blocks
__device__ __forceinline__ int ens_member(const EnsMember* __restrict__ mem, int nm, int pass, unsigned b) {
  int lo = 0, hi = nm - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mem[mid].start[pass] <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

template <typename T>
__global__ void __launch_bounds__(kBlock2) k_ens_zinv(const EnsMember* __restrict__ mem, int nm) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[ens_member(mem, nm, 0, b)];
  const unsigned lb = b - e.start[0];
  switch (e.n) {
#define PDR_EC(n)                                                                                                \
  case n:                                                                                                        \
    k2_zinv_r_body<T, n>(lb, e.g, e.cf, (const cx<T>*)e.u[0], (const cx<T>*)e.u[1], (const cx<T>*)e.u[2],        \
                         (cx<T>*)e.w1, (const cx<T>*)e.twz, e.nt[0]);                                            \
    break;
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      break;
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock2) k_ens_yinv(const EnsMember* __restrict__ mem, int nm) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[ens_member(mem, nm, 1, b)];
  const unsigned lb = b - e.start[1];
  switch (e.n) {
#define PDR_EC(n)                                                                                                \
  case n:                                                                                                        \
    k2_yinv_body<T, n, true, false>(lb, e.g, (const cx<T>*)e.w1, (cx<T>*)e.w2, (const cx<T>*)e.twy, e.nt[1], 0, e.g.nz,      \
                       e.fpb_y);                                                                                 \
    break;
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      break;
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock2) k_ens_xpass(const EnsMember* __restrict__ mem, int nm) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[ens_member(mem, nm, 2, b)];
  const unsigned lb = b - e.start[2];
  switch (e.n) {
#define PDR_EC(n)                                                                                                \
  case n:                                                                                                        \
    k2_xpass_body<T, n, 0>(lb, e.g, e.cf, (cx<T>*)e.w2, (T*)nullptr, 0, 0, e.umax, (const cx<T>*)e.twx,      \
                               e.nt[2], 0, nullptr);                                                             \
    break;
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      break;
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock2) k_ens_yfwd(const EnsMember* __restrict__ mem, int nm) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[ens_member(mem, nm, 3, b)];
  const unsigned lb = b - e.start[3];
  switch (e.n) {
#define PDR_EC(n)                                                                                                \
  case n:                                                                                                        \
    k2_yfwd_body<T, n, true>(lb, e.g, (const cx<T>*)e.w2, (cx<T>*)e.w1, (const cx<T>*)e.twy, e.nt[3], 0, e.g.nz,      \
                       e.fpb_yf);                                                                                \
    break;
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      break;
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock2) k_ens_zfwd_formf(const EnsMember* __restrict__ mem, int nm, double beta,
                                                          double gamma) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const EnsMember& e = mem[ens_member(mem, nm, 4, b)];
  const unsigned lb = b - e.start[4];
  const double gdt = gamma * e.dt;
  switch (e.n) {
#define PDR_EC(n)                                                                                                \
  case n:                                                                                                        \
    k2_zfwd_formf_body<T, n, kBlock2, 0>(lb, e.g, e.cf, (const cx<T>*)e.w1, 1, (cx<T>*)e.u[0], (cx<T>*)e.u[1],  \
                             (cx<T>*)e.u[2], (cx<T>*)e.rk[0], (cx<T>*)e.rk[1], (cx<T>*)e.rk[2], nullptr, 0, 0.0, \
                             beta, gdt,                                                                          \
                             (const cx<T>*)e.twz, e.nt[4], T(e.norm));                                           \
    break;
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      break;
  }
}

template <typename T, int N>
int ens_tiles_n(const Geo& g, int fpb_y, int fpb_yf, int nt[5], unsigned blocks[5]) {
  nt[0] = (g.nkj + zinv_lines<T>(N) - 1) / zinv_lines<T>(N);
  constexpr int PP = y_planes<T>(N);
  nt[1] = PP ? (g.nz + PP - 1) / PP : (g.nki + y_lines<T>(N) - 1) / y_lines<T>(N);
  nt[2] = (g.ny + xrows<T>(N) - 1) / xrows<T>(N);
  nt[3] = PP ? (g.nz + PP - 1) / PP : (g.nki + y_lines_fwd<T>(N) - 1) / y_lines_fwd<T>(N);
  nt[4] = (g.nkj + tile_lines_fwd<T>(N) - 1) / tile_lines_fwd<T>(N);
  blocks[0] = unsigned(nt[0] * g.nki);
  blocks[1] = unsigned(nt[1] * (PP ? 1 : g.nz) * (6 / fpb_y));
  blocks[2] = unsigned(nt[2] * g.nz);
  blocks[3] = unsigned(nt[3] * (PP ? 1 : g.nz) * (3 / fpb_yf));
  blocks[4] = unsigned(nt[4] * g.nki);
  return 0;
}

template <typename T, int N>
size_t ens_lds_n(int pass) {
  switch (pass) {
    case 0: return size_t(lds_zinv_bytes<T>(N));
    case 1: return size_t(lds_y_bytes<T>(N));
    case 2: return lds_x<T, N>();
    case 3: return size_t(lds_yf_bytes<T>(N));
    default: return lds_fwd<T, N>();
  }
}

}  // namespace

bool ens_size_supported(int n) {
  switch (n) {
#define PDR_EC(n) case n:
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    return true;
    default:
      return false;
  }
}

int ens_tiles(int prec, int n, const Geo& g, int fpb_y, int fpb_yf, int nt[5], unsigned blocks[5]) {
  switch (n) {
#define PDR_EC(n)                                                                                     \
  case n:                                                                                             \
    return prec ? ens_tiles_n<float, n>(g, fpb_y, fpb_yf, nt, blocks)                                 \
                : ens_tiles_n<double, n>(g, fpb_y, fpb_yf, nt, blocks);
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      return -1;
  }
}

size_t ens_lds(int prec, int n, int pass) {
  switch (n) {
#define PDR_EC(n) \
  case n:         \
    return prec ? ens_lds_n<float, n>(pass) : ens_lds_n<double, n>(pass);
    PDR_ENS_SIZES(PDR_EC)
#undef PDR_EC
    default:
      return 0;
  }
}

template <typename T>
static hipError_t ens_prepare_t(size_t lds_max) {
  const void* fns[5] = {(const void*)k_ens_zinv<T>, (const void*)k_ens_yinv<T>, (const void*)k_ens_xpass<T>,
                        (const void*)k_ens_yfwd<T>, (const void*)k_ens_zfwd_formf<T>};
  for (const void* f : fns) {
    hipError_t e = big_lds(f, lds_max);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t ens_prepare(int prec, size_t lds_max) {
  return prec ? ens_prepare_t<float>(lds_max) : ens_prepare_t<double>(lds_max);
}

template <typename T>
static void ens_launch_t(int pass, const EnsMember* mem, int nm, unsigned nblk, size_t lds, double beta,
                         double gamma, hipStream_t s) {
  const dim3 grid(nblk);
  switch (pass) {
    case 0: k_ens_zinv<T><<<grid, kBlock2, lds, s>>>(mem, nm); break;
    case 1: k_ens_yinv<T><<<grid, kBlock2, lds, s>>>(mem, nm); break;
    case 2: k_ens_xpass<T><<<grid, kBlock2, lds, s>>>(mem, nm); break;
    case 3: k_ens_yfwd<T><<<grid, kBlock2, lds, s>>>(mem, nm); break;
    default: k_ens_zfwd_formf<T><<<grid, kBlock2, lds, s>>>(mem, nm, beta, gamma); break;
  }
}

hipError_t launch_ens_pass(int prec, int pass, const EnsMember* mem, int nm, unsigned nblk, size_t lds,
                           double beta, double gamma, hipStream_t s) {
  if (prec)
    ens_launch_t<float>(pass, mem, nm, nblk, lds, beta, gamma, s);
  else
    ens_launch_t<double>(pass, mem, nm, nblk, lds, beta, gamma, s);
  return hipGetLastError();
}

}  // namespace pdr
