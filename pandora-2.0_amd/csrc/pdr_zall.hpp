// pdr_zall.hpp -- the z passes of short lines with every field of a tile of lines in LDS
// at once: the z forward transform with FormF and the RK update (f_RK3SolveNavierStokes,
// src/pf_rk3.f90:2067-2130), the vorticity and inverse z transform of the next stage
// (f_RK3PrepareRealSpace, 269-700), or both in one kernel with the mode's new velocity
// kept in registers between them.
//
// A tile of a short line is little work: the kernels that take its fields one after
// another spend a small box's time on the chain of six (three) loads, transforms and
// stores, each with its barriers and its own copy of the transform's code to fetch.
// Here one transform runs over 6 L (3 L) lines, a thread holds one or two modes, and
// a stage's end and the next one's start need no launch and no read of the velocity
// between them.
#pragma once
#include "pdr_passes.hpp"

// Longest lines: up to here the joined kernel beats the two it replaces in a box of few
// lines (us a launch by events: 64 points 12.4 against 12.3 + 11.8 in FP64 and 11.0 against
// 12.4 + 11.0 in FP32-mixed, 128 points FP32-mixed 25.5 against 19.1 + 16.5; 128 points FP64
// 44.0 against 19.0 + 21.5); zall_most has the lines.
#ifndef PDR_ZALL_MAX_F32
#define PDR_ZALL_MAX_F32 128
#endif
#ifndef PDR_ZALL_MAX_F64
#define PDR_ZALL_MAX_F64 96
#endif

namespace pdr {

namespace {

// Lines (consecutive j) of a tile; 0: the line length runs the other z passes.
template <typename T>
constexpr int zall_lines(int n) {
  return n > (sizeof(T) == 4 ? PDR_ZALL_MAX_F32 : PDR_ZALL_MAX_F64) ? 0 : (sizeof(T) == 4 && n > 64 ? 8 : 4);
}
// Most z lines (i, j) of a single box that takes them.  Up to 80 points they win at any
// number (us a step, the separate passes -> these: 256 x 256 x 64 FP64 594 -> 539, 256 x 256
// x 80 FP64 731 -> 720); above, a workgroup's tile is half the LDS of a CU or more, and the
// separate passes' smaller ones move more at a time once there are lines enough for them
// (90 to 96 points FP64: 96 x 96 x 96, 2145 lines, 229 / 230, 128 x 128, 3655 lines, 271 ->
// 296, 256 x 256, 14706 lines, 906 -> 989; FP32-mixed: 96 points 128 x 128 194 -> 178, 192 x
// 128, 5525 lines, 254 / 254, 256 x 256 512 -> 563, 128 points 192 x 128 304 -> 301, 192 x
// 192, 8385 lines, 433 -> 446).
template <typename T>
constexpr long long zall_most(int n) {
  return n <= 80 ? (1ll << 40) : sizeof(T) == 4 ? 6000 : 3000;
}
template <typename T>
constexpr int zall_lds_bytes(int n) {
  return (n + 6 * zall_lines<T>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
// Threads: one per mode of the tile and per butterfly of the inverse transform's first
// pass, up to 1024.
template <typename T>
constexpr int zall_threads(int n) {
  const int l = zall_lines<T>(n) ? zall_lines<T>(n) : 1;
  const int m = l * (2 * (n / 3) + 1), b = 6 * l * (n / plan_radix(n, 0));
  const int t = ((m > b ? m : b) + 63) / 64 * 64;
  return t > 1024 ? 1024 : t;
}

// FWD: z forward of the three NL fields at nlw (the sum of `parts` addends), FormF with
// cf and the RK update.  INV: vorticity with the operator cn and inverse z transforms of
// the six fields into w1.  nlw may be w1: a tile's lines are its own.
template <typename T, int N, bool FWD, bool INV, int FRC>
__device__ __forceinline__ void zall_body(unsigned bid, const Geo& g, const Coef& cf, const Coef& cn,
                                          const cx<T>* nlw, int parts, cx<T>* w1, cx<T>* __restrict__ u0,
                                          cx<T>* __restrict__ u1, cx<T>* __restrict__ u2, cx<T>* __restrict__ r0,
                                          cx<T>* __restrict__ r1, cx<T>* __restrict__ r2,
                                          const double2* __restrict__ frc, int fnk, double fkf, double beta,
                                          double gdt, const cx<T>* __restrict__ twg, int ntile, T norm) {
  constexpr int L = zall_lines<T>(N);
  constexpr int NT = zall_threads<T>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKK = 2 * K + 1;
  constexpr int EM = L * NKK, QM = (EM + NT - 1) / NT;  // modes
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* const tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* const buf = tw + N;
  const int tile = int(bid % unsigned(ntile));
  const int i = int(bid / unsigned(ntile));
  const int j0 = tile * L;
  const int nkj = g.nkj;
  const int lines = (nkj - j0) < L ? (nkj - j0) : L;
  const long long e0 = ((long long)i * nkj + j0) * NKK;
  cx<T> un[QM][3];
  if constexpr (FWD) {
    constexpr int E = 3 * L * N, Q = (E + NT - 1) / NT;
    const cx<T>* src = nlw + (long long)i * N * g.ldj + j0;
    cx<T> v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      const int line = e % L, z = (e / L) % N, f = e / (L * N);
      v[q] = ((E % NT == 0 || e < E) && line < lines) ? src[(long long)f * g.m1 + z * g.ldj + line] : czero<T>();
    }
    // the plane pass left NL as up to kNlParts addends: all of their loads in flight at once
    cx<T> v2[kNlParts - 1][Q];
#pragma unroll
    for (int p = 1; p < kNlParts; ++p) {
      const cx<T>* sp = src + 3 * p * g.m1;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = int(threadIdx.x) + NT * q;
        const int line = e % L, z = (e / L) % N, f = e / (L * N);
        v2[p - 1][q] = (p < parts && (E % NT == 0 || e < E) && line < lines) ? sp[(long long)f * g.m1 + z * g.ldj + line]
                                                                           : czero<T>();
      }
    }
    if (parts > 1) {
#pragma unroll
      for (int p = 1; p < kNlParts; ++p)
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = add(v[q], v2[p - 1][q]);
    }
    load_tw<T, N, NT>(tw, twg);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      const int line = e % L, z = (e / L) % N, f = e / (L * N);
      if (E % NT == 0 || e < E) buf[(f * L + line) * LD + lds_off<T>(z)] = v[q];
    }
    __syncthreads();
    fft_ip<T, N, 3 * L, LD, -1, true, NT>(buf, tw);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      const int line = e / NKK, k = e - line * NKK;
      const int zz = (k <= K) ? k : N - NKK + k;
      if (e < lines * NKK) {
        const cx<T>* b = buf + line * LD + lds_off<T>(zz);
        formf_mode<T, FRC>(g, cf, i, j0 + line, k, e0 + e, scl(b[0], norm), scl(b[L * LD], norm),
                           scl(b[2 * L * LD], norm), u0, u1, u2, r0, r1, r2, frc, fnk, fkf, beta, gdt,
                           INV ? un[q] : nullptr);
      } else if (INV) {
        un[q][0] = un[q][1] = un[q][2] = czero<T>();
      }
    }
    if (INV) __syncthreads();
  } else {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      const bool in = e < lines * NKK;
      un[q][0] = in ? u0[e0 + e] : czero<T>();
      un[q][1] = in ? u1[e0 + e] : czero<T>();
      un[q][2] = in ? u2[e0 + e] : czero<T>();
    }
    load_tw<T, N, NT>(tw, twg);
  }
  if constexpr (INV) {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      if (EM % NT == 0 || e < EM) {
        const int line = e / NKK, k = e - line * NKK;
        cx<T>* b = buf + line * LD + lds_off<T>((k <= K) ? k : k + (N - NKK));
        // w_c = i sum_n (G[c][n] . k) u_n, the same operations as k2_zinv
        const double kv[3] = {double(i), wvn2(j0 + line, g.kj), wvn2(k, K)};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          cx<T> acc = czero<T>();
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            const double* G = &cn.G[(c * 3 + n) * 3];
            if ((G[0] != 0.0) || (G[1] != 0.0) || (G[2] != 0.0))
              acc = add(acc, scl(un[q][n], T(G[0] * kv[0] + G[1] * kv[1] + G[2] * kv[2])));
          }
          b[c * L * LD] = un[q][c];
          b[(3 + c) * L * LD] = mk<T>(-acc.y, acc.x);
        }
      }
    }
    zero_band_edges<T, N, 6 * L, LD, K, NT>(buf);
    __syncthreads();
    fft_ip<T, N, 6 * L, LD, +1, true, NT, K>(buf, tw);
    constexpr int E = 6 * L * N, Q = (E + NT - 1) / NT;
    cx<T>* dst = w1 + (long long)i * N * g.ldj + j0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int e = int(threadIdx.x) + NT * q;
      const int line = e % L, z = (e / L) % N, f = e / (L * N);
      if ((E % NT == 0 || e < E) && line < lines)
        put<kNtZinv && !small_store(N)>(&dst[(long long)f * g.m1 + z * g.ldj + line], buf[(f * L + line) * LD + lds_off<T>(z)]);
    }
  }
}

template <typename T, int N, bool FWD, bool INV, int FRC>
__global__ void __launch_bounds__((zall_threads<T>(N)))
    k2_zall(Geo g, Coef cf, Coef cn, const cx<T>* nlw, int parts, cx<T>* w1, cx<T>* __restrict__ u0,
            cx<T>* __restrict__ u1, cx<T>* __restrict__ u2, cx<T>* __restrict__ r0, cx<T>* __restrict__ r1,
            cx<T>* __restrict__ r2, const double2* __restrict__ frc, int fnk, double fkf, double beta, double gdt,
            const cx<T>* __restrict__ twg, int ntile, T norm) {
  zall_body<T, N, FWD, INV, FRC>(xcd_remap(blockIdx.x, gridDim.x), g, cf, cn, nlw, parts, w1, u0, u1, u2, r0, r1, r2,
                                 frc, fnk, fkf, beta, gdt, twg, ntile, norm);
}

template <typename T, int N, bool FWD, bool INV, int FRC>
hipError_t zall_launch(pdr_ctx* c, const Coef& cf, const Coef& cn, double beta, double gdt) {
  const Geo& g = c->g;
  constexpr int L = zall_lines<T>(N);
  const int nt = (g.nkj + L - 1) / L;
  const size_t lds = size_t(zall_lds_bytes<T>(N));
  hipError_t e = big_lds((const void*)k2_zall<T, N, FWD, INV, FRC>, lds);
  if (e != hipSuccess) return e;
  const double norm = 1.0 / (double(g.nx) * double(g.ny) * double(g.nz));
  k2_zall<T, N, FWD, INV, FRC><<<dim3(unsigned(nt * g.nki)), zall_threads<T>(N), lds, c->stream>>>(
      g, cf, cn, (const cx<T>*)(c->nl_parts > 1 ? c->w2 : c->w1), c->nl_parts, (cx<T>*)c->w1, (cx<T>*)c->u[0],
      (cx<T>*)c->u[1], (cx<T>*)c->u[2], (cx<T>*)c->rk[0], (cx<T>*)c->rk[1], (cx<T>*)c->rk[2],
      FRC ? (const double2*)c->force : nullptr, FRC ? c->force_nk : 0, FRC ? c->p.force_kf : 0.0, beta, gdt,
      (const cx<T>*)c->tab.twz, nt, T(norm));
  return hipGetLastError();
}

template <typename T, int N>
hipError_t zall_inv_n(pdr_ctx* c, const Coef& cn) {
  return zall_launch<T, N, false, true, 0>(c, cn, cn, 0.0, 0.0);
}
// next: the operator of the stage that follows, whose inverse z pass is then done too (or null)
template <typename T, int N>
hipError_t zall_fwd_n(pdr_ctx* c, const Coef& cf, const Coef* next, double beta, double gdt) {
  auto go = [&](auto frc_c) -> hipError_t {
    constexpr int F = decltype(frc_c)::value;
    return next ? zall_launch<T, N, true, true, F>(c, cf, *next, beta, gdt)
                : zall_launch<T, N, true, false, F>(c, cf, cf, beta, gdt);
  };
  if (!c->forcing) return go(std::integral_constant<int, 0>{});
  if (cf.fdef) return go(std::integral_constant<int, 2>{});
  return go(std::integral_constant<int, 1>{});
}

}  // namespace

}  // namespace pdr
