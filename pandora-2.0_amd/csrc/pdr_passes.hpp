// pdr_passes.hpp -- length-specialised pass kernels (the default path for the
// grid sizes that pdr_spec.hip instantiates).  Same work split and data layouts as pdr_kernels.hip
// (pass 1 k_zinv ... pass 5 k_zfwd); see that file for the reference routines
// each pass replaces.  Differences: compile-time transform length and tile
// height, in-place LDS transforms, twiddles in LDS, 128-byte tile chunks on
// 16-element-padded strides, XCD-aware tile order, several x rows per block.
#pragma once
#include <type_traits>

#include "pdr_fft2.hpp"
#include "pdr_internal.hpp"
#include "pdr_rsstats.hpp"
#include "pdr_formf.hpp"

namespace pdr {

namespace {

__device__ __forceinline__ double wvn2(int k, int kmax) {
  return (k <= kmax) ? double(k) : double(k - (2 * kmax + 1));
}

template <typename T>
__device__ __forceinline__ cx<T> czero() {
  return mk<T>(T(0), T(0));
}
// i k a for the stored mode k (0..K, then -K..-1)
template <typename T>
__device__ __forceinline__ cx<T> mul_ik(cx<T> a, int k, int K) {
  const T w = T(k <= K ? k : k - (2 * K + 1));
  return mk<T>(-w * a.y, w * a.x);
}

// *m = max(*m, v), with the atomic only where v is larger than what is there already (a
// value that has gone stale is a smaller one): thousands of workgroups queued on one
// address (6400 of a 160^3 FP32-mixed box: the x pass of stage 1 some 45 us longer, a step
// 506 against 460).
__device__ __forceinline__ void raise_max(unsigned long long* m, unsigned long long v) {
  if (v > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(m, v);
}

// Tile shapes.  Lines per tile of the y/z kernels and rows per block of the x
// kernel; the build may override the FP32 / FP64 values for lengths <= 512
// (PDR_LINES_F32, PDR_LINES_F64, PDR_XROWS_F32, PDR_XROWS_F64) and the FP32
// heights of longer lines (PDR_LINES_MID_F32 and PDR_LINES_MID_FWD_F32 for
// 512 < n <= 1024, PDR_LINES_LONG_F32 and PDR_LINES_LONG_FWD_F32 above) to tune.
// Longer lines keep at least 8 lines in the inverse kernels, whose global
// accesses are runs of one element of each line (64-byte runs at 8 FP32 lines;
// 1.45 against 1.26 steps/s at 1536^3 with 4), while the forward kernels of
// lines above 1024 run faster with the two workgroups per CU that 4 lines allow.
#ifndef PDR_LINES_F32
#define PDR_LINES_F32 16
#endif
#ifndef PDR_LINES_F64
#define PDR_LINES_F64 8
#endif
#ifndef PDR_XROWS_F32
#define PDR_XROWS_F32 2
#endif
#ifndef PDR_XROWS_F64
#define PDR_XROWS_F64 2
#endif
#ifndef PDR_LINES_MID_F32
#define PDR_LINES_MID_F32 8
#endif
#ifndef PDR_LINES_LONG_F32
#define PDR_LINES_LONG_F32 8
#endif
template <typename T>
constexpr int tile_lines(int n) {
  return sizeof(T) == 4 ? (n <= 512 ? PDR_LINES_F32 : (n <= 1024 ? PDR_LINES_MID_F32 : PDR_LINES_LONG_F32))
                        : (n <= 512 ? PDR_LINES_F64 : (n <= 1024 ? 4 : 2));
}
// forward y/z kernels (3 fields per tile) may use their own FP32 tile height
#ifndef PDR_LINES_FWD_F32
#define PDR_LINES_FWD_F32 8
#endif
#ifndef PDR_LINES_MID_FWD_F32
#define PDR_LINES_MID_FWD_F32 8
#endif
#ifndef PDR_LINES_LONG_FWD_F32
#define PDR_LINES_LONG_FWD_F32 4
#endif
template <typename T>
constexpr int tile_lines_fwd(int n) {
  return sizeof(T) != 4 ? tile_lines<T>(n)
                        : (n <= 512 ? PDR_LINES_FWD_F32 : (n <= 1024 ? PDR_LINES_MID_FWD_F32 : PDR_LINES_LONG_FWD_F32));
}
// y passes of short lines: a workgroup takes PP whole z planes (all NKI
// i-lines of each) instead of a tile of i-lines of one plane, so that it
// moves about three thousand points and no tile is left part-empty
// (PP = 0: tiles of tile_lines i-lines within one plane).
// PL selects these plane tiles; they take the i-lines per plane from the pass's own
// length (NKI = NY/3 + 1), so boxes with NX/3 != NY/3 run the tiles of i-lines.
template <typename T, bool PL = true>
constexpr int y_planes(int n) {
  return !PL ? 0 : n <= 32 ? 8 : (n <= 48 ? 4 : (n <= 64 ? 2 : (n <= 96 ? 1 : 0)));
}
template <typename T, bool PL = true>
constexpr int y_lines(int n) {
  return y_planes<T, PL>(n) ? y_planes<T, PL>(n) * (n / 3 + 1) : tile_lines<T>(n);
}
template <typename T, bool PL = true>
constexpr int y_lines_fwd(int n) {
  return y_planes<T, PL>(n) ? y_planes<T, PL>(n) * (n / 3 + 1) : tile_lines_fwd<T>(n);
}

// Short lines take more rows per workgroup, so that a workgroup still moves
// about a thousand points (2 rows of 512; 16 rows of 64), and then fewer as soon as the CU
// gains more by workgroups at different phases than it loses by threads without a
// butterfly (us a launch, 8 -> 4 rows at 128^3: FP64 39.8 -> 36.4, FP32-mixed 26.3 -> 24.2;
// 4 -> 2 rows in FP64 at 250^3 362 -> 321, 256^3 300 -> 256, but 240^3 253 -> 264;
// FP32-mixed 160^3 42.8 -> 47.8, 192^3 65.7 -> 75.1, 256^3 129.9 / 128.6).
// With the moments (RS) the tile keeps the rows where it then holds the threads' sums for
// their reduction (us a call of pdr_rs_stats, rows as above -> kept: 100^3 FP64 109 -> 101,
// FP32-mixed 91 -> 81, 128^3 138 -> 130 and 101 -> 86, 144^3 FP32-mixed 167 -> 158, 256^3
// FP64 724 -> 716; but 144^3 FP64, two tiles of eight rows to a CU, 207 -> 210).
template <typename T, bool RS = false>
constexpr int xrows(int n) {
  constexpr bool f32 = sizeof(T) == 4;
  if (RS && n > 96 && n <= 256) return n <= (f32 ? 144 : 128) ? 8 : 4;
  return n <= 64 ? 16 : n <= 96 ? 8 : n <= (f32 ? 256 : 240) ? 4 : n <= 512 ? (f32 ? PDR_XROWS_F32 : PDR_XROWS_F64) : 2;
}

// LDS bytes of a workgroup, and the waves per SIMD that the 160 KB of LDS of a
// CU admit (each 256-thread workgroup puts one wave on each of the 4 SIMDs).
// The kernels declare that occupancy, capped at two, to the register
// allocator: it then keeps within 256 registers per lane (without the hint it
// takes more, and one wave per SIMD), and still uses fewer where it can.
constexpr int kLdsPerCu = 160 * 1024;
template <typename T>
constexpr int lds_lines_bytes(int n) {
  return (n + tile_lines<T>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
template <typename T>
constexpr int lds_fwd_bytes(int n) {
  return (n + tile_lines_fwd<T>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
template <typename T, bool PL = true>
constexpr int lds_y_bytes(int n) {
  return (n + y_lines<T, PL>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
template <typename T, bool PL = true>
constexpr int lds_yf_bytes(int n) {
  return (n + y_lines_fwd<T, PL>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
// The x tile of lines longer than PDR_X_TWG_MIN points reads its twiddles from
// the global table (through the caches) instead of staging them in LDS: that
// frees N complex of LDS, so two 2-row FP32 tiles of 1536 points fit one CU
// and the FP64 one fits at all.
#ifndef PDR_X_TWG_MIN
#define PDR_X_TWG_MIN 1024
#endif
template <typename T>
constexpr bool x_tw_global(int n) { return n > PDR_X_TWG_MIN; }
template <typename T, bool RS = false>
constexpr int lds_x_bytes(int n) {
  return ((x_tw_global<T>(n) ? 0 : n) + 3 * xrows<T, RS>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>)) +
         (kBlock2 / 64) * int(sizeof(T));
}
// Threads of the x pass: 512 for the tiles of which the CU's LDS holds fewer than four (FP64
// 192 points 42 KB, 512 points 60 KB; FP32-mixed 768 points 45 KB), so that it still has
// sixteen waves (us a launch, 256 -> 512 threads: 512^3 FP64 2418 -> 2168, 768^3 FP64
// 16050 -> 12020, 768 x 128 x 1024 FP32-mixed 1206 -> 950, 640^3 2573 -> 2542).  The moments'
// reductions are written for 256.
template <typename T, int RS>
constexpr int xthreads(int n) {
  return RS == 0 && 4 * lds_x_bytes<T>(n) > kLdsPerCu ? 2 * kBlock2 : kBlock2;
}
template <typename T, int RS>
constexpr int xwaves(int n) {
  return (kLdsPerCu / lds_x_bytes<T, RS != 0>(n) < 2 ? 1 : 2) * (xthreads<T, RS>(n) / kBlock2);
}
// Streaming (non-temporal) stores per kernel, bit mask: 1 zinv, 2 yinv,
// 4 xpass, 8 yfwd, 16 zfwd.  Every pass writes data that only the next pass
// reads, long after the caches have turned over: streaming stores keep the
// caches for the re-read inputs (measured 73.1 -> 75.4 steps/s at 512^3).
#ifndef PDR_NT_WRITES
#define PDR_NT_WRITES 31
#endif
// Streaming loads of single-use inputs, bit mask: 1 zinv (register form),
// 2 yinv, 4 xpass, 8 yfwd, 16 zfwd.
#ifndef PDR_NT_READS
#define PDR_NT_READS 0
#endif
constexpr bool kNrZinv = (PDR_NT_READS & 1) != 0;
constexpr bool kNrYinv = (PDR_NT_READS & 2) != 0;
constexpr bool kNrXpass = (PDR_NT_READS & 4) != 0;
constexpr bool kNrYfwd = (PDR_NT_READS & 8) != 0;
constexpr bool kNrZfwd = (PDR_NT_READS & 16) != 0;
constexpr bool kNtZinv = (PDR_NT_WRITES & 1) != 0;
constexpr bool kNtYinv = (PDR_NT_WRITES & 2) != 0;
constexpr bool kNtXpass = (PDR_NT_WRITES & 4) != 0;
constexpr bool kNtYfwd = (PDR_NT_WRITES & 8) != 0;
constexpr bool kNtZfwd = (PDR_NT_WRITES & 16) != 0;
// The fused kernels of short lines store through the caches: a small box's arrays are
// still there for the next kernel (16 members of 64 points, us a step: 314 -> 299
// FP32-mixed, 560 -> 543 FP64).
#ifndef PDR_SMALL_STORE_MAX
#define PDR_SMALL_STORE_MAX 64
#endif
constexpr bool small_store(int n) { return n <= PDR_SMALL_STORE_MAX; }

[[maybe_unused]] constexpr int waves_for(int lds) {
  return kLdsPerCu / lds < 2 ? 1 : 2;
}
// Threads of the passes of lines above 512 points: 512, since a CU holds two or three of
// their tiles (us a launch, 256 -> 512: z forward 768 x 128 x 1024 FP32-mixed 243 -> 216,
// 640^3 625 -> 547, 768^3 FP64 1916 -> 1717; y forward 640^3 FP32-mixed 978 -> 851, 768^3
// FP64 2812 -> 2601).  The inverse z pass, which keeps the velocity's loads of a field in
// registers, only where two fit (768 x 128 x 1024 490 -> 435, 768^3 FP64 3632 -> 3305; but
// 640^3 FP32-mixed 1380 -> 1449).
constexpr int zthreads(int n) { return n > 512 ? 2 * kBlock2 : kBlock2; }
template <typename T>
constexpr int zinv_threads(int n) {
  return 3 * lds_lines_bytes<T>(n) > kLdsPerCu ? zthreads(n) : kBlock2;
}
#define PDR_FWD_WAVES __attribute__((amdgpu_waves_per_eu(waves_for(lds_fwd_bytes<T>(N)))))

// Line kernels issue all global loads of a field (QE elements per thread)
// before the LDS stores of that field, so that one HBM latency is exposed per
// field rather than one per element.  (Loading field f+1 during the transform
// of field f was measured slower: it needs more registers than the occupancy
// leaves and spills.)

// ---------------------------------------------------------------------------
// pass 1: vorticity + inverse z FFT, (i, j-tile) per block
// ---------------------------------------------------------------------------
template <typename T, int N>
__global__ void __launch_bounds__((zinv_threads<T>(N))) __attribute__((amdgpu_waves_per_eu(waves_for(lds_lines_bytes<T>(N)) * (zinv_threads<T>(N) / kBlock2))))
    k2_zinv(Geo g, Coef cf, const cx<T>* __restrict__ u0, const cx<T>* __restrict__ u1,
            const cx<T>* __restrict__ u2, cx<T>* __restrict__ w1, const cx<T>* __restrict__ twg, int ntile) {
  constexpr int ZT = zinv_threads<T>(N);
  constexpr int L = tile_lines<T>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKK = 2 * K + 1;
  constexpr int QE = (L * N + ZT - 1) / ZT;
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const unsigned bid = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = int(bid % unsigned(ntile));
  const int i = int(bid / unsigned(ntile));
  const int j0 = tile * L;
  const int nkj = g.nkj;
  load_tw<T, N, ZT>(tw, twg);
  const double wi = double(i);
  bool need[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const double* G = &cf.G[(c * 3 + n) * 3];
      need[c][n] = (G[0] != 0.0) || (G[1] != 0.0) || (G[2] != 0.0);
    }
  const long long base = ((long long)i * nkj + j0) * NKK;
  const cx<T>* uu[3] = {u0 + base, u1 + base, u2 + base};
  // velocity fields: QE elements per thread, loaded in one batch
  cx<T> pre[QE];
  auto load_u = [&](int f) {
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = int(threadIdx.x) + ZT * q;
      const int line = idx / N;
      const int z = idx - line * N;
      const int k = (z <= K) ? z : ((z >= N - K) ? z - (N - NKK) : -1);
      pre[q] = ((L * N % ZT == 0 || idx < L * N) && j0 + line < nkj && k >= 0) ? uu[f][line * NKK + k]
                                                                                    : czero<T>();
    }
  };
  // vorticity fields need two or three components per element: computed and
  // stored to LDS in chunks of VC elements to bound the registers in flight
  constexpr int VC0 = sizeof(T) == 4 ? 8 : 4;
  constexpr int VC = QE < VC0 ? QE : VC0;
  auto fill_w = [&](int c) {
#pragma unroll 1
    for (int q0 = 0; q0 < QE; q0 += VC) {
      cx<T> a[VC][3];
#pragma unroll
      for (int qq = 0; qq < VC; ++qq) {
        const int idx = int(threadIdx.x) + ZT * (q0 + qq);
        const int line = idx / N;
        const int z = idx - line * N;
        const int k = (z <= K) ? z : ((z >= N - K) ? z - (N - NKK) : -1);
        const bool ok = (QE % VC == 0 || q0 + qq < QE) && (L * N % ZT == 0 || idx < L * N) &&
                        j0 + line < nkj && k >= 0;
#pragma unroll
        for (int n = 0; n < 3; ++n) a[qq][n] = (ok && need[c][n]) ? uu[n][line * NKK + k] : czero<T>();
      }
#pragma unroll
      for (int qq = 0; qq < VC; ++qq) {
        const int idx = int(threadIdx.x) + ZT * (q0 + qq);
        if ((QE % VC == 0 || q0 + qq < QE) && (L * N % ZT == 0 || idx < L * N)) {
          const int line = idx / N;
          const int z = idx - line * N;
          const int k = (z <= K) ? z : ((z >= N - K) ? z - (N - NKK) : 0);
          const double kv[3] = {wi, wvn2(j0 + line, g.kj), wvn2(k, K)};
          cx<T> acc = czero<T>();
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            if (need[c][n]) {
              const double* G = &cf.G[(c * 3 + n) * 3];
              acc = add(acc, scl(a[qq][n], T(G[0] * kv[0] + G[1] * kv[1] + G[2] * kv[2])));
            }
          }
          buf[line * LD + lds_off<T>(z)] = mk<T>(-acc.y, acc.x);
        }
      }
    }
  };
  const int nf = cf.y3 ? 5 : 6;  // y3: the inverse y pass forms the last vorticity component
  for (int f = 0; f < nf; ++f) {
    if (f < 3) {
      load_u(f);
#pragma unroll
      for (int q = 0; q < QE; ++q) {
        const int idx = int(threadIdx.x) + ZT * q;
        if (L * N % ZT == 0 || idx < L * N) {
          const int line = idx / N;
          buf[line * LD + lds_off<T>(idx - line * N)] = pre[q];
        }
      }
    } else {
      fill_w(f - 3);
    }
    __syncthreads();
    fft_ip<T, N, L, LD, +1, true, ZT>(buf, tw);
    cx<T>* dst = w1 + (long long)f * g.m1 + (long long)i * N * g.ldj + j0;
    for (int idx = threadIdx.x; idx < L * N; idx += ZT) {
      const int z = idx / L;
      const int line = idx - z * L;
      if (j0 + line < nkj) put<kNtZinv>(&dst[z * g.ldj + line], buf[line * LD + lds_off<T>(z)]);
    }
    __syncthreads();
  }
}

// The thread index of a phase of the z passes.  FRESH: formed anew (fresh_tid), so that the
// indices of all phases together do not take the registers that another workgroup on the CU
// needs; it lengthens a workgroup's own chain, and is for lengths whose registers it brings
// below that line, in boxes of more workgroups than the CUs hold otherwise.
template <bool FRESH>
__device__ __forceinline__ int phase_tid() {
  return FRESH ? fresh_tid() : int(threadIdx.x);
}
constexpr int kCus = 256;

// ---------------------------------------------------------------------------
// pass 1, register form: the three velocity fields of a tile are loaded once
// and kept in registers; the vorticity fields are formed from them, so the
// velocity is read from HBM exactly once.  Narrower tiles (PDR_ZINV_LINES)
// keep the registers per thread within two waves per SIMD.
// ---------------------------------------------------------------------------
#ifndef PDR_ZINV_LINES_F32
#define PDR_ZINV_LINES_F32 8
#endif
#ifndef PDR_ZINV_LINES_F64
#define PDR_ZINV_LINES_F64 4
#endif
#ifndef PDR_ZINV_REG
#define PDR_ZINV_REG 1
#endif
template <typename T>
constexpr int zinv_lines(int n) {
  return n <= 512 ? (sizeof(T) == 4 ? PDR_ZINV_LINES_F32 : PDR_ZINV_LINES_F64) : tile_lines<T>(n);
}
template <typename T>
constexpr int lds_zinv_bytes(int n) {
  return (n + zinv_lines<T>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
#define PDR_ZINV_WAVES __attribute__((amdgpu_waves_per_eu(waves_for(lds_zinv_bytes<T>(N)))))
// The single-box register z inverse runs 512-thread workgroups over twice the
// lines (16 FP32 / 8 FP64): each thread keeps the same velocity elements as
// with 256 threads and 8 / 4 lines, and occupancy stays two waves per SIMD, but
// a tile's store of one z row is a whole 128-byte line of the 1r2w array
// instead of half of one (which the neighbouring tile wrote at another time).
// Batched ensembles keep the 256-thread form.
#ifndef PDR_ZINV_THREADS
#define PDR_ZINV_THREADS 512
#endif
template <typename T, int ZT>
constexpr int zinv_lines_t(int n) {
  return zinv_lines<T>(n) * (ZT / kBlock2);
}
template <typename T, int ZT>
constexpr int lds_zinv_bytes_t(int n) {
  return (n + zinv_lines_t<T, ZT>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
// Two workgroups per CU, where the LDS admits them, need the velocity modes and the indices
// in 128 registers: up to 256 points they fit, above only with FRESH indices (512^3
// FP32-mixed 189 -> 122), of which 360, 432 and 480 points in FP32 spill.  Up to one
// workgroup per CU there is no second to make room for (us a launch, FRESH -> not: 64 x 64 x
// 512 FP32-mixed 45.4 -> 34.4, 96 x 96 x 384 43.0 -> 33.4, 64 x 64 x 384 FP64 33.0 -> 28.0;
// more workgroups: 512^3 FP32-mixed 440 -> 464, FP64 748 -> 801, 192 x 192 x 384 FP64 101 ->
// 119; 256^3 FP32-mixed 57.3 -> 50.1, FP64 98.2 -> 88.0; 320 x 320 x 480 FP32-mixed 264 ->
// 222).
template <typename T>
constexpr bool zinv_fresh(int n) {
  return n > 256 && !(sizeof(T) == 4 && (n == 360 || n == 432 || n == 480));
}
// waves per SIMD declared to the register allocator
template <typename T, bool FRESH>
constexpr int zinv_waves_t(int n) {
  return PDR_ZINV_THREADS / kBlock2 * (FRESH || n < 256 ? waves_for(lds_zinv_bytes_t<T, PDR_ZINV_THREADS>(n)) : 1);
}

template <typename T, int N, int ZT = kBlock2, bool FRESH = false>
__device__ __forceinline__ void k2_zinv_r_body(unsigned bid, const Geo& g, const Coef& cf, const cx<T>* __restrict__ u0, const cx<T>* __restrict__ u1,
              const cx<T>* __restrict__ u2, cx<T>* __restrict__ w1, const cx<T>* __restrict__ twg, int ntile) {
  constexpr int L = zinv_lines_t<T, ZT>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKK = 2 * K + 1;
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const int tile = int(bid % unsigned(ntile));
  const int i = int(bid / unsigned(ntile));
  const int j0 = tile * L;
  const int nkj = g.nkj;
  load_tw<T, N, ZT>(tw, twg);
  const long long base = ((long long)i * nkj + j0) * NKK;
  const cx<T>* uu[3] = {u0 + base, u1 + base, u2 + base};
  // A thread keeps the stored modes e = tid + ZT q of the tile (line e / NKK,
  // mode k = e % NKK): the tile's velocity is one contiguous run of L NKK modes
  // per component, and of the truncated band of each line only the positions
  // the first FFT pass reads are written (zeros).
  constexpr int EM = L * NKK;
  constexpr int QM = (EM + ZT - 1) / ZT;
  cx<T> ua[QM], ub[QM], uc[QM];  // u1, u2, u3 of this thread's modes
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int e = int(threadIdx.x) + ZT * q;
    const int line = e / NKK;
    const bool ok = (EM % ZT == 0 || e < EM) && j0 + line < nkj;
    ua[q] = ok ? get<kNrZinv>(&uu[0][e]) : czero<T>();
    ub[q] = ok ? get<kNrZinv>(&uu[1][e]) : czero<T>();
    uc[q] = ok ? get<kNrZinv>(&uu[2][e]) : czero<T>();
  }
  const double wi = double(i);
#pragma unroll
  for (int f = 0; f < 6; ++f) {  // unrolled: every field selection is static
    if (f == 5 && cf.y3) break;  // the inverse y pass forms the last vorticity component
    const int t0 = phase_tid<FRESH>();
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int e = t0 + ZT * q;
      if (EM % ZT == 0 || e < EM) {
        const int line = e / NKK;
        const int k = e - line * NKK;
        const int z = (k <= K) ? k : k + (N - NKK);
        const cx<T> un[3] = {ua[q], ub[q], uc[q]};
        cx<T> v;
        if (f < 3) {
          v = un[f];
        } else {
          // w_c = i sum_n (G[c][n] . k) u_n, the same operations as k2_zinv
          const int c = f - 3;
          const double kv[3] = {wi, wvn2(j0 + line, g.kj), wvn2(k, K)};
          cx<T> acc = czero<T>();
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            const double* G = &cf.G[(c * 3 + n) * 3];
            if ((G[0] != 0.0) || (G[1] != 0.0) || (G[2] != 0.0))
              acc = add(acc, scl(un[n], T(G[0] * kv[0] + G[1] * kv[1] + G[2] * kv[2])));
          }
          v = mk<T>(-acc.y, acc.x);
        }
        buf[line * LD + lds_off<T>(z)] = v;
      }
    }
    zero_band_edges<T, N, L, LD, K, ZT>(buf, t0);
    __syncthreads();
    fft_ip<T, N, L, LD, +1, true, ZT, K>(buf, tw, phase_tid<FRESH>());
    cx<T>* dst = w1 + (long long)f * g.m1 + (long long)i * N * g.ldj + j0;
    for (int idx = phase_tid<FRESH>(); idx < L * N; idx += ZT) {
      const int z = idx / L;
      const int line = idx - z * L;
      if (j0 + line < nkj) put<kNtZinv>(&dst[z * g.ldj + line], buf[line * LD + lds_off<T>(z)]);
    }
    __syncthreads();
  }
}

template <typename T, int N, bool FRESH>
__global__ void __launch_bounds__(PDR_ZINV_THREADS) __attribute__((amdgpu_waves_per_eu(zinv_waves_t<T, FRESH>(N))))
    k2_zinv_r(Geo g, Coef cf, const cx<T>* __restrict__ u0, const cx<T>* __restrict__ u1,
              const cx<T>* __restrict__ u2, cx<T>* __restrict__ w1, const cx<T>* __restrict__ twg, int ntile) {
  k2_zinv_r_body<T, N, PDR_ZINV_THREADS, FRESH>(xcd_remap(blockIdx.x, gridDim.x), g, cf, u0, u1, u2, w1, twg, ntile);
}

// ---------------------------------------------------------------------------
// pass 2: inverse y FFT, (z, i-tile) per block
// ---------------------------------------------------------------------------
// DY: nine fields instead of six, fields 6..8 being d/dy of fields 0..2 (their modes
// times i k2 on the way in)
// W3: the last vorticity component, i sum_n (G[2][n] . k) u_n, has no k3 in it (the
// frame maps k3 to the third laboratory direction alone), so the z pass need not
// transform it: this pass forms it from the modes of the three velocity fields that it
// loads anyway, kept in registers meanwhile.  Five fields then go through the z pass and
// over memory to this one instead of six (us a launch, z and y: 512^3 FP64 932 + 1457 ->
// 749 + 1350, 256^3 FP64 105 + 223 -> 99 + 212, 768 x 128 x 1024 FP32-mixed 594 + 605 ->
// 488 + 590, 512^3 FP32-mixed 542 + 772 -> 441 + 737).
struct YVort {
  double a[3], b[3];  // factors of k1 and k2 for u_1, u_2, u_3
};
template <typename T, int N, bool PL, bool DY, int YT = kBlock2, bool W3 = false>
__device__ __forceinline__ void k2_yinv_body(unsigned bid, const Geo& g, const cx<T>* __restrict__ w1, cx<T>* __restrict__ w2, const cx<T>* __restrict__ twg,
            int ntile, int z0, int nzc, int fpb, const YVort& vort = YVort()) {
  constexpr int PP = y_planes<T, PL>(N);
  constexpr int L = y_lines<T, PL>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKJ = 2 * K + 1;
  constexpr int QE = (L * N + YT - 1) / YT;
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const int tile = int(bid % unsigned(ntile));
  const int zg = int(bid / unsigned(ntile));
  const int zl = PP ? 0 : zg % nzc;   // plane within the chunk (PP: tile = group of PP planes)
  const int fg = PP ? zg : zg / nzc;  // field group
  const int z = z0 + zl;
  const int i0 = PP ? 0 : tile * L;
  const int nki = g.nki;
  const int lstride = g.nz * g.ldj;
  load_tw<T, N, YT>(tw, twg);
  // Tiles of i-lines: a thread takes the stored modes e = tid + YT q of the tile
  // (line e / NKJ, mode j = e % NKJ); of the truncated band of each line only
  // the positions the first FFT pass reads are written (zeros).  Whole-plane
  // tiles fill every position the first pass reads.
  constexpr int EM = L * NKJ;
  constexpr int QM = PP > 0 ? QE : (EM + YT - 1) / YT;
  cx<T> pre[QM];
  // (W3 keeps a field in registers: no room for indices kept from phase to phase)
  auto tid = [&]() { return W3 ? fresh_tid() : int(threadIdx.x); };
  // (the transform's and the stores' fit in FP32: formed anew there too, 785 us a launch
  // at 512^3 against 737)
  auto tid2 = [&]() { return W3 && sizeof(T) == 8 ? fresh_tid() : int(threadIdx.x); };
  auto load = [&](int f) {
    const cx<T>* src = w1 + (long long)(DY && f >= 6 ? f - 6 : f) * g.m1 + ((long long)i0 * g.nz + z) * g.ldj;
    if constexpr (PP == 0) {
      const int t0 = tid();
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int e = t0 + YT * q;
        const int line = e / NKJ;
        cx<T> v = czero<T>();
        if ((EM % YT == 0 || e < EM) && i0 + line < nki) v = get<kNrYinv>(&src[line * lstride + (e - line * NKJ)]);
        pre[q] = DY && f >= 6 ? mul_ik<T>(v, e - line * NKJ, K) : v;
      }
    } else {
#pragma unroll
      for (int q = 0; q < QE; ++q) {
        const int idx = int(threadIdx.x) + YT * q;
        const int line = idx / N;
        const int y = idx - line * N;
        const int j = (y <= K) ? y : ((y >= N - K) ? y - (N - NKJ) : -1);
        const int p = line / (K + 1);
        const int i = line - p * (K + 1);
        const int zz = tile * PP + p;
        cx<T> v = czero<T>();
        if ((L * N % YT == 0 || idx < L * N) && zz < nzc && j >= 0)
          v = get<kNrYinv>(&src[((long long)i * g.nz + zz) * g.ldj + j]);
        pre[q] = DY && f >= 6 ? mul_ik<T>(v, j, K) : v;
      }
    }
  };
  static_assert(!W3 || (PP == 0 && !DY), "W3 is a form of the tiles of i-lines");
  constexpr int QW = W3 ? QM : 1;
  cx<T> acc[QW];
  for (int f = fg * fpb; f < (fg + 1) * fpb; ++f) {
    if (W3 && f == 5) {
#pragma unroll
      for (int q = 0; q < QW; ++q) pre[q] = mk<T>(-acc[q].y, acc[q].x);
    } else {
      load(f);
    }
    if constexpr (PP == 0) {
      // into the tile; W3: times factor(line, j) into acc, the z pass's operations
      auto fill = [&](auto factor) {
        const int t0 = tid();
#pragma unroll
        for (int q = 0; q < QM; ++q) {
          const int e = t0 + YT * q;
          if (EM % YT == 0 || e < EM) {
            const int line = e / NKJ;
            const int j = e - line * NKJ;
            buf[line * LD + lds_off<T>((j <= K) ? j : j + (N - NKJ))] = pre[q];
            if constexpr (W3 && !std::is_same_v<decltype(factor), int>) acc[q] = add(acc[q], scl(pre[q], T(factor(line, j))));
          }
        }
        zero_band_edges<T, N, L, LD, K, YT>(buf, t0);
      };
      if constexpr (W3) {
        if (f == 0) {
#pragma unroll
          for (int q = 0; q < QW; ++q) acc[q] = czero<T>();
        }
        const double ga = f < 3 ? vort.a[f] : 0.0, gb = f < 3 ? vort.b[f] : 0.0;
        // (a frame has one of the two for most components)
        if (ga != 0.0 && gb != 0.0)
          fill([&](int line, int j) { return ga * double(i0 + line) + gb * wvn2(j, K); });
        else if (ga != 0.0)
          fill([&](int line, int) { return ga * double(i0 + line); });
        else if (gb != 0.0)
          fill([&](int, int j) { return gb * wvn2(j, K); });
        else
          fill(0);
      } else {
        fill(0);
      }
    } else {
      // whole-plane tiles: every position but those of the skipped band blocks
      // (the band's other positions hold the zeros of the load)
#pragma unroll
      for (int q = 0; q < QE; ++q) {
        const int idx = int(threadIdx.x) + YT * q;
        if (L * N % YT == 0 || idx < L * N) {
          const int line = idx / N;
          const int y = idx - line * N;
          if (!in_skipped_block<N, K>(y)) buf[line * LD + lds_off<T>(y)] = pre[q];
        }
      }
    }
    __syncthreads();
    fft_ip<T, N, L, LD, +1, true, YT, K>(buf, tw, tid2());
    cx<T>* dst = w2 + (long long)f * g.m2 + (long long)zl * N * g.ldi + i0;
    for (int idx = tid2(); idx < L * N; idx += YT) {
      const int y = idx / L;
      const int line = idx - y * L;
      if constexpr (PP > 0) {
        const int p = line / (K + 1);
        const int zz = tile * PP + p;
        if (zz < nzc)
          put<kNtYinv>(&dst[((long long)zz * N + y) * g.ldi + (line - p * (K + 1))], buf[line * LD + lds_off<T>(y)]);
      } else {
        if (i0 + line < nki) put<kNtYinv>(&dst[y * g.ldi + line], buf[line * LD + lds_off<T>(y)]);
      }
    }
    __syncthreads();
  }
}

// The single-box inverse y pass of tiles of i-lines runs 512-thread workgroups
// over the same tile: half the elements per thread, so the registers of a wave
// fall below half of what 256 threads need and the CU holds twice the waves
// (the tile's LDS then bounds it) to keep more loads in flight.  The
// batched ensembles keep 256 threads.
// Lines of up to 128 points take 256: their tile is a butterfly or less per thread of
// 512, and more tiles fit a CU (us a launch, 512 -> 256 threads: 128^3 FP64 31.3 -> 29.0,
// 128^3 FP32-mixed 20.1 -> 17.9, 768 x 128 x 1024 FP32-mixed 590 -> 551, 120 x 48 x 96 FP64
// 20.8 -> 15.1; but 160^3 FP32-mixed 33.2 -> 36.9).
#ifndef PDR_YINV_THREADS
#define PDR_YINV_THREADS 512
#endif
#ifndef PDR_YINV_SHORT
#define PDR_YINV_SHORT 128
#endif
// FP64 whole-plane tiles (some 50 KB of LDS, three to a CU) take 512 as well, in both
// directions (us a launch, 256 -> 512: inverse at 96^3 22.8 -> 18.2, nine fields 27.7 -> 24.2);
// the batched ensembles keep 256.
template <typename T>
constexpr int yplane_threads() {
  return sizeof(T) == 8 ? 2 * kBlock2 : kBlock2;
}
template <typename T, int N, bool PL>
constexpr int yinv_threads() {
  return y_planes<T, PL>(N) ? yplane_threads<T>() : N <= PDR_YINV_SHORT ? kBlock2 : PDR_YINV_THREADS;
}
// waves per SIMD declared to the register allocator: as for the other passes
// (at most two 256-thread workgroups), or the two waves per SIMD of each
// 512-thread workgroup times the workgroups the LDS admits, at most four
template <typename T, int N, bool PL>
constexpr int yinv_waves() {
  if (!y_planes<T, PL>(N) && N <= PDR_YINV_SHORT) return 4;
  constexpr int wg = kLdsPerCu / lds_y_bytes<T, PL>(N) < 1 ? 1 : kLdsPerCu / lds_y_bytes<T, PL>(N);
  return yinv_threads<T, N, PL>() == kBlock2 ? waves_for(lds_y_bytes<T, PL>(N))
                                          : (wg * (yinv_threads<T, N, PL>() / kBlock2) > 4 ? 4 : wg * (yinv_threads<T, N, PL>() / kBlock2));
}

template <typename T, int N, bool PL, bool DY>
__global__ void __launch_bounds__((yinv_threads<T, N, PL>())) __attribute__((amdgpu_waves_per_eu(yinv_waves<T, N, PL>())))
    k2_yinv(Geo g, const cx<T>* __restrict__ w1, cx<T>* __restrict__ w2, const cx<T>* __restrict__ twg,
            int ntile, int z0, int nzc, int fpb) {
  k2_yinv_body<T, N, PL, DY, yinv_threads<T, N, PL>()>(xcd_remap(blockIdx.x, gridDim.x), g, w1, w2, twg, ntile, z0, nzc, fpb);
}

// the five fields of a z pass with y3 (YVort)
template <typename T, int N>
__global__ void __launch_bounds__((yinv_threads<T, N, false>())) __attribute__((amdgpu_waves_per_eu(yinv_waves<T, N, false>())))
    k2_yinv5(Geo g, YVort vort, const cx<T>* __restrict__ w1, cx<T>* __restrict__ w2, const cx<T>* __restrict__ twg,
             int ntile, int z0, int nzc) {
  k2_yinv_body<T, N, false, false, yinv_threads<T, N, false>(), true>(xcd_remap(blockIdx.x, gridDim.x), g, w1, w2, twg,
                                                                    ntile, z0, nzc, 6, vort);
}

// ---------------------------------------------------------------------------
// pass 3: RB rows (z, y0..y0+RB-1) per block: c2r, product, r2c
// ---------------------------------------------------------------------------
// Real-space moments (RS): 0 none; a thread's own points summed in FP32 (1) or FP64 (2).
template <typename T, int N, int RS, int XT = kBlock2>
__device__ __forceinline__ void k2_xpass_body(unsigned bid, const Geo& g, const Coef& cf, cx<T>* __restrict__ w2, T* __restrict__ ur, int want_tr, int want_cfl,
             unsigned long long* __restrict__ umax, const cx<T>* __restrict__ twg, int ntile, int z0,
             double* __restrict__ rsp) {
  constexpr int RB = xrows<T, RS != 0>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int KI = N / 3;
  constexpr int NKI = KI + 1;
  constexpr int IT = (RB * N + XT - 1) / XT;  // product items per thread
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ T red[XT / 64];  // the CFL maximum of each wave
  constexpr bool TWG = x_tw_global<T>(N);
  cx<T>* const lds0 = reinterpret_cast<cx<T>*>(smem);
  const cx<T>* const tw = TWG ? twg : lds0;
  cx<T>* const buf = TWG ? lds0 : lds0 + N;
  const int tile = int(bid % unsigned(ntile));
  const int zl = int(bid / unsigned(ntile));  // plane within the chunk
  const int z = z0 + zl;
  const int y0 = tile * RB;
  const int ny = g.ny;
  if constexpr (!TWG) load_tw<T, N, XT>(lds0, twg);
  cx<T>* rowp = w2 + ((long long)zl * ny + y0) * g.ldi;
  // fill: the 3 * RB lines pack pairs of real inputs (p = 0: u1 + i u2,
  // 1: u3 + i w1, 2: w2 + i w3).  Each stored mode m' = 0..KI of a pair (a, b) is
  // loaded once and written to both m' and its Hermitian image N - m'
  // (conj(a) + i conj(b)); c2r uses only the real part of the DC term; the band
  // KI < m < N - KI is zero, and only its positions that the first FFT pass
  // reads are written.  All loads of a thread precede its LDS stores.
  if constexpr (NKI >= 128) {
    // long lines: thread m takes mode m of every line, so the global row bases
    // are workgroup-uniform, the LDS line offsets compile-time constants and
    // the per-element index arithmetic is one address add
    constexpr int NL = 3 * RB;
    const cx<T>* fa[NL];
#pragma unroll
    for (int line = 0; line < NL; ++line) fa[line] = rowp + (long long)(2 * (line % 3)) * g.m2 + (line / 3) * g.ldi;
    for (int m0 = 0; m0 < NKI; m0 += XT) {
      const int m = m0 + int(threadIdx.x);
      if (m < NKI) {
        cx<T> A[NL], B[NL];
#pragma unroll
        for (int line = 0; line < NL; ++line) {
          A[line] = czero<T>();
          B[line] = czero<T>();
          if (y0 + line / 3 < ny) {
            A[line] = get<kNrXpass>(&fa[line][m]);
            B[line] = get<kNrXpass>(&fa[line][g.m2 + m]);
          }
        }
        const int om = lds_off<T>(m), on = lds_off<T>(N - m);
#pragma unroll
        for (int line = 0; line < NL; ++line) {
          cx<T>* row = buf + line * LD;
          if (m == 0) {
            row[0] = mk<T>(A[line].x, B[line].x);
          } else {
            row[om] = mk<T>(A[line].x - B[line].y, A[line].y + B[line].x);
            row[on] = mk<T>(A[line].x + B[line].y, B[line].x - A[line].y);
          }
        }
      }
    }
  } else {
    constexpr int EL = 3 * RB * NKI;
    constexpr int QL = (EL + XT - 1) / XT;
    cx<T> A[QL], B[QL];
#pragma unroll
    for (int q = 0; q < QL; ++q) {
      const int idx = int(threadIdx.x) + XT * q;
      const int line = idx / NKI;
      const int m = idx - line * NKI;
      const int r = line / 3;
      const int p = line - 3 * r;
      A[q] = czero<T>();
      B[q] = czero<T>();
      if ((EL % XT == 0 || idx < EL) && y0 + r < ny) {
        const cx<T>* fa = rowp + (long long)(2 * p) * g.m2 + r * g.ldi;
        A[q] = get<kNrXpass>(&fa[m]);
        B[q] = get<kNrXpass>(&fa[g.m2 + m]);
      }
    }
#pragma unroll
    for (int q = 0; q < QL; ++q) {
      const int idx = int(threadIdx.x) + XT * q;
      if (EL % XT == 0 || idx < EL) {
        const int line = idx / NKI;
        const int m = idx - line * NKI;
        cx<T>* row = buf + line * LD;
        if (m == 0) {
          row[0] = mk<T>(A[q].x, B[q].x);
        } else {
          row[lds_off<T>(m)] = mk<T>(A[q].x - B[q].y, A[q].y + B[q].x);
          row[lds_off<T>(N - m)] = mk<T>(A[q].x + B[q].y, B[q].x - A[q].y);
        }
      }
    }
  }
  zero_band_edges<T, N, 3 * RB, LD, KI, XT>(buf);
  __syncthreads();
  fft_ip<T, N, 3 * RB, LD, +1, !TWG, XT, KI>(buf, tw);
  T V[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    if constexpr (sizeof(T) == 4)
      V[q] = cf.Vf[q];
    else
      V[q] = T(cf.V[q]);
  }
  T nl[IT][3];
  T lmax = T(0);
  T* urow = ur + ((long long)z * ny + y0) * N * 3;
  using RA = std::conditional_t<RS == 2, double, T>;
  RsAccT<RA> acc;
  if (RS) rs_init(acc);
  // the product, with the frame's form a compile-time choice (no per-point select)
  auto product = [&](auto form_c) {
    constexpr bool FORM = decltype(form_c)::value;
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int idx = int(threadIdx.x) + XT * q;
    if ((RB * N) % XT == 0 || idx < RB * N) {
      const int r = idx / N;
      const int x = idx - r * N;
      const cx<T> a = buf[(3 * r) * LD + lds_off<T>(x)], b = buf[(3 * r + 1) * LD + lds_off<T>(x)],
                  c = buf[(3 * r + 2) * LD + lds_off<T>(x)];
      const T u1 = a.x, u2 = a.y, u3 = b.x, o1 = b.y, o2 = c.x, o3 = c.y;
      const T v1 = V[0] * u1 + V[1] * u2 + V[2] * u3;
      const T v2 = V[3] * u1 + V[4] * u2 + V[5] * u3;
      const T v3 = V[6] * u1 + V[7] * u2 + V[8] * u3;
      // omega x (binv u) (BF_ROT), or omega x u (isotropic with binv = I, R_ROT)
      const T w1 = FORM ? u1 : v1, w2 = FORM ? u2 : v2, w3 = FORM ? u3 : v3;
      nl[q][0] = o2 * w3 - o3 * w2;
      nl[q][1] = o3 * w1 - o1 * w3;
      nl[q][2] = o1 * w2 - o2 * w1;
      if (want_tr && y0 + r < ny) {
        T* d = urow + idx * 3;
        put1<kNtXpass>(d, u1);
        put1<kNtXpass>(d + 1, u2);
        put1<kNtXpass>(d + 2, u3);
      }
      if (want_cfl) {
        const T s = fabs(v1) + fabs(v2) + fabs(v3);  // lab-frame velocity (src/pf_fluidstats.f90:853-866, 914)
        lmax = s > lmax ? s : lmax;
      }
      if (RS && y0 + r < ny) rs_add(acc, RA(v1), RA(v2), RA(v3), RA(o1), RA(o2), RA(o3));
    }
  }
  };
  if (cf.form)
    product(std::true_type{});
  else
    product(std::false_type{});
  if constexpr (RS != 0) {
    // partial of this workgroup at its place in the whole box: (z, tile); where
    // the x tile can hold the threads' partials (the product has read it), they
    // are reduced through it
    double* const rso = rsp + ((long long)z * ntile + tile) * kRsWidth;
    __shared__ double rs_lds[kRsWidth * 4];
    if constexpr (kRsWidth * (XT + 1) * sizeof(RA) <= 3 * RB * LD * sizeof(cx<T>)) {
      __syncthreads();
      rs_block_out_lds<XT>(acc, reinterpret_cast<RA*>(buf), rs_lds, rso);
    } else {
      static_assert(kRsWidth * (XT / 64) <= kRsWidth * 4, "rs_block_out's LDS");
      rs_block_out(acc, rs_lds, rso);
    }
  }
  __syncthreads();
  // forward lines: r -> n1 + i n2 of row r; RB + r/2 -> n3 of rows (r, r+1)
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int idx = int(threadIdx.x) + XT * q;
    if ((RB * N) % XT == 0 || idx < RB * N) {
      const int r = idx / N;
      const int x = idx - r * N;
      buf[r * LD + lds_off<T>(x)] = mk<T>(nl[q][0], nl[q][1]);
      cx<T>* p3 = &buf[(RB + r / 2) * LD + lds_off<T>(x)];
      if (r & 1)
        p3->y = nl[q][2];
      else
        p3->x = nl[q][2];
    }
  }
  __syncthreads();
  fft_ip<T, N, 3 * RB / 2, LD, -1, !TWG, XT>(buf, tw);
  // unpack the pairs: row r of n1 + i n2 and half of line RB + r/2 give the
  // stored modes m = 0..KI of the three forward fields
  auto unpack = [&](int r, int m, int om, int omr) {
    const cx<T> Z = buf[r * LD + om], Zr = buf[r * LD + omr];
    const cx<T> W = buf[(RB + r / 2) * LD + om], Wr = buf[(RB + r / 2) * LD + omr];
    cx<T>* d0 = rowp + r * g.ldi + m;
    put<kNtXpass>(d0, mk<T>(T(0.5) * (Z.x + Zr.x), T(0.5) * (Z.y - Zr.y)));
    put<kNtXpass>(d0 + g.m2, mk<T>(T(0.5) * (Z.y + Zr.y), T(-0.5) * (Z.x - Zr.x)));
    if (r & 1)
      put<kNtXpass>(d0 + 2 * g.m2, mk<T>(T(0.5) * (W.y + Wr.y), T(-0.5) * (W.x - Wr.x)));
    else
      put<kNtXpass>(d0 + 2 * g.m2, mk<T>(T(0.5) * (W.x + Wr.x), T(0.5) * (W.y - Wr.y)));
  };
  if constexpr (NKI >= 128) {
    for (int m0 = 0; m0 < NKI; m0 += XT) {
      const int m = m0 + int(threadIdx.x);
      if (m < NKI) {
        const int om = lds_off<T>(m), omr = lds_off<T>((m == 0) ? 0 : N - m);
#pragma unroll
        for (int r = 0; r < RB; ++r)
          if (y0 + r < ny) unpack(r, m, om, omr);
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < RB * NKI; idx += XT) {
      const int r = idx / NKI;
      const int m = idx - r * NKI;
      if (y0 + r >= ny) continue;
      const int mr = (m == 0) ? 0 : N - m;
      unpack(r, m, lds_off<T>(m), lds_off<T>(mr));
    }
  }
  if (want_cfl) {
    // maximum over the wave, then over the XT / 64 waves of the workgroup
    T m = lmax;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const T o = __shfl_xor(m, off);
      m = o > m ? o : m;
    }
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      T r = red[0];
      for (int w = 1; w < XT / 64; ++w) r = red[w] > r ? red[w] : r;
      raise_max(umax, (unsigned long long)__double_as_longlong(double(r)));
    }
  }
}

template <typename T, int N, int RS>
__global__ void __launch_bounds__((xthreads<T, RS>(N))) __attribute__((amdgpu_waves_per_eu(xwaves<T, RS>(N))))
    k2_xpass(Geo g, Coef cf, cx<T>* __restrict__ w2, T* __restrict__ ur, int want_tr, int want_cfl,
             unsigned long long* __restrict__ umax, const cx<T>* __restrict__ twg, int ntile, int z0,
             double* __restrict__ rsp) {
  k2_xpass_body<T, N, RS, xthreads<T, RS>(N)>(xcd_remap(blockIdx.x, gridDim.x), g, cf, w2, ur, want_tr, want_cfl, umax, twg, ntile, z0,
                          rsp);
}

// ---------------------------------------------------------------------------
// pass 3, NS_R_CONV: the y pass hands over u, du/dz and du/dy (fields 0..2, 3..5 and
// 6..8); du/dx is formed here, its modes times i k1 on the way into the tile.  RB rows
// per block, six complex lines of two real rows each: (u1, u2), (u3, dz u1),
// (dz u2, dz u3), (dy u1, dy u2), (dy u3, dx u1), (dx u2, dx u3); then
// NL_i = sum_j sum_k bmat(k,j) du_i/dx_k u_j (f_RK3ComputeNonlinearRConv,
// src/pf_rk3.f90:1717-1774) and the forward lines of k2_xpass.  Forming each
// derivative in its own pass moves 6 fields through the z pass and 9 through the y
// pass, where transforming u and nine gradients from the z pass on moves 18 and 18
// (three sweeps of six): ten FP64 steps at 96^3 14.7 -> 3.39 ms against the
// runtime-radix kernels' three sweeps (launch_conv_front).  The moments take u, binv u and du/dx, as the reference's
// f_FluidstatsRs2D reads u4..u6 (src/pf_fluidstats.f90:846-917), summed in FP64.
// ---------------------------------------------------------------------------
template <typename T>
constexpr int xrows_conv(int n) {  // half the rows of k2_xpass: twice the lines a row
  if (sizeof(T) == 4 && n > 96 && n <= 128) return 4;  // (128^3: 33.4 us a launch against 35.7 with 2; FP64 57.3 with 2, 68.6 with 4)
  return xrows<T>(n) > 4 ? xrows<T>(n) / 2 : 2;
}
template <typename T>
constexpr int lds_xc_bytes(int n) {
  return ((x_tw_global<T>(n) ? 0 : n) + 6 * xrows_conv<T>(n) * lds_ld<T>(n)) * int(sizeof(cx<T>));
}
#define PDR_XC_WAVES __attribute__((amdgpu_waves_per_eu(waves_for(lds_xc_bytes<T>(N)))))

template <typename T, int N, bool RS>
__global__ void __launch_bounds__(kBlock2) PDR_XC_WAVES
    k2_xpass_conv(Geo g, Coef cf, cx<T>* __restrict__ w2, T* __restrict__ ur, int want_tr, int want_cfl,
                  unsigned long long* __restrict__ umax, const cx<T>* __restrict__ twg, int ntile,
                  double* __restrict__ rsp) {
  constexpr int RB = xrows_conv<T>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int KI = N / 3;
  constexpr int NKI = KI + 1;
  constexpr int IT = (RB * N + kBlock2 - 1) / kBlock2;  // product items per thread
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ T red[kBlock2 / 64];
  constexpr bool TWG = x_tw_global<T>(N);
  cx<T>* const lds0 = reinterpret_cast<cx<T>*>(smem);
  const cx<T>* const tw = TWG ? twg : lds0;
  cx<T>* const buf = TWG ? lds0 : lds0 + N;
  const unsigned bid = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = int(bid % unsigned(ntile));
  const int z = int(bid / unsigned(ntile));
  const int y0 = tile * RB;
  const int ny = g.ny;
  if constexpr (!TWG) load_tw<T, N>(lds0, twg);
  cx<T>* rowp = w2 + ((long long)z * ny + y0) * g.ldi;
  // one (row, mode) per thread: nine modes in, twelve out as six packed lines, each
  // at its mode and its Hermitian image (c2r uses only the real part of the DC term)
  for (int idx = threadIdx.x; idx < RB * NKI; idx += kBlock2) {
    const int r = idx / NKI;
    const int m = idx - r * NKI;
    cx<T> f[12];
#pragma unroll
    for (int q = 0; q < 9; ++q) f[q] = (y0 + r < ny) ? rowp[(long long)q * g.m2 + r * g.ldi + m] : czero<T>();
#pragma unroll
    for (int q = 0; q < 3; ++q) f[9 + q] = mk<T>(-T(m) * f[q].y, T(m) * f[q].x);
    cx<T>* row = buf + 6 * r * LD;
    const int om = lds_off<T>(m), on = lds_off<T>(N - m);
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      const cx<T> A = f[2 * p], B = f[2 * p + 1];
      if (m == 0) {
        row[p * LD] = mk<T>(A.x, B.x);
      } else {
        row[p * LD + om] = mk<T>(A.x - B.y, A.y + B.x);
        row[p * LD + on] = mk<T>(A.x + B.y, B.x - A.y);
      }
    }
  }
  zero_band_edges<T, N, 6 * RB, LD, KI>(buf);
  __syncthreads();
  fft_ip<T, N, 6 * RB, LD, +1, !TWG, kBlock2, KI>(buf, tw);
  T V[9], Bk[9];  // masked binv; bmat as [k][j]
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    V[q] = T(cf.V[q]);
    Bk[q] = T(cf.Bm[q]);
  }
  T nl[IT][3];
  T lmax = T(0);
  T* urow = ur + ((long long)z * ny + y0) * N * 3;
  RsAcc acc;
  if (RS) rs_init(acc);
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int idx = int(threadIdx.x) + kBlock2 * q;
    if ((RB * N) % kBlock2 == 0 || idx < RB * N) {
      const int r = idx / N;
      const int x = idx - r * N;
      T f[12];  // u, du/dz, du/dy, du/dx
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        const cx<T> v = buf[(6 * r + p) * LD + lds_off<T>(x)];
        f[2 * p] = v.x;
        f[2 * p + 1] = v.y;
      }
      const int at[3] = {9, 6, 3};  // d/dx, d/dy, d/dz
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        T a = T(0);
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int k = 0; k < 3; ++k) a = a + (Bk[3 * k + j] * f[at[k] + i] * f[j]);
        nl[q][i] = a;
      }
      if (want_tr && y0 + r < ny) {
        T* d = urow + idx * 3;
        put1<kNtXpass>(d, f[0]);
        put1<kNtXpass>(d + 1, f[1]);
        put1<kNtXpass>(d + 2, f[2]);
      }
      if (want_cfl || RS) {
        const T v1 = V[0] * f[0] + V[1] * f[1] + V[2] * f[2];
        const T v2 = V[3] * f[0] + V[4] * f[1] + V[5] * f[2];
        const T v3 = V[6] * f[0] + V[7] * f[1] + V[8] * f[2];
        const T s = fabs(v1) + fabs(v2) + fabs(v3);
        lmax = s > lmax ? s : lmax;
        if (RS && y0 + r < ny)
          rs_add(acc, double(v1), double(v2), double(v3), double(f[9]), double(f[10]), double(f[11]));
      }
    }
  }
  if constexpr (RS) {
    __shared__ double rs_lds[kRsWidth * (kBlock2 / 64)];
    rs_block_out(acc, rs_lds, rsp + ((long long)z * ntile + tile) * kRsWidth);
  }
  __syncthreads();
  // forward lines and stored modes as in k2_xpass: r -> n1 + i n2 of row r,
  // RB + r/2 -> n3 of rows (r, r+1)
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int idx = int(threadIdx.x) + kBlock2 * q;
    if ((RB * N) % kBlock2 == 0 || idx < RB * N) {
      const int r = idx / N;
      const int x = idx - r * N;
      buf[r * LD + lds_off<T>(x)] = mk<T>(nl[q][0], nl[q][1]);
      cx<T>* p3 = &buf[(RB + r / 2) * LD + lds_off<T>(x)];
      if (r & 1)
        p3->y = nl[q][2];
      else
        p3->x = nl[q][2];
    }
  }
  __syncthreads();
  fft_ip<T, N, 3 * RB / 2, LD, -1, !TWG>(buf, tw);
  for (int idx = threadIdx.x; idx < RB * NKI; idx += kBlock2) {
    const int r = idx / NKI;
    const int m = idx - r * NKI;
    if (y0 + r >= ny) continue;
    const int om = lds_off<T>(m), omr = lds_off<T>((m == 0) ? 0 : N - m);
    const cx<T> Z = buf[r * LD + om], Zr = buf[r * LD + omr];
    const cx<T> W = buf[(RB + r / 2) * LD + om], Wr = buf[(RB + r / 2) * LD + omr];
    cx<T>* d0 = rowp + r * g.ldi + m;
    put<kNtXpass>(d0, mk<T>(T(0.5) * (Z.x + Zr.x), T(0.5) * (Z.y - Zr.y)));
    put<kNtXpass>(d0 + g.m2, mk<T>(T(0.5) * (Z.y + Zr.y), T(-0.5) * (Z.x - Zr.x)));
    if (r & 1)
      put<kNtXpass>(d0 + 2 * g.m2, mk<T>(T(0.5) * (W.y + Wr.y), T(-0.5) * (W.x - Wr.x)));
    else
      put<kNtXpass>(d0 + 2 * g.m2, mk<T>(T(0.5) * (W.x + Wr.x), T(0.5) * (W.y - Wr.y)));
  }
  if (want_cfl) {
    T m = lmax;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const T o = __shfl_xor(m, off);
      m = o > m ? o : m;
    }
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      T r = red[0];
      for (int w = 1; w < kBlock2 / 64; ++w) r = red[w] > r ? red[w] : r;
      raise_max(umax, (unsigned long long)__double_as_longlong(double(r)));
    }
  }
}

// ---------------------------------------------------------------------------
// pass 4: forward y FFT + truncation, (z, i-tile) per block
// ---------------------------------------------------------------------------
template <typename T, int N, bool PL, int YT = kBlock2>
__device__ __forceinline__ void k2_yfwd_body(unsigned bid, const Geo& g, const cx<T>* __restrict__ w2, cx<T>* __restrict__ w1, const cx<T>* __restrict__ twg,
            int ntile, int z0, int nzc, int fpb) {
  constexpr int PP = y_planes<T, PL>(N);
  constexpr int L = y_lines_fwd<T, PL>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKJ = 2 * K + 1;
  constexpr int QE = (L * N + YT - 1) / YT;
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const int tile = int(bid % unsigned(ntile));
  const int zg = int(bid / unsigned(ntile));
  const int zl = PP ? 0 : zg % nzc;   // PP: tile = group of PP planes
  const int fg = PP ? zg : zg / nzc;
  const int z = z0 + zl;
  const int i0 = PP ? 0 : tile * L;
  const int nki = g.nki;
  const int lstride = g.nz * g.ldj;
  load_tw<T, N, YT>(tw, twg);
  cx<T> pre[QE];
  auto load = [&](int f) {
    const cx<T>* src = w2 + (long long)f * g.m2 + (long long)zl * N * g.ldi + i0;
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = int(threadIdx.x) + YT * q;
      const int y = idx / L;
      const int line = idx - y * L;
      if constexpr (PP > 0) {
        const int p = line / (K + 1);
        const int zz = tile * PP + p;
        pre[q] = ((L * N % YT == 0 || idx < L * N) && zz < nzc)
                     ? get<kNrYfwd>(&src[((long long)zz * N + y) * g.ldi + (line - p * (K + 1))])
                     : czero<T>();
      } else {
        pre[q] = ((L * N % YT == 0 || idx < L * N) && i0 + line < nki) ? get<kNrYfwd>(&src[y * g.ldi + line])
                                                                          : czero<T>();
      }
    }
  };
  for (int f = fg * fpb; f < (fg + 1) * fpb; ++f) {
    load(f);
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = int(threadIdx.x) + YT * q;
      if (L * N % YT == 0 || idx < L * N) {
        const int y = idx / L;
        buf[(idx - y * L) * LD + lds_off<T>(y)] = pre[q];
      }
    }
    __syncthreads();
    fft_ip<T, N, L, LD, -1, true, YT>(buf, tw);
    cx<T>* dst = w1 + (long long)f * g.m1 + ((long long)i0 * g.nz + z) * g.ldj;
    for (int idx = threadIdx.x; idx < L * NKJ; idx += YT) {
      const int line = idx / NKJ;
      const int j = idx - line * NKJ;
      const int yy = (j <= K) ? j : N - NKJ + j;
      if constexpr (PP > 0) {
        const int p = line / (K + 1);
        const int zz = tile * PP + p;
        if (zz < nzc)
          put<kNtYfwd>(&dst[((long long)(line - p * (K + 1)) * g.nz + zz) * g.ldj + j], buf[line * LD + lds_off<T>(yy)]);
      } else {
        if (i0 + line < nki) put<kNtYfwd>(&dst[line * lstride + j], buf[line * LD + lds_off<T>(yy)]);
      }
    }
    __syncthreads();
  }
}

template <typename T, int N, bool PL>
constexpr int yfwd_threads() {
  return y_planes<T, PL>(N) ? yplane_threads<T>() : zthreads(N);
}
template <typename T, int N, bool PL>
__global__ void __launch_bounds__((yfwd_threads<T, N, PL>()))
    __attribute__((amdgpu_waves_per_eu(waves_for(lds_yf_bytes<T, PL>(N)) * (yfwd_threads<T, N, PL>() / kBlock2))))
    k2_yfwd(Geo g, const cx<T>* __restrict__ w2, cx<T>* __restrict__ w1, const cx<T>* __restrict__ twg,
            int ntile, int z0, int nzc, int fpb) {
  k2_yfwd_body<T, N, PL, yfwd_threads<T, N, PL>()>(xcd_remap(blockIdx.x, gridDim.x), g, w2, w1, twg, ntile, z0, nzc, fpb);
}

// ---------------------------------------------------------------------------
// pass 5: forward z FFT, normalisation, truncation -> NL [c][i][j][k]
// ---------------------------------------------------------------------------
template <typename T, int N>
__global__ void __launch_bounds__((zthreads(N))) __attribute__((amdgpu_waves_per_eu(waves_for(lds_fwd_bytes<T>(N)) * (zthreads(N) / kBlock2))))
    k2_zfwd(Geo g, const cx<T>* __restrict__ w1, cx<T>* __restrict__ nl, const cx<T>* __restrict__ twg,
            int ntile, T norm) {
  constexpr int ZT = zthreads(N);
  constexpr int L = tile_lines_fwd<T>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKK = 2 * K + 1;
  constexpr int QE = (L * N + ZT - 1) / ZT;
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const unsigned bid = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = int(bid % unsigned(ntile));
  const int i = int(bid / unsigned(ntile));
  const int j0 = tile * L;
  const int nkj = g.nkj;
  load_tw<T, N, ZT>(tw, twg);
  cx<T> pre[QE];
  auto load = [&](int f) {
    const cx<T>* src = w1 + (long long)f * g.m1 + (long long)i * N * g.ldj + j0;
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = int(threadIdx.x) + ZT * q;
      const int z = idx / L;
      const int line = idx - z * L;
      pre[q] = ((L * N % ZT == 0 || idx < L * N) && j0 + line < nkj) ? get<kNrZfwd>(&src[z * g.ldj + line]) : czero<T>();
    }
  };
  for (int f = 0; f < 3; ++f) {
    load(f);
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = int(threadIdx.x) + ZT * q;
      if (L * N % ZT == 0 || idx < L * N) {
        const int z = idx / L;
        buf[(idx - z * L) * LD + lds_off<T>(z)] = pre[q];
      }
    }
    __syncthreads();
    fft_ip<T, N, L, LD, -1, true, ZT>(buf, tw);
    cx<T>* dst = nl + (long long)f * g.mw + ((long long)i * nkj + j0) * NKK;
    const int nl_lines = (nkj - j0) < L ? (nkj - j0) : L;
    for (int idx = threadIdx.x; idx < nl_lines * NKK; idx += ZT) {
      const int line = idx / NKK;
      const int k = idx - line * NKK;
      const int zz = (k <= K) ? k : N - NKK + k;
      put<kNtZfwd>(&dst[idx], scl(buf[line * LD + lds_off<T>(zz)], norm));
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// pass 5 + FormF: forward z FFT of the three NL fields of an (i, j-tile), then
// FormF / RK3 / continuity fix of the tile's modes straight from registers:
// NL never goes through HBM (f_RK3SolveNavierStokes, src/pf_rk3.f90:2067-2130,
// does the same per i slice).  The modes of a tile, (i, j0..j0+L-1, all k), are
// contiguous in the wave arrays.
// ---------------------------------------------------------------------------
#ifndef PDR_ZFF_PF
#define PDR_ZFF_PF 1
#endif
// FRESH indices where they bring the compiled kernel's registers from two workgroups of 256
// threads per CU to three, which depends on the length and on the forcing's code (FRC as
// below); in boxes of more than two per CU (us a launch, FRESH -> not: unforced 512^3
// FP32-mixed 533 -> 568, 320 x 320 x 480 224 -> 252, 192 x 128 x 256 FP64 57.8 -> 64.3, forced
// 384^3 FP32-mixed 249 -> 267; two per CU 64 x 64 x 512 FP32-mixed 32.5 -> 28.9, 128 x 96 x 256
// FP64 33.2 -> 30.9; two, or three, in both forms 256^3 FP32-mixed 80.9 -> 75.0, 384^3
// 252 -> 239, FP64 499 -> 486, forced 512^3 FP32-mixed 584 -> 563).
template <typename T>
constexpr bool zff_fresh(int n, int frc) {
  if (sizeof(T) == 8) return n == 256 && frc == 0;
  const int longest = frc == 0 ? 512 : frc == 1 ? 432 : 384;
  const int three = frc == 0 ? 384 : frc == 1 ? 320 : 256;  // multiples of 32 up to here have three
  return n > 256 && n <= longest && (n % 32 != 0 || n > three);
}
template <typename T, int N, int FT = kBlock2, int FRC = 2, bool FRESH = false>
__device__ __forceinline__ void k2_zfwd_formf_body(unsigned bid, const Geo& g, const Coef& cf, const cx<T>* __restrict__ w1, cx<T>* __restrict__ u0, cx<T>* __restrict__ u1,
                  cx<T>* __restrict__ u2, cx<T>* __restrict__ r0, cx<T>* __restrict__ r1, cx<T>* __restrict__ r2,
                  const double2* __restrict__ frc, int fnk, double fkf, double beta, double gdt,
                  const cx<T>* __restrict__ twg, int ntile, T norm) {
  constexpr int L = tile_lines_fwd<T>(N);
  constexpr int LD = lds_ld<T>(N);
  constexpr int K = N / 3;
  constexpr int NKK = 2 * K + 1;
  constexpr int QE = (L * N + FT - 1) / FT;
  constexpr int QF = (L * NKK + FT - 1) / FT;  // modes per thread
  extern __shared__ __align__(16) unsigned char smem[];
  cx<T>* tw = reinterpret_cast<cx<T>*>(smem);
  cx<T>* buf = tw + N;
  const int tile = int(bid % unsigned(ntile));
  const int i = int(bid / unsigned(ntile));
  const int j0 = tile * L;
  const int nkj = g.nkj;
  const int nl_lines = (nkj - j0) < L ? (nkj - j0) : L;
  load_tw<T, N, FT>(tw, twg);
  cx<T> pre[QE];
  cx<T> nlv[3][QF];
  auto load = [&](int f) {
    const cx<T>* src = w1 + (long long)f * g.m1 + (long long)i * N * g.ldj + j0;
    const int t0 = phase_tid<FRESH>();
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = t0 + FT * q;
      const int z = idx / L;
      const int line = idx - z * L;
      pre[q] = ((L * N % FT == 0 || idx < L * N) && j0 + line < nkj) ? src[z * g.ldj + line] : czero<T>();
    }
  };
  // FP32 lines of 256..512 points: the next field's loads are issued before
  // this field's transform, whose work then hides their latency (the registers
  // of one field's elements fit beside the transform's)
  constexpr bool PF = PDR_ZFF_PF && sizeof(T) == 4 && N >= 256 && N <= 512;
  if constexpr (PF) load(0);
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    if constexpr (!PF) load(f);
    const int ts = phase_tid<FRESH>();
#pragma unroll
    for (int q = 0; q < QE; ++q) {
      const int idx = ts + FT * q;
      if (L * N % FT == 0 || idx < L * N) {
        const int z = idx / L;
        buf[(idx - z * L) * LD + lds_off<T>(z)] = pre[q];
      }
    }
    __syncthreads();
    if constexpr (PF) {
      if (f < 2) load(f + 1);
    }
    fft_ip<T, N, L, LD, -1, true, FT>(buf, tw, phase_tid<FRESH>());
    const int tm = phase_tid<FRESH>();
#pragma unroll
    for (int q = 0; q < QF; ++q) {
      const int idx = tm + FT * q;
      const int line = idx / NKK;
      const int k = idx - line * NKK;
      const int zz = (k <= K) ? k : N - NKK + k;
      nlv[f][q] = (idx < nl_lines * NKK) ? scl(buf[line * LD + lds_off<T>(zz)], norm) : czero<T>();
    }
    __syncthreads();
  }
  const long long e0 = ((long long)i * nkj + j0) * NKK;
  const int te = phase_tid<FRESH>();
#pragma unroll
  for (int q = 0; q < QF; ++q) {
    const int idx = te + FT * q;
    if (idx < nl_lines * NKK) {
      const int line = idx / NKK;
      formf_mode<T, FRC>(g, cf, i, j0 + line, idx - line * NKK, e0 + idx, nlv[0][q], nlv[1][q], nlv[2][q], u0, u1, u2,
                    r0, r1, r2, frc, fnk, fkf, beta, gdt);
    }
  }
}

// FRC: 0 unforced, 1 isotropic forcing, 2 deformed isotropic forcing
template <typename T, int N, int FRC, bool FRESH>
__global__ void __launch_bounds__(kBlock2) PDR_FWD_WAVES
    k2_zfwd_formf(Geo g, Coef cf, const cx<T>* __restrict__ w1, cx<T>* __restrict__ u0, cx<T>* __restrict__ u1,
                  cx<T>* __restrict__ u2, cx<T>* __restrict__ r0, cx<T>* __restrict__ r1, cx<T>* __restrict__ r2,
                  const double2* __restrict__ frc, int fnk, double fkf, double beta, double gdt,
                  const cx<T>* __restrict__ twg, int ntile, T norm) {
  k2_zfwd_formf_body<T, N, kBlock2, FRC, FRESH>(xcd_remap(blockIdx.x, gridDim.x), g, cf, w1, u0, u1, u2, r0, r1, r2, frc,
                                         fnk, fkf, beta, gdt, twg, ntile, norm);
}

template <typename T, int N>
size_t lds_lines() {
  return size_t(lds_lines_bytes<T>(N));
}
template <typename T, int N>
size_t lds_fwd() {
  return size_t(lds_fwd_bytes<T>(N));
}
template <typename T, int N>
size_t lds_y() {
  size_t m = 0;
  for (int b : {lds_y_bytes<T, true>(N), lds_yf_bytes<T, true>(N), lds_y_bytes<T, false>(N), lds_yf_bytes<T, false>(N)})
    m = size_t(b) > m ? size_t(b) : m;
  return m;
}
template <typename T, int N, bool RS = false>
size_t lds_x() {
  return size_t(lds_x_bytes<T, RS>(N) - (kBlock2 / 64) * int(sizeof(T)));  // dynamic part
}

hipError_t big_lds(const void* fn, size_t bytes) {
  if (bytes <= 65536) return hipSuccess;
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
}

template <typename T, int N>
hipError_t zinv_n(pdr_ctx* c, const Coef& cf) {
  const Geo& g = c->g;
  if constexpr (PDR_ZINV_REG && N <= 512) {  // longer lines hold too many values per thread
    constexpr int L = zinv_lines_t<T, PDR_ZINV_THREADS>(N);
    const int nt = (g.nkj + L - 1) / L;
    const size_t lds = size_t(lds_zinv_bytes_t<T, PDR_ZINV_THREADS>(N));
    auto launch = [&](auto fresh_c) -> hipError_t {
      constexpr bool FRESH = decltype(fresh_c)::value;
      hipError_t e = big_lds((const void*)k2_zinv_r<T, N, FRESH>, lds);
      if (e != hipSuccess) return e;
      k2_zinv_r<T, N, FRESH><<<dim3(unsigned(nt * g.nki)), PDR_ZINV_THREADS, lds, c->stream>>>(
          g, cf, (const cx<T>*)c->u[0], (const cx<T>*)c->u[1], (const cx<T>*)c->u[2], (cx<T>*)c->w1,
          (const cx<T>*)c->tab.twz, nt);
      return hipGetLastError();
    };
    if constexpr (zinv_fresh<T>(N)) {
      if (nt * g.nki > kCus) return launch(std::true_type{});
    }
    return launch(std::false_type{});
  } else {
    constexpr int L = tile_lines<T>(N);
    const int nt = (g.nkj + L - 1) / L;
    const size_t lds = lds_lines<T, N>();
    hipError_t e = big_lds((const void*)k2_zinv<T, N>, lds);
    if (e != hipSuccess) return e;
    k2_zinv<T, N><<<dim3(unsigned(nt * g.nki)), zinv_threads<T>(N), lds, c->stream>>>(
        g, cf, (const cx<T>*)c->u[0], (const cx<T>*)c->u[1], (const cx<T>*)c->u[2], (cx<T>*)c->w1,
        (const cx<T>*)c->tab.twz, nt);
    return hipGetLastError();
  }
}

template <typename T, int N, bool PL, bool DY>
hipError_t yinv_t(pdr_ctx* c, int z0, int nzc) {
  const Geo& g = c->g;
  constexpr int PP = y_planes<T, PL>(N);
  constexpr int L = y_lines<T, PL>(N);
  const int nt = PP ? (nzc + PP - 1) / PP : (g.nki + L - 1) / L;
  const size_t lds = size_t(lds_y_bytes<T, PL>(N));
  hipError_t e = big_lds((const void*)k2_yinv<T, N, PL, DY>, lds);
  if (e != hipSuccess) return e;
  // nine fields split over workgroups by one or three
  const int fpb = DY ? (c->fpb_y >= 3 ? 3 : 1) : c->fpb_y;
  k2_yinv<T, N, PL, DY>
      <<<dim3(unsigned(nt * (PP ? 1 : nzc) * ((DY ? 9 : 6) / fpb))), yinv_threads<T, N, PL>(), lds, c->stream>>>(
          g, (const cx<T>*)c->w1, (cx<T>*)c->w2, (const cx<T>*)c->tab.twy, nt, z0, nzc, fpb);
  return hipGetLastError();
}

template <typename T, int N>
hipError_t yinv5_n(pdr_ctx* c, const Coef& cf, int z0, int nzc) {
  const Geo& g = c->g;
  constexpr int L = y_lines<T, false>(N);
  const int nt = (g.nki + L - 1) / L;
  const size_t lds = size_t(lds_y_bytes<T, false>(N));
  hipError_t e = big_lds((const void*)k2_yinv5<T, N>, lds);
  if (e != hipSuccess) return e;
  YVort v;
  for (int n = 0; n < 3; ++n) {
    v.a[n] = cf.G[18 + 3 * n];
    v.b[n] = cf.G[18 + 3 * n + 1];
  }
  k2_yinv5<T, N><<<dim3(unsigned(nt * nzc)), yinv_threads<T, N, false>(), lds, c->stream>>>(
      g, v, (const cx<T>*)c->w1, (cx<T>*)c->w2, (const cx<T>*)c->tab.twy, nt, z0, nzc);
  return hipGetLastError();
}

template <typename T, int N, bool DY>
hipError_t yinv_n(pdr_ctx* c, int z0, int nzc) {
  if constexpr (y_planes<T>(N) > 0) {
    if (c->g.nki == N / 3 + 1) return yinv_t<T, N, true, DY>(c, z0, nzc);
  }
  return yinv_t<T, N, false, DY>(c, z0, nzc);
}

// FP32-mixed boxes whose moments a thread sums in FP32 over its own points: cubes
// and long boxes of 2^a or 3 2^a points; every other shape sums them in FP64 (the
// sums across threads are FP64 in both).
constexpr bool rs_fp32_len(int n) {
  return n >= 32 && ((n & (n - 1)) == 0 || (n % 3 == 0 && ((n / 3) & (n / 3 - 1)) == 0));
}
inline bool rs_fp32_box(const Geo& g) {
  return rs_fp32_len(g.nx) && rs_fp32_len(g.ny) && rs_fp32_len(g.nz) && (g.ny > 96 || g.nx / 3 == g.ny / 3);
}

template <typename T, int N>
hipError_t xpass_n(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, int z0, int nzc, double* rsp) {
  const Geo& g = c->g;
  auto launch = [&](auto rs_c) -> hipError_t {
    constexpr int RS = decltype(rs_c)::value;
    constexpr int RB = xrows<T, RS != 0>(N);
    const int nt = (g.ny + RB - 1) / RB;
    const size_t lds = lds_x<T, N, RS != 0>();
    hipError_t e = big_lds((const void*)k2_xpass<T, N, RS>, lds);
    if (e != hipSuccess) return e;
    k2_xpass<T, N, RS><<<dim3(unsigned(nt * nzc)), xthreads<T, RS>(N), lds, c->stream>>>(
        g, cf, (cx<T>*)c->w2, (T*)c->ur, tr ? 1 : 0, cfl ? 1 : 0, c->umax, (const cx<T>*)c->tab.twx, nt, z0, rsp);
    return hipGetLastError();
  };
  if (!rsp) return launch(std::integral_constant<int, 0>{});
  if constexpr (sizeof(T) == 4 && rs_fp32_len(N)) {
    if (rs_fp32_box(g)) return launch(std::integral_constant<int, 1>{});
  }
  return launch(std::integral_constant<int, 2>{});
}

template <typename T, int N>
hipError_t xpass_conv_n(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, double* rsp) {
  const Geo& g = c->g;
  constexpr int RB = xrows_conv<T>(N);
  const int nt = (g.ny + RB - 1) / RB;
  const size_t lds = size_t(lds_xc_bytes<T>(N));
  auto launch = [&](auto rs_c) -> hipError_t {
    constexpr bool RS = decltype(rs_c)::value;
    hipError_t e = big_lds((const void*)k2_xpass_conv<T, N, RS>, lds);
    if (e != hipSuccess) return e;
    k2_xpass_conv<T, N, RS><<<dim3(unsigned(nt * g.nz)), kBlock2, lds, c->stream>>>(
        g, cf, (cx<T>*)c->w2, (T*)c->ur, tr ? 1 : 0, cfl ? 1 : 0, c->umax, (const cx<T>*)c->tab.twx, nt, rsp);
    return hipGetLastError();
  };
  return rsp ? launch(std::true_type{}) : launch(std::false_type{});
}

template <typename T, int N, bool PL>
hipError_t yfwd_t(pdr_ctx* c, int z0, int nzc) {
  const Geo& g = c->g;
  constexpr int PP = y_planes<T, PL>(N);
  constexpr int L = y_lines_fwd<T, PL>(N);
  const int nt = PP ? (nzc + PP - 1) / PP : (g.nki + L - 1) / L;
  const size_t lds = size_t(lds_yf_bytes<T, PL>(N));
  hipError_t e = big_lds((const void*)k2_yfwd<T, N, PL>, lds);
  if (e != hipSuccess) return e;
  k2_yfwd<T, N, PL><<<dim3(unsigned(nt * (PP ? 1 : nzc) * (3 / c->fpb_yf))), yfwd_threads<T, N, PL>(), lds, c->stream>>>(
      g, (const cx<T>*)c->w2, (cx<T>*)c->w1, (const cx<T>*)c->tab.twy, nt, z0, nzc, c->fpb_yf);
  return hipGetLastError();
}

template <typename T, int N>
hipError_t yfwd_n(pdr_ctx* c, int z0, int nzc) {
  if constexpr (y_planes<T>(N) > 0) {
    if (c->g.nki == N / 3 + 1) return yfwd_t<T, N, true>(c, z0, nzc);
  }
  return yfwd_t<T, N, false>(c, z0, nzc);
}

template <typename T, int N>
hipError_t zfwd_n(pdr_ctx* c) {
  const Geo& g = c->g;
  constexpr int L = tile_lines_fwd<T>(N);
  const int nt = (g.nkj + L - 1) / L;
  const size_t lds = lds_fwd<T, N>();
  hipError_t e = big_lds((const void*)k2_zfwd<T, N>, lds);
  if (e != hipSuccess) return e;
  const double norm = 1.0 / (double(g.nx) * double(g.ny) * double(g.nz));
  k2_zfwd<T, N><<<dim3(unsigned(nt * g.nki)), zthreads(N), lds, c->stream>>>(
      g, (const cx<T>*)c->w1, (cx<T>*)c->nl, (const cx<T>*)c->tab.twz, nt, T(norm));
  return hipGetLastError();
}

template <typename T, int N>
hipError_t zfwd_formf_n(pdr_ctx* c, const Coef& cf, double beta, double gdt) {
  if constexpr (N > 512) {  // not used above 512 points per line (see pdr_create)
    return hipErrorNotSupported;
  } else {
  const Geo& g = c->g;
  constexpr int L = tile_lines_fwd<T>(N);
  const int nt = (g.nkj + L - 1) / L;
  const size_t lds = lds_fwd<T, N>();
  const double norm = 1.0 / (double(g.nx) * double(g.ny) * double(g.nz));
  auto launch_f = [&](auto frc_c, auto fresh_c) -> hipError_t {
    constexpr int F = decltype(frc_c)::value;
    constexpr bool FRESH = decltype(fresh_c)::value;
    hipError_t e = big_lds((const void*)k2_zfwd_formf<T, N, F, FRESH>, lds);
    if (e != hipSuccess) return e;
    k2_zfwd_formf<T, N, F, FRESH><<<dim3(unsigned(nt * g.nki)), kBlock2, lds, c->stream>>>(
        g, cf, (const cx<T>*)c->w1, (cx<T>*)c->u[0], (cx<T>*)c->u[1],
        (cx<T>*)c->u[2], (cx<T>*)c->rk[0], (cx<T>*)c->rk[1], (cx<T>*)c->rk[2], F ? (const double2*)c->force : nullptr, F ? c->force_nk : 0,
        F ? c->p.force_kf : 0.0, beta, gdt, (const cx<T>*)c->tab.twz, nt, T(norm));
    return hipGetLastError();
  };
  auto launch = [&](auto frc_c) -> hipError_t {
    if constexpr (zff_fresh<T>(N, decltype(frc_c)::value)) {
      if (nt * g.nki > 2 * kCus) return launch_f(frc_c, std::true_type{});
    }
    return launch_f(frc_c, std::false_type{});
  };
  if (!c->forcing) return launch(std::integral_constant<int, 0>{});
  if (cf.fdef) return launch(std::integral_constant<int, 2>{});
  return launch(std::integral_constant<int, 1>{});
  }
}

}  // namespace

}  // namespace pdr
