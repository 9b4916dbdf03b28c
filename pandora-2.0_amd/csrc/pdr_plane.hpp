// pdr_plane.hpp -- passes 2 to 4 of a z plane in one workgroup: inverse y FFT, x c2r,
// product, x r2c and forward y FFT (f_RK3RealSpace, src/pf_rk3.f90:960-1237) with the
// plane kept in LDS from the 1r2w array back to the 1r2w array.
//
// The separate passes write and read the x-pencil array between them, 18 of the 45
// field passes over memory that a stage makes, and a small box spends their three
// launches mostly waiting.  A plane's six fields fit a workgroup's LDS for short
// lines; where the x tile of the whole plane does not (three packed complex lines a
// row), the plane is taken in S parts of the rows y = s, s + S, ...: part s of the
// inverse y transform is a transform of N / S points of the modes folded onto each
// other, b_s[j'] = sum over j = j' mod N/S of a[j] w^{js}, and the forward transform
// is the sum over the parts of w^{-js} G_s[j mod N/S], kept in registers, or left as
// addends for the z forward pass where the parts of a plane go to several workgroups.
// A part is a chain of some 26 barriers (6 us at 32 and 11 us at 64 points FP64, however
// many run), so a small box gives each of its parts a workgroup of its own.
#pragma once
#include "pdr_passes.hpp"

// Longest planes of a single box: beyond them a plane's parts, one workgroup to a CU, keep
// fewer lanes busy than the separate passes' many small workgroups (us by events, inverse y
// + x + forward y against one launch: 32 points FP64 8.8 + 7.6 + 8.6 / 12.0, 64 points
// 12.4 + 11.2 + 9.4 / 21.2, FP32-mixed 9.7 + 9.4 + 8.7 / 16.7; 72 points FP64
// 13.2 + 15.9 + 9.3 / 45, 96 points FP32-mixed 13.4 + 18.0 + 10.7 / 56).
#ifndef PDR_PLANE_MAX
#define PDR_PLANE_MAX 64
#endif

namespace pdr {

namespace {

// Bytes of a workgroup that takes a plane of n x n points in s parts.
template <typename T>
constexpr int plane_lds_bytes(int n, int s) {
  const int m = n / s, nki = n / 3 + 1;
  const int x = 3 * m * lds_ld<T>(n), y = 6 * nki * lds_ld<T>(m);
  return (n + (s > 1 ? n + m : 0) + (x > y ? x : y)) * int(sizeof(cx<T>));
}
// Deepest boxes that take them: with a plane in parts, an under-filled chip's worth of planes
// (us a step, separate passes -> these: 32 points FP64 64 planes 76 -> 56, 96 planes 87 -> 85,
// 160 151 -> 150, 256 183 -> 196, 64 points FP64 64 planes 104 -> 91, 72 121 -> 137, 256
// 254 -> 272, 512 431 -> 495; FP32-mixed 48 points 128 planes 117 -> 105, 144 182 -> 184, 256
// 222 -> 230, 64 points 80 planes 102 -> 93, 96 107 -> 110, 256 218 -> 238); planes in one
// part at any depth (24 points FP64 512 planes 259 -> 212).
template <typename T>
constexpr int plane_most(int n, int s) {
  if (s == 1) return 1 << 30;
  return sizeof(T) == 4 ? (n > 60 ? 80 : 128) : (n > 48 ? 64 : 96);
}
// Threads: the first x pass's butterflies in as few equal rounds as 1024 threads allow.
constexpr int plane_threads(int n, int s) {
  const int b = 3 * (n / s) * (n / plan_radix(n, 0));
  const int rounds = (b + 1023) / 1024;
  return ((b + rounds - 1) / rounds + 63) / 64 * 64;
}
// Bytes of the kernel's own arrays, the CFL maxima and the moments' sums of its waves.
template <typename T>
constexpr int plane_static_bytes(int n, int s) {
  return (plane_threads(n, s) / 64 * (kRsWidth * int(sizeof(double)) + int(sizeof(T))) + 15) / 16 * 16;
}
// The longest planes taken this way, and the parts a plane is taken in (0: the
// separate passes run): the fewest, at least `least`, that the LDS of a CU holds.
template <typename T, bool ENS = false>
constexpr int plane_parts(int n, int least) {
  if (!ENS && n > PDR_PLANE_MAX) return 0;
  for (int s = least; 8 * s <= n + 7; ++s)
    if (n % s == 0 && plane_lds_bytes<T>(n, s) + plane_static_bytes<T>(n, s) <= kLdsPerCu) return s;
  return least > 1 ? plane_parts<T, ENS>(n, 1) : 0;
}
// Parts of a single box's planes: enough for the groups below to fill the chip
// where the planes alone do not.
template <typename T>
constexpr int plane_parts_box(int n) {
  const int want = (256 + n - 1) / n;
  return plane_parts<T>(n, want < 4 ? want : 4);
}

// Parts gr, gr + ng, ... of plane z, from w1 into the three fields at dst (w1 itself
// if this is the plane's only workgroup).
template <typename T, int N, int S, bool RS>
__device__ __forceinline__ void plane_body(int z, int gr, int ng, const Geo& g, const Coef& cf,
                                           const cx<T>* w1, cx<T>* dst, T* __restrict__ ur,
                                           int want_tr, int want_cfl, unsigned long long* __restrict__ umax,
                                           const cx<T>* __restrict__ twg, double* __restrict__ rsp) {
  constexpr int NT = plane_threads(N, S);
  constexpr int M = N / S;            // rows of a part
  constexpr int LD = lds_ld<T>(N);    // x lines
  constexpr int LY = lds_ld<T>(M);    // y lines
  constexpr int K = N / 3;
  constexpr int NKI = K + 1, NKJ = 2 * K + 1;
  constexpr int IT = (M * N + NT - 1) / NT;          // product points per thread
  constexpr int QO = (3 * NKI * NKJ + NT - 1) / NT;  // output modes per thread
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ T red[(NT + 63) / 64];
  cx<T>* const tw = reinterpret_cast<cx<T>*>(smem);  // of N points
  cx<T>* const twp = S > 1 ? tw + N : tw;            // the plain table exp(-2 pi i m / N)
  cx<T>* const twy = S > 1 ? tw + 2 * N : tw;        // of M points
  cx<T>* const buf = tw + N + (S > 1 ? N + M : 0);
  load_tw<T, N, NT>(tw, twg);
  if constexpr (S > 1) {
    load_tw<T, M, NT, S>(twy, twg);
    for (int m = threadIdx.x; m < N; m += NT) twp[m] = twg[m];
  }
  // modes (f, i, j) of the plane at f m1 + i nz ldj + j; 32-bit byte offsets (plane_offsets_fit),
  // so that a load in flight holds one register of address
  const char* const wz = reinterpret_cast<const char*>(w1 + (long long)z * g.ldj);
  char* const dz = reinterpret_cast<char*>(dst + (long long)z * g.ldj);
  const unsigned fstr = unsigned(g.m1), istr = unsigned(g.nz * g.ldj);
  auto at = [&](int f, int i, int j) {
    return (unsigned(f) * fstr + unsigned(i) * istr + unsigned(j)) * unsigned(sizeof(cx<T>));
  };
  auto load = [&](int f, int i, int j) { return *reinterpret_cast<const cx<T>*>(wz + at(f, i, j)); };
  T lmax = T(0);
  cx<T> out[QO];
#pragma unroll 1
  for (int s = gr; s < S; s += ng) {
    if (S > 1 && s != gr) __syncthreads();
    if constexpr (S == 1) {
      // the stored modes, and zeros at the band positions that the first pass reads
      constexpr int E = 6 * NKI * NKJ, Q = (E + NT - 1) / NT;
      const int tid = fresh_tid();
      cx<T> v[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        const int line = e / NKJ, f = line / NKI;
        v[q] = (E % NT == 0 || e < E) ? load(f, line - f * NKI, e - line * NKJ) : czero<T>();
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        const int line = e / NKJ, j = e - line * NKJ;
        if (E % NT == 0 || e < E) buf[line * LY + lds_off<T>(j <= K ? j : j + (N - NKJ))] = v[q];
      }
      zero_band_edges<T, N, 6 * NKI, LY, K, NT>(buf, tid);
      __syncthreads();
      fft_ip<T, N, 6 * NKI, LY, +1, true, NT, K>(buf, tw, fresh_tid());
    } else {
      // folded modes: b[j'] = sum over q of a[y] w^{y s}, y = j' + q M the positions of stored
      // modes; CH positions' loads in flight per thread
      constexpr int E = 6 * NKI * M, Q = (E + NT - 1) / NT;
      constexpr int CH0 = NT <= 512 ? 6 : (sizeof(T) == 4 ? 32 : 16) / S;
      constexpr int CH = CH0 < 1 ? 1 : (CH0 > Q ? Q : CH0);
      const int tid = fresh_tid();
#pragma unroll 1
      for (int c0 = 0; c0 < Q; c0 += CH) {
        cx<T> a[CH][S];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const int e = tid + NT * (c0 + c);
          const int line = e / M, j = e - line * M, f = line / NKI;
          const int i = line - f * NKI;
#pragma unroll
          for (int q = 0; q < S; ++q) {
            if (q * M > K && q * M + M - 1 < N - K) continue;  // all in the truncated band
            const int y = j + q * M;
            a[c][q] = (e < E && (y <= K || y >= N - K)) ? load(f, i, y <= K ? y : y - (N - NKJ)) : czero<T>();
          }
        }
        if (c0 == 0 && s == gr) __syncthreads();  // the tables
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const int e = tid + NT * (c0 + c);
          const int line = e / M, j = e - line * M;
          if (e < E) {
            cx<T> v = czero<T>();
#pragma unroll
            for (int q = 0; q < S; ++q) {
              if (q * M > K && q * M + M - 1 < N - K) continue;
              const cx<T> w = twp[((j + q * M) * s) % N];
              v = add(v, mul(a[c][q], mk<T>(w.x, -w.y)));
            }
            buf[line * LY + lds_off<T>(j)] = v;
          }
        }
      }
      __syncthreads();
      fft_ip<T, M, 6 * NKI, LY, +1, true, NT>(buf, twy, fresh_tid());
    }
    // y lines to packed x lines (3 r + p: fields 2 p and 2 p + 1 of row r), as k2_xpass fills them
    {
      constexpr int E = 3 * M * NKI, Q = (E + NT - 1) / NT;
      const int tid = fresh_tid();
      cx<T> A[Q], B[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        const int line = e / NKI, m = e - line * NKI;
        const int r = line / 3, p = line - 3 * r;
        if (E % NT == 0 || e < E) {
          A[q] = buf[((2 * p) * NKI + m) * LY + lds_off<T>(r)];
          B[q] = buf[((2 * p + 1) * NKI + m) * LY + lds_off<T>(r)];
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        if (E % NT == 0 || e < E) {
          const int line = e / NKI, m = e - line * NKI;
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
    zero_band_edges<T, N, 3 * M, LD, K, NT>(buf, fresh_tid());
    __syncthreads();
    fft_ip<T, N, 3 * M, LD, +1, true, NT, K>(buf, tw, fresh_tid());
    T V[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      if constexpr (sizeof(T) == 4)
        V[q] = cf.Vf[q];
      else
        V[q] = T(cf.V[q]);
    }
    const bool form = cf.form != 0;
    T nl[IT][3];
    RsAcc acc;
    if (RS) rs_init(acc);
    {
      const int tid = fresh_tid();
#pragma unroll
      for (int q = 0; q < IT; ++q) {
        const int idx = tid + NT * q;
        if ((M * N) % NT == 0 || idx < M * N) {
          const int r = idx / N;
          const int x = idx - r * N;
          const cx<T>* row = buf + 3 * r * LD + lds_off<T>(x);
          const cx<T> a = row[0], b = row[LD], c = row[2 * LD];
          const T u1 = a.x, u2 = a.y, u3 = b.x, o1 = b.y, o2 = c.x, o3 = c.y;
          const T v1 = V[0] * u1 + V[1] * u2 + V[2] * u3;
          const T v2 = V[3] * u1 + V[4] * u2 + V[5] * u3;
          const T v3 = V[6] * u1 + V[7] * u2 + V[8] * u3;
          // omega x (binv u) (BF_ROT), or omega x u (isotropic with binv = I, R_ROT)
          const T p1 = form ? u1 : v1, p2 = form ? u2 : v2, p3 = form ? u3 : v3;
          nl[q][0] = o2 * p3 - o3 * p2;
          nl[q][1] = o3 * p1 - o1 * p3;
          nl[q][2] = o1 * p2 - o2 * p1;
          if (want_tr) {
            T* d = ur + (((long long)z * N + (S * r + s)) * N + x) * 3;
            put1<kNtXpass>(d, u1);
            put1<kNtXpass>(d + 1, u2);
            put1<kNtXpass>(d + 2, u3);
          }
          if (want_cfl) {
            const T sm = fabs(v1) + fabs(v2) + fabs(v3);  // lab-frame velocity (src/pf_fluidstats.f90:853-866, 914)
            lmax = sm > lmax ? sm : lmax;
          }
          if (RS) rs_add(acc, double(v1), double(v2), double(v3), double(o1), double(o2), double(o3));
        }
      }
    }
    if constexpr (RS) {
      __shared__ double rs_lds[kRsWidth * ((NT + 63) / 64)];
      rs_block_out(acc, rs_lds, rsp + (z * S + s) * kRsWidth);
    }
    __syncthreads();
    // forward lines: r -> n1 + i n2 of row r; M + r/2 -> n3 of rows (r, r+1)
    constexpr int NF = M + (M + 1) / 2;
    {
    const int tid = fresh_tid();
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int idx = tid + NT * q;
      if ((M * N) % NT == 0 || idx < M * N) {
        const int r = idx / N;
        const int x = idx - r * N;
        buf[r * LD + lds_off<T>(x)] = mk<T>(nl[q][0], nl[q][1]);
        cx<T>* p3 = &buf[(M + r / 2) * LD + lds_off<T>(x)];
        if (r & 1)
          p3->y = nl[q][2];
        else
          p3->x = nl[q][2];
        if (M % 2 == 1 && r == M - 1) p3->y = T(0);
      }
    }
    }
    __syncthreads();
    fft_ip<T, N, NF, LD, -1, true, NT>(buf, tw, fresh_tid());
    // unpacked modes (r, m) to the y lines c NKI + m
    {
      constexpr int E = M * NKI, Q = (E + NT - 1) / NT;
      const int tid = fresh_tid();
      cx<T> n[Q][3];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        if (E % NT == 0 || e < E) {
          const int r = e / NKI, m = e - r * NKI;
          const int om = lds_off<T>(m), omr = lds_off<T>(m == 0 ? 0 : N - m);
          const cx<T> Z = buf[r * LD + om], Zr = buf[r * LD + omr];
          const cx<T> W = buf[(M + r / 2) * LD + om], Wr = buf[(M + r / 2) * LD + omr];
          n[q][0] = mk<T>(T(0.5) * (Z.x + Zr.x), T(0.5) * (Z.y - Zr.y));
          n[q][1] = mk<T>(T(0.5) * (Z.y + Zr.y), T(-0.5) * (Z.x - Zr.x));
          n[q][2] = (r & 1) ? mk<T>(T(0.5) * (W.y + Wr.y), T(-0.5) * (W.x - Wr.x))
                            : mk<T>(T(0.5) * (W.x + Wr.x), T(0.5) * (W.y - Wr.y));
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int e = tid + NT * q;
        if (E % NT == 0 || e < E) {
          const int r = e / NKI, m = e - r * NKI;
#pragma unroll
          for (int c = 0; c < 3; ++c) buf[(c * NKI + m) * LY + lds_off<T>(r)] = n[q][c];
        }
      }
    }
    __syncthreads();
    fft_ip<T, M, 3 * NKI, LY, -1, true, NT>(buf, twy, fresh_tid());
    const int otid = fresh_tid();
#pragma unroll
    for (int q = 0; q < QO; ++q) {
      const int e = otid + NT * q;
      if ((3 * NKI * NKJ) % NT == 0 || e < 3 * NKI * NKJ) {
        const int line = e / NKJ, j = e - line * NKJ;
        const int y = j <= K ? j : j + (N - NKJ);
        if constexpr (S == 1) {
          out[q] = buf[line * LY + lds_off<T>(y)];
        } else {
          const cx<T> v = mul(buf[line * LY + lds_off<T>(y % M)], twp[(y * s) % N]);
          out[q] = s == gr ? v : add(out[q], v);
        }
      }
    }
  }
  // (a plane with one workgroup: its inputs have been read, NL replaces fields 0..2)
  const int tid = fresh_tid();
#pragma unroll
  for (int q = 0; q < QO; ++q) {
    const int e = tid + NT * q;
    if ((3 * NKI * NKJ) % NT == 0 || e < 3 * NKI * NKJ) {
      const int line = e / NKJ, f = line / NKI;
      put<kNtYfwd && !small_store(N)>(reinterpret_cast<cx<T>*>(dz + at(f, line - f * NKI, e - line * NKJ)), out[q]);
    }
  }
  if (want_cfl) {
    T m = lmax;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const T o = __shfl_xor(m, off);
      m = o > m ? o : m;
    }
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
      T r = red[0];
      for (int w = 1; w < NT / 64; ++w) r = red[w] > r ? red[w] : r;
      raise_max(umax, (unsigned long long)__double_as_longlong(double(r)));
    }
  }
}

template <typename T, int N, int S, bool RS>
__global__ void __launch_bounds__((plane_threads(N, S)))
    k2_plane(Geo g, Coef cf, const cx<T>* w1, cx<T>* dst, T* __restrict__ ur, int want_tr, int want_cfl,
             unsigned long long* __restrict__ umax, const cx<T>* __restrict__ twg, double* __restrict__ rsp, int ng) {
  // the groups of a plane nz apart: on one XCD, and its L2, where nz divides by 8
  const int z = int(blockIdx.x) % g.nz, gr = int(blockIdx.x) / g.nz;
  plane_body<T, N, S, RS>(z, gr, ng, g, cf, w1, dst + 3 * (long long)gr * g.m1, ur, want_tr, want_cfl, umax, twg, rsp);
}

template <typename T, int N>
hipError_t plane_n(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, double* rsp) {
  if constexpr (plane_parts_box<T>(N) == 0) {
    return hipErrorNotSupported;
  } else {
    constexpr int S = plane_parts_box<T>(N);
    const Geo& g = c->g;
    const size_t lds = size_t(plane_lds_bytes<T>(N, S));
    const int ng = c->nl_parts;
    auto launch = [&](auto rs_c) -> hipError_t {
      constexpr bool RS = decltype(rs_c)::value;
      hipError_t e = big_lds((const void*)k2_plane<T, N, S, RS>, lds);
      if (e != hipSuccess) return e;
      k2_plane<T, N, S, RS><<<dim3(unsigned(g.nz * ng)), plane_threads(N, S), lds, c->stream>>>(
          g, cf, (const cx<T>*)c->w1, (cx<T>*)(ng > 1 ? c->w2 : c->w1), (T*)c->ur, tr ? 1 : 0, cfl ? 1 : 0, c->umax,
          (const cx<T>*)c->tab.twx, rsp, ng);
      return hipGetLastError();
    };
    return rsp ? launch(std::true_type{}) : launch(std::false_type{});
  }
}

}  // namespace

}  // namespace pdr
