// pdr_spec.hpp -- what one (precision, line length) of the specialised path offers:
// the host launchers of its passes and the shapes they take.
#pragma once
#include "pdr_internal.hpp"

namespace pdr {

struct SpecOps {
  int prec, n;
  hipError_t (*zinv)(pdr_ctx*, const Coef&);
  hipError_t (*yinv)(pdr_ctx*, int z0, int nzc);
  // the same from the five fields of a z pass with Coef::y3
  hipError_t (*yinv5)(pdr_ctx*, const Coef&, int z0, int nzc);
  int y_planes;  // > 0: boxes with NX/3 = NY/3 take whole z planes per y-pass workgroup
  hipError_t (*xpass)(pdr_ctx*, const Coef&, bool tr, bool cfl, int z0, int nzc, double* rsp);
  hipError_t (*yinv_conv)(pdr_ctx*, int z0, int nzc);  // NS_R_CONV: also d/dy of the velocity
  hipError_t (*xpass_conv)(pdr_ctx*, const Coef&, bool tr, bool cfl, double* rsp);
  hipError_t (*yfwd)(pdr_ctx*, int z0, int nzc);
  hipError_t (*zfwd)(pdr_ctx*);
  // next: the operator of the stage that follows, whose inverse z pass is then done in the
  // same kernel; only where zz is true, else null
  hipError_t (*zfwd_formf)(pdr_ctx*, const Coef&, const Coef* next, double beta, double gdt);
  bool zz;
  // passes 2 to 4 of n x n planes in one launch (pdr_plane.hpp), null where they do not fit
  hipError_t (*plane)(pdr_ctx*, const Coef&, bool tr, bool cfl, double* rsp);
  size_t lds_plane;  // the kernel's own arrays included
  int plane_parts;
  size_t lds_z, lds_y, lds_x, lds_xc;  // the largest workgroup of the z, y, x and NS_R_CONV x passes
  int xrows, xrows_conv;       // rows of an x tile
  int x_tw_global;             // 1: the x tile reads its twiddles from the global table
  int zinv_register;           // 1: register z inverse
  int zinv_lines;              // lines of a z inverse tile
};

// The specialised path of a line length, or null (pdr_spec_dispatch.hip).
const SpecOps* spec_ops(int prec, int n);

// Lengths of the translation units that pdr_spec.hip is compiled into, one per
// PDR_SPEC_TU, the long and costly ones spread over them: every even length of
// 24 .. 512 points that a 2^a 3^b 5^c box of the reference's form 2^a {1, 3, 5}
// or with one more factor 3 or 5 has, and 640 .. 1536.  Other lengths, and tiles
// beyond a workgroup's LDS, run the runtime-radix kernels of pdr_kernels.hip, which
// ping-pong two LDS buffers with run-time index divisions: twelve FP32 steps of a
// 160^3 box with the CFL time step, spherical truncation and the state read back
// take 20.2 ms there and 9.0 ms here, twelve FP64 steps of 120 x 48 x 96 with 5000
// tracers 7.2 against 3.7 ms.
#define PDR_SPEC_SIZES_0(X) X(32) X(128) X(512) X(180) X(300)
#define PDR_SPEC_SIZES_1(X) X(48) X(192) X(384) X(24) X(320)
#define PDR_SPEC_SIZES_2(X) X(64) X(256) X(768) X(36) X(360)
#define PDR_SPEC_SIZES_3(X) X(96) X(100) X(1024) X(40) X(200)
#define PDR_SPEC_SIZES_4(X) X(60) X(108) X(1536) X(400) X(160)
#define PDR_SPEC_SIZES_5(X) X(72) X(80) X(1280) X(240) X(432)
#define PDR_SPEC_SIZES_6(X) X(120) X(640) X(288) X(480) X(216)
#define PDR_SPEC_SIZES_7(X) X(144) X(960) X(150) X(250) X(90) X(30)
constexpr int kSpecTus = 8;

// The table of translation unit K and its length.
#define PDR_SPEC_TABLE(K) const SpecOps* spec_table_##K(int* count)
PDR_SPEC_TABLE(0);
PDR_SPEC_TABLE(1);
PDR_SPEC_TABLE(2);
PDR_SPEC_TABLE(3);
PDR_SPEC_TABLE(4);
PDR_SPEC_TABLE(5);
PDR_SPEC_TABLE(6);
PDR_SPEC_TABLE(7);

}  // namespace pdr
