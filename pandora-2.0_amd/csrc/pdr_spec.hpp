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
  hipError_t (*zfwd_formf)(pdr_ctx*, const Coef&, double beta, double gdt);
  // the z passes of short lines with every field of a tile in LDS (pdr_zall.hpp), null where
  // there are none; next: the operator of the stage that follows, whose inverse z pass is
  // then done in the same kernel, or null
  hipError_t (*zall_inv)(pdr_ctx*, const Coef&);
  hipError_t (*zall_fwd)(pdr_ctx*, const Coef&, const Coef* next, double beta, double gdt);
  long long zall_most;  // most z lines of a box that runs them
  // passes 2 to 4 of n x n planes in one launch (pdr_plane.hpp), null where they do not fit
  hipError_t (*plane)(pdr_ctx*, const Coef&, bool tr, bool cfl, double* rsp);
  size_t lds_plane;  // the kernel's own arrays included
  int plane_parts;
  int plane_most;  // most planes of a box that takes them
  size_t lds_z, lds_y, lds_x, lds_xc;  // the largest workgroup of the z, y, x and NS_R_CONV x passes
  int xrows, xrows_rs, xrows_conv;  // rows of an x tile; with the moments; NS_R_CONV
  int x_tw_global;             // 1: the x tile reads its twiddles from the global table
  int zinv_register;           // 1: the velocity tile of a z inverse is kept in registers
  int zinv_lines, zall_lines;  // lines of a z inverse tile
};

// The specialised path of a line length, or null (pdr_spec_dispatch.hip).
const SpecOps* spec_ops(int prec, int n);

// The lengths with specialised kernels, a chosen set: 2^a {1, 3, 5} and 2^a 15 from 24 to
// 1536 points, and up to 512 points the other even 2^a 3^b 5^c except 50, 54, 162, 270, 324,
// 450, 486 and 500.  Those, the odd ones, the shorter ones and the rest of the longer ones,
// and tiles beyond a workgroup's LDS, run the runtime-radix kernels of
// pdr_kernels.hip, which ping-pong two LDS buffers with run-time index divisions: twelve FP32
// steps of a 160^3 box with the CFL time step, spherical truncation and the state read back
// take 20.2 ms there and 7.2 ms here, twelve FP64 steps of 120 x 48 x 96 with 5000 tracers
// 7.2 against 2.7 ms.
//
// pdr_spec.hip is compiled once for each length and precision (build_lib.py reads them
// here), which makes each a code object of its own: the runtime loads a code object whole at
// the first launch from it, some 60 us for every kernel in it, so a program pays for the
// lengths that it steps.  First step of a 32^3 FP32-mixed box in a process 1.3 ms; 11.4 with
// eight code objects of five lengths in both precisions each, of which boxes of 32, 48, 64 and
// 96 points then take four (five steps of 64 such boxes, loads included, 53 -> 21 ms).
#define PDR_SPEC_LENGTHS(X) X(24) X(30) X(32) X(36) X(40) X(48) X(60) X(64) X(72) X(80) X(90) X(96) X(100) \
   X(108) X(120) X(128) X(144) X(150) X(160) X(180) X(192) X(200) X(216) X(240) X(250) X(256) X(288) X(300) \
   X(320) X(360) X(384) X(400) X(432) X(480) X(512) X(640) X(768) X(960) X(1024) X(1280) X(1536)

#define PDR_ROW(n)                   \
  const SpecOps* spec_ops_f32_##n(); \
  const SpecOps* spec_ops_f64_##n();
PDR_SPEC_LENGTHS(PDR_ROW)
#undef PDR_ROW

}  // namespace pdr
