// pdr_spec_dispatch.hip -- from a box's line lengths to the specialised passes.
#include "pdr_spec.hpp"

namespace pdr {

const SpecOps* spec_ops(int prec, int n) {
  switch (n) {
#define PDR_ROW(n) \
  case n:          \
    return prec ? spec_ops_f32_##n() : spec_ops_f64_##n();
    PDR_SPEC_LENGTHS(PDR_ROW)
#undef PDR_ROW
    default:
      return nullptr;
  }
}

// Finds the passes of the box's three lengths; false: a length has none, or its
// tiles do not fit the LDS of a workgroup.
bool spec_find(pdr_ctx* c) {
  c->ops_x = spec_ops(c->prec, c->g.nx);
  c->ops_y = spec_ops(c->prec, c->g.ny);
  c->ops_z = spec_ops(c->prec, c->g.nz);
  c->zall = c->ops_z && c->ops_z->zall_inv && (long long)c->g.nki * c->g.nkj <= c->ops_z->zall_most;
  return c->ops_x && c->ops_y && c->ops_z && (conv_form(c) ? c->ops_x->lds_xc : c->ops_x->lds_x) <= c->lds_max && c->ops_y->lds_y <= c->lds_max &&
         c->ops_z->lds_z <= c->lds_max;
}

// Forms the passes of this box take (pdr_kernel_forms): x rows that a workgroup takes
// at a time, 1 if the x tile reads its twiddles from the global table, 1 for a z inverse
// with the velocity tile in registers, lines per z-inverse tile.
void spec_forms(const pdr_ctx* c, int out[4]) {
  out[0] = conv_form(c) ? c->ops_x->xrows_conv : plane_fused(c) ? c->g.ny / c->ops_x->plane_parts : c->ops_x->xrows;
  out[1] = c->ops_x->x_tw_global;
  out[2] = c->ops_z->zinv_register;
  out[3] = c->zall ? c->ops_z->zall_lines : c->ops_z->zinv_lines;
}

// The plane kernel reaches the modes of a plane by 32-bit byte offsets into six fields.
static bool plane_offsets_fit(const pdr_ctx* c) { return 6 * size_t(c->g.m1) * c->csz <= size_t(UINT32_MAX); }
// Whether the y and x passes of a plane run as one kernel: square planes of a length
// that has it, unless the environment asks for the chunked passes or their streams.
bool plane_fused(const pdr_ctx* c) {
  return c->spec && !conv_form(c) && !c->plane_separate && c->g.nx == c->g.ny && c->ops_x->plane &&
         c->g.nz <= c->ops_x->plane_most && c->ops_x->lds_plane <= c->lds_max && plane_offsets_fit(c) &&
         c->g.zc == c->g.nz;
}
hipError_t launch2_plane(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, double* rsp) {
  return c->ops_x->plane(c, cf, tr, cfl, rsp);
}

// rows of moment partials per z plane: x-pass workgroups, or the parts of a fused plane
int xpass_tiles(const pdr_ctx* c) {
  if (plane_fused(c)) return c->ops_x->plane_parts;
  const int rb = conv_form(c) ? c->ops_x->xrows_conv : c->ops_x->xrows_rs;
  return (c->g.ny + rb - 1) / rb;
}

hipError_t launch2_zinv(pdr_ctx* c, const Coef& cf) { return c->zall ? c->ops_z->zall_inv(c, cf) : c->ops_z->zinv(c, cf); }
hipError_t launch2_yinv(pdr_ctx* c, const Coef& cf, int z0, int nzc) {
  return cf.y3 ? c->ops_y->yinv5(c, cf, z0, nzc) : c->ops_y->yinv(c, z0, nzc);
}
// Whether five fields go through the z pass and the y pass forms the last vorticity
// component: where it has no k3 (every frame of the library itself; not one set by hand
// with k3 in another direction, in NS_R_ROT), and where one y workgroup takes all six
// fields of its tile of i-lines, so that it has the velocity's modes in any case (with the
// fields split over workgroups, or whole-plane tiles, they would be read once more).
bool z5_fields(const pdr_ctx* c, const Coef& cf) {
  return c->spec && !conv_form(c) && !plane_fused(c) && !c->zall && c->fpb_y == 6 &&
         !(c->ops_y->y_planes > 0 && c->g.nki == c->g.ny / 3 + 1) && cf.G[20] == 0.0 && cf.G[23] == 0.0 &&
         cf.G[26] == 0.0;
}
hipError_t launch2_xpass(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, int z0, int nzc, double* rsp) {
  return c->ops_x->xpass(c, cf, tr, cfl, z0, nzc, rsp);
}
hipError_t launch2_yinv_conv(pdr_ctx* c) { return c->ops_y->yinv_conv(c, 0, c->g.nz); }
hipError_t launch2_xpass_conv(pdr_ctx* c, const Coef& cf, bool tr, bool cfl, double* rsp) {
  return c->ops_x->xpass_conv(c, cf, tr, cfl, rsp);
}
hipError_t launch2_yfwd(pdr_ctx* c, int z0, int nzc) { return c->ops_y->yfwd(c, z0, nzc); }
hipError_t launch2_zfwd(pdr_ctx* c) { return c->ops_z->zfwd(c); }
// Whether the z forward pass can go on with the next stage's z inverse
bool zz_fused(const pdr_ctx* c) { return c->spec && !conv_form(c) && c->fuse_zf && c->zall; }
hipError_t launch2_zfwd_formf(pdr_ctx* c, const Coef& cf, const Coef* next, double beta, double gdt) {
  return c->zall ? c->ops_z->zall_fwd(c, cf, next, beta, gdt) : c->ops_z->zfwd_formf(c, cf, beta, gdt);
}

}  // namespace pdr
