// pdr_ens_ops.hpp -- the batched ensemble passes of one (precision, line length).
#pragma once
#include "pdr_internal.hpp"

namespace pdr {

// Launchers over nm members of one line length, on stream s.
struct EnsOps {
  int prec, n;
  bool zz;     // zend can go on with the next stage's inverse z pass (join)
  bool split;  // mid has y passes, whose fields may be split over workgroups
  hipError_t (*prepare)();  // once, outside a capture
  hipError_t (*zinv)(const EnsMember* mem, int nm, hipStream_t s);
  hipError_t (*mid)(const EnsMember* mem, int nm, int fpb_y, int fpb_yf, hipStream_t s);
  hipError_t (*zend)(const EnsMember* mem, int nm, double beta, double gamma, bool join, hipStream_t s);
};

// Null: no member may have this line length.
const EnsOps* ens_ops(int prec, int n);

}  // namespace pdr
