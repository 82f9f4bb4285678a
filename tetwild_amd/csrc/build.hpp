// build.hpp -- the device build of the envelope tree (build.hip).
#pragma once

#include <algorithm>

#include "twg_bvh.hpp"
#include "twg_internal.hpp"

namespace twg {

// Builds B (its memory, order and scalars) over the host arrays V (nv x 3) and
// F (nf x 3); *bad: the first corner of F whose id lies outside [0, nv), -1
// when there is none (else B holds no usable tree).  Synchronous.
int bvh_build_device(twg_ctx* ctx, const double* V, int64_t nv, const int32_t* F, int64_t nf, twg_bvh* B,
                     int64_t* bad);

}  // namespace twg
