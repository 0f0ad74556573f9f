// k2d_pipe_r3.hip -- the level-pipelined 2-D kernels of radius 3 (k2d_pipe_body.h).
#include "k2d_pipe_body.h"

namespace cs {

// ids 900000 + (star) * 10000 + R * 1000 + KF.  Depths measured at 8192^2 (kernel alone,
// GStencil/s): star 1 x 8 1208 (1 x 4: 1029; 2 x 4 spills: 264), box 1 x 4 458 (1 x 2: 383; 1 x 8,
// one workgroup per CU: 457).
static const Variant kVariantsPipeR3[] = {
    CS_VP2D(913008, 3, SHAPE_STAR, 8, 1, 8, 2, 3),
    CS_VP2D(913004, 3, SHAPE_STAR, 8, 1, 4, 2, 2),
    CS_VP2D(903004, 3, SHAPE_BOX, 8, 1, 4, 1, 2),
    CS_VP2D(903002, 3, SHAPE_BOX, 8, 1, 2, 1, 2),
};

const Variant *variants_2d_pipe_r3(int *count) {
  *count = (int)(sizeof(kVariantsPipeR3) / sizeof(kVariantsPipeR3[0]));
  return kVariantsPipeR3;
}

}  // namespace cs
