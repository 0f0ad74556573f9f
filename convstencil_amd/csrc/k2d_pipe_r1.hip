// k2d_pipe_r1.hip -- the level-pipelined 2-D kernels of radius 1 (k2d_pipe_body.h).
#include "k2d_pipe_body.h"

namespace cs {

// ids 900000 + (star) * 10000 + R * 1000 + KF.  Depths measured at 10240^2 (kernel alone,
// GStencil/s): box 3 x 4 2290 (2 x 4: 1936; 4 x 4 spills in the first wave: 1858), star 4 x 4
// 3440 (3 x 4: 3170, 2 x 4: 2312).
static const Variant kVariantsPipeR1[] = {
    CS_VP2D(901012, 1, SHAPE_BOX, 8, 3, 4, 2, 3),  CS_VP2D(901008, 1, SHAPE_BOX, 8, 2, 4, 2, 3),
    CS_VP2D(901004, 1, SHAPE_BOX, 8, 1, 4, 2, 3),  CS_VP2D(911016, 1, SHAPE_STAR, 8, 4, 4, 2, 1),
    CS_VP2D(911012, 1, SHAPE_STAR, 8, 3, 4, 2, 3), CS_VP2D(911008, 1, SHAPE_STAR, 8, 2, 4, 2, 3),
    CS_VP2D(911004, 1, SHAPE_STAR, 8, 1, 4, 2, 3),
};

const Variant *variants_2d_pipe_r1(int *count) {
  *count = (int)(sizeof(kVariantsPipeR1) / sizeof(kVariantsPipeR1[0]));
  return kVariantsPipeR1;
}

}  // namespace cs
