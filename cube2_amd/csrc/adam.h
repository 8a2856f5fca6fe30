// One Adam update of an FP32 weight (c1, c2: the bias corrections of the
// step), shared by the per-tensor and the whole-network kernel so that both
// round alike.
#pragma once
#include "common.h"

namespace cube2 {
__device__ inline float adam_update(float w, float g, float& m, float& v, float lr, float b1,
                                    float b2, float eps, float c1, float c2) {
#pragma clang fp contract(off)
    m = fmaf(1.f - b1, g, b1 * m);
    v = fmaf(g, (1.f - b2) * g, b2 * v);
    return w - lr * (m / c1) / (sqrtf(v / c2) + eps);
}
}  // namespace cube2
