#pragma once
#include <hip/hip_runtime.h>

namespace vx {

// (cos, sin) of dimension pair j of a head at a position (backend/cpu/cpu.go:226-303).
__device__ __forceinline__ float2 rope_angle(int position, int j, int head_dim, float theta) {
    const double ex = (double)(2 * j) / (double)head_dim;
    const float freq = (float)(1.0 / pow((double)theta, ex));
    const float angle = __fmul_rn((float)position, freq);
    return make_float2((float)cos((double)angle), (float)sin((double)angle));
}

}  // namespace vx
