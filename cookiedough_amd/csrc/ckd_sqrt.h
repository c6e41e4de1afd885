// ckd_sqrt.h -- the square root of the raymarched effects' steps.
#pragma once

#include <hip/hip_runtime.h>

// sqrtf, correctly rounded: the reciprocal root's product with x and one Newton
// step on its residual, which the fused multiply-add leaves exact.  An estimate
// an ulp off can miss at a few mantissas, so this holds by the card's own
// v_rsq_f32: tests/test_gpu_sqrt.py compares every float of the range.  The
// rest, 0 among it, takes sqrtf.  7 instructions instead of 15 of a march step's
// 125.
__device__ __forceinline__ float st_sqrt(float x)
{
    if (!(x > 0x1p-96f && x < 0x1p96f)) return sqrtf(x);
    const float y = __builtin_amdgcn_rsqf(x), s = x * y;
    return fmaf(fmaf(-s, s, x), 0.5f * y, s);
}
