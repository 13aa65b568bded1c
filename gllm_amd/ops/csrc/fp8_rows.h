// e4m3 rows as the fp8 products take them: a scale per row and 128 columns,
// [columns / 128, rows], and bytes. What a kernel leaves in this form is what
// per_token_group_quant_fp8 makes of its bf16 result: a launch less in front of
// each product (a two-layer step of 64 rows of 5120, seven of eight launches:
// 473 -> 458 us).
#pragma once

#include "common.h"

struct Fp8Out {
  unsigned char *q;  // [M, N]; null: not wanted
  float *scales;     // [N / 128, M]
};

// scale of a group whose largest value is amax
DEV_INLINE float fp8_scale(float amax) { return fmaxf(amax, 1e-4f) / 448.f; }

DEV_INLINE unsigned fp8_byte(float v) { return __hip_fp8_e4m3(v).__x; }

DEV_INLINE unsigned fp8_bytes(const float (&v)[4], float inv) {
  return fp8_byte(v[0] * inv) | fp8_byte(v[1] * inv) << 8 |
         fp8_byte(v[2] * inv) << 16 | fp8_byte(v[3] * inv) << 24;
}
