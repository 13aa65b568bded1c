// fp32 parts of a product and how their readers sum them; rows of a merged
// q | k | v projection brought to biased, rotated bf16 columns.
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(4))) float part_f4;

DEV_INLINE short to_bf16(float v) {
  return __builtin_bit_cast(short, __float2bfloat16(v));
}

DEV_INLINE float bf16_value(float v) {
  return __bfloat162float(__float2bfloat16(v));
}

// sums of the S parts of V groups of four columns, in the order of S. Loads of
// nine parts are in flight, and no part is read twice: a workgroup that reads
// a row's parts is bound by its CU's 64 B a cycle.
template <int V>
DEV_INLINE void part_sums(const float *const (&p)[V], long stride, int S,
                          part_f4 (&v)[V]) {
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = *reinterpret_cast<const part_f4 *>(p[j]);
  for (int s = 1; s < S; s += 8) {
    part_f4 b[8][V];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s + i < S) {
#pragma unroll
        for (int j = 0; j < V; ++j)
          b[i][j] =
              *reinterpret_cast<const part_f4 *>(p[j] + (s + i) * stride);
      }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s + i < S) {
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] += b[i][j];
      }
  }
}

// Rows [M, (Hq + 2 Hkv) D] before their bias and rotation: fp32 parts [S, M,
// N], or bf16 rows `stride` apart.
struct QkvRows {
  const void *src;
  long stride;
  const __hip_bfloat16 *bias;
  const long *positions;
  const float *cos_sin;  // [position, rot]
  int M, S, rot, rounded;
};

// 4 + 4 columns of a head: a rotated pair block, or eight plain ones
struct QkvUnit {
  int d1, d2;
  shortx4 o1, o2;
};

// Unit u (of D / 8) of head h of H, row t; turned: a query or key head
// (rotate-half on the first `rot` columns).
template <bool PARTS>
DEV_INLINE QkvUnit qkv_unit(const QkvRows &R, long t, int h, int u,
                            bool turned, int H, int D) {
  QkvUnit x;
  turned = turned && u < R.rot / 8;
  x.d1 = turned ? u * 4 : u * 8;
  x.d2 = turned ? R.rot / 2 + u * 4 : u * 8 + 4;
  const int c1 = h * D + x.d1, c2 = h * D + x.d2, N = H * D;
  const float *cs = R.cos_sin + R.positions[t] * R.rot;
  part_f4 v[2];
  if (PARTS) {
    const float *p = (const float *)R.src + t * N;
    part_sums<2>({p + c1, p + c2}, (long)R.M * N, R.S, v);
  } else {
    const __hip_bfloat16 *p = (const __hip_bfloat16 *)R.src + t * R.stride;
    const shortx4 a = *reinterpret_cast<const shortx4 *>(p + c1);
    const shortx4 b = *reinterpret_cast<const shortx4 *>(p + c2);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[0][r] = __bfloat162float(
          __builtin_bit_cast(__hip_bfloat16, (short)a[r]));
      v[1][r] = __bfloat162float(
          __builtin_bit_cast(__hip_bfloat16, (short)b[r]));
    }
  }
  if (R.bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[0][r] += __bfloat162float(R.bias[c1 + r]);
      v[1][r] += __bfloat162float(R.bias[c2 + r]);
    }
  }
  if (R.rounded) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[0][r] = bf16_value(v[0][r]);
      v[1][r] = bf16_value(v[1][r]);
    }
  }
  if (turned) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float c = cs[x.d1 + r], s = cs[R.rot / 2 + x.d1 + r];
      const float a = v[0][r], b = v[1][r];
      v[0][r] = a * c - b * s;
      v[1][r] = b * c + a * s;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    x.o1[r] = to_bf16(v[0][r]);
    x.o2[r] = to_bf16(v[1][r]);
  }
  return x;
}
