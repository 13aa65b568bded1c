// Gated DeltaNet (GDN) kernels for gfx950: ragged chunk prefill, the
// one-token step, the gated norm.
//
// Reference parity: the vendored FLA Triton kernels' chunk and
// fused_recurrent_gated_delta_rule paths + causal_conv1d_update +
// gated RMSNorm (layers/ops/fla/fused_recurrent.py:16,
// layers/ops/mamba/causal_conv1d_triton.py:584, fused_norm_gate.py).
// A whole batch is one launch per op; a step streams each recurrent state
// S [Dv, Dk] exactly once (read + write).
//
// Recurrence per (seq, v-head), single token:
//   Sk   = exp(g) * (S_old @ k)
//   u    = beta * (v - Sk)            (per v-row)
//   S    = exp(g) * S_old + u k^T
//   o    = S @ q

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

// ---------------------------------------------------------- conv update
// x [B, C] input token; weight [C, K]; conv_state [slots, C, K-1]
// (rolls in place); out [B, C] = silu(conv).
template <int K>
__global__ void gdn_conv_update_kernel(
    __hip_bfloat16 *__restrict__ out, const __hip_bfloat16 *__restrict__ x,
    const __hip_bfloat16 *__restrict__ weight,
    __hip_bfloat16 *__restrict__ conv_state,
    const long *__restrict__ slots, int C, long state_stride) {
  const int b = blockIdx.x;
  const long slot = slots[b];
  __hip_bfloat16 *st = conv_state + slot * state_stride;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < C;
       c += gridDim.y * blockDim.x) {
    float ctx[K];
#pragma unroll
    for (int j = 0; j < K - 1; ++j)
      ctx[j] = __bfloat162float(st[(long)c * (K - 1) + j]);
    ctx[K - 1] = __bfloat162float(x[(long)b * C + c]);
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < K; ++j)
      acc += ctx[j] * __bfloat162float(weight[(long)c * K + j]);
#pragma unroll
    for (int j = 0; j < K - 1; ++j)
      st[(long)c * (K - 1) + j] = __float2bfloat16(ctx[j + 1]);
    const float s = acc / (1.f + __expf(-acc));
    out[(long)b * C + c] = __float2bfloat16(s);
  }
}

// ---------------------------------------------------------- delta decode
// qn/kn [B, Hv, Dk] fp32 (L2-normalized, q pre-scaled); v [B, Hv, Dv]
// fp32; g, beta [B, Hv] fp32; state pool [slots, Hv, Dv, Dk] fp32.
template <int DK>
__global__ __launch_bounds__(256) void gdn_decode_kernel(
    __hip_bfloat16 *__restrict__ o,        // [B, Hv, Dv]
    const float *__restrict__ qn, const float *__restrict__ kn,
    const float *__restrict__ v, const float *__restrict__ g,
    const float *__restrict__ beta, float *__restrict__ state,
    const long *__restrict__ slots, int Hv, int Dv, long slot_stride,
    long head_stride) {
  const int b = blockIdx.x;
  const int h = blockIdx.y;
  const long slot = slots[b];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  constexpr int PER_LANE = DK / 64;  // float2 for DK=128

  float *S = state + slot * slot_stride + h * head_stride;
  const float eg = __expf(g[(long)b * Hv + h]);
  const float bt = beta[(long)b * Hv + h];

  float kf[PER_LANE], qf[PER_LANE];
#pragma unroll
  for (int j = 0; j < PER_LANE; ++j) {
    kf[j] = kn[((long)b * Hv + h) * DK + lane * PER_LANE + j];
    qf[j] = qn[((long)b * Hv + h) * DK + lane * PER_LANE + j];
  }

  for (int row = wave; row < Dv; row += 4) {
    float *srow = S + (long)row * DK + lane * PER_LANE;
    float s[PER_LANE];
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      s[j] = srow[j];
      dot += s[j] * kf[j];
    }
    dot = wave_reduce_sum(dot);
    const float u = bt * (v[((long)b * Hv + h) * Dv + row] - eg * dot);
    float od = 0.f;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      s[j] = eg * s[j] + u * kf[j];
      srow[j] = s[j];
      od += s[j] * qf[j];
    }
    od = wave_reduce_sum(od);
    if (lane == 0)
      o[((long)b * Hv + h) * Dv + row] = __float2bfloat16(od);
  }
}

// ---------------------------------------------------------- gated norm
// out = rmsnorm(x) * w * silu(z); rows [N, D], one wave per row.
__global__ void rmsnorm_gated_kernel(__hip_bfloat16 *__restrict__ out,
                                     const __hip_bfloat16 *__restrict__ x,
                                     const __hip_bfloat16 *__restrict__ z,
                                     const __hip_bfloat16 *__restrict__ w,
                                     float eps, long N, int D) {
  const long row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= N) return;
  const int lane = threadIdx.x & 63;
  const __hip_bfloat16 *xr = x + row * D;
  const __hip_bfloat16 *zr = z + row * D;
  float ss = 0.f;
  for (int i = lane; i < D; i += 64) {
    const float xv = __bfloat162float(xr[i]);
    ss += xv * xv;
  }
  ss = wave_reduce_sum(ss);
  const float inv = rsqrtf(ss / D + eps);
  for (int i = lane; i < D; i += 64) {
    const float xv = __bfloat162float(xr[i]);
    const float zv = __bfloat162float(zr[i]);
    const float sz = zv / (1.f + __expf(-zv));
    out[row * D + i] =
        __float2bfloat16(xv * inv * __bfloat162float(w[i]) * sz);
  }
}


// ------------------------------------------------- chunked WY prefill
// Chunk-parallel gated delta rule (WY form) over a ragged batch, all in fp32
// (V_MFMA_F32_16X16X4_F32), in two kernels:
//
//   local   one workgroup per (64-token chunk, v-head), all chunks at once:
//           unit keys, A = strict tril(beta_t exp(b_t - b_i) k_t k_i), and
//           X = (I + A)^-1 [beta B k | beta v] by blocks of 16 rows (their
//           inverses by substitution, the rest as products), att =
//           tril(exp(b_t - b_i) q_t k_i). b is the running log decay.
//   carry   one workgroup per (sequence, v-head, DVS value columns), chunk
//           after chunk: U = X_v - X_k S^T, o = B q S^T + att U,
//           S = B_last S + (exp(b_last - b) U)^T k, with its columns of S in
//           accumulators and LDS and the next chunk's operands on their way
//           into registers.
// Only what needs the state is serial: 224 matrix instructions a wave and
// chunk at 32 columns. One kernel that did all of it chunk after chunk, a
// workgroup per (sequence, head, 64 columns) and the substitution on one
// wave, took 922 us for 4096 tokens in four prompts, 16 heads of 128; these
// take 212 (local; five rounds of workgroups, one per CU by its LDS) and
// 200 us (carry; the serial chain of the longest prompt, 3 us of matrix
// instructions a chunk). X and att are 168 MB of traffic, 34 us.
typedef __attribute__((ext_vector_type(4))) float gdn_f4;

constexpr int C = 64;     // tokens of a chunk
constexpr int D = 128;    // key and value size of a head
constexpr int KS = 132;   // LDS row of 128 floats: rows 4 banks apart
constexpr int AS = 68;    // of 64 floats
constexpr int XS = 272;   // of 256 floats: rows 16 banks apart
constexpr int US = 48;    // of 32 floats

DEV_INLINE gdn_f4 mma4(float a, float b, gdn_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

DEV_INLINE float sigmoid_f(float x) { return 1.f / (1.f + __expf(-x)); }

// log decay and write strength of a token and head, either given or formed
// from the projections (g = -exp(A_log) softplus(a + dt), beta = sigmoid(b))
struct Gates {
  const float *g, *beta;            // [T, Hv]
  const __hip_bfloat16 *ba;         // rows of b | a
  long ba_stride;
  const float *A_log, *dt;          // [Hv]
  DEV_INLINE void at(long t, int h, int Hv, float &gv, float &bv) const {
    if (g) {
      gv = g[t * Hv + h];
      bv = beta[t * Hv + h];
      return;
    }
    const float a = __bfloat162float(ba[t * ba_stride + Hv + h]) + dt[h];
    const float sp = a > 20.f ? a : log1pf(expf(a));
    gv = -expf(A_log[h]) * sp;
    bv = 1.f / (1.f + expf(-__bfloat162float(ba[t * ba_stride + h])));
  }
};

__global__ __launch_bounds__(256) void gdn_local_kernel(
    float *__restrict__ wk, float *__restrict__ u0,  // X_k, X_v [T, Hv, D]
    float *__restrict__ att,                         // [T, Hv, C]
    float *__restrict__ scal,                        // [3, T, Hv]: b, 1/|k|, scale/|q|
    const __hip_bfloat16 *__restrict__ q, const __hip_bfloat16 *__restrict__ k,
    const __hip_bfloat16 *__restrict__ v, long qk_stride, long v_stride,
    Gates gates, const int *__restrict__ qsl, long T, int Hk, int Hv,
    float scale) {
  const int seq = blockIdx.y, h = blockIdx.z;
  const int start = qsl[seq] + blockIdx.x * C;
  const int len = min(C, qsl[seq + 1] - start);
  if (len <= 0) return;
  const int hk = h / (Hv / Hk);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  __shared__ float Kt[C * KS];
  __shared__ float X[C * XS];     // q first, the solution afterwards
  __shared__ float Am[C * AS];
  __shared__ float Di[4][16 * 20];
  __shared__ float bb[C], btv[C];
  float *Qt = X;

  // ---- 16 rows of a wave: unit keys and queries
  unsigned kr[16], qr[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int t = wave * 16 + r;
    const long row = (long)(start + min(t, len - 1)) * qk_stride + hk * D;
    kr[r] = reinterpret_cast<const unsigned *>(k + row)[lane];
    qr[r] = reinterpret_cast<const unsigned *>(q + row)[lane];
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int t = wave * 16 + r;
    float k0 = __uint_as_float(kr[r] << 16);
    float k1 = __uint_as_float(kr[r] & 0xffff0000u);
    float q0 = __uint_as_float(qr[r] << 16);
    float q1 = __uint_as_float(qr[r] & 0xffff0000u);
    const float live = t < len ? 1.f : 0.f;
    const float rk = live * rsqrtf(wave_reduce_sum(k0 * k0 + k1 * k1) + 1e-6f);
    const float rq =
        live * rsqrtf(wave_reduce_sum(q0 * q0 + q1 * q1) + 1e-6f) * scale;
    *reinterpret_cast<floatx2 *>(Kt + t * KS + lane * 2) =
        floatx2{k0 * rk, k1 * rk};
    *reinterpret_cast<floatx2 *>(Qt + t * KS + lane * 2) =
        floatx2{q0 * rq, q1 * rq};
    if (lane == 0 && t < len) {
      scal[(T + start + t) * Hv + h] = rk;
      scal[(2 * T + start + t) * Hv + h] = rq;
    }
  }
  if (wave == 0) {  // running log decay
    float gv = 0.f, bv = 0.f;
    if (lane < len) gates.at(start + lane, h, Hv, gv, bv);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float prev = __shfl_up(gv, off, 64);
      if (lane >= off) gv += prev;
    }
    bb[lane] = gv;
    btv[lane] = bv;
    if (lane < len) scal[(long)(start + lane) * Hv + h] = gv;
  }
  __syncthreads();

  // ---- rows 16 w .. + 15 of A and att (blocks on and below the diagonal)
  for (int it = 0; it <= wave; ++it) {
    gdn_f4 a = {0, 0, 0, 0}, s = {0, 0, 0, 0};
#pragma unroll 8
    for (int ks = 0; ks < D / 4; ++ks) {
      const float ki = Kt[(it * 16 + l16) * KS + ks * 4 + lhi];
      a = mma4(Kt[(wave * 16 + l16) * KS + ks * 4 + lhi], ki, a);
      s = mma4(Qt[(wave * 16 + l16) * KS + ks * 4 + lhi], ki, s);
    }
    const int i = it * 16 + l16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = wave * 16 + lhi * 4 + r;
      const float d = i <= t ? __expf(bb[t] - bb[i]) : 0.f;
      Am[t * AS + i] = i < t ? btv[t] * d * a[r] : 0.f;
      if (t < len) att[((long)(start + t) * Hv + h) * C + i] = d * s[r];
    }
  }
  // right hand sides: waves 0, 1 the keys' columns, 2, 3 the values'
  gdn_f4 x[4][4];
  const int c0 = (wave & 1) * 64;
#pragma unroll
  for (int R = 0; R < 4; ++R)
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = R * 16 + lhi * 4 + r, c = c0 + n * 16 + l16;
        if (wave < 2) {
          x[R][n][r] = btv[t] * __expf(bb[t]) * Kt[t * KS + c];
        } else {
          const float vv = __bfloat162float(
              v[(long)(start + min(t, len - 1)) * v_stride + h * D + c]);
          x[R][n][r] = btv[t] * vv;  // (rows past the end: beta 0)
        }
      }
  __syncthreads();  // A is there; q is not needed any more
  {  // inverse of this wave's diagonal block, a column per lane
    float y[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = i == l16 ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j)
        acc -= Am[(wave * 16 + i) * AS + wave * 16 + j] * y[j];
      y[i] = acc;
    }
    if (lhi == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) Di[wave][i * 20 + l16] = y[i];
    }
  }
  __syncthreads();
  float *xw = X + wave * 64;  // this wave's columns
  float *dst = wave < 2 ? wk : u0;
#pragma unroll
  for (int R = 0; R < 4; ++R) {
    for (int ks = 0; ks < R * 4; ++ks) {
      const float a = -Am[(R * 16 + l16) * AS + ks * 4 + lhi];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        x[R][n] = mma4(a, xw[(ks * 4 + lhi) * XS + n * 16 + l16], x[R][n]);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        xw[(R * 16 + lhi * 4 + r) * XS + n * 16 + l16] = x[R][n][r];
    __syncthreads();
    gdn_f4 y[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) y[n] = gdn_f4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const float a = Di[R][l16 * 20 + ks * 4 + lhi];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        y[n] = mma4(a, xw[(R * 16 + ks * 4 + lhi) * XS + n * 16 + l16], y[n]);
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = R * 16 + lhi * 4 + r;
        xw[t * XS + n * 16 + l16] = y[n][r];
        if (t < len)
          dst[((long)(start + t) * Hv + h) * D + c0 + n * 16 + l16] = y[n][r];
      }
    __syncthreads();
  }
}

// DVS value columns of a (sequence, head)
template <int DVS>
__global__ __launch_bounds__(256, 1) void gdn_carry_kernel(
    __hip_bfloat16 *__restrict__ o,  // [T, Hv, D]
    float *__restrict__ states,      // [slots, Hv, D, D], in place
    const float *__restrict__ wk, const float *__restrict__ u0,
    const float *__restrict__ att, const float *__restrict__ scal,
    const __hip_bfloat16 *__restrict__ q, const __hip_bfloat16 *__restrict__ k,
    long qk_stride, const long *__restrict__ slots,
    const int *__restrict__ has_init, const int *__restrict__ qsl, long T,
    int Hk, int Hv) {
  constexpr int VT = DVS / 16;
  const int seq = blockIdx.x, h = blockIdx.y, z = blockIdx.z;
  const int begin = qsl[seq], end = qsl[seq + 1];
  if (begin >= end) return;
  const int hk = h / (Hv / Hk);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  __shared__ float Ws[C * KS], Ks[C * KS], Qs[C * KS], At[C * AS];
  __shared__ float Ss[DVS * KS], Us[C * US];
  __shared__ float bb[C];

  // S rows (values) vt * 16 + lhi * 4 + r, columns (keys) of this wave's
  // two tiles
  float *sg = states + ((slots[seq] * Hv + h) * D + z * DVS) * D;
  gdn_f4 s[VT][2];
  const bool init = has_init[seq] != 0;
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int vr = vt * 16 + lhi * 4 + r, d = (wave * 2 + dt) * 16 + l16;
        s[vt][dt][r] = init ? sg[(long)vr * D + d] : 0.f;
        Ss[vr * KS + d] = s[vt][dt][r];
      }

  // operands of a chunk, on their way in registers
  floatx4 wr[8], ar[4];
  shortx8 kr[4], qr[4];
  float rk[4], rq[4], ur[VT][4], br;
  auto fetch = [&](int start) {
    const int len = min(C, end - start);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int u = j * 256 + tid, row = u >> 5, c = (u & 31) * 4;
      wr[j] = row < len ? *reinterpret_cast<const floatx4 *>(
                              wk + ((long)(start + row) * Hv + h) * D + c)
                        : floatx4{0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = j * 256 + tid, row = u >> 4, c = u & 15;
      const bool live = row < len;
      const long t = start + min(row, len - 1);
      // (columns above the diagonal block are never read)
      ar[j] = live ? *reinterpret_cast<const floatx4 *>(
                         att + (t * Hv + h) * C + c * 4)
                   : floatx4{0, 0, 0, 0};
      kr[j] = *reinterpret_cast<const shortx8 *>(k + t * qk_stride + hk * D +
                                                 c * 8);
      qr[j] = *reinterpret_cast<const shortx8 *>(q + t * qk_stride + hk * D +
                                                 c * 8);
      rk[j] = live ? scal[(T + t) * Hv + h] : 0.f;
      rq[j] = live ? scal[(2 * T + t) * Hv + h] : 0.f;
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = wave * 16 + lhi * 4 + r;
        ur[vt][r] = t < len ? u0[((long)(start + t) * Hv + h) * D + z * DVS +
                                 vt * 16 + l16]
                            : 0.f;
      }
    br = scal[(long)(start + min(lane, len - 1)) * Hv + h];
  };
  fetch(begin);
  for (int start = begin; start < end; start += C) {
    const int len = min(C, end - start);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int u = j * 256 + tid;
      *reinterpret_cast<floatx4 *>(Ws + (u >> 5) * KS + (u & 31) * 4) = wr[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = j * 256 + tid, row = u >> 4, c = u & 15;
      *reinterpret_cast<floatx4 *>(At + row * AS + c * 4) = ar[j];
      float kf[8], qf[8];
      unpack8<__hip_bfloat16>(kr[j], kf);
      unpack8<__hip_bfloat16>(qr[j], qf);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        kf[e] *= rk[j];
        qf[e] *= rq[j];
      }
      st8<float>(Ks + row * KS + c * 8, kf);
      st8<float>(Qs + row * KS + c * 8, qf);
    }
    if (wave == 0) bb[lane] = br;
    gdn_f4 u[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
      u[vt] = gdn_f4{ur[vt][0], ur[vt][1], ur[vt][2], ur[vt][3]};
    __syncthreads();
    if (start + C < end) fetch(start + C);

    // ---- U = X_v - X_k S^T and B q S^T, rows 16 w ..
    gdn_f4 qs[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) qs[vt] = gdn_f4{0, 0, 0, 0};
#pragma unroll 8
    for (int ks = 0; ks < D / 4; ++ks) {
      const float w = -Ws[(wave * 16 + l16) * KS + ks * 4 + lhi];
      const float qv = Qs[(wave * 16 + l16) * KS + ks * 4 + lhi];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const float sv = Ss[(vt * 16 + l16) * KS + ks * 4 + lhi];
        u[vt] = mma4(w, sv, u[vt]);
        qs[vt] = mma4(qv, sv, qs[vt]);
      }
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Us[(wave * 16 + lhi * 4 + r) * US + vt * 16 + l16] = u[vt][r];
        qs[vt][r] *= __expf(bb[wave * 16 + lhi * 4 + r]);
      }
    __syncthreads();
    // ---- o = that + att U (columns up to the diagonal block)
    for (int ks = 0; ks < (wave + 1) * 4; ++ks) {
      const float a = At[(wave * 16 + l16) * AS + ks * 4 + lhi];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
        qs[vt] = mma4(a, Us[(ks * 4 + lhi) * US + vt * 16 + l16], qs[vt]);
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = wave * 16 + lhi * 4 + r;
        if (t < len)
          o[((long)(start + t) * Hv + h) * D + z * DVS + vt * 16 + l16] =
              __float2bfloat16(qs[vt][r]);
      }
    // ---- S = B_last S + (exp(b_last - b) U)^T k
    const float last = bb[len - 1], keep = __expf(last);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[vt][dt][r] *= keep;
#pragma unroll 4
    for (int ks = 0; ks < C / 4; ++ks) {
      const int t = ks * 4 + lhi;
      const float wc = __expf(last - bb[t]);
      float kv[2];
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
        kv[dt] = Ks[t * KS + (wave * 2 + dt) * 16 + l16];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const float uv = wc * Us[t * US + vt * 16 + l16];
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
          s[vt][dt] = mma4(uv, kv[dt], s[vt][dt]);
      }
    }
    __syncthreads();  // everybody is done with this chunk's operands and S
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          Ss[(vt * 16 + lhi * 4 + r) * KS + (wave * 2 + dt) * 16 + l16] =
              s[vt][dt][r];
  }
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sg[(long)(vt * 16 + lhi * 4 + r) * D + (wave * 2 + dt) * 16 + l16] =
            s[vt][dt][r];
}

// ------------------------------------------------- one token per sequence
// From the convolved projection: unit q and k, gates, and one pass over the
// state (16 lanes per state row, four rows per wave and step). Bound by the
// state's bytes (64 KB read and written per head). It stands for the slices,
// norms, repeats and conversions (about 20 launches) in front of gdn_decode.
__global__ __launch_bounds__(256) void gdn_step_kernel(
    __hip_bfloat16 *__restrict__ o, float *__restrict__ states,
    const __hip_bfloat16 *__restrict__ q, const __hip_bfloat16 *__restrict__ k,
    const __hip_bfloat16 *__restrict__ v, long qk_stride, long v_stride,
    Gates gates, const long *__restrict__ slots, int Hk, int Hv,
    float scale) {
  const long b = blockIdx.x;
  const int h = blockIdx.y, hk = h / (Hv / Hk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int l16 = lane & 15, sub = lane >> 4;
  float kf[8], qf[8], nk = 0.f, nq = 0.f;
  ld8<__hip_bfloat16>(k + b * qk_stride + hk * D + l16 * 8, kf);
  ld8<__hip_bfloat16>(q + b * qk_stride + hk * D + l16 * 8, qf);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    nk += kf[e] * kf[e];
    nq += qf[e] * qf[e];
  }
  const float rk = rsqrtf(lanes_sum<16>(nk) + 1e-6f);
  const float rq = rsqrtf(lanes_sum<16>(nq) + 1e-6f) * scale;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    kf[e] *= rk;
    qf[e] *= rq;
  }
  float gv, bt;
  gates.at(b, h, Hv, gv, bt);
  const float eg = __expf(gv);
  float *S = states + (slots[b] * Hv + h) * (long)D * D + l16 * 8;
#pragma unroll 4
  for (int it = 0; it < D / 16; ++it) {
    const int row = it * 16 + wave * 4 + sub;
    float s[8], dot = 0.f, od = 0.f;
    ld8<float>(S + (long)row * D, s);
#pragma unroll
    for (int e = 0; e < 8; ++e) dot += s[e] * kf[e];
    dot = lanes_sum<16>(dot);
    const float u =
        bt * (__bfloat162float(v[b * v_stride + h * D + row]) - eg * dot);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] = eg * s[e] + u * kf[e];
      od += s[e] * qf[e];
    }
    st8<float>(S + (long)row * D, s);
    od = lanes_sum<16>(od);
    if (l16 == 0) o[(b * Hv + h) * D + row] = __float2bfloat16(od);
  }
}

// out = rmsnorm(o) * w * silu(z) per head of 128; z may be a column slice.
// 16 lanes per head.
__global__ __launch_bounds__(256) void gdn_gate_kernel(
    __hip_bfloat16 *__restrict__ out, const __hip_bfloat16 *__restrict__ o,
    const __hip_bfloat16 *__restrict__ z, long z_stride,
    const __hip_bfloat16 *__restrict__ w, float eps, long rows, int H) {
  const long row = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (row >= rows) return;
  const int l16 = threadIdx.x & 15;
  const long t = row / H;
  const int h = row % H;
  float x[8], zf[8], wf[8], ss = 0.f;
  ld8<__hip_bfloat16>(o + row * D + l16 * 8, x);
  ld8<__hip_bfloat16>(z + t * z_stride + h * D + l16 * 8, zf);
  ld8<__hip_bfloat16>(w + l16 * 8, wf);
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
  const float inv = rsqrtf(lanes_sum<16>(ss) / D + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e)
    x[e] = x[e] * inv * wf[e] * (zf[e] * sigmoid_f(zf[e]));
  st8<__hip_bfloat16>(out + row * D + l16 * 8, x);
}

}  // namespace

void gdn_conv_update(torch::Tensor out, torch::Tensor x,
                     torch::Tensor weight, torch::Tensor conv_state,
                     torch::Tensor slots) {
  const int B = x.size(0), C = x.size(1);
  const int K = weight.size(1);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_contiguous());
  TORCH_CHECK(conv_state.scalar_type() == at::kBFloat16);
  TORCH_CHECK(conv_state.stride(1) == K - 1,
              "conv_state rows must be contiguous");
  TORCH_CHECK(slots.scalar_type() == at::kLong);
  auto stream = at::cuda::getCurrentCUDAStream();
  const int ygrid = std::min(16, (C + 255) / 256);
  TORCH_CHECK(K == 4, "gdn conv: kernel width 4 expected");
  hipLaunchKernelGGL((gdn_conv_update_kernel<4>), dim3(B, ygrid),
                     dim3(256), 0, stream,
                     (__hip_bfloat16 *)out.data_ptr(),
                     (const __hip_bfloat16 *)x.data_ptr(),
                     (const __hip_bfloat16 *)weight.data_ptr(),
                     (__hip_bfloat16 *)conv_state.data_ptr(),
                     slots.data_ptr<long>(), C, conv_state.stride(0));
  HIP_CHECK_KERNEL();
}

void gdn_decode(torch::Tensor o, torch::Tensor qn, torch::Tensor kn,
                torch::Tensor v, torch::Tensor g, torch::Tensor beta,
                torch::Tensor state, torch::Tensor slots) {
  const int B = qn.size(0), Hv = qn.size(1), Dk = qn.size(2);
  const int Dv = v.size(2);
  TORCH_CHECK(qn.scalar_type() == at::kFloat && qn.is_contiguous());
  TORCH_CHECK(state.scalar_type() == at::kFloat);
  TORCH_CHECK(state.stride(3) == 1 && state.stride(2) == Dk,
              "state head must be contiguous [Dv, Dk]");
  TORCH_CHECK(Dk == 128, "gdn decode: Dk=128 expected");
  TORCH_CHECK(slots.scalar_type() == at::kLong);
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL((gdn_decode_kernel<128>), dim3(B, Hv), dim3(256), 0,
                     stream, (__hip_bfloat16 *)o.data_ptr(),
                     qn.data_ptr<float>(), kn.data_ptr<float>(),
                     v.data_ptr<float>(), g.data_ptr<float>(),
                     beta.data_ptr<float>(), state.data_ptr<float>(),
                     slots.data_ptr<long>(), Hv, Dv, state.stride(0),
                     state.stride(1));
  HIP_CHECK_KERNEL();
}

void rmsnorm_gated(torch::Tensor out, torch::Tensor x, torch::Tensor z,
                   torch::Tensor w, double eps) {
  const long N = x.size(0);
  const int D = x.size(1);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_contiguous());
  TORCH_CHECK(z.is_contiguous() && out.is_contiguous());
  auto stream = at::cuda::getCurrentCUDAStream();
  const long grid = (N + 3) / 4;
  hipLaunchKernelGGL(rmsnorm_gated_kernel, dim3(grid), dim3(256), 0,
                     stream, (__hip_bfloat16 *)out.data_ptr(),
                     (const __hip_bfloat16 *)x.data_ptr(),
                     (const __hip_bfloat16 *)z.data_ptr(),
                     (const __hip_bfloat16 *)w.data_ptr(), (float)eps, N,
                     D);
  HIP_CHECK_KERNEL();
}

namespace {

bool rows16(const torch::Tensor &t) {
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 &&
         t.stride(-1) == 1 &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

void run_chunks(torch::Tensor &o, const void *q, const void *k,
                const void *v, long qk_stride, long v_stride,
                const Gates &gates, torch::Tensor &states, const long *slots,
                const int *has_init, const int *qsl, long T, int B,
                int max_len, int Hk, int Hv, double scale) {
  auto opts = states.options();
  auto wk = torch::empty({T, (long)Hv, (long)D}, opts);
  auto u0 = torch::empty({T, (long)Hv, (long)D}, opts);
  auto att = torch::empty({T, (long)Hv, (long)C}, opts);
  auto scal = torch::empty({3, T, (long)Hv}, opts);
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(gdn_local_kernel, dim3((max_len + C - 1) / C, B, Hv),
                     dim3(256), 0, stream, wk.data_ptr<float>(),
                     u0.data_ptr<float>(), att.data_ptr<float>(),
                     scal.data_ptr<float>(), (const __hip_bfloat16 *)q,
                     (const __hip_bfloat16 *)k, (const __hip_bfloat16 *)v,
                     qk_stride, v_stride, gates, qsl, T, Hk, Hv,
                     (float)scale);
  HIP_CHECK_KERNEL();
#define RUN(DVS)                                                             \
  hipLaunchKernelGGL((gdn_carry_kernel<DVS>), dim3(B, Hv, D / DVS),          \
                     dim3(256), 0, stream, (__hip_bfloat16 *)o.data_ptr(),   \
                     states.data_ptr<float>(), wk.data_ptr<float>(),         \
                     u0.data_ptr<float>(), att.data_ptr<float>(),            \
                     scal.data_ptr<float>(), (const __hip_bfloat16 *)q,      \
                     (const __hip_bfloat16 *)k, qk_stride, slots, has_init,  \
                     qsl, T, Hk, Hv)
  // (narrower columns shorten the serial chain as long as CUs are free)
  if ((long)B * Hv * 4 < 256) RUN(16); else RUN(32);
#undef RUN
  HIP_CHECK_KERNEL();
}

}  // namespace

// the padded form: q, k [B, T, Hk, 128], v [B, T, Hv, 128], g and beta [B, T,
// Hv], states [B, Hv, 128, 128] in place
void gdn_chunk_prefill(torch::Tensor o, torch::Tensor q, torch::Tensor k,
                       torch::Tensor v, torch::Tensor g, torch::Tensor beta,
                       torch::Tensor states, double scale) {
  const int B = q.size(0), T = q.size(1), Hk = q.size(2);
  const int Hv = v.size(2);
  TORCH_CHECK(q.size(3) == 128 && v.size(3) == 128,
              "gdn prefill: Dk = Dv = 128");
  TORCH_CHECK(Hv % Hk == 0);
  TORCH_CHECK(q.is_contiguous() && k.is_contiguous() && v.is_contiguous() &&
              o.is_contiguous() && rows16(q) && rows16(k) && rows16(v));
  TORCH_CHECK(g.is_contiguous() && beta.is_contiguous() &&
              g.scalar_type() == at::kFloat &&
              beta.scalar_type() == at::kFloat);
  TORCH_CHECK(states.is_contiguous() &&
              states.scalar_type() == at::kFloat);
  if (B == 0 || T == 0) return;
  auto ints = q.options().dtype(at::kInt);
  auto qsl = torch::arange(0, (long)(B + 1) * T, (long)T, ints);
  auto ones = torch::ones({(long)B}, ints);
  auto slots = torch::arange((long)B, q.options().dtype(at::kLong));
  const Gates gates = {g.data_ptr<float>(), beta.data_ptr<float>(), nullptr,
                       0, nullptr, nullptr};
  run_chunks(o, q.data_ptr(), k.data_ptr(), v.data_ptr(), (long)Hk * D,
             (long)Hv * D, gates, states, slots.data_ptr<long>(),
             ones.data_ptr<int>(), qsl.data_ptr<int>(), (long)B * T, B, T,
             Hk, Hv, scale);
}

namespace {

// conv [T, (2 Hk + Hv) 128] rows of q | k | v; ba [T, 2 Hv] rows of b | a
Gates check_rows(const torch::Tensor &conv, const torch::Tensor &ba,
                 const torch::Tensor &A_log, const torch::Tensor &dt_bias,
                 const torch::Tensor &states, const torch::Tensor &slots,
                 int Hk) {
  const int Hv = states.size(1);
  TORCH_CHECK(rows16(conv) && conv.dim() == 2 && conv.stride(0) % 8 == 0 &&
              conv.size(1) == (2L * Hk + Hv) * D && Hk > 0 && Hv % Hk == 0,
              "gdn: conv rows of q | k | v, heads of 128");
  TORCH_CHECK(ba.is_cuda() && ba.scalar_type() == at::kBFloat16 &&
              ba.dim() == 2 && ba.stride(1) == 1 &&
              ba.size(0) == conv.size(0) && ba.size(1) == 2L * Hv);
  TORCH_CHECK(A_log.scalar_type() == at::kFloat && A_log.numel() == Hv &&
              dt_bias.scalar_type() == at::kFloat && dt_bias.numel() == Hv &&
              A_log.is_contiguous() && dt_bias.is_contiguous());
  TORCH_CHECK(states.dim() == 4 && states.is_contiguous() &&
              states.scalar_type() == at::kFloat && states.size(2) == D &&
              states.size(3) == D, "gdn: state [slots, Hv, 128, 128] fp32");
  TORCH_CHECK(slots.scalar_type() == at::kLong && slots.is_contiguous());
  return {nullptr, nullptr, (const __hip_bfloat16 *)ba.data_ptr(),
          (long)ba.stride(0), A_log.data_ptr<float>(),
          dt_bias.data_ptr<float>()};
}

}  // namespace

// ragged prompt portions and decode tokens; returns [T, Hv, 128]
torch::Tensor gdn_varlen(torch::Tensor conv, torch::Tensor ba,
                         torch::Tensor A_log, torch::Tensor dt_bias,
                         torch::Tensor states, torch::Tensor slots,
                         torch::Tensor has_init, torch::Tensor qsl, long Hk,
                         long max_len, double scale) {
  const Gates gates =
      check_rows(conv, ba, A_log, dt_bias, states, slots, Hk);
  const long T = conv.size(0), B = slots.numel();
  const int Hv = states.size(1);
  TORCH_CHECK(has_init.scalar_type() == at::kInt && has_init.numel() == B &&
              qsl.scalar_type() == at::kInt && qsl.numel() >= B + 1);
  auto o = torch::empty({T, (long)Hv, (long)D}, conv.options());
  if (T == 0) return o;
  const auto *p = (const __hip_bfloat16 *)conv.data_ptr();
  run_chunks(o, p, p + Hk * D, p + 2 * Hk * D, conv.stride(0),
             conv.stride(0), gates, states, slots.data_ptr<long>(),
             has_init.data_ptr<int>(), qsl.data_ptr<int>(), T, (int)B,
             (int)max_len, (int)Hk, Hv, scale);
  return o;
}

// one token per sequence on carried state; returns [B, Hv, 128]
torch::Tensor gdn_step(torch::Tensor conv, torch::Tensor ba,
                       torch::Tensor A_log, torch::Tensor dt_bias,
                       torch::Tensor states, torch::Tensor slots, long Hk,
                       double scale) {
  const Gates gates =
      check_rows(conv, ba, A_log, dt_bias, states, slots, Hk);
  const long B = conv.size(0);
  const int Hv = states.size(1);
  TORCH_CHECK(slots.numel() == B);
  auto o = torch::empty({B, (long)Hv, (long)D}, conv.options());
  if (B == 0) return o;
  const auto *p = (const __hip_bfloat16 *)conv.data_ptr();
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(gdn_step_kernel, dim3(B, Hv), dim3(256), 0, stream,
                     (__hip_bfloat16 *)o.data_ptr(), states.data_ptr<float>(),
                     p, p + Hk * D, p + 2 * Hk * D, (long)conv.stride(0),
                     (long)conv.stride(0), gates, slots.data_ptr<long>(),
                     (int)Hk, Hv, (float)scale);
  HIP_CHECK_KERNEL();
  return o;
}

// rmsnorm(o) * w * silu(z): o [T, H, 128], z [T, H * 128] (a column slice of
// a wider projection is fine) -> [T, H * 128]
torch::Tensor gdn_gate(torch::Tensor o, torch::Tensor z, torch::Tensor w,
                       double eps) {
  const long T = o.size(0), H = o.size(1);
  TORCH_CHECK(rows16(o) && o.is_contiguous() && o.size(2) == D);
  TORCH_CHECK(rows16(z) && z.dim() == 2 && z.size(0) == T &&
              z.size(1) == H * D && z.stride(0) % 8 == 0);
  TORCH_CHECK(rows16(w) && w.numel() == D);
  auto out = torch::empty({T, H * D}, o.options());
  if (T == 0) return out;
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(gdn_gate_kernel, dim3((T * H + 15) / 16), dim3(256), 0,
                     stream, (__hip_bfloat16 *)out.data_ptr(),
                     (const __hip_bfloat16 *)o.data_ptr(),
                     (const __hip_bfloat16 *)z.data_ptr(),
                     (long)z.stride(0), (const __hip_bfloat16 *)w.data_ptr(),
                     (float)eps, T * H, (int)H);
  HIP_CHECK_KERNEL();
  return out;
}
