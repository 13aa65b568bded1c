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
// Chunk-parallel gated delta rule (WY form) over a ragged batch, in two
// kernels (t, i: rows of a chunk; k, q: the unit keys and queries):
//
//   local   one workgroup per (64-token chunk, v-head), all chunks at once:
//           A = strict tril(beta_t exp(b_t - b_i) k_t k_i), T = (I + A)^-1 by
//           blocks of 16 rows, X = T [beta B k | beta v] and att =
//           tril(exp(b_t - b_i) q_t k_i). b is the running log decay.
//   carry   one workgroup per (sequence, v-head, 16 value columns), chunk
//           after chunk: U = X_v - X_k S^T, o = B q S^T + att U,
//           S = B_last S + (exp(b_last - b) U)^T k, with its columns of S in
//           accumulators and the next chunk's operands on their way into
//           the registers that this one has used.
//
// Keys, queries and values are bf16 and enter the matrix instructions as they
// are, their norms as fp32 factors of the sums; an fp32 operand (T, X_k, att,
// U, S) is the sum of three bf16 numbers, 24 bits in all, and a product of
// two such takes the six partial products above 2^-24. That is 3 (6)
// instructions of 16 cycles for 32 terms where fp32 ones take 8 of 32.
// Accumulation, T and the state stay fp32. Error of the state against 64
// bits, 64 to 1500 tokens, weak and strong decay: 1.1e-7 to 5.2e-7 (1.7e-7 to
// 5.3e-7 with fp32 instructions, mean 2.5e-7 against 2.9e-7).
//
// 4096 tokens in four prompts of 682 to 1365, 16 heads of 128: 44 + 68 us;
// with the same results, of carry's 118 us 91 were left when its operands
// stood in runs of 1 KB (see below; local 55 -> 48), 89 with 16 columns and
// two workgroups a CU for 32 and one (the next chunk's operands in registers
// that are free by then, 220 for 332: what follows a barrier or an LDS read
// in one workgroup is hidden by the other), 75 with sequences spread over the
// XCDs and 68 with the longest first. One prompt of 4096: 253 -> 152, 64 of
// 16: 98 -> 73, 30 tokens beside 700 + 900 + 15: 135 -> 58. (Queries and keys
// in rows of another stride, sums of att and state in turn: no faster.)
// local is bound by its chain of barriers and by its stores (X, att: 105 MB):
// with 36 KB of LDS four workgroups a CU, 44 us where 73 KB and two took 52 (54
// KB and three 46). carry is bound by what a CU takes in as much as by a
// chunk's chain (products of U, split, barrier, products of the state, split,
// barrier): 103 KB of operands a workgroup and chunk, the same for the eight of
// a sequence and head, 0.87 GB in 7.6 million reads of the L2, five of six of
// which hit. That is 49 KB a us and CU, 2.4 us a chunk alone and 4 us for two
// workgroups on a CU.
typedef __attribute__((ext_vector_type(4))) float gdn_f4;
typedef __attribute__((ext_vector_type(8))) __bf16 gdn_bf8;
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

union GdnFrag {
  gdn_bf8 v;
  shortx8 s;
  shortx4 h[2];
};

constexpr int C = 64;     // tokens of a chunk
constexpr int D = 128;    // key and value size of a head
constexpr int AS = 68;    // LDS row of 64 floats: rows 4 banks apart
constexpr int KB = 144;   // of 128 bf16, for transposed reads: 8 banks
constexpr int SB = 136;   // of 128 bf16: 4 banks
constexpr int UB = 72;    // of 64 bf16
constexpr int DVS = 16;   // value columns of a workgroup of carry

// What local leaves for carry stands as carry's waves take it, a block of 16
// rows and a head after the other and in it the 16 bytes of lane 0, 1, .. of
// each load: a load is one run of 1 KB. With rows of all heads side by side
// it was 16 runs of 64 bytes 4 KB apart, which share a channel of the L2, and
// local's stores 16 runs of 32 bytes.
constexpr int XK = 16 * D;  // X_k, of 3 parts: columns ks * 32 .. at ks * 512
constexpr int XV = 16 * D;  // X_v: value columns n * 16 .. at n * 256
constexpr int AT = 16 * C;  // att, of 3 parts: columns kk * 32 .. at kk * 512
// A sequence's first block there: blocks of 16 rows from row `start` on end
// before the next sequence's begin, T / 16 + sequences in all.
DEV_INLINE long first_block(int start, int seq) { return start / 16 + seq; }

DEV_INLINE gdn_f4 mma4(float a, float b, gdn_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

DEV_INLINE gdn_f4 mma32(const GdnFrag &a, const GdnFrag &b, gdn_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

// terms of a product of two numbers of three parts each, small ones first
constexpr int TERM_A[6] = {2, 0, 1, 1, 0, 0}, TERM_B[6] = {0, 2, 1, 0, 1, 0};

// x as a sum of three bf16 numbers
DEV_INLINE void split3(float x, short &h, short &m, short &l) {
  const __hip_bfloat16 a = __float2bfloat16(x);
  x -= __bfloat162float(a);
  const __hip_bfloat16 b = __float2bfloat16(x);
  x -= __bfloat162float(b);
  h = __builtin_bit_cast(short, a);
  m = __builtin_bit_cast(short, b);
  l = __builtin_bit_cast(short, __float2bfloat16(x));
}

DEV_INLINE void split3(gdn_f4 x, shortx4 (&p)[3]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    short h, m, l;
    split3(x[r], h, m, l);
    p[0][r] = h;
    p[1][r] = m;
    p[2][r] = l;
  }
}

// fragment of the transpose of an LDS tile with rows of `ld`: lane l16 is
// column col0 + l16, elements rows row0 + 4 lhi + 0..3 and + 16
DEV_INLINE void read_tr(GdnFrag &f, const short *tile, int ld, int row0,
                        int col0, int l16, int lhi) {
#pragma unroll
  for (int half = 0; half < 2; ++half)
    f.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_shortx4 *)(tile +
                        (row0 + half * 16 + lhi * 4 + (l16 >> 2)) * ld +
                        col0 + (l16 & 3) * 4));
}

DEV_INLINE float sigmoid_f(float x) { return 1.f / (1.f + __expf(-x)); }

// log decay and write strength of a token and head, either given or formed
// from the projections (g = -exp(A_log) softplus(a + dt), beta = sigmoid(b))
struct Gates {
  const float *g, *beta;            // [T, Hv]
  const __hip_bfloat16 *ba;         // rows of b | a
  long ba_stride;
  const float *A_log, *dt;          // [Hv]
  const __hip_bfloat16 *dt16;       // or dt in 16 bits, where dt is null
  DEV_INLINE void at(long t, int h, int Hv, float &gv, float &bv) const {
    if (g) {
      gv = g[t * Hv + h];
      bv = beta[t * Hv + h];
      return;
    }
    const float a = __bfloat162float(ba[t * ba_stride + Hv + h]) +
                    (dt ? dt[h] : __bfloat162float(dt16[h]));
    const float sp = a > 20.f ? a : log1pf(expf(a));
    gv = -expf(A_log[h]) * sp;
    bv = 1.f / (1.f + expf(-__bfloat162float(ba[t * ba_stride + h])));
  }
};

__global__ __launch_bounds__(512, 8) void gdn_local_kernel(
    short *__restrict__ wk,    // X_k, bf16 [blocks, Hv, 3, XK]
    float *__restrict__ u0,    // X_v [blocks, Hv, XV]
    short *__restrict__ att,   // bf16 [blocks, Hv, 3, AT]
    float *__restrict__ scal,  // [3, T, Hv]: b, 1/|k|, scale/|q|
    int *__restrict__ order,   // [B] sequences, the longest first
    const __hip_bfloat16 *__restrict__ q, const __hip_bfloat16 *__restrict__ k,
    const __hip_bfloat16 *__restrict__ v, long qk_stride, long v_stride,
    Gates gates, const int *__restrict__ qsl, long T, int Hk, int Hv,
    float scale) {
  const int seq = blockIdx.y, h = blockIdx.z;
  if (blockIdx.x == 0 && h == 0) {
    const int B = gridDim.y, own = qsl[seq + 1] - qsl[seq];
    int rank = 0;
    for (int j0 = 0; j0 < B; j0 += 512) {
      const int j = min(j0 + (int)threadIdx.x, B - 1);
      const int other = qsl[j + 1] - qsl[j];
      rank += __syncthreads_count(j0 + (int)threadIdx.x < B &&
                                  (other > own || (other == own && j < seq)));
    }
    if (threadIdx.x == 0) order[rank] = seq;
  }
  const int start = qsl[seq] + blockIdx.x * C;
  const int len = min(C, qsl[seq + 1] - start);
  if (len <= 0) return;
  const int hk = h / (Hv / Hk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lhi = lane >> 4;
  // block R of the chunk: + R * Hv times a block's size
  const long block =
      (first_block(qsl[seq], seq) + blockIdx.x * (C / 16)) * Hv + h;
  // (36 KB: four workgroups a CU. T takes the keys' place, whose columns X
  // wants are in registers by then, and the values A's)
  static_assert(C * SB * sizeof(short) == C * AS * sizeof(float));
  __shared__ __attribute__((aligned(16))) float Am[C * AS], Tm[C * AS];
  short *Kt = reinterpret_cast<short *>(Tm);
  short *Vt = reinterpret_cast<short *>(Am);
  __shared__ __attribute__((aligned(16))) float bb[C], btv[C], rkv[C],
      rqv[C], ck[C];

  // ---- keys to LDS (rows past the end: the last one, factors 0), norms of
  // keys and queries: 16 lanes per row
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int u = j * 512 + tid, t = u >> 4, c = (u & 15) * 8;
    const long row = start + min(t, len - 1);
    const shortx8 kr = *reinterpret_cast<const shortx8 *>(
        k + row * qk_stride + hk * D + c);
    const shortx8 qr = *reinterpret_cast<const shortx8 *>(
        q + row * qk_stride + hk * D + c);
    *reinterpret_cast<shortx8 *>(Kt + t * SB + c) = kr;
    float kf[8], qf[8], nk = 0.f, nq = 0.f;
    unpack8<__hip_bfloat16>(kr, kf);
    unpack8<__hip_bfloat16>(qr, qf);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      nk += kf[e] * kf[e];
      nq += qf[e] * qf[e];
    }
    const float live = t < len ? 1.f : 0.f;
    const float rk = live * rsqrtf(lanes_sum<16>(nk) + 1e-6f);
    const float rq = live * rsqrtf(lanes_sum<16>(nq) + 1e-6f) * scale;
    if (c == 0) {
      rkv[t] = rk;
      rqv[t] = rq;
      if (t < len) {
        scal[(T + row) * Hv + h] = rk;
        scal[(2 * T + row) * Hv + h] = rq;
      }
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
  if (tid < C) ck[tid] = btv[tid] * __expf(bb[tid]) * rkv[tid];

  // ---- blocks on and below the diagonal of A and att, a wave each
  for (int blk = wave; blk < 12; blk += 8) {
    // 0..9: (R, I) row by row; 10, 11: (0, 1) and (2, 3), zero
    int R = blk < 1 ? 0 : blk < 3 ? 1 : blk < 6 ? 2 : 3;
    int I = blk - R * (R + 1) / 2;
    if (blk >= 10) {
      R = (blk - 10) * 2;
      I = R + 1;
    }
    gdn_f4 a = {0, 0, 0, 0}, s = {0, 0, 0, 0};
    if (blk < 10) {
      const long qrow = start + min(R * 16 + l16, len - 1);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        GdnFrag ki, kt, qt;
        const int c = ks * 32 + lhi * 8;
        ki.s = *reinterpret_cast<const shortx8 *>(Kt + (I * 16 + l16) * SB + c);
        kt.s = *reinterpret_cast<const shortx8 *>(Kt + (R * 16 + l16) * SB + c);
        qt.s = *reinterpret_cast<const shortx8 *>(q + qrow * qk_stride +
                                                  hk * D + c);
        a = mma32(kt, ki, a);  // lane: i = l16, t = 4 lhi + r
        s = mma32(ki, qt, s);  // lane: t = l16, i = 4 lhi + r
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = R * 16 + lhi * 4 + r, i = I * 16 + l16;
      const float d = i < t ? __expf(bb[t] - bb[i]) : 0.f;
      Am[t * AS + i] = i < t ? btv[t] * d * rkv[t] * rkv[i] * a[r] : 0.f;
    }
    const int t = R * 16 + l16, i0 = I * 16 + lhi * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      s[r] = i0 + r <= t ? __expf(bb[t] - bb[i0 + r]) * rqv[t] *
                               rkv[i0 + r] * s[r]
                         : 0.f;
    if (R * 16 < len) {  // (rows past the end are zero)
      shortx4 p[3];
      split3(s, p);
#pragma unroll
      for (int j = 0; j < 3; ++j)
        *reinterpret_cast<shortx4 *>(
            att + ((block + R * Hv) * 3 + j) * AT + (I >> 1) * 512 +
            (((I & 1) * 2 + (lhi >> 1)) * 16 + l16) * 8 + (lhi & 1) * 4) =
            p[j];
    }
  }
  const int c0 = (wave & 3) * 32;
  GdnFrag cols[2][2];
  auto columns = [&](const short *src) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int n = 0; n < 2; ++n)
        read_tr(cols[kk][n], src, SB, kk * 32, c0 + n * 16, l16, lhi);
  };
  if (wave < 4) columns(Kt);
  __syncthreads();
  // ---- T: inverses of the diagonal blocks, a column per lane
  if (wave >= 4 && wave < 6) {  // (0, 1) and (2, 3) are zero
    const int R = (wave - 4) * 2;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      Tm[(R * 16 + lhi * 4 + r) * AS + (R + 1) * 16 + l16] = 0.f;
  }
  if (wave < 4) {
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
      for (int i = 0; i < 16; ++i)
        Tm[(wave * 16 + i) * AS + wave * 16 + l16] = y[i];
    }
  }
  __syncthreads();
  // then the blocks below it: T_RI = -T_RR sum_J A_RJ T_JI
  for (int d = 1; d < 4; ++d) {
    const int I = wave, R = I + d;
    gdn_f4 y = {0, 0, 0, 0};
    if (R < 4) {
      for (int c = I * 16; c < R * 16; c += 4)
        y = mma4(Am[(R * 16 + l16) * AS + c + lhi],
                 Tm[(c + lhi) * AS + I * 16 + l16], y);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Tm[(R * 16 + lhi * 4 + r) * AS + I * 16 + l16] = y[r];
    }
    __syncthreads();
    if (R < 4) {
      y = gdn_f4{0, 0, 0, 0};
#pragma unroll
      for (int c = 0; c < 16; c += 4)
        y = mma4(-Tm[(R * 16 + l16) * AS + R * 16 + c + lhi],
                 Tm[(R * 16 + c + lhi) * AS + I * 16 + l16], y);
    }
    __syncthreads();
    if (R < 4) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Tm[(R * 16 + lhi * 4 + r) * AS + I * 16 + l16] = y[r];
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int u = j * 512 + tid;
    const long row = start + min(u >> 4, len - 1);
    *reinterpret_cast<shortx8 *>(Vt + (u >> 4) * SB + (u & 15) * 8) =
        *reinterpret_cast<const shortx8 *>(v + row * v_stride + h * D +
                                           (u & 15) * 8);
  }
  __syncthreads();
  // ---- X: waves 0..3 the keys' columns (transposed: a lane has four of a
  // row), 4..7 the values' (four rows of a column)
  const float *fac = wave < 4 ? ck : btv;
  if (wave >= 4) columns(Vt);
#pragma unroll
  for (int R = 0; R < 4; ++R) {
    gdn_f4 x[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int kk = 0; kk <= R / 2; ++kk) {
      GdnFrag tf[3];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int i = kk * 32 + half * 16 + lhi * 4;
        gdn_f4 tv = *reinterpret_cast<const gdn_f4 *>(
            Tm + (R * 16 + l16) * AS + i);
        tv *= *reinterpret_cast<const gdn_f4 *>(fac + i);
        shortx4 p[3];
        split3(tv, p);
#pragma unroll
        for (int j = 0; j < 3; ++j) tf[j].h[half] = p[j];
      }
#pragma unroll
      for (int j = 2; j >= 0; --j)
#pragma unroll
        for (int n = 0; n < 2; ++n)
          x[n] = wave < 4 ? mma32(cols[kk][n], tf[j], x[n])
                          : mma32(tf[j], cols[kk][n], x[n]);
    }
    if (R * 16 >= len) break;  // (rows past the end are zero)
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      if (wave < 4) {
        shortx4 p[3];
        split3(x[n], p);
#pragma unroll
        for (int j = 0; j < 3; ++j)
          *reinterpret_cast<shortx4 *>(
              wk + ((block + R * Hv) * 3 + j) * XK + wave * 512 +
              ((n * 2 + (lhi >> 1)) * 16 + l16) * 8 + (lhi & 1) * 4) = p[j];
      } else {
        *reinterpret_cast<gdn_f4 *>(
            u0 + (block + R * Hv) * XV + ((wave & 3) * 2 + n) * 256 +
            lane * 4) = x[n];
      }
    }
  }
}

// bytes from p on
template <typename T_>
DEV_INLINE __amdgpu_buffer_rsrc_t rows_of(const T_ *p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, bytes, 0x00020000);
}

__global__ __launch_bounds__(256, 2) void gdn_carry_kernel(
    __hip_bfloat16 *__restrict__ o,  // [T, Hv, D]
    float *__restrict__ states,      // [slots, Hv, D, D], in place
    const short *__restrict__ wk, const float *__restrict__ u0,
    const short *__restrict__ att, const float *__restrict__ scal,
    const __hip_bfloat16 *__restrict__ q, const __hip_bfloat16 *__restrict__ k,
    long qk_stride, const long *__restrict__ slots,
    const int *__restrict__ has_init, const int *__restrict__ qsl,
    const int *__restrict__ order, long T, int B, int Hk, int Hv,
    bool snake) {
  // workgroups go to the 8 XCDs in turn
  const int turn = blockIdx.x >> 3, z = turn % (D / DVS);
  const int pair = turn / (D / DVS) * 8 + (blockIdx.x & 7);
  if (pair >= B * Hv) return;
  int at_seq = pair / Hv;
  if (snake && at_seq >= (B + 1) / 2) at_seq = B - 1 - (at_seq - (B + 1) / 2);
  const int h = pair % Hv, seq = order[at_seq];
  const int begin = qsl[seq], end = qsl[seq + 1];
  if (begin >= end) return;
  const int hk = h / (Hv / Hk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lhi = lane >> 4;
  __shared__ __attribute__((aligned(16))) short Kt[2][C * KB];
  __shared__ __attribute__((aligned(16))) short Sp[3][DVS * SB];
  // U and, for the state, exp(b_last - b) U / |k|; rows are value columns
  __shared__ __attribute__((aligned(16))) short Up[6][DVS * UB];
  __shared__ float sc[2][3][C];  // b, 1/|k|, scale/|q|

  // S transposed: lane value column l16, keys (wave * 2 + dt) * 16 + lhi * 4
  // + r
  float *sg = states + ((slots[seq] * Hv + h) * D + z * DVS) * D;
  gdn_f4 s[2];
  const bool init = has_init[seq] != 0;
  auto put_state = [&]() {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
      shortx4 p[3];
      split3(s[dt], p);
#pragma unroll
      for (int j = 0; j < 3; ++j)
        *reinterpret_cast<shortx4 *>(Sp[j] + l16 * SB +
                                     (wave * 2 + dt) * 16 + lhi * 4) = p[j];
    }
  };
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
    s[dt] = init ? *reinterpret_cast<const gdn_f4 *>(
                       sg + l16 * D + (wave * 2 + dt) * 16 + lhi * 4)
                 : gdn_f4{0, 0, 0, 0};
  put_state();

  // operands of a chunk; the next one's are on their way as soon as their
  // registers are free: keys, then X and queries, then att
  GdnFrag w[4][3], at[2][3] = {}, qf[4];
  shortx8 kr[4];
  gdn_f4 u;
  float sr;
  // Rows of a chunk by descriptors that end with it (what lies past is zero):
  // addresses are a lane's fixed offsets, where 64 bits and a branch for each
  // load were a third of the loop's instructions.
  const int row_b = Hv * D * 2, key_b = (int)qk_stride * 2;
  const int q_at = (wave * 16 + l16) * key_b + lhi * 16;
  const int k_at = (tid >> 4) * key_b + (tid & 15) * 16;
  auto load16 = [](__amdgpu_buffer_rsrc_t r, int at) {
    return __builtin_bit_cast(
        shortx8, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
  };
  // the wave's block of rows in the chunk at `start`
  const long block0 = (first_block(begin, seq) + wave) * Hv + h;
  auto block_of = [&](int start) {
    return block0 + (long)((start - begin) / 16) * Hv;
  };
  auto fetch_keys = [&](int start) {
    const int len = min(C, end - start);
    const __amdgpu_buffer_rsrc_t rk =
        rows_of(k + start * qk_stride + hk * D, (len - 1) * key_b + D * 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) kr[j] = load16(rk, k_at + j * 16 * key_b);
    sr = scal[(min(wave, 2) * T + start + min(lane, len - 1)) * Hv + h];
  };
  auto fetch_rows = [&](int start) {
    const int len = min(C, end - start);
    if (wave * 16 >= len) {
      // no row of this wave (loads that all fall outside: 7 % of 64 prompts
      // of 16 rows)
      const shortx8 none = {};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
        for (int j = 0; j < 3; ++j) w[ks][j].s = none;
        qf[ks].s = none;
      }
      u = gdn_f4{0, 0, 0, 0};
      return;
    }
    const long block = block_of(start);
    const __amdgpu_buffer_rsrc_t rw = rows_of(wk + block * 3 * XK, 6 * XK);
    const __amdgpu_buffer_rsrc_t ru =
        rows_of(u0 + block * XV + z * 256, 1024);
    const __amdgpu_buffer_rsrc_t rq =
        rows_of(q + start * qk_stride + hk * D, (len - 1) * key_b + D * 2);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        w[ks][j].s = load16(rw, (j * XK + ks * 512) * 2 + lane * 16);
      qf[ks].s = load16(rq, q_at + ks * 64);
    }
    u = __builtin_bit_cast(gdn_f4, load16(ru, lane * 16));
  };
  auto fetch_att = [&](int start) {
    if (wave * 16 >= end - start) {
      const shortx8 none = {};
#pragma unroll
      for (int j = 0; j < 3; ++j) at[0][j].s = at[1][j].s = none;
      return;
    }
    const __amdgpu_buffer_rsrc_t ra =
        rows_of(att + block_of(start) * 3 * AT, 6 * AT);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      at[0][j].s = load16(ra, j * AT * 2 + lane * 16);
      // (blocks past the diagonal's pair are never written, nor read)
      if (wave >= 2) at[1][j].s = load16(ra, (j * AT + 512) * 2 + lane * 16);
    }
  };
  auto put_keys = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = j * 256 + tid;
      *reinterpret_cast<shortx8 *>(Kt[buf] + (u >> 4) * KB + (u & 15) * 8) =
          kr[j];
    }
    if (wave < 3) sc[buf][wave][lane] = sr;
  };
  fetch_keys(begin);
  fetch_rows(begin);
  fetch_att(begin);
  put_keys(0);
  __syncthreads();
  int cur = 0;
  for (int start = begin; start < end; start += C) {
    const int len = min(C, end - start);
    const bool more = start + C < end;
    if (more) fetch_keys(start + C);

    // ---- U = X_v - X_k S^T and q S^T, rows 16 w ..
    // (two waves per SIMD hide little of the latency of an LDS read, so
    // fragments are read a step ahead)
    gdn_f4 xs = {0, 0, 0, 0}, qs = {0, 0, 0, 0};
    GdnFrag sf[2][3];
    auto read_state = [&](int ks) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        sf[ks & 1][j].s = *reinterpret_cast<const shortx8 *>(
            Sp[j] + l16 * SB + ks * 32 + lhi * 8);
    };
    read_state(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) read_state(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        xs = mma32(w[ks][TERM_A[i]], sf[ks & 1][TERM_B[i]], xs);
        if (i % 2 == 0) qs = mma32(qf[ks], sf[ks & 1][2 - i / 2], qs);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const float last = sc[cur][0][len - 1];
    gdn_f4 wc, eb;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = wave * 16 + lhi * 4 + r;
      wc[r] = __expf(last - sc[cur][0][t]) * sc[cur][1][t];
      eb[r] = __expf(sc[cur][0][t]) * sc[cur][2][t];
    }
    u -= xs;
    qs *= eb;
    {
      shortx4 p[3], pw[3];
      split3(u, p);
      split3(u * wc, pw);
      const int at_u = l16 * UB + wave * 16 + lhi * 4;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        *reinterpret_cast<shortx4 *>(Up[j] + at_u) = p[j];
        *reinterpret_cast<shortx4 *>(Up[3 + j] + at_u) = pw[j];
      }
    }
    if (more) fetch_rows(start + C);
    __syncthreads();
    // ---- o = B q S^T + att U
    GdnFrag uf[2][3], kf[2][2], wf[2][3];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        uf[kk][j].s = *reinterpret_cast<const shortx8 *>(
            Up[j] + l16 * UB + kk * 32 + lhi * 8);
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
        read_tr(kf[kk][dt], Kt[cur], KB, kk * 32, (wave * 2 + dt) * 16, l16,
                lhi);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int half = 0; half < 2; ++half)
          wf[kk][j].h[half] = *reinterpret_cast<const shortx4 *>(
              Up[3 + j] + l16 * UB + kk * 32 + half * 16 + lhi * 4);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk > wave / 2) continue;
#pragma unroll
      for (int i = 0; i < 6; ++i)
        qs = mma32(at[kk][TERM_A[i]], uf[kk][TERM_B[i]], qs);
    }
    if (more) fetch_att(start + C);
    // (rows past the end fall outside: with a branch around each store the
    // wait for the next chunk's operands would be one for these stores too)
    const __amdgpu_buffer_rsrc_t ro =
        rows_of(o + ((long)start * Hv + h) * D + z * DVS,
                (len - 1) * row_b + DVS * 2);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __builtin_amdgcn_raw_buffer_store_b16(
          __builtin_bit_cast(short, __float2bfloat16(qs[r])), ro,
          (wave * 16 + lhi * 4 + r) * row_b + l16 * 2, 0, 0);
    // ---- S = B_last S + (exp(b_last - b) U)^T k
    const float keep = __expf(last);
    s[0] *= keep;
    s[1] *= keep;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 2; j >= 0; --j) {
        s[0] = mma32(kf[kk][0], wf[kk][j], s[0]);
        s[1] = mma32(kf[kk][1], wf[kk][j], s[1]);
      }
    put_state();
    if (more) put_keys(cur ^ 1);
    cur ^= 1;
    __syncthreads();  // S is there, this chunk's U and keys have been read
  }
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
    *reinterpret_cast<gdn_f4 *>(sg + l16 * D + (wave * 2 + dt) * 16 +
                                lhi * 4) = s[dt];
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

// What local leaves for carry: 26 KB for each value head and block of 16 rows,
// T / 16 + B blocks (a sequence of one row fills one too), and 12 bytes a row.
// 1024 decode rows beside 8192 of prompts, 16 heads: 0.7 GB.
struct Left {
  torch::Tensor wk, u0, att, scal, order;
  Left(long T, long B, long Hv, const torch::TensorOptions &opts) {
    const auto bf = opts.dtype(at::kBFloat16);
    const long blocks = T / 16 + B;
    wk = torch::empty({blocks, Hv, 3, (long)XK}, bf);
    u0 = torch::empty({blocks, Hv, (long)XV}, opts.dtype(at::kFloat));
    att = torch::empty({blocks, Hv, 3, (long)AT}, bf);
    scal = torch::empty({3, T, Hv}, opts.dtype(at::kFloat));
    order = torch::empty({B}, opts.dtype(at::kInt));
  }
};

void run_chunks(torch::Tensor &o, const void *q, const void *k,
                const void *v, long qk_stride, long v_stride,
                const Gates &gates, torch::Tensor &states, const long *slots,
                const int *has_init, const int *qsl, long T, int B,
                int max_len, int Hk, int Hv, double scale) {
  const Left left(T, B, Hv, states.options());
  const auto &[wk, u0, att, scal, order] = left;
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(gdn_local_kernel, dim3((max_len + C - 1) / C, B, Hv),
                     dim3(512), 0, stream, (short *)wk.data_ptr(),
                     u0.data_ptr<float>(), (short *)att.data_ptr(),
                     scal.data_ptr<float>(), order.data_ptr<int>(),
                     (const __hip_bfloat16 *)q, (const __hip_bfloat16 *)k,
                     (const __hip_bfloat16 *)v,
                     qk_stride, v_stride, gates, qsl, T, Hk, Hv,
                     (float)scale);
  HIP_CHECK_KERNEL();
  const long pairs = (long)B * Hv;
  hipLaunchKernelGGL(
      gdn_carry_kernel, dim3((pairs + 7) / 8 * 8 * (D / DVS)), dim3(256), 0,
      stream, (__hip_bfloat16 *)o.data_ptr(), states.data_ptr<float>(),
      (const short *)wk.data_ptr(), u0.data_ptr<float>(),
      (const short *)att.data_ptr(), scal.data_ptr<float>(),
      (const __hip_bfloat16 *)q, (const __hip_bfloat16 *)k, qk_stride, slots,
      has_init, qsl, order.data_ptr<int>(), T, B, Hk, Hv,
      pairs * (D / DVS) <= 512);
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
                       0, nullptr, nullptr, nullptr};
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
              (dt_bias.scalar_type() == at::kFloat ||
               dt_bias.scalar_type() == at::kBFloat16) &&
              dt_bias.numel() == Hv && A_log.is_contiguous() &&
              dt_bias.is_contiguous());
  TORCH_CHECK(states.dim() == 4 && states.is_contiguous() &&
              states.scalar_type() == at::kFloat && states.size(2) == D &&
              states.size(3) == D, "gdn: state [slots, Hv, 128, 128] fp32");
  TORCH_CHECK(slots.scalar_type() == at::kLong && slots.is_contiguous());
  const bool wide = dt_bias.scalar_type() == at::kFloat;
  return {nullptr, nullptr, (const __hip_bfloat16 *)ba.data_ptr(),
          (long)ba.stride(0), A_log.data_ptr<float>(),
          wide ? dt_bias.data_ptr<float>() : nullptr,
          wide ? nullptr : (const __hip_bfloat16 *)dt_bias.data_ptr()};
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

// takes and gives back what gdn_varlen of T rows in B sequences works on
void gdn_reserve(torch::Tensor like, long T, long B, long Hv) {
  TORCH_CHECK(like.is_cuda() && T >= 0 && B >= 0 && Hv > 0);
  const Left left(T, B, Hv, like.options());
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
