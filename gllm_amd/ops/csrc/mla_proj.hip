// What stands around the absorbed latent attention (bf16, latent 512 +
// rotated part 64, 128 unrotated query dims and 128 value dims a head):
//
//   mla_prepare   one workgroup per token: the latent row is RMS-normed, its
//                 rotated part turned, both written to their slot of the
//                 paged cache; the queries' rotated parts turned
//   mla_queries   the same into the attention's query rows, and beside it (in
//                 front of it where rows are many)
//                 q_lat[t, h, :] = q_nope[t, h, :] W_uk[h]
//   mla_project   out[t, h, :] = o_lat[t, h, :] W_uv[h]^T
//
// Bound by launches and by fp32 copies where it was torch: three slices
// copied, a norm, a rotation, two concatenations, the scatter, and two
// batched products that converted their weights to fp32 in every layer (22
// launches). The products take bf16 operands with fp32 sums: the same
// products, exact in fp32.
// A layer of 128 decoding requests, 16 heads: 7 + 8 us where these launches
// took 105 (rows and absorbed products, which need nothing of each other, by a
// launch each: 5 + 5); of 4096 prompt tokens: 53 + 89 us for 390. (The products
// from the parts of the split projection, without its sum: 2 us less at 128
// rows, level at 64, 2 to 4 us more with few heads.)

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mp_bf8;
typedef __attribute__((ext_vector_type(4))) float mp_f4;

namespace {

typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int LORA = 512, ROPE = 64, DK = LORA + ROPE;
constexpr int NOPE = 128, DV = 128;
constexpr int QD = NOPE + ROPE;          // a head's columns of q
constexpr int WROWS = NOPE + DV;         // a head's rows of the weight
constexpr int TOK = 64;                  // tokens of a workgroup
constexpr int CHUNK = 128;               // latent columns of a workgroup
constexpr int VCH = 32;                  // value columns of a workgroup

union MpFrag {
  mp_bf8 v;
  shortx4 h[2];
};

DEV_INLINE short bf16_bits(float v) {
  return __builtin_bit_cast(short, __float2bfloat16(v));
}

// rotate-half of 8 neighbouring pairs: x1 = dims d .. d + 7, x2 = + 32
DEV_INLINE void rotate8(const __hip_bfloat16 *src, __hip_bfloat16 *dst,
                        const float *cs, int d) {
  float a[8], b[8], x[8], y[8];
  ld8<__hip_bfloat16>(src + d, a);
  ld8<__hip_bfloat16>(src + 32 + d, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float c = cs[d + i], s = cs[32 + d + i];
    x[i] = a[i] * c - b[i] * s;
    y[i] = b[i] * c + a[i] * s;
  }
  st8<__hip_bfloat16>(dst + d, x);
  st8<__hip_bfloat16>(dst + 32 + d, y);
}

// 4 waves: wave 0 the latent row, waves 1 to 3 the queries. PROMPT: the latent
// goes to lat and pe too, and the queries are turned where they are.
template <typename TW, bool PROMPT>
DEV_INLINE void prepare_row(
    const long t, __hip_bfloat16 *__restrict__ qf,  // [T, H, DK] (dims LORA..)
    __hip_bfloat16 *__restrict__ lat,       // [T, LORA]
    __hip_bfloat16 *__restrict__ pe,        // [T, ROPE]
    __hip_bfloat16 *__restrict__ k_cache,   // [slots, DK]
    __hip_bfloat16 *q, long q_stride,
    const __hip_bfloat16 *__restrict__ kv, long kv_stride,
    const TW *__restrict__ norm_w, float eps,
    const long *__restrict__ positions, const float *__restrict__ cos_sin,
    const long *__restrict__ slots, int H) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float *cs = cos_sin + positions[t] * ROPE;
  if (wave == 0) {
    const __hip_bfloat16 *row = kv + t * kv_stride;
    __hip_bfloat16 *dst = k_cache + slots[t] * DK;
    float x[8], w[8], ss = 0.f;
    ld8<__hip_bfloat16>(row + lane * 8, x);
    ld8<TW>(norm_w + lane * 8, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
    const float inv = rsqrtf(wave_reduce_sum(ss) / LORA + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = x[i] * inv * w[i];
    st8<__hip_bfloat16>(dst + lane * 8, x);
    if (PROMPT) st8<__hip_bfloat16>(lat + t * LORA + lane * 8, x);
    if (lane < 4) rotate8(row + LORA, dst + LORA, cs, lane * 8);
    if (PROMPT && lane < 4) rotate8(row + LORA, pe + t * ROPE, cs, lane * 8);
    return;
  }
  for (int i = threadIdx.x - 64; i < H * 4; i += 192) {
    const int h = i >> 2;
    __hip_bfloat16 *src = q + t * q_stride + h * QD + NOPE;
    rotate8(src, PROMPT ? src : qf + (t * H + h) * (long)DK + LORA, cs,
            (i & 3) * 8);
  }
}

template <typename TW, bool PROMPT>
__global__ __launch_bounds__(256) void mla_prepare_kernel(
    __hip_bfloat16 *__restrict__ qf, __hip_bfloat16 *__restrict__ lat,
    __hip_bfloat16 *__restrict__ pe, __hip_bfloat16 *__restrict__ k_cache,
    __hip_bfloat16 *q, long q_stride,
    const __hip_bfloat16 *__restrict__ kv, long kv_stride,
    const TW *__restrict__ norm_w, float eps,
    const long *__restrict__ positions, const float *__restrict__ cos_sin,
    const long *__restrict__ slots, int H) {
  prepare_row<TW, PROMPT>(blockIdx.x, qf, lat, pe, k_cache, q, q_stride, kv,
                          kv_stride, norm_w, eps, positions, cos_sin, slots,
                          H);
}

// A workgroup per 64 tokens (16 per wave), head and 128 latent columns, and
// behind those (of a longer grid) one per token for its row. The weight block
// [128 k][128 columns] sits in LDS as two column blocks of [128][128 B] (16 B
// units permuted by k & 7) and is read transposed; the products are W^T q^T, so
// a lane holds four neighbouring columns of a token.
template <typename TW>
__global__ __launch_bounds__(256) void mla_queries_kernel(
    __hip_bfloat16 *__restrict__ qf,       // [T, H, DK]
    __hip_bfloat16 *__restrict__ k_cache, __hip_bfloat16 *q, long q_stride,
    const __hip_bfloat16 *__restrict__ kv, long kv_stride,
    const TW *__restrict__ norm_w, float eps,
    const long *__restrict__ positions, const float *__restrict__ cos_sin,
    const long *__restrict__ slots,
    const __hip_bfloat16 *__restrict__ w,  // [H, WROWS, LORA]
    int T, int H) {
  __shared__ __attribute__((aligned(16))) char wt[NOPE * CHUNK * 2];
  const int tiles = (T + TOK - 1) / TOK, block = blockIdx.x;
  if (block >= tiles * H * (LORA / CHUNK)) {
    prepare_row<TW, false>(block - tiles * H * (LORA / CHUNK), qf, nullptr,
                           nullptr, k_cache, q, q_stride, kv, kv_stride,
                           norm_w, eps, positions, cos_sin, slots, H);
    return;
  }
  const int t0 = block % tiles * TOK, h = block / tiles % H;
  const int n0 = block / tiles / H * CHUNK;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  const __hip_bfloat16 *wh = w + (long)h * WROWS * LORA + n0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // 32 KB in units of [8 k][128 B]
    const int u = wave * 8 + j, cb = u >> 4, k = (u & 15) * 8 + (lane >> 3);
    const int col = cb * 64 + ((lane & 7) ^ (lane >> 3)) * 8;
    __builtin_amdgcn_global_load_lds(
        reinterpret_cast<const unsigned int *>(wh + (long)k * LORA + col),
        reinterpret_cast<unsigned int *>(wt + u * 1024), 16, 0, 0);
  }
  const int tok = t0 + wave * 16 + l16;
  const __hip_bfloat16 *qp =
      q + min(tok, T - 1) * q_stride + h * QD + lhi * 4;
  MpFrag qfr[NOPE / 32];
#pragma unroll
  for (int kk = 0; kk < NOPE / 32; ++kk)
#pragma unroll
    for (int half = 0; half < 2; ++half)
      qfr[kk].h[half] = *reinterpret_cast<const shortx4 *>(
          qp + kk * 32 + half * 16);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;
  __hip_bfloat16 *op = qf + ((long)tok * H + h) * DK + n0 + lhi * 4;
#pragma unroll
  for (int nt = 0; nt < CHUNK / 16; ++nt) {
    mp_f4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < NOPE / 32; ++kk) {
      MpFrag wf;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int row = kk * 32 + half * 16 + tr_row;
        wf.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_shortx4 *)(wt + (nt >> 2) * (NOPE * 128) + row * 128 +
                            (((nt & 3) * 32 + tr_col) ^ ((row & 7) << 4))));
      }
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, qfr[kk].v, acc, 0,
                                                    0, 0);
    }
    if (tok < T) {
      shortx4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = bf16_bits(acc[r]);
      *reinterpret_cast<shortx4 *>(op + nt * 16) = o;
    }
  }
}

// Workgroup = 64 tokens (16 per wave), one head, 32 value columns; both
// operands lie as the products want them and come from memory (the weight
// rows of a head are read by the four waves through L1).
__global__ __launch_bounds__(256) void mla_project_kernel(
    __hip_bfloat16 *__restrict__ out,          // [T, H * DV]
    const __hip_bfloat16 *__restrict__ o_lat,  // [T, H, LORA]
    const __hip_bfloat16 *__restrict__ w,      // [H, WROWS, LORA]
    int T, int H) {
  const int t0 = blockIdx.x * TOK, h = blockIdx.y, n0 = blockIdx.z * VCH;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  const int tok = t0 + wave * 16 + l16;
  const __hip_bfloat16 *ap =
      o_lat + ((long)min(tok, T - 1) * H + h) * LORA + lhi * 8;
  const __hip_bfloat16 *wp =
      w + ((long)h * WROWS + NOPE + n0 + l16) * LORA + lhi * 8;
  mp_f4 acc[VCH / 16];
#pragma unroll
  for (int n = 0; n < VCH / 16; ++n) acc[n] = mp_f4{0, 0, 0, 0};
#pragma unroll 8
  for (int kk = 0; kk < LORA / 32; ++kk) {
    const mp_bf8 a = *reinterpret_cast<const mp_bf8 *>(ap + kk * 32);
#pragma unroll
    for (int n = 0; n < VCH / 16; ++n) {
      const mp_bf8 b =
          *reinterpret_cast<const mp_bf8 *>(wp + n * 16 * LORA + kk * 32);
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc[n], 0, 0, 0);
    }
  }
  if (tok >= T) return;
  __hip_bfloat16 *op = out + ((long)tok * H + h) * DV + n0 + lhi * 4;
#pragma unroll
  for (int n = 0; n < VCH / 16; ++n) {
    shortx4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = bf16_bits(acc[n][r]);
    *reinterpret_cast<shortx4 *>(op + n * 16) = o;
  }
}

void check16(const torch::Tensor &t, const char *what) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16 &&
              reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, what);
}

// What mla_queries and mla_prompt_rows take: q [T, H * 192], kv [T, 576] (row
// views allowed), norm_w [512] fp32 or bf16
void check_rows(const torch::Tensor &q, const torch::Tensor &kv,
                const torch::Tensor &norm_w, const torch::Tensor &positions,
                const torch::Tensor &cos_sin, const torch::Tensor &k_cache,
                const torch::Tensor &slots) {
  const long T = q.size(0);
  check16(q, "q: bf16, 16 B aligned");
  check16(kv, "kv: bf16, 16 B aligned");
  check16(k_cache, "k_cache: bf16, 16 B aligned");
  const int H = q.size(1) / QD;
  TORCH_CHECK(q.dim() == 2 && q.size(1) == (long)H * QD && H > 0 &&
              q.stride(1) == 1 && q.stride(0) % 8 == 0);
  TORCH_CHECK(kv.dim() == 2 && kv.size(0) == T && kv.size(1) == DK &&
              kv.stride(1) == 1 && kv.stride(0) % 8 == 0);
  TORCH_CHECK(k_cache.is_contiguous() && k_cache.size(-1) == DK);
  TORCH_CHECK(positions.scalar_type() == at::kLong &&
              positions.is_contiguous() && positions.numel() == T);
  TORCH_CHECK(slots.scalar_type() == at::kLong && slots.is_contiguous() &&
              slots.numel() == T);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat &&
              cos_sin.is_contiguous() && cos_sin.size(-1) == ROPE);
  TORCH_CHECK(norm_w.is_contiguous() && norm_w.numel() == LORA &&
              reinterpret_cast<uintptr_t>(norm_w.data_ptr()) % 16 == 0 &&
              (norm_w.scalar_type() == at::kFloat ||
               norm_w.scalar_type() == at::kBFloat16),
              "norm_w: fp32 or bf16");
}

}  // namespace

// w_kvb [H * 256, 512]; writes the cache rows of `slots`, returns the query
// rows [T, H, 576].
torch::Tensor mla_queries(torch::Tensor q, torch::Tensor kv,
                          torch::Tensor norm_w, double eps,
                          torch::Tensor positions, torch::Tensor cos_sin,
                          torch::Tensor w_kvb, torch::Tensor k_cache,
                          torch::Tensor slots) {
  check_rows(q, kv, norm_w, positions, cos_sin, k_cache, slots);
  const long T = q.size(0);
  const int H = q.size(1) / QD;
  check16(w_kvb, "w_kvb: bf16, 16 B aligned");
  TORCH_CHECK(w_kvb.is_contiguous() && w_kvb.size(0) == (long)H * WROWS &&
              w_kvb.size(1) == LORA);
  auto qf = torch::empty({T, (long)H, (long)DK}, q.options());
  if (T == 0) return qf;
  // The rows by a launch of their own where they are many: beside the products
  // a row's workgroup holds LDS for the products too, and there is no longer a
  // launch's time to save by it (us, apart / beside: 2 heads, 3000 rows 10.2 /
  // 9.4, 4096 11.2 / 11.6, 16384 31.5 / 42.9; 16 heads, 4096 42.4 / 41.5, 8192
  // 77.8 / 79.2, 16384 179 / 194; 32 heads, 4096 77.4 / 74.5, 8192 184 / 184).
  const bool apart = T > (H < 8 ? 3072 : 4096);
  const long blocks =
      (T + TOK - 1) / TOK * H * (LORA / CHUNK) + (apart ? 0 : T);
  TORCH_CHECK(blocks < 1L << 31);
#define ROWS(TW)                                                             \
  (__hip_bfloat16 *)k_cache.data_ptr(), (__hip_bfloat16 *)q.data_ptr(),      \
      (long)q.stride(0), (const __hip_bfloat16 *)kv.data_ptr(),              \
      (long)kv.stride(0), (const TW *)norm_w.data_ptr(), (float)eps,         \
      positions.data_ptr<long>(), cos_sin.data_ptr<float>(),                 \
      slots.data_ptr<long>()
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(TW)                                                              \
  do {                                                                       \
    if (apart)                                                               \
      hipLaunchKernelGGL((mla_prepare_kernel<TW, false>), dim3(T),           \
                         dim3(256), 0, stream,                               \
                         (__hip_bfloat16 *)qf.data_ptr(), nullptr, nullptr,  \
                         ROWS(TW), H);                                       \
    hipLaunchKernelGGL((mla_queries_kernel<TW>), dim3(blocks), dim3(256), 0, \
                       stream, (__hip_bfloat16 *)qf.data_ptr(), ROWS(TW),    \
                       (const __hip_bfloat16 *)w_kvb.data_ptr(), (int)T, H); \
  } while (0)
  if (norm_w.scalar_type() == at::kFloat) RUN(float);
  else RUN(__hip_bfloat16);
#undef RUN
  HIP_CHECK_KERNEL();
  return qf;
}

// Rows of prompts: turns the rotated parts of q in place, writes the cache
// rows of `slots`, returns the normed latents [T, 512] and the shared rotated
// key parts [T, 64].
std::vector<torch::Tensor> mla_prompt_rows(
    torch::Tensor q, torch::Tensor kv, torch::Tensor norm_w, double eps,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor k_cache,
    torch::Tensor slots) {
  check_rows(q, kv, norm_w, positions, cos_sin, k_cache, slots);
  const long T = q.size(0);
  auto lat = torch::empty({T, (long)LORA}, q.options());
  auto pe = torch::empty({T, (long)ROPE}, q.options());
  if (T == 0) return {lat, pe};
#define RUN(TW)                                                              \
  hipLaunchKernelGGL((mla_prepare_kernel<TW, true>), dim3(T), dim3(256), 0,  \
                     at::cuda::getCurrentCUDAStream(),                       \
                     nullptr, (__hip_bfloat16 *)lat.data_ptr(),              \
                     (__hip_bfloat16 *)pe.data_ptr(), ROWS(TW),              \
                     (int)(q.size(1) / QD))
  if (norm_w.scalar_type() == at::kFloat) RUN(float);
  else RUN(__hip_bfloat16);
#undef RUN
#undef ROWS
  HIP_CHECK_KERNEL();
  return {lat, pe};
}

// o_lat [T, H, 512] -> [T, H * 128]
torch::Tensor mla_values(torch::Tensor o_lat, torch::Tensor w_kvb) {
  const long T = o_lat.size(0), H = o_lat.size(1);
  check16(o_lat, "o_lat: bf16, 16 B aligned");
  check16(w_kvb, "w_kvb: bf16, 16 B aligned");
  TORCH_CHECK(o_lat.dim() == 3 && o_lat.is_contiguous() &&
              o_lat.size(2) == LORA);
  TORCH_CHECK(w_kvb.is_contiguous() && w_kvb.size(0) == H * WROWS &&
              w_kvb.size(1) == LORA);
  auto out = torch::empty({T, H * DV}, o_lat.options());
  if (T == 0) return out;
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(mla_project_kernel,
                     dim3((T + TOK - 1) / TOK, H, DV / VCH), dim3(256), 0,
                     stream, (__hip_bfloat16 *)out.data_ptr(),
                     (const __hip_bfloat16 *)o_lat.data_ptr(),
                     (const __hip_bfloat16 *)w_kvb.data_ptr(), (int)T,
                     (int)H);
  HIP_CHECK_KERNEL();
  return out;
}
