// fp8 (OCP e4m3) execution path for gfx950: per-token-group activation
// quant, block-scale weight-streaming GEMM (decode), block-scale grouped
// MoE GEMM. Replaces the reference's DeepGEMM / flashinfer / Triton
// w8a8 chain (layers/quantization/fp8.py:33-158,556-676) with native
// CDNA4 fp8 MFMA (V_MFMA_F32_16X16X32_FP8_FP8).
//
// Layouts (exactly what layers/quantization/fp8.py loads):
//   weights    e4m3 [N, K], scale_inv fp32 [ceil(N/128), ceil(K/128)]
//   activation e4m3 [M, K], scales    fp32 [M, K/128] (per token-group)
// Scales are applied PER 128-K BLOCK in the accumulator: each BK=128
// tile accumulates into a fresh sub-accumulator through 4 fp8 MFMA
// k-steps, then folds into the fp32 accumulator scaled by
// a_scale[m, kb] * w_scale[nblk, kb]. The fp8 stream halves the weight
// bytes — decode GEMMs are weight-bandwidth-bound, so this is ~2x.

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f8_f4;

namespace {

constexpr int BLOCK = 256;
constexpr int BN = 64;
constexpr int BK = 128;         // one scale block per K tile
constexpr int ROW_B = BK;       // tile row bytes (128 fp8)
constexpr int GROUP = 128;

DEV_INLINE int swz(int row, int byte_off) {
  return byte_off ^ ((row & 7) << 4);
}

DEV_INLINE float fp8_to_f32(unsigned char v) {
  __hip_fp8_e4m3 h;
  h.__x = v;
  return (float)h;
}

// ------------------------------------------------- activation quant
// x [T, K] bf16 -> q [T, K] e4m3 + scales [T, K/128]. One wave per
// (token, group): 2 elems per lane.
__global__ void per_token_group_quant_kernel(
    const __hip_bfloat16 *__restrict__ x, unsigned char *__restrict__ q,
    float *__restrict__ scales, float *__restrict__ scales_t,
    long n_groups, int k_groups, int K, bool ue8m0) {
  const long g0 = blockIdx.x * (long)(blockDim.x / 64) + (threadIdx.x >> 6);
  if (g0 >= n_groups) return;
  const int lane = threadIdx.x & 63;
  const long t = g0 / k_groups;
  const int kg = g0 % k_groups;
  const __hip_bfloat16 *src = x + t * (long)K + kg * GROUP + lane * 2;
  float v0 = __bfloat162float(src[0]);
  float v1 = __bfloat162float(src[1]);
  float amax = fmaxf(fabsf(v0), fabsf(v1));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  amax = fmaxf(amax, 1e-4f);
  float scale = amax / 448.f;
  if (ue8m0) scale = exp2f(ceilf(log2f(scale)));
  const float inv = 1.f / scale;
  __hip_fp8_e4m3 q0(v0 * inv), q1(v1 * inv);
  unsigned char *dst = q + t * (long)K + kg * GROUP + lane * 2;
  dst[0] = q0.__x;
  dst[1] = q1.__x;
  if (lane == 0) {
    scales[t * (long)k_groups + kg] = scale;
    // column-major copy [k_groups, T] for the skinny GEMM: a stage's
    // M scales become ONE contiguous glds line-run instead of a
    // 64-line strided gather inside the counted-vmcnt ring
    if (scales_t)
      scales_t[(long)kg * (n_groups / k_groups) + t] = scale;
  }
}

// ------------------------------------------------- fp8 grouped MoE GEMM
// moe.hip's pipeline with fp8 operands + block scales. LDS-tiled like
// the bf16 version (BKm = 128 elems = one scale block per k tile).
constexpr int MOE_BK = 128;

template <int BM, int MOE_BN, bool SCATTER>
__global__ __launch_bounds__(BLOCK) void moe_gemm_fp8_kernel(
    __hip_bfloat16 *__restrict__ C,
    const unsigned char *__restrict__ A,   // [Ta, K] e4m3
    const float *__restrict__ As,          // [Ta, K/128]
    const unsigned char *__restrict__ W,   // [E, Nd, K] e4m3
    const float *__restrict__ Ws,          // [E, ceil(Nd/128), K/128]
    const int *__restrict__ sorted_ids, const int *__restrict__ expert_blocks,
    const int *__restrict__ n_post_pad,
    const float *__restrict__ topk_w, int n_pairs, int K, int Nd,
    int topk) {
  const int mb = blockIdx.x;
  if (mb * BM >= n_post_pad[0]) return;
  const int nb = blockIdx.y;
  const int e = expert_blocks[mb];
  const int kgroups = K / MOE_BK;
  const int nblocks = (Nd + 127) / 128;

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lhi = lane >> 4;

  constexpr int WM = BM / 16;
  constexpr int WN_TILES = MOE_BN * WM / 64;
  const int wm = wave % WM;
  const int wn = wave / WM;

  constexpr int APAD = 16;
  __shared__ unsigned char a_tile[2][BM * (MOE_BK + APAD)];
  __shared__ unsigned char w_tile[2][MOE_BN * (MOE_BK + APAD)];

  const int g0 = mb * BM;
  constexpr int A_CH = BM * MOE_BK / 16;  // 16-B chunks
  constexpr int W_CH = MOE_BN * MOE_BK / 16;
  typedef __attribute__((ext_vector_type(4))) int int4v;
  int4v areg[(A_CH + BLOCK - 1) / BLOCK];
  int4v wreg[(W_CH + BLOCK - 1) / BLOCK];

  const long w_base = (long)e * Nd * K;

  auto load_tiles = [&](int kb) {
#pragma unroll
    for (int it = 0; it < (A_CH + BLOCK - 1) / BLOCK; ++it) {
      const int idx = tid + it * BLOCK;
      if (idx < A_CH) {
        const int m = idx / (MOE_BK / 16);
        const int c = idx % (MOE_BK / 16);
        const int g = g0 + m;
        const int pair = sorted_ids[g];
        const bool valid = pair < n_pairs;
        long arow = SCATTER ? g : (valid ? pair / topk : 0);
        if (valid)
          areg[it] = *reinterpret_cast<const int4v *>(
              A + arow * (long)K + kb * MOE_BK + c * 16);
        else
          areg[it] = int4v{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int it = 0; it < (W_CH + BLOCK - 1) / BLOCK; ++it) {
      const int idx = tid + it * BLOCK;
      if (idx < W_CH) {
        const int n = idx / (MOE_BK / 16);
        const int c = idx % (MOE_BK / 16);
        if (nb * MOE_BN + n < Nd) {
          const int4v *wp = reinterpret_cast<const int4v *>(
              W + w_base + (long)(nb * MOE_BN + n) * K + kb * MOE_BK +
              c * 16);
          // nt measured NEGATIVE here (DeepSeek fp8 MoE B256: many
          // experts span 2 m-blocks, nt kills the W reuse) — cached
          wreg[it] = *wp;
        } else
          wreg[it] = int4v{0, 0, 0, 0};
      }
    }
  };
  auto write_tiles = [&](int buf) {
#pragma unroll
    for (int it = 0; it < (A_CH + BLOCK - 1) / BLOCK; ++it) {
      const int idx = tid + it * BLOCK;
      if (idx < A_CH) {
        const int m = idx / (MOE_BK / 16);
        const int c = idx % (MOE_BK / 16);
        *reinterpret_cast<int4v *>(
            &a_tile[buf][m * (MOE_BK + APAD) + c * 16]) = areg[it];
      }
    }
#pragma unroll
    for (int it = 0; it < (W_CH + BLOCK - 1) / BLOCK; ++it) {
      const int idx = tid + it * BLOCK;
      if (idx < W_CH) {
        const int n = idx / (MOE_BK / 16);
        const int c = idx % (MOE_BK / 16);
        *reinterpret_cast<int4v *>(
            &w_tile[buf][n * (MOE_BK + APAD) + c * 16]) = wreg[it];
      }
    }
  };

  f8_f4 acc[WN_TILES];
#pragma unroll
  for (int t = 0; t < WN_TILES; ++t) acc[t] = f8_f4{0, 0, 0, 0};

  load_tiles(0);
  write_tiles(0);
  __syncthreads();

  int cur = 0;
  const int nkb = K / MOE_BK;
  for (int kb = 0; kb < nkb; ++kb) {
    if (kb + 1 < nkb) load_tiles(kb + 1);

    f8_f4 sub[WN_TILES];
#pragma unroll
    for (int t = 0; t < WN_TILES; ++t) sub[t] = f8_f4{0, 0, 0, 0};
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < MOE_BK / 32; ++ks) {
      const long afrag = *reinterpret_cast<const long *>(
          &a_tile[cur][(wm * 16 + l16) * (MOE_BK + APAD) + ks * 32 +
                       lhi * 8]);
#pragma unroll
      for (int t = 0; t < WN_TILES; ++t) {
        const long bfrag = *reinterpret_cast<const long *>(
            &w_tile[cur][((wn * WN_TILES + t) * 16 + l16) * (MOE_BK + APAD) +
                         ks * 32 + lhi * 8]);
        sub[t] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
            afrag, bfrag, sub[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);

    // fold scales: A row per acc row r, W block per n tile
    float asc[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int g = g0 + wm * 16 + lhi * 4 + r;
      const int pair = sorted_ids[min(g, (int)(mb * BM + BM - 1))];
      const bool valid = pair < n_pairs;
      long arow = SCATTER ? g : (valid ? pair / topk : 0);
      asc[r] = valid ? As[arow * (long)kgroups + kb] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < WN_TILES; ++t) {
      const int nblk = (nb * MOE_BN + (wn * WN_TILES + t) * 16) / 128;
      const float wsc =
          Ws[((long)e * nblocks + min(nblk, nblocks - 1)) * kgroups + kb];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] += sub[t][r] * asc[r] * wsc;
    }

    __syncthreads();
    if (kb + 1 < nkb) {
      write_tiles(cur ^ 1);
      cur ^= 1;
      __syncthreads();
    }
  }

#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = wm * 16 + lhi * 4 + r;
    const int g = g0 + m;
    const int pair = sorted_ids[g];
    if (pair >= n_pairs) continue;
    long crow = SCATTER ? (long)pair : (long)g;
    float scalew = 1.f;
    if (SCATTER && topk_w != nullptr) scalew = topk_w[pair];
#pragma unroll
    for (int t = 0; t < WN_TILES; ++t) {
      const int n = nb * MOE_BN + (wn * WN_TILES + t) * 16 + l16;
      if (n < Nd)
        C[crow * (long)Nd + n] = __float2bfloat16(acc[t][r] * scalew);
    }
  }
}

}  // namespace

void per_token_group_quant_fp8(torch::Tensor x, torch::Tensor q,
                               torch::Tensor scales,
                               c10::optional<torch::Tensor> scales_t,
                               bool ue8m0) {
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_contiguous());
  TORCH_CHECK(q.is_contiguous() && scales.is_contiguous());
  const long T = x.size(0);
  const int K = x.size(1);
  TORCH_CHECK(K % GROUP == 0, "K must be a multiple of 128");
  const int kg = K / GROUP;
  const long n_groups = T * kg;
  float *st = nullptr;
  if (scales_t.has_value()) {
    TORCH_CHECK(scales_t->is_contiguous() &&
                scales_t->numel() == n_groups);
    st = scales_t->data_ptr<float>();
  }
  const int wpb = 4;  // waves per block
  const long grid = (n_groups + wpb - 1) / wpb;
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(per_token_group_quant_kernel, dim3(grid),
                     dim3(wpb * 64), 0, stream,
                     (const __hip_bfloat16 *)x.data_ptr(),
                     (unsigned char *)q.data_ptr(),
                     scales.data_ptr<float>(), st, n_groups, kg, K, ue8m0);
  HIP_CHECK_KERNEL();
}

void moe_gemm_fp8(torch::Tensor C, torch::Tensor A, torch::Tensor As,
                  torch::Tensor W, torch::Tensor Ws,
                  torch::Tensor sorted_ids, torch::Tensor expert_blocks,
                  torch::Tensor n_post_pad,
                  c10::optional<torch::Tensor> topk_weights, long n_pairs,
                  long topk, long block_m, bool scatter) {
  TORCH_CHECK(A.is_contiguous() && W.is_contiguous() && C.is_contiguous());
  const int K = W.size(2);
  const int Nd = W.size(1);
  TORCH_CHECK(A.size(-1) == K);
  TORCH_CHECK(K % MOE_BK == 0, "fp8 moe: K must be a multiple of 128");
  const int max_blocks = expert_blocks.numel();
  const float *tw = nullptr;
  if (topk_weights.has_value()) tw = topk_weights->data_ptr<float>();
  auto stream = at::cuda::getCurrentCUDAStream();
#define LAUNCH_M(BM, BNV, SC)                                                \
  hipLaunchKernelGGL((moe_gemm_fp8_kernel<BM, BNV, SC>),                     \
                     dim3(max_blocks, (Nd + BNV - 1) / BNV),                 \
                     dim3(BLOCK), 0, stream,                                 \
                     (__hip_bfloat16 *)C.data_ptr(),                         \
                     (const unsigned char *)A.data_ptr(),                    \
                     As.data_ptr<float>(),                                   \
                     (const unsigned char *)W.data_ptr(),                    \
                     Ws.data_ptr<float>(), sorted_ids.data_ptr<int>(),       \
                     expert_blocks.data_ptr<int>(),                          \
                     n_post_pad.data_ptr<int>(), tw, (int)n_pairs, K, Nd,    \
                     (int)topk)
  if (block_m == 16) {
    if (scatter) LAUNCH_M(16, 64, true); else LAUNCH_M(16, 64, false);
  } else if (block_m == 32) {
    if (scatter) LAUNCH_M(32, 64, true); else LAUNCH_M(32, 64, false);
  } else if (block_m == 64) {
    if (scatter) LAUNCH_M(64, 64, true); else LAUNCH_M(64, 64, false);
  } else if (block_m == 164) {  // BM=64, BN=256 (dense prefill)
    if (scatter) LAUNCH_M(64, 256, true); else LAUNCH_M(64, 256, false);
  } else {
    TORCH_CHECK(false, "moe_gemm_fp8: block_m must be 16/32/64/164");
  }
#undef LAUNCH_M
  HIP_CHECK_KERNEL();
}
