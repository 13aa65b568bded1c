// Fused-MoE kernel family for gfx950: device-side token alignment,
// grouped MFMA GEMM over sorted (token, expert) pairs, weighted combine.
//
// Reference semantics: moe_align_block_size (_custom_ops.py:424-451),
// fused_moe_kernel (fused_moe_triton/fused_moe.py:210), moe_sum
// (_custom_ops.py:393-421). MI355X-native: everything stays on device
// (no per-layer host sync), so MoE decode steps are hipGraph-capturable.
//
// Pipeline per MoE layer:
//   moe_align(topk_ids)           -> sorted_ids, expert_blocks, n_post[1]
//   gate and up, activation       -> inter_act [rows_pad, I]   (sorted)
//   down, scatter y*w             -> pair_out [T*K, H]
//   moe_sum                       -> out [T, H]
// The two products are moe_tiled.hip's where both contractions are a
// multiple of 64, else moe_gemm below (the first one then writes
// inter1 [rows_pad, 2I] and the activation is a kernel of its own).

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mfma_bf8;
typedef __attribute__((ext_vector_type(4))) float mfma_f4;

namespace {

// ---------------------------------------------------------------- align
// One workgroup: histogram -> padded prefix sum -> scatter. E_local <= 1024.
// Bound by its chain of barriers, so every phase is parallel: thread e owns
// expert e in the prefix sum and writes its block entries, a wave per expert
// writes the padding, and the pairs are scattered without another pass over
// the table (64 experts: 768 pairs 4.6 us, 24576 pairs 20.5 us; one thread
// walking the experts and a fill of the whole table took 9.7 and 35 us).
constexpr int ALIGN_BLOCK = 1024;
constexpr int MAX_E = 1024;

__global__ __launch_bounds__(ALIGN_BLOCK) void moe_align_kernel(
    const int *__restrict__ ids,  // [N] global expert id per (token,k) pair
    int N, int E_local, int expert_start, int BM,
    int *__restrict__ sorted_ids,     // [cap] pair indices, N = pad sentinel
    int *__restrict__ expert_blocks,  // [max_blocks] local expert per block
    int *__restrict__ n_post_pad) {   // [1]
  __shared__ int cnt[MAX_E], fill[MAX_E], first[MAX_E];
  __shared__ int wave_sum[ALIGN_BLOCK / 64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  cnt[tid] = 0;
  __syncthreads();
  for (int i = tid; i < N; i += ALIGN_BLOCK) {
    const int e = ids[i] - expert_start;
    if (0 <= e && e < E_local) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  const int c = cnt[tid];  // 0 past E_local
  const int nb = (c + BM - 1) / BM;
  int run = nb;  // blocks up to and with this expert
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(run, off, 64);
    if (lane >= off) run += o;
  }
  if (lane == 63) wave_sum[wave] = run;
  __syncthreads();
  for (int w = 0; w < wave; ++w) run += wave_sum[w];
  const int block0 = run - nb;
  first[tid] = block0 * BM;
  fill[tid] = block0 * BM;
  for (int b = 0; b < nb; ++b) expert_blocks[block0 + b] = tid;
  if (tid == ALIGN_BLOCK - 1) n_post_pad[0] = run * BM;
  __syncthreads();
  for (int e = wave; e < E_local; e += ALIGN_BLOCK / 64) {
    const int n = cnt[e];
    const int end = (n + BM - 1) / BM * BM;
    for (int i = n + lane; i < end; i += 64) sorted_ids[first[e] + i] = N;
  }
  for (int i = tid; i < N; i += ALIGN_BLOCK) {
    const int e = ids[i] - expert_start;
    if (0 <= e && e < E_local) sorted_ids[atomicAdd(&fill[e], 1)] = i;
  }
}

// ---------------------------------------------------------------- gemm
// C[m, n] = sum_k A[row(m), k] * W[e, n, k]  (W row-major over k).
// GATHER (gemm1): row(m) = sorted_ids[g]/topk into x; C row = g (sorted).
// SCATTER (gemm2): row(m) = g (sorted inter buffer); C row =
//   sorted_ids[g] (pair index), scaled by topk_w[pair].
constexpr int BK = 64;
constexpr int GEMM_BLOCK = 256;

// The form for K that is not a multiple of 64 (moe_tiled.hip has the rest):
// tiles pass through registers, so a K tail can be zero-filled.
template <int BM, int BN, bool SCATTER>
__global__ __launch_bounds__(GEMM_BLOCK) void moe_gemm_kernel(
    __hip_bfloat16 *__restrict__ C,
    const __hip_bfloat16 *__restrict__ A,
    const __hip_bfloat16 *__restrict__ W,  // [E_local, Nd, K]
    const int *__restrict__ sorted_ids, const int *__restrict__ expert_blocks,
    const int *__restrict__ n_post_pad,
    const float *__restrict__ topk_w,  // [n_pairs] (SCATTER only, may be 0)
    int n_pairs, int K, int Nd, int topk) {
  const int mb = blockIdx.x;
  if (mb * BM >= n_post_pad[0]) return;
  const int nb = blockIdx.y;
  const int e = expert_blocks[mb];

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lhi = lane >> 4;

  // wave tiling over the BM x BN block: (BM/16) x (BN/16) tiles over
  // 4 waves; wave owns one m sub-tile row and BN*WM/64 n tiles
  constexpr int WM = BM / 16;            // m sub-tiles (1, 2 or 4)
  constexpr int WN_TILES = BN * WM / 64; // 16-wide n tiles per wave
  const int wm = wave % WM;
  const int wn = wave / WM;              // n-tile group (4/WM groups)

  constexpr int APAD = 8;
  __shared__ __hip_bfloat16 a_tile[2][BM * (BK + APAD)];
  __shared__ __hip_bfloat16 w_tile[2][BN * (BK + APAD)];

  // per-row source/destination ids
  const int g0 = mb * BM;

  // ---- staging lambdas: 16-B chunks across the block ----
  // A tile: BM rows x BK cols; W tile: BN rows x BK cols
  constexpr int A_CH = BM * BK / 8;         // 16-B chunks
  constexpr int W_CH = BN * BK / 8;
  shortx8 areg[(A_CH + GEMM_BLOCK - 1) / GEMM_BLOCK];
  shortx8 wreg[W_CH / GEMM_BLOCK];

  const long w_base = (long)e * Nd * K;

  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int it = 0; it < (A_CH + GEMM_BLOCK - 1) / GEMM_BLOCK; ++it) {
      const int idx = tid + it * GEMM_BLOCK;
      if (idx < A_CH) {
        const int m = idx / (BK / 8);
        const int c = idx % (BK / 8);
        const int g = g0 + m;
        const int pair = sorted_ids[g];
        long arow;
        bool valid = pair < n_pairs;
        if (SCATTER) arow = g;           // sorted-order inter buffer
        else arow = valid ? pair / topk : 0;
        if (valid && k0 + c * 8 < K)
          areg[it] = *reinterpret_cast<const shortx8 *>(
              A + arow * (long)K + k0 + c * 8);
        else
          areg[it] = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int it = 0; it < W_CH / GEMM_BLOCK; ++it) {
      const int idx = tid + it * GEMM_BLOCK;
      const int n = idx / (BK / 8);
      const int c = idx % (BK / 8);
      if (nb * BN + n < Nd && k0 + c * 8 < K) {
        const shortx8 *wp = reinterpret_cast<const shortx8 *>(
            W + w_base + (long)(nb * BN + n) * K + k0 + c * 8);
        // decode tiles (BM<=32, ~1 m-block per expert) stream each W
        // row exactly once: non-temporal keeps the small A tile L2-
        // resident (guide "nt-weights"); prefill re-reads W -> cached
        if constexpr (BM <= 32)
          wreg[it] = __builtin_nontemporal_load(wp);
        else
          wreg[it] = *wp;
      } else
        wreg[it] = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  };
  auto write_tiles = [&](int buf) {
#pragma unroll
    for (int it = 0; it < (A_CH + GEMM_BLOCK - 1) / GEMM_BLOCK; ++it) {
      const int idx = tid + it * GEMM_BLOCK;
      if (idx < A_CH) {
        const int m = idx / (BK / 8);
        const int c = idx % (BK / 8);
        *reinterpret_cast<shortx8 *>(&a_tile[buf][m * (BK + APAD) + c * 8]) =
            areg[it];
      }
    }
#pragma unroll
    for (int it = 0; it < W_CH / GEMM_BLOCK; ++it) {
      const int idx = tid + it * GEMM_BLOCK;
      const int n = idx / (BK / 8);
      const int c = idx % (BK / 8);
      *reinterpret_cast<shortx8 *>(&w_tile[buf][n * (BK + APAD) + c * 8]) =
          wreg[it];
    }
  };

  mfma_f4 acc[WN_TILES];
#pragma unroll
  for (int t = 0; t < WN_TILES; ++t) acc[t] = mfma_f4{0, 0, 0, 0};

  load_tiles(0);
  write_tiles(0);
  __syncthreads();

  int cur = 0;
  for (int k0 = 0; k0 < K; k0 += BK) {
    if (k0 + BK < K) load_tiles(k0 + BK);

    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      mfma_bf8 afrag = *reinterpret_cast<const mfma_bf8 *>(
          &a_tile[cur][(wm * 16 + l16) * (BK + APAD) + ks * 32 + lhi * 8]);
#pragma unroll
      for (int t = 0; t < WN_TILES; ++t) {
        mfma_bf8 wfrag = *reinterpret_cast<const mfma_bf8 *>(
            &w_tile[cur][((wn * WN_TILES + t) * 16 + l16) * (BK + APAD) +
                         ks * 32 + lhi * 8]);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            afrag, wfrag, acc[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);

    __syncthreads();
    if (k0 + BK < K) {
      write_tiles(cur ^ 1);
      cur ^= 1;
      __syncthreads();
    }
  }

  // ---- epilogue: C rows lhi*4+r of the wave's m tile ----
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
      const int n = nb * BN + (wn * WN_TILES + t) * 16 + l16;
      if (n < Nd)
        C[crow * (long)Nd + n] = __float2bfloat16(acc[t][r] * scalew);
    }
  }
}

// ---------------------------------------------------------------- sum
// out[t, :] = sum_k pair_out[t*K + k, :] over the pairs whose expert is one
// of the local ones (rows of the others were never written)
template <typename T>
__global__ void moe_sum_kernel(T *__restrict__ out,
                               const T *__restrict__ pair_out,
                               const int *__restrict__ ids, int expert_start,
                               int E_local, long TH, int topk, int H) {
  const int nvec = H / 8;
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
       idx < TH * nvec; idx += (long)gridDim.x * blockDim.x) {
    const long t = idx / nvec;
    const int c = idx % nvec;
    float accv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < topk; ++k) {
      const int e = ids[t * topk + k] - expert_start;
      if (e < 0 || e >= E_local) continue;
      shortx8 v = reinterpret_cast<const shortx8 *>(
          pair_out + (t * topk + k) * (long)H)[c];
      float f[8];
      unpack8<T>(v, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) accv[j] += f[j];
    }
    reinterpret_cast<shortx8 *>(out + t * (long)H)[c] = pack8<T>(accv);
  }
}

// A workgroup per token: residual += (sum of its pairs, rounded) + shared
// (each step rounded as if it were stored), out = RMS norm of the stored
// residual. Bound by the pairs' bytes and by launches: a sum, an addition and
// a norm that each read and wrote the rows took 23 + 9 + 14 us for 4096 tokens
// of 2048 with 6 experts and 5.7 + 4.9 + 4.5 for 128; this takes 29 and 4.7.
template <int V, typename TW>
__global__ __launch_bounds__(256) void moe_sum_norm_kernel(
    __hip_bfloat16 *__restrict__ out, __hip_bfloat16 *__restrict__ residual,
    const __hip_bfloat16 *__restrict__ pair_out, const int *__restrict__ ids,
    const __hip_bfloat16 *__restrict__ shared, const TW *__restrict__ w,
    float eps, int expert_start, int E_local, int topk, int H) {
  typedef __hip_bfloat16 T;
  constexpr int KU = 4;  // pairs on their way at once
  __shared__ float red[4];
  const long t = blockIdx.x;
  const int *row_ids = ids + t * topk;
  const T *pairs = pair_out + t * topk * H;
  const int nvec = H / 8;
  float x[V][8], ss = 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int c = j * 256 + threadIdx.x;
    if (c >= nvec) continue;
    const shortx8 old = reinterpret_cast<const shortx8 *>(residual + t * H)[c];
    shortx8 sh = {0, 0, 0, 0, 0, 0, 0, 0};
    if (shared) sh = reinterpret_cast<const shortx8 *>(shared + t * H)[c];
    float a[8] = {0, 0, 0, 0, 0, 0, 0, 0}, f[8];
    for (int k0 = 0; k0 < topk; k0 += KU) {
      shortx8 v[KU];
      bool used[KU];
#pragma unroll
      for (int i = 0; i < KU; ++i) {
        const int k = min(k0 + i, topk - 1), e = row_ids[k] - expert_start;
        used[i] = k0 + i < topk && 0 <= e && e < E_local;
        v[i] = reinterpret_cast<const shortx8 *>(pairs + (long)k * H)[c];
      }
#pragma unroll
      for (int i = 0; i < KU; ++i) {
        unpack8<T>(v[i], f);
#pragma unroll
        for (int r = 0; r < 8; ++r) a[r] = used[i] ? a[r] + f[r] : a[r];
      }
    }
    unpack8<T>(pack8<T>(a), a);
    if (shared) {
      unpack8<T>(sh, f);
#pragma unroll
      for (int r = 0; r < 8; ++r) a[r] += f[r];
      unpack8<T>(pack8<T>(a), a);
    }
    unpack8<T>(old, f);
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] += f[r];
    const shortx8 sum = pack8<T>(a);
    reinterpret_cast<shortx8 *>(residual + t * H)[c] = sum;
    unpack8<T>(sum, x[j]);
#pragma unroll
    for (int r = 0; r < 8; ++r) ss += x[j][r] * x[j][r];
  }
  ss = block_reduce_sum<256>(ss, red);
  const float inv = rsqrtf(ss / H + eps);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int c = j * 256 + threadIdx.x;
    if (c >= nvec) continue;
    float wv[8];
    ld8<TW>(w + c * 8, wv);
#pragma unroll
    for (int r = 0; r < 8; ++r) x[j][r] = x[j][r] * inv * wv[r];
    reinterpret_cast<shortx8 *>(out + t * H)[c] = pack8<T>(x[j]);
  }
}

}  // namespace

void moe_align(torch::Tensor topk_ids, long E_local, long expert_start,
               long block_m, torch::Tensor sorted_ids,
               torch::Tensor expert_blocks, torch::Tensor n_post_pad) {
  const int N = topk_ids.numel();
  TORCH_CHECK(topk_ids.scalar_type() == at::kInt);
  TORCH_CHECK(topk_ids.is_contiguous());
  TORCH_CHECK(E_local <= MAX_E);
  TORCH_CHECK(sorted_ids.numel() >=
              N + E_local * (block_m - 1) + 1);
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(ALIGN_BLOCK), 0, stream,
                     topk_ids.data_ptr<int>(), N, (int)E_local,
                     (int)expert_start, (int)block_m,
                     sorted_ids.data_ptr<int>(),
                     expert_blocks.data_ptr<int>(),
                     n_post_pad.data_ptr<int>());
  HIP_CHECK_KERNEL();
}

void moe_gemm(torch::Tensor C, torch::Tensor A, torch::Tensor W,
              torch::Tensor sorted_ids, torch::Tensor expert_blocks,
              torch::Tensor n_post_pad,
              c10::optional<torch::Tensor> topk_weights, long n_pairs,
              long topk, long block_m, bool scatter) {
  TORCH_CHECK(A.scalar_type() == at::kBFloat16 &&
              W.scalar_type() == at::kBFloat16);
  TORCH_CHECK(A.is_contiguous() && W.is_contiguous() && C.is_contiguous());
  const int K = W.size(2);
  const int Nd = W.size(1);
  TORCH_CHECK(A.size(-1) == K);
  TORCH_CHECK(K % 8 == 0, "moe_gemm: K must be a multiple of 8");
  const int max_blocks = expert_blocks.numel();
  const float *tw = nullptr;
  if (topk_weights.has_value()) {
    TORCH_CHECK(topk_weights->scalar_type() == at::kFloat);
    tw = topk_weights->data_ptr<float>();
  }
  auto stream = at::cuda::getCurrentCUDAStream();
#define LAUNCH(BM, BNV, SC)                                                 \
  hipLaunchKernelGGL((moe_gemm_kernel<BM, BNV, SC>),                        \
                     dim3(max_blocks, (Nd + BNV - 1) / BNV),                \
                     dim3(GEMM_BLOCK), 0, stream,                           \
                     (__hip_bfloat16 *)C.data_ptr(),                        \
                     (const __hip_bfloat16 *)A.data_ptr(),                  \
                     (const __hip_bfloat16 *)W.data_ptr(),                  \
                     sorted_ids.data_ptr<int>(),                            \
                     expert_blocks.data_ptr<int>(),                         \
                     n_post_pad.data_ptr<int>(), tw, (int)n_pairs, K, Nd,   \
                     (int)topk)
  if (block_m == 16) {
    if (scatter) LAUNCH(16, 64, true); else LAUNCH(16, 64, false);
  } else if (block_m == 32) {
    if (scatter) LAUNCH(32, 64, true); else LAUNCH(32, 64, false);
  } else if (block_m == 64) {
    if (scatter) LAUNCH(64, 64, true); else LAUNCH(64, 64, false);
  } else {
    TORCH_CHECK(false, "moe_gemm: block_m must be 16/32/64");
  }
#undef LAUNCH
  HIP_CHECK_KERNEL();
}

void moe_sum(torch::Tensor out, torch::Tensor pair_out, torch::Tensor ids,
             long expert_start, long E_local, long topk) {
  TORCH_CHECK(out.scalar_type() == at::kBFloat16 &&
              pair_out.scalar_type() == at::kBFloat16);
  TORCH_CHECK(ids.scalar_type() == at::kInt && ids.is_contiguous() &&
              ids.numel() == out.size(0) * topk);
  TORCH_CHECK(out.is_contiguous() && pair_out.is_contiguous());
  const long T = out.size(0);
  const int H = out.size(-1);
  TORCH_CHECK(H % 8 == 0);
  const long total = T * (H / 8);
  const int block = 256;
  const long grid = std::min<long>((total + block - 1) / block, 4096);
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL((moe_sum_kernel<__hip_bfloat16>), dim3(grid),
                     dim3(block), 0, stream,
                     (__hip_bfloat16 *)out.data_ptr(),
                     (const __hip_bfloat16 *)pair_out.data_ptr(),
                     ids.data_ptr<int>(), (int)expert_start, (int)E_local, T,
                     (int)topk, H);
  HIP_CHECK_KERNEL();
}

// residual (bf16 [T, H], in place) += the tokens' sums (+ shared); returns its
// RMS norm
torch::Tensor moe_sum_norm(torch::Tensor pair_out, torch::Tensor ids,
                           long expert_start, long E_local, long topk,
                           c10::optional<torch::Tensor> shared,
                           torch::Tensor residual, torch::Tensor norm_w,
                           double eps) {
  auto rows_ok = [&](const torch::Tensor &t) {
    return t.is_cuda() && t.scalar_type() == at::kBFloat16 &&
           t.is_contiguous() &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  TORCH_CHECK(residual.dim() == 2 && rows_ok(residual) && rows_ok(pair_out),
              "moe_sum_norm: contiguous bf16 rows, 16 B aligned");
  const long T = residual.size(0), H = residual.size(1);
  TORCH_CHECK(H % 8 == 0 && H <= 8192 && topk > 0 &&
              pair_out.numel() == T * topk * H);
  TORCH_CHECK(ids.scalar_type() == at::kInt && ids.is_contiguous() &&
              ids.numel() == T * topk);
  TORCH_CHECK(!shared.has_value() ||
              (rows_ok(*shared) && shared->numel() == T * H));
  TORCH_CHECK(norm_w.is_cuda() && norm_w.is_contiguous() &&
              norm_w.numel() == H &&
              reinterpret_cast<uintptr_t>(norm_w.data_ptr()) % 16 == 0);
  auto out = torch::empty_like(residual);
  if (T == 0) return out;
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(V, TW)                                                           \
  hipLaunchKernelGGL((moe_sum_norm_kernel<V, TW>), dim3(T), dim3(256), 0,    \
                     stream, (__hip_bfloat16 *)out.data_ptr(),               \
                     (__hip_bfloat16 *)residual.data_ptr(),                  \
                     (const __hip_bfloat16 *)pair_out.data_ptr(),            \
                     ids.data_ptr<int>(),                                    \
                     shared.has_value()                                      \
                         ? (const __hip_bfloat16 *)shared->data_ptr()        \
                         : nullptr,                                          \
                     (const TW *)norm_w.data_ptr(), (float)eps,              \
                     (int)expert_start, (int)E_local, (int)topk, (int)H)
#define COLS(TW)                                                             \
  do {                                                                       \
    if (H <= 2048) RUN(1, TW);                                               \
    else if (H <= 4096) RUN(2, TW);                                          \
    else RUN(4, TW);                                                         \
  } while (0)
  if (norm_w.scalar_type() == at::kFloat) COLS(float);
  else if (norm_w.scalar_type() == at::kBFloat16) COLS(__hip_bfloat16);
  else TORCH_CHECK(false, "norm_w: fp32 or bf16");
#undef COLS
#undef RUN
  HIP_CHECK_KERNEL();
  return out;
}

// ---------------------------------------------------------------------
// Top-k of the router LOGITS, softmax over the chosen ones only.
// One wave per token row: lane l holds logits l, l + 64, ... (E <= 512);
// k rounds of a wave-wide arg-max (ties go to the lower index) pick the
// experts in descending order, lane r keeps the r-th pick, and the
// softmax over the k picks is one more wave reduction.
namespace {

constexpr int TK_MAXJ = 8;  // logits per lane: E <= 64 * TK_MAXJ

// Order of floats as unsigned numbers, for picks on which all lanes of a
// wave agree whatever the values are (with a NaN, comparisons of the floats
// themselves leave lanes with different picks): 0 is no candidate, a NaN
// stands behind every number, -0 equals 0.
DEV_INLINE unsigned pick_key(float v) {
  if (v != v) return 1u;
  const unsigned u = __float_as_uint(v + 0.f);
  return u & 0x80000000u ? ~u : u | 0x80000000u;
}

DEV_INLINE float key_value(unsigned k) {
  return __uint_as_float(k == 1u ? 0x7fc00000u
                         : k & 0x80000000u ? k ^ 0x80000000u : ~k);
}

// the largest of the wave's keys
DEV_INLINE unsigned wave_max_key(unsigned x) {
#define STEP(CTRL, ROWS)                                                     \
  x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS,    \
                                                   0xf, false))
  STEP(0x111, 0xf);  // row_shr 1, 2, 4, 8; then the rows before
  STEP(0x112, 0xf);
  STEP(0x114, 0xf);
  STEP(0x118, 0xf);
  STEP(0x142, 0xa);
  STEP(0x143, 0xc);
#undef STEP
  return __builtin_amdgcn_readlane(x, 63);
}

// Takes the wave's largest key (lane: indexes lane + 64 j) out of the
// candidates; its index, the lowest of equals. (us, eight of 128 experts, 128
// rows 6.0, 8192 rows 13.1; with key and index passed from lane to lane 8.6 and
// 17.2.)
template <int J>
DEV_INLINE int take_best(unsigned (&key)[J], unsigned &best) {
  unsigned mine = key[0];
#pragma unroll
  for (int j = 1; j < J; ++j) mine = max(mine, key[j]);
  best = wave_max_key(mine);
  int idx = -1;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const unsigned long long m = __ballot(key[j] == best);
    if (idx < 0 && m) idx = 64 * j + __ffsll(m) - 1;
  }
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (idx == (int)(threadIdx.x & 63) + 64 * j) key[j] = 0u;
  return idx;
}

__global__ __launch_bounds__(256) void topk_softmax_rows_kernel(
    float *__restrict__ weights, int *__restrict__ ids,
    const float *__restrict__ logits, long rows, int E, int k) {
  const long r = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  const float *row = logits + r * E;
  unsigned key[TK_MAXJ];
#pragma unroll
  for (int j = 0; j < TK_MAXJ; ++j) {
    const int e = lane + 64 * j;
    key[j] = e < E ? pick_key(row[e]) : 0u;
  }
  float my_val = -INFINITY;
  int my_idx = 0;
  for (int it = 0; it < k; ++it) {
    unsigned best;
    const int bidx = take_best(key, best);
    if (lane == it) { my_val = key_value(best); my_idx = bidx; }
  }
  const float top = __shfl(my_val, 0, 64);  // the first pick is the largest
  const float p = lane < k ? expf(my_val - top) : 0.f;
  const float sum = wave_reduce_sum(p);
  if (lane < k) {
    weights[r * k + lane] = p / sum;
    ids[r * k + lane] = my_idx;
  }
}

// Softmax over ALL experts, then the top k of the probabilities, in
// descending order (ties to the lower index); renorm: over their sum.
// Bound by launches, not by work: it stands for a cast, a softmax, a top-k,
// a sort, a sum, a division and a cast (8 experts: 64 tokens 5.3 us for 48,
// 5000 tokens 7.8 us for 57). A wave per row, as above, J experts per lane;
// with one, a pick is a maximum over lanes and the first lane that has it.
template <typename T, int J>
__global__ __launch_bounds__(256) void softmax_topk_rows_kernel(
    float *__restrict__ weights, int *__restrict__ ids,
    const T *__restrict__ logits, long rows, int E, int k, bool renorm) {
  const long r = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  const T *row = logits + r * E;
  float v[J], mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int e = lane + 64 * j;
    v[j] = e < E ? ScalarOps<T>::to_f32(row[e]) : -INFINITY;
    mx = fmaxf(mx, v[j]);
  }
  mx = wave_reduce_max(mx);
  float sum = 0.f;
  unsigned key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const bool live = lane + 64 * j < E;
    const float p = expf(v[j] - mx);
    key[j] = live ? pick_key(p) : 0u;
    if (live) sum += p;
  }
  sum = wave_reduce_sum(sum);
  float my_val = 0.f;
  int my_idx = 0;
  for (int it = 0; it < k; ++it) {
    unsigned best;
    const int bidx = take_best(key, best);
    if (lane == it) { my_val = key_value(best) / sum; my_idx = bidx; }
  }
  if (renorm) my_val /= wave_reduce_sum(lane < k ? my_val : 0.f);
  if (lane < k) {
    weights[r * k + lane] = my_val;
    ids[r * k + lane] = my_idx;
  }
}

// Sigmoid router with a selection-only correction and group limits.
// One wave per token, up to 64 * TK_MAXJ experts, lane l holds experts
// l, l + 64, ...: s = sigmoid(logit) weighs, c = s + correction chooses.
// Experts form n_group equal groups of neighbours; a group scores the
// sum of its two largest c and only experts of the `keep` best groups
// stay eligible (the rest count as -inf). k rounds of a wave-wide
// arg-max (ties to the lower index) pick the experts; weights are the
// chosen s over their sum (+ 1e-20), times scale.
// The per-wave LDS row holds c for the group scan.
__global__ __launch_bounds__(256) void sigmoid_group_topk_kernel(
    float *__restrict__ weights, int *__restrict__ ids,
    const float *__restrict__ logits, const float *__restrict__ correction,
    long rows, int E, int k, int n_group, int keep, float scale) {
  extern __shared__ float sg_lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long r = (long)blockIdx.x * 4 + wave;
  if (r >= rows) return;  // no block-wide barrier below
  float *crow = sg_lds + (size_t)wave * (E + n_group);
  float *gsc = crow + E;
  const float *row = logits + r * E;
  float c[TK_MAXJ];
#pragma unroll
  for (int j = 0; j < TK_MAXJ; ++j) {
    const int e = lane + 64 * j;
    if (e < E) {
      c[j] = 1.0f / (1.0f + expf(-row[e])) +
             (correction ? correction[e] : 0.f);
      crow[e] = c[j];
    } else {
      c[j] = -INFINITY;
    }
  }
  if (n_group > 1) {
    const int per = E / n_group;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // LDS writes of this wave landed
    for (int g = lane; g < n_group; g += 64) {
      float b0 = -INFINITY, b1 = -INFINITY;
      for (int i = 0; i < per; ++i) {
        const float x = crow[g * per + i];
        if (x > b0) { b1 = b0; b0 = x; }
        else if (x > b1) b1 = x;
      }
      gsc[g] = per > 1 ? b0 + b1 : b0;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0xc07f);
#pragma unroll
    for (int j = 0; j < TK_MAXJ; ++j) {
      const int e = lane + 64 * j;
      if (e < E) {
        const int g = e / per;
        const float mine = gsc[g];
        int rank = 0;  // groups ahead of mine; ties go to the lower index
        for (int o = 0; o < n_group; ++o) {
          const float x = gsc[o];
          rank += (x > mine || (x == mine && o < g)) ? 1 : 0;
        }
        if (rank >= keep) c[j] = -INFINITY;
      }
    }
  }
  unsigned key[TK_MAXJ];
#pragma unroll
  for (int j = 0; j < TK_MAXJ; ++j)
    key[j] = lane + 64 * j < E ? pick_key(c[j]) : 0u;
  int my_idx = 0;
  for (int it = 0; it < k; ++it) {
    unsigned best;
    const int bidx = take_best(key, best);
    if (lane == it) my_idx = bidx;
  }
  const float my_w = lane < k ? 1.0f / (1.0f + expf(-row[my_idx])) : 0.f;
  const float sum = wave_reduce_sum(my_w);
  if (lane < k) {
    weights[r * k + lane] = my_w / (sum + 1e-20f) * scale;
    ids[r * k + lane] = my_idx;
  }
}

}  // namespace

void sigmoid_group_topk(torch::Tensor weights, torch::Tensor ids,
                        torch::Tensor logits,
                        c10::optional<torch::Tensor> correction,
                        long n_group, long keep, double scale) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 &&
              logits.is_contiguous() && logits.scalar_type() == at::kFloat,
              "logits: fp32 [rows, experts]");
  const long rows = logits.size(0);
  const int E = logits.size(1);
  TORCH_CHECK(weights.dim() == 2 && weights.size(0) == rows &&
              weights.is_contiguous() && weights.scalar_type() == at::kFloat);
  const int k = weights.size(1);
  TORCH_CHECK(ids.is_contiguous() && ids.scalar_type() == at::kInt &&
              ids.numel() == rows * k);
  TORCH_CHECK(E >= 1 && E <= 64 * TK_MAXJ && k >= 1 && k <= 64 && k <= E,
              "sigmoid_group_topk: experts <= ", 64 * TK_MAXJ,
              ", top <= min(64, experts)");
  TORCH_CHECK(n_group >= 1 && E % n_group == 0 && keep >= 1 &&
              keep <= n_group, "sigmoid_group_topk: bad groups");
  TORCH_CHECK(k <= keep * (E / n_group),
              "sigmoid_group_topk: the kept groups hold fewer experts "
              "than are chosen");
  const float *cp = nullptr;
  if (correction.has_value()) {
    TORCH_CHECK(correction->is_cuda() && correction->is_contiguous() &&
                correction->scalar_type() == at::kFloat &&
                correction->numel() == E, "correction: fp32 [experts]");
    cp = correction->data_ptr<float>();
  }
  if (rows == 0) return;
  auto stream = at::cuda::getCurrentCUDAStream();
  const size_t lds = 4 * (size_t)(E + n_group) * sizeof(float);
  hipLaunchKernelGGL(sigmoid_group_topk_kernel, dim3((rows + 3) / 4),
                     dim3(256), lds, stream, weights.data_ptr<float>(),
                     ids.data_ptr<int>(), logits.data_ptr<float>(), cp, rows,
                     E, k, (int)n_group, (int)keep, (float)scale);
  HIP_CHECK_KERNEL();
}

// logits: fp32, bf16 or fp16 [rows, experts]
void softmax_topk_rows(torch::Tensor weights, torch::Tensor ids,
                       torch::Tensor logits, bool renorm) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 &&
              logits.is_contiguous(), "logits: [rows, experts]");
  const long rows = logits.size(0);
  const int E = logits.size(1);
  TORCH_CHECK(weights.dim() == 2 && weights.size(0) == rows &&
              weights.is_contiguous() && weights.scalar_type() == at::kFloat);
  const int k = weights.size(1);
  TORCH_CHECK(ids.is_contiguous() && ids.scalar_type() == at::kInt &&
              ids.numel() == rows * k);
  TORCH_CHECK(E >= 1 && E <= 64 * TK_MAXJ && k >= 1 && k <= 64 && k <= E,
              "softmax_topk_rows: experts <= ", 64 * TK_MAXJ,
              ", top <= min(64, experts)");
  if (rows == 0) return;
  auto stream = at::cuda::getCurrentCUDAStream();
#define ROWS(T, J)                                                           \
  hipLaunchKernelGGL((softmax_topk_rows_kernel<T, J>), dim3((rows + 3) / 4), \
                     dim3(256), 0, stream, weights.data_ptr<float>(),        \
                     ids.data_ptr<int>(), (const T *)logits.data_ptr(), rows,\
                     E, k, renorm)
#define RUN(T)                                                               \
  do {                                                                       \
    if (E <= 64) ROWS(T, 1);                                                 \
    else ROWS(T, TK_MAXJ);                                                   \
  } while (0)
  if (logits.scalar_type() == at::kFloat) RUN(float);
  else if (logits.scalar_type() == at::kBFloat16) RUN(__hip_bfloat16);
  else if (logits.scalar_type() == at::kHalf) RUN(__half);
  else TORCH_CHECK(false, "softmax_topk_rows: fp32, bf16 or fp16 logits");
#undef RUN
#undef ROWS
  HIP_CHECK_KERNEL();
}

void topk_softmax_rows(torch::Tensor weights, torch::Tensor ids,
                       torch::Tensor logits) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 &&
              logits.is_contiguous() && logits.scalar_type() == at::kFloat,
              "logits: fp32 [rows, experts]");
  const long rows = logits.size(0);
  const int E = logits.size(1);
  TORCH_CHECK(weights.dim() == 2 && weights.size(0) == rows &&
              weights.is_contiguous() && weights.scalar_type() == at::kFloat);
  const int k = weights.size(1);
  TORCH_CHECK(ids.is_contiguous() && ids.scalar_type() == at::kInt &&
              ids.numel() == rows * k);
  TORCH_CHECK(E >= 1 && E <= 64 * TK_MAXJ && k >= 1 && k <= 64 && k <= E,
              "topk_softmax_rows: experts <= ", 64 * TK_MAXJ,
              ", top <= min(64, experts)");
  if (rows == 0) return;
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(topk_softmax_rows_kernel, dim3((rows + 3) / 4),
                     dim3(256), 0, stream, weights.data_ptr<float>(),
                     ids.data_ptr<int>(), logits.data_ptr<float>(), rows, E,
                     k);
  HIP_CHECK_KERNEL();
}
