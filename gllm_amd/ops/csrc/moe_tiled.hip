// Grouped MoE GEMM of wide tiles for gfx950 (bf16, K a multiple of 64).
//
// The same (token, expert) blocks as moe.hip: rows sorted by expert, every
// block of block_m rows belongs to one expert. Three forms:
//   gated    act[row, i] = f(x W_gate^T)(x W_up^T), rows gathered by token
//   plain    act[row, n] = f(x W^T), rows gathered by token
//   scatter  out[pair, n] = w[pair] * act W^T
// The activation is applied to the fp32 accumulators: the [rows, 2I]
// intermediate is never written.
//
// Both operands go straight to LDS (global_load_lds, 16 B per lane) in rows
// of 128 B whose 16 B units are permuted by row & 7, so the fragment reads
// (16 rows, one unit each) fall on all banks. Products are W A^T: a lane
// holds four neighbouring columns of one row, and the gate and up columns
// of a pair (rows of the staged W tile alternate in groups of 16) sit in
// the same lane.
//
// The tile follows the rows per expert, because two things bound this:
//  * few rows: the weights' bytes. 32 x 128 and 64 x 128 tiles keep three
//    and two tiles of a ring in flight (80 KB and 72 KB of LDS: two
//    workgroups per CU) and read weights non-temporally. 8 experts of
//    4096 x 14336, 64 tokens: 289 + 178 us (6.5 and 5.3 TB/s) where the
//    former 32 x 64 tiles through registers took 504 + 339 us. 64 experts
//    of 2048 x 1408, 128 tokens: 131 + 60 us (168 + 86 us). 32 rows hold
//    an expert's share up to 12 per expert; at 16, where popular experts
//    have more, 64 rows take 2732 us for a step of four layers, 32 rows
//    2875 us; at 24 the two are within 3 %, at 32 64 rows take 299 + 184 us
//    against 375 + 230 us.
//  * many rows: the matrix cores. Blocks of 256 rows go to tile_gemm.hip,
//    which takes operands below 2 GiB (8 experts of 4096 x 14336, 10000 rows:
//    1910 + 990 us); for larger ones 256 x 256 tiles on eight waves of 128 x
//    64, one workgroup each (2226 + 1177 us).
//  * between (40 to 128 rows per expert): 128 x 128 tiles on four waves;
//    64 rows per expert 375 + 192 us against 442 + 251 us (64 x 128) and
//    475 + 379 us (256 x 256); 192 rows 287 + 182 us against 226 + 163 us
//    for 256 x 256.
// A shared expert's tiles come first in the same launch: they are the longest
// of the second product, and what they wait for is hidden by the routed ones'.
// (Two of 2048 x 1408 for 128 rows beside 64 routed ones, with sum and norm:
// 214 us by launches of their own, 207 so; 32 rows 203, 194.)
// Workgroups go to the eight dies in turn; each die gets a contiguous run
// of tiles, row blocks fastest within groups, so that the tiles which
// share weights meet in one L2.

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "tile_gemm.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mt_bf8;
typedef __attribute__((ext_vector_type(4))) float mt_f4;

namespace {

constexpr int BK = 64;
constexpr int ROW_B = BK * 2;  // LDS row bytes

enum Form { GATED = 0, PLAIN = 1, SCATTER = 2 };
enum Act { NONE = 0, SILU = 1, CLAMP = 2, RELU2 = 3 };

// AUX 2: non-temporal
template <int AUX>
DEV_INLINE void glds16(const __hip_bfloat16 *gsrc, char *lds_ptr) {
  __builtin_amdgcn_global_load_lds(
      reinterpret_cast<const unsigned int *>(gsrc),
      reinterpret_cast<unsigned int *>(lds_ptr), 16, 0, AUX);
}

DEV_INLINE short to_bf16(float v) {
  return __builtin_bit_cast(short, __float2bfloat16(v));
}

// An expert that all rows pass, of a size of its own and in row order, beside
// the routed ones in the same launch.
struct Shared {
  __hip_bfloat16 *C;
  const __hip_bfloat16 *A, *W;  // [rows, K], [N, K]
  int rows, K, N, nbm, nbn;
  int slice;  // columns of K of one sum, see SUMS below
};

// WM x WN waves share a BM x BN tile; a ring of ST stages of BK columns
template <int BM, int BN, int WM, int WN, int ST, int AUX, int FORM, int ACT,
          bool SHARED = false>
__global__ __launch_bounds__(WM *WN * 64) void moe_tiled_kernel(
    __hip_bfloat16 *__restrict__ C, const __hip_bfloat16 *__restrict__ A,
    const __hip_bfloat16 *__restrict__ W,  // [E_local, Nd, K]
    const int *__restrict__ sorted_ids, const int *__restrict__ expert_blocks,
    const int *__restrict__ n_post_pad,
    const float *__restrict__ topk_w,  // [n_pairs] (SCATTER only, may be 0)
    int n_pairs, int K, int Nd, int topk, int nbn, float limit,
    float alpha, const Shared shared) {
  constexpr int THREADS = WM * WN * 64;
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;  // 16 x 16 per wave
  constexpr int A_B = BM * ROW_B, STAGE = A_B + BN * ROW_B;
  constexpr int AL = BM * ROW_B / (THREADS * 16);  // loads per thread
  constexpr int BL = BN * ROW_B / (THREADS * 16);
  constexpr int LD = AL + BL;
  static_assert(AL * THREADS * 16 == BM * ROW_B, "whole loads");
  static_assert(BL * THREADS * 16 == BN * ROW_B, "whole loads");
  static_assert(ST >= 2 && ST <= 4, "waits below");
  __shared__ __attribute__((aligned(16))) char smem[ST * STAGE];

  const int nblk = n_post_pad[0] / BM;
  const int total = nblk * nbn;
  const int pid = blockIdx.x;
  const int xcd = pid & 7;
  int t = pid >> 3, mb, nb, e = 0;
  bool sh = false;  // a tile of the shared expert: each die's first ones
  // Its second product by itself is formed of sums over shares of K, added in
  // their order (stream_gemm). So is this one: the same bits, and sums as
  // short. (64 experts of 2048 x 1408, shared 2816, in one sum / in four: 128
  // rows 208 / 208 us, 32 rows 195 / 195.)
  constexpr bool SUMS = SHARED && FORM == SCATTER;
  if (SHARED) {
    const int s_total = shared.nbm * shared.nbn;
    const int s0 = xcd * s_total >> 3, s1 = (xcd + 1) * s_total >> 3;
    sh = t < s1 - s0;
    if (sh) {
      mb = (s0 + t) % shared.nbm;
      nb = (s0 + t) / shared.nbm;
      A = shared.A;
      W = shared.W;
      C = shared.C;
      K = shared.K;
      Nd = shared.N;
    }
    t -= s1 - s0;
  }
  if (!sh) {
    const int per = total >> 3;
    if (t >= per + (xcd < (total & 7))) return;
    t += xcd * per + min(xcd, total & 7);
    constexpr int GM = BM >= 256 ? 4 : 8;  // row blocks of a group
    const int grp = t / (GM * nbn), in_g = t - grp * GM * nbn;
    const int gm = min(GM, nblk - grp * GM);
    mb = grp * GM + in_g % gm;
    nb = in_g / gm;
    e = expert_blocks[mb];
  }
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int g0 = mb * BM;
  const int I = FORM == GATED ? Nd >> 1 : Nd;  // columns of C

  // sources of this thread's 16 B units
  const __hip_bfloat16 *asrc[AL], *bsrc[BL];
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    const int u = j * THREADS + tid, row = u >> 3;
    long r = g0 + row;  // (padding rows of a sorted buffer are not used)
    if (sh) {
      r = min(g0 + row, shared.rows - 1);
    } else if (FORM != SCATTER) {
      const int pair = sorted_ids[g0 + row];
      r = pair < n_pairs ? pair / topk : 0;
    }
    asrc[j] = A + r * (long)K + ((u & 7) ^ (row & 7)) * 8;
  }
  const __hip_bfloat16 *we = W + (long)e * Nd * K;
#pragma unroll
  for (int j = 0; j < BL; ++j) {
    const int u = j * THREADS + tid, row = u >> 3;
    int n;
    if (FORM == GATED) {  // 16 gate rows, their 16 up rows, the next 16
      const int col = min(nb * (BN / 2) + (row >> 5) * 16 + (row & 15), I - 1);
      n = (row & 16) ? I + col : col;
    } else {
      n = min(nb * BN + row, Nd - 1);
    }
    bsrc[j] = we + (long)n * K + ((u & 7) ^ (row & 7)) * 8;
  }
  auto stage = [&](int slot) {
    char *base = smem + slot * STAGE + wave * 1024;
#pragma unroll
    for (int j = 0; j < AL; ++j) {
      glds16<0>(asrc[j], base + j * THREADS * 16);
      asrc[j] += BK;
    }
#pragma unroll
    for (int j = 0; j < BL; ++j) {
      glds16<AUX>(bsrc[j], base + A_B + j * THREADS * 16);
      bsrc[j] += BK;
    }
  };
  mt_f4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = mt_f4{0, 0, 0, 0};
  mt_f4 sum[SUMS ? NT : 1][MT] = {};

  const int nkt = K / BK;
  const int share = SUMS && sh ? shared.slice / BK : nkt;
  int border = share;
#pragma unroll
  for (int i = 0; i < ST - 1; ++i)
    if (i < nkt) stage(i);
  int cur = 0, nxt = ST - 1;  // slots of this stage and of the newest
  for (int kt = 0; kt < nkt; ++kt) {
    // this wave's loads of stage kt have landed; `ahead` later stages may
    // still be on their way (fewer near the end)
    const int ahead = min(nkt - 1 - kt, ST - 2);
    if (ST >= 4 && ahead == 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * LD) : "memory");
    else if (ST >= 3 && ahead == 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LD) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // everybody's loads of stage kt are there, and everybody has read
    // stage kt - 1, whose slot the next stage takes
    __builtin_amdgcn_s_barrier();
    if (kt + ST - 1 < nkt) stage(nxt);
    if (SUMS && kt == border) {
      border += share;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          sum[SUMS ? n : 0][m] += acc[n][m];
          acc[n][m] = mt_f4{0, 0, 0, 0};
        }
    }
    const char *ab = smem + cur * STAGE + (wm * MT * 16 + l16) * ROW_B;
    const char *bb = smem + cur * STAGE + A_B + (wn * NT * 16 + l16) * ROW_B;
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      const int off = ((ks * 4 + lhi) ^ (l16 & 7)) << 4;
      mt_bf8 bf[NT], af[MT];
#pragma unroll
      for (int n = 0; n < NT; ++n)
        bf[n] = *reinterpret_cast<const mt_bf8 *>(bb + n * 16 * ROW_B + off);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        af[m] = *reinterpret_cast<const mt_bf8 *>(ab + m * 16 * ROW_B + off);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              bf[n], af[m], acc[n][m], 0, 0, 0);
    }
    if (BM >= 128) {
      // reads (0x100) between products (0x008): the second half of the
      // rows and the next 32 columns arrive under the products before
      __builtin_amdgcn_sched_group_barrier(0x100, NT + MT / 2, 0);
#pragma unroll
      for (int i = 0; i < MT / 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
#pragma unroll
      for (int i = 0; i < MT / 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, (NT + MT) / (MT / 2), 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NT * MT, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    cur = cur + 1 == ST ? 0 : cur + 1;
    nxt = nxt + 1 == ST ? 0 : nxt + 1;
  }

  // lane: row l16 of each row tile, columns lhi * 4 + r
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int g = g0 + (wm * MT + m) * 16 + l16;
    const int pair = sh ? g : sorted_ids[g];
    if (pair >= (sh ? shared.rows : n_pairs)) continue;
    const float sc = FORM == SCATTER && topk_w && !sh ? topk_w[pair] : 1.f;
    __hip_bfloat16 *crow = C + (long)(FORM == SCATTER ? pair : g) * I;
#pragma unroll
    for (int n = 0; n < NT; n += FORM == GATED ? 2 : 1) {
      const int tile = wn * NT + n;
      const int col = nb * (FORM == GATED ? BN / 2 : BN) +
                      tile * (FORM == GATED ? 8 : 16) + lhi * 4;
      if (col >= I) continue;
      shortx4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = acc[n][m][r];
        if (SUMS) x += sum[SUMS ? n : 0][m][r];
        if (FORM == GATED) {
          float u = acc[n + (NT > 1 ? 1 : 0)][m][r];
          if (ACT == CLAMP) {
            x = fminf(x, limit);
            u = fminf(fmaxf(u, -limit), limit) + 1.f;
            x = x / (1.f + __expf(-alpha * x)) * u;
          } else {
            x = x / (1.f + __expf(-x)) * u;
          }
        } else if (ACT == RELU2) {
          x = fmaxf(x, 0.f);
          x = x * x;
        } else {
          x *= sc;
        }
        o[r] = to_bf16(x);
      }
      *reinterpret_cast<shortx4 *>(crow + col) = o;
    }
  }
}

}  // namespace

// act: 0 none (scatter), 1 silu_glu, 2 clamped swiglu (limit, alpha), 3
// relu^2. block_m: the row block of the tables, 32, 64, 128 or 256.
static void run_tiled(const torch::Tensor &C, const torch::Tensor &A,
                      const torch::Tensor &W, const torch::Tensor &sorted_ids,
                      const torch::Tensor &expert_blocks,
                      const torch::Tensor &n_post_pad,
                      const c10::optional<torch::Tensor> &topk_weights,
                      long n_pairs, long topk, long block_m, long act,
                      double limit, double alpha, Shared shared) {
  TORCH_CHECK(A.scalar_type() == at::kBFloat16 &&
              W.scalar_type() == at::kBFloat16 &&
              C.scalar_type() == at::kBFloat16);
  TORCH_CHECK(A.is_contiguous() && W.is_contiguous() && C.is_contiguous() &&
              W.dim() == 3 && C.dim() == 2);
  const int K = W.size(2), Nd = W.size(1);
  const bool gated = act == SILU || act == CLAMP, scatter = act == NONE;
  const int cols = gated ? Nd / 2 : Nd;
  TORCH_CHECK(A.size(-1) == K && K > 0 && K % BK == 0,
              "moe_gemm_tiled: K must be a multiple of ", BK);
  TORCH_CHECK(cols % 8 == 0 && (!gated || Nd % 2 == 0) && C.size(1) == cols,
              "moe_gemm_tiled: columns must be a multiple of 8");
  for (const auto *p : {&A, &W, &C})
    TORCH_CHECK(reinterpret_cast<uintptr_t>(p->data_ptr()) % 16 == 0);
  const long max_blocks = expert_blocks.numel();
  // rows of the sorted buffer: at most n_pairs and a block less one row of
  // padding per expert (padding rows are read but not used in A and never
  // written in C)
  const long sorted = n_pairs + W.size(0) * (block_m - 1);
  TORCH_CHECK(max_blocks >= (n_pairs + block_m - 1) / block_m && topk >= 1 &&
              sorted_ids.numel() >= sorted);
  TORCH_CHECK(scatter ? C.size(0) >= n_pairs && A.size(0) >= sorted
                      : A.size(0) * topk >= n_pairs && C.size(0) >= sorted);
  const float *tw = nullptr;
  if (topk_weights.has_value()) {
    TORCH_CHECK(topk_weights->scalar_type() == at::kFloat &&
                topk_weights->is_contiguous() &&
                topk_weights->numel() >= n_pairs);
    tw = topk_weights->data_ptr<float>();
  }
  if (block_m == 256 &&
      tile_gemm_grouped_ok(A.numel(), n_pairs, Nd, K, (int)act)) {
    tile_gemm_grouped(C.data_ptr(), A.data_ptr(), W.data_ptr(),
                      sorted_ids.data_ptr<int>(),
                      expert_blocks.data_ptr<int>(),
                      n_post_pad.data_ptr<int>(), tw, max_blocks, n_pairs,
                      topk, Nd, K, A.numel() / K, (int)act, (float)limit,
                      (float)alpha,
                      TileShared{shared.C, shared.A, shared.W, shared.rows,
                                 shared.K, shared.N});
    return;
  }
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(BM, BN, WM, WN, ST, AUX, FORM, ACT, ...)                         \
  do {                                                                       \
    const int nbn = ((FORM == GATED ? 2 * cols : cols) + BN - 1) / BN;       \
    shared.nbm = (shared.rows + BM - 1) / BM;                                \
    shared.nbn = (shared.N + BN - 1) / BN;                                   \
    /* (a die has at most one tile of each kind more than another) */        \
    const long tiles = max_blocks * nbn +                                    \
                       (shared.C ? shared.nbm * shared.nbn + 8L : 0);        \
    hipLaunchKernelGGL(                                                      \
        (moe_tiled_kernel<BM, BN, WM, WN, ST, AUX, FORM, ACT                 \
                          __VA_OPT__(,) __VA_ARGS__>),                       \
        dim3((tiles + 7) / 8 * 8), dim3(WM * WN * 64), 0, stream,            \
        (__hip_bfloat16 *)C.data_ptr(), (const __hip_bfloat16 *)A.data_ptr(),\
        (const __hip_bfloat16 *)W.data_ptr(), sorted_ids.data_ptr<int>(),    \
        expert_blocks.data_ptr<int>(), n_post_pad.data_ptr<int>(), tw,       \
        (int)n_pairs, K, Nd, (int)topk, nbn, (float)limit, (float)alpha,     \
        shared);                                                             \
  } while (0)
#define FORMS(BM, BN, WM, WN, ST, AUX)                                       \
  do {                                                                       \
    if (act == NONE) RUN(BM, BN, WM, WN, ST, AUX, SCATTER, NONE);            \
    else if (act == SILU) RUN(BM, BN, WM, WN, ST, AUX, GATED, SILU);         \
    else if (act == CLAMP) RUN(BM, BN, WM, WN, ST, AUX, GATED, CLAMP);       \
    else if (act == RELU2) RUN(BM, BN, WM, WN, ST, AUX, PLAIN, RELU2);       \
    else TORCH_CHECK(false, "moe_gemm_tiled: act ", act);                    \
  } while (0)
#define WITH(BM, BN, WM, WN, ST, AUX)                                        \
  do {                                                                       \
    if (act == NONE) RUN(BM, BN, WM, WN, ST, AUX, SCATTER, NONE, true);      \
    else RUN(BM, BN, WM, WN, ST, AUX, GATED, SILU, true);                    \
  } while (0)
  if (shared.C && block_m == 32) WITH(32, 128, 1, 4, 4, 2);
  else if (shared.C && block_m == 64) WITH(64, 128, 1, 4, 3, 2);
  else if (shared.C && block_m == 128) WITH(128, 128, 2, 2, 3, 0);
  else if (block_m == 32) FORMS(32, 128, 1, 4, 4, 2);
  else if (block_m == 64) FORMS(64, 128, 1, 4, 3, 2);
  else if (block_m == 128) FORMS(128, 128, 2, 2, 3, 0);
  else if (block_m == 256) FORMS(256, 256, 2, 4, 2, 0);
  else TORCH_CHECK(false, "moe_gemm_tiled: block_m must be 32/64/128/256");
#undef WITH
#undef FORMS
#undef RUN
  HIP_CHECK_KERNEL();
}

void moe_gemm_tiled(torch::Tensor C, torch::Tensor A, torch::Tensor W,
                    torch::Tensor sorted_ids, torch::Tensor expert_blocks,
                    torch::Tensor n_post_pad,
                    c10::optional<torch::Tensor> topk_weights, long n_pairs,
                    long topk, long block_m, long act, double limit,
                    double alpha) {
  run_tiled(C, A, W, sorted_ids, expert_blocks, n_post_pad, topk_weights,
            n_pairs, topk, block_m, act, limit, alpha, Shared{});
}

// moe_gemm_tiled of act 1 or 0 with a shared expert's product beside it:
// silu(gate) * up of all rows for w = gate rows over up rows, [rows, N / 2], or
// rows w^T, [rows, N].
torch::Tensor moe_gemm_tiled_shared(
    torch::Tensor C, torch::Tensor A, torch::Tensor W,
    torch::Tensor sorted_ids, torch::Tensor expert_blocks,
    torch::Tensor n_post_pad, c10::optional<torch::Tensor> topk_weights,
    long n_pairs, long topk, long block_m, long act, torch::Tensor rows,
    torch::Tensor w) {
  TORCH_CHECK(act == NONE || act == SILU);
  TORCH_CHECK(block_m == 32 || block_m == 64 || block_m == 128 ||
              block_m == 256,
              "moe_gemm_tiled_shared: block_m must be 32/64/128/256");
  for (const auto *t : {&rows, &w})
    TORCH_CHECK(t->is_cuda() && t->dim() == 2 && t->is_contiguous() &&
                t->scalar_type() == at::kBFloat16 &&
                reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0,
                "moe_gemm_tiled_shared: 16 B aligned bf16 rows");
  const long T = rows.size(0), K = rows.size(1), N = w.size(0);
  const long cols = act == SILU ? N / 2 : N;
  TORCH_CHECK(w.size(1) == K && K > 0 && K % BK == 0 && cols > 0 &&
              cols % 8 == 0 && (act == NONE || N % 2 == 0) && T > 0 &&
              T < 1L << 20 && N < 1L << 20 && N * K < 1L << 30,
              "moe_gemm_tiled_shared: K a multiple of 64, columns of 8");
  TORCH_CHECK(block_m != 256 ||
              tile_gemm_grouped_ok(A.numel(), n_pairs, W.size(1), W.size(2),
                                   (int)act),
              "moe_gemm_tiled_shared: operands below 2 GiB");
  auto out = torch::empty({T, cols}, rows.options());
  const int slice = act == NONE && T <= 256 ? stream_slice(T, N, K) : 0;
  run_tiled(C, A, W, sorted_ids, expert_blocks, n_post_pad, topk_weights,
            n_pairs, topk, block_m, act, 0.0, 0.0,
            Shared{(__hip_bfloat16 *)out.data_ptr(),
                   (const __hip_bfloat16 *)rows.data_ptr(),
                   (const __hip_bfloat16 *)w.data_ptr(), (int)T, (int)K,
                   (int)N, 0, 0, slice > 0 ? slice : (int)K});
  return out;
}
