// Products of few rows (M <= 256) with a weight matrix: x [M, K] W[N, K]^T,
// bf16 in, fp32 sums (K a multiple of 64).
//
// Bound by the weights' bytes, so the job is to keep them coming: 16 B
// global -> LDS loads (non-temporal: a weight row is used by one workgroup)
// into a ring that holds several 64-column stages in flight, two workgroups
// per CU where LDS allows. LDS rows are 128 B with their 16 B units permuted
// by row & 7, so fragment reads fall on all banks; products are W x^T, so a
// lane ends with four neighbouring columns of one row.
//
// A weight with few tiles is also split along K (parts_plan: into one full
// round of workgroups); the fp32 parts [S, M, N] are then summed by whatever
// comes next, in the order of S:
//   stream_gemm           bias, bf16
//   stream_add_norm       residual += sum, RMS norm of it (attention and
//                         feed-forward outputs)
//   qkv_finish            bias, rotation, keys and values to their cache
//                         slots, queries out
// and a gated feed-forward (gate and up rows of W alternate in the staged
// tile) leaves silu(gate) * up straight from the sums.
// (us against hipBLASLt and against the kernel before this one, which split
// K into up to 16 and summed the parts one load at a time:) 5120 x 27648, 64
// rows 60 for 159 and 79, 256 rows 83 for 266 and 160; 7168 x 5120, 1 row
// 13.5 for 24; 28672 x 4096 gated, 1 row 40 for 61 + 5. Weights come at 4.2
// to 6.6 TB/s from 35 MB on, below that the launch and the ring's first
// stages are most of the time (2048 x 2048: 5 + 3 us). Parts of large weights
// with more than 64 rows (32 if K is long) come from tile_gemm.hip, where 256
// columns share their rows (tile_parts_plan has both sides of the line).

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "fp8_rows.h"
#include "qkv_rows.h"
#include "tile_gemm.h"

typedef __attribute__((ext_vector_type(8))) __bf16 st_bf8;
typedef part_f4 st_f4;

namespace {

constexpr int BK = 64;
constexpr int ROW_B = BK * 2;  // LDS row bytes
constexpr int MAX_SPLIT = 16;

enum Form { GATED = 0, PLAIN = 1, PART = 2 };

// AUX 2: non-temporal
template <int AUX>
DEV_INLINE void glds16(const __hip_bfloat16 *gsrc, char *lds_ptr) {
  __builtin_amdgcn_global_load_lds(
      reinterpret_cast<const unsigned int *>(gsrc),
      reinterpret_cast<unsigned int *>(lds_ptr), 16, 0, AUX);
}

// wait until at most AHEAD stages of LD loads are on their way
template <int AHEAD, int LD>
DEV_INLINE void wait_stages(int ahead) {
  if (ahead >= AHEAD)
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(AHEAD * LD) : "memory");
  else if constexpr (AHEAD > 0)
    wait_stages<AHEAD - 1, LD>(ahead);
}

// WM x WN waves share a BM x BN tile; a ring of ST stages of BK columns
template <int BM, int BN, int WM, int WN, int ST, int FORM>
__global__ __launch_bounds__(WM *WN * 64) void stream_gemm_kernel(
    void *__restrict__ C,  // bf16 [M, N or N / 2], PART: fp32 [S, M, N]
    const __hip_bfloat16 *__restrict__ A, long lda,
    const __hip_bfloat16 *__restrict__ W,  // [N, K]
    const __hip_bfloat16 *__restrict__ bias, int M, int N, int K,
    int k_slice, int nbm, int nbn) {
  constexpr int THREADS = WM * WN * 64;
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int A_B = BM * ROW_B, STAGE = A_B + BN * ROW_B;
  constexpr int A_UNITS = A_B / 1024, B_UNITS = BN * ROW_B / 1024;
  constexpr int WAVES = WM * WN;
  // BM = 16: two waves bring the rows, the other two only weights
  constexpr int AL = (A_UNITS + WAVES - 1) / WAVES;
  constexpr int BL = B_UNITS / WAVES;
  static_assert(BL * WAVES == B_UNITS, "whole loads");
  static_assert(A_UNITS % WAVES == 0 || A_UNITS < WAVES, "whole loads");
  __shared__ __attribute__((aligned(16))) char smem[ST * STAGE];

  // eight dies take workgroups in turn: each gets a contiguous run of tiles,
  // row blocks fastest (they share weights)
  const int total = nbm * nbn;
  const int pid = blockIdx.x, xcd = pid & 7, per = total >> 3;
  const int t = xcd * per + min(xcd, total & 7) + (pid >> 3);
  const int mb = t % nbm, nb = t / nbm;
  const int z = blockIdx.y;
  const int k0 = z * k_slice;
  const int nkt = min(K - k0, k_slice) / BK;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int NC = FORM == GATED ? N >> 1 : N;  // columns of C

  // sources: unit u of 1 KB = 8 rows, lane = row u * 8 + lane / 8
  const int sub = lane >> 3, col = ((lane & 7) ^ sub) * 8;
  const bool a_wave = A_UNITS >= WAVES || wave < A_UNITS;
  const __hip_bfloat16 *asrc[AL], *bsrc[BL];
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    const int row = min((j * WAVES + wave) * 8 + sub, BM - 1);
    asrc[j] = A + (long)min(mb * BM + row, M - 1) * lda + k0 + col;
  }
#pragma unroll
  for (int j = 0; j < BL; ++j) {
    const int row = (j * WAVES + wave) * 8 + sub;
    int n;
    if (FORM == GATED) {  // 16 gate rows, their 16 up rows, the next 16
      const int c = min(nb * (BN / 2) + (row >> 5) * 16 + (row & 15), NC - 1);
      n = (row & 16) ? NC + c : c;
    } else {
      n = min(nb * BN + row, N - 1);
    }
    bsrc[j] = W + (long)n * K + k0 + col;
  }
  auto stage = [&](int slot) {
    char *base = smem + slot * STAGE + wave * 1024;
    if (a_wave) {
#pragma unroll
      for (int j = 0; j < AL; ++j) {
        glds16<0>(asrc[j], base + j * WAVES * 1024);
        asrc[j] += BK;
      }
    }
#pragma unroll
    for (int j = 0; j < BL; ++j) {
      glds16<2>(bsrc[j], base + A_B + j * WAVES * 1024);
      bsrc[j] += BK;
    }
  };
  st_f4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = st_f4{0, 0, 0, 0};

#pragma unroll
  for (int i = 0; i < ST - 1; ++i)
    if (i < nkt) stage(i);
  int cur = 0, nxt = ST - 1;
  for (int kt = 0; kt < nkt; ++kt) {
    // this wave's loads of stage kt have landed, later ones may fly
    const int ahead = min(nkt - 1 - kt, ST - 2);
    if (a_wave) wait_stages<ST - 2, AL + BL>(ahead);
    else wait_stages<ST - 2, BL>(ahead);
    // everybody's are there, and stage kt - 1 (the slot that the next one
    // takes) has been read
    __builtin_amdgcn_s_barrier();
    if (kt + ST - 1 < nkt) stage(nxt);
    const char *ab = smem + cur * STAGE + (wm * MT * 16 + l16) * ROW_B;
    const char *bb = smem + cur * STAGE + A_B + (wn * NT * 16 + l16) * ROW_B;
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      const int off = ((ks * 4 + lhi) ^ (l16 & 7)) << 4;
      st_bf8 bf[NT], af[MT];
#pragma unroll
      for (int n = 0; n < NT; ++n)
        bf[n] = *reinterpret_cast<const st_bf8 *>(bb + n * 16 * ROW_B + off);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        af[m] = *reinterpret_cast<const st_bf8 *>(ab + m * 16 * ROW_B + off);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              bf[n], af[m], acc[n][m], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    cur = cur + 1 == ST ? 0 : cur + 1;
    nxt = nxt + 1 == ST ? 0 : nxt + 1;
  }

  // lane: row l16 of each row tile, columns lhi * 4 + r
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = mb * BM + (wm * MT + m) * 16 + l16;
    if (row >= M) continue;
#pragma unroll
    for (int n = 0; n < NT; n += FORM == GATED ? 2 : 1) {
      const int tile = wn * NT + n;
      const int c = nb * (FORM == GATED ? BN / 2 : BN) +
                    tile * (FORM == GATED ? 8 : 16) + lhi * 4;
      if (c >= NC) continue;
      if (FORM == PART) {
        *reinterpret_cast<st_f4 *>((float *)C + ((long)z * M + row) * N + c) =
            acc[n][m];
        continue;
      }
      shortx4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[n][m][r];
        if (FORM == GATED)
          v = v / (1.f + __expf(-v)) * acc[n + (NT > 1 ? 1 : 0)][m][r];
        else if (bias)
          v += __bfloat162float(bias[c + r]);
        o[r] = to_bf16(v);
      }
      *reinterpret_cast<shortx4 *>((__hip_bfloat16 *)C + (long)row * NC + c) =
          o;
    }
  }
}

template <typename TB>
__global__ __launch_bounds__(256) void stream_sum_kernel(
    __hip_bfloat16 *__restrict__ out, const float *__restrict__ part,
    const TB *__restrict__ bias, long MN, int N, int S) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  st_f4 sum[1];
  part_sums<1>({part + i}, MN, S, sum);
  const st_f4 v = sum[0];
  const int n = i % N;
  shortx4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    o[r] = to_bf16(v[r] + (bias ? ScalarOps<TB>::to_f32(bias[n + r]) : 0.f));
  *reinterpret_cast<shortx4 *>(out + i) = o;
}

// A workgroup per row: residual += sum of the parts (rounded as stored),
// out = RMS norm of the stored residual. V x 4 columns per thread. Bound by
// one chain of memory latencies: with all loads ahead of the sums, and each
// part read once, 64 x 5120 in four parts takes 5.7 us (7.6 with the groups
// of columns in turn), 256 x 5120 in six 10.4 (11.1), 1 x 4096 4.5 (4.8).
// FP8 (N a multiple of 128): the result's e4m3 rows too.
template <int V, typename TW, bool FP8>
__global__ __launch_bounds__(512) void stream_add_norm_kernel(
    __hip_bfloat16 *__restrict__ out, __hip_bfloat16 *__restrict__ residual,
    const float *__restrict__ part, const TW *__restrict__ w, float eps,
    int M, int N, int S, int rounded, const Fp8Out fp8) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  const long MN = (long)M * N;
  // every load goes out before the first sum (columns past the row's end
  // repeat its last four; threads with none of their own load nothing)
  shortx4 old[V] = {};
  float wv[V][4] = {};
  st_f4 v[V] = {};
  if (V > 1 || (int)threadIdx.x * 4 < N) {
    const float *p[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int c = min((j * 512 + (int)threadIdx.x) * 4, N - 4);
      p[j] = part + row * N + c;
      old[j] = *reinterpret_cast<const shortx4 *>(residual + row * N + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) wv[j][r] = ScalarOps<TW>::to_f32(w[c + r]);
    }
    part_sums<V>(p, MN, S, v);
  }
  float x[V][4], ss = 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int c = (j * 512 + threadIdx.x) * 4;
    if (rounded) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[j][r] = bf16_value(v[j][r]);
    }
    shortx4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[r] = to_bf16(v[j][r] + __bfloat162float(__builtin_bit_cast(
                                   __hip_bfloat16, (short)old[j][r])));
      x[j][r] =
          __bfloat162float(__builtin_bit_cast(__hip_bfloat16, (short)o[r]));
      if (c < N) ss += x[j][r] * x[j][r];
    }
    if (c < N)
      *reinterpret_cast<shortx4 *>(residual + row * N + c) = o;
  }
  ss = block_reduce_sum<512>(ss, red);
  const float inv = rsqrtf(ss / N + eps);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int c = (j * 512 + threadIdx.x) * 4;
    if (c >= N) continue;
    shortx4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = to_bf16(x[j][r] * inv * wv[j][r]);
    *reinterpret_cast<shortx4 *>(out + row * N + c) = o;
    if constexpr (FP8) {  // a group is the columns of 32 lanes
      float v8[4], amax = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v8[r] =
            __bfloat162float(__builtin_bit_cast(__hip_bfloat16, (short)o[r]));
        amax = fmaxf(amax, fabsf(v8[r]));
      }
#pragma unroll
      for (int off = 16; off > 0; off >>= 1)
        amax = fmaxf(amax, __shfl_xor(amax, off, 64));
      const float scale = fp8_scale(amax);
      *reinterpret_cast<unsigned *>(fp8.q + row * N + c) =
          fp8_bytes(v8, 1.f / scale);
      if ((threadIdx.x & 31) == 0) fp8.scales[(long)(c >> 7) * M + row] = scale;
    }
  }
}

// Workgroups along the columns of a token, a thread per unit. PARTS: the rows
// are fp32 parts [S, M, N].
template <bool PARTS>
__global__ __launch_bounds__(256) void qkv_finish_kernel(
    __hip_bfloat16 *__restrict__ q_out, __hip_bfloat16 *__restrict__ k_cache,
    __hip_bfloat16 *__restrict__ v_cache, const QkvRows rows,
    const long *__restrict__ slots, int Hq, int Hkv, int D) {
  const long t = blockIdx.x;
  const long slot = slots[t];
  const int i = blockIdx.y * 256 + threadIdx.x, per = D / 8;
  if (i >= (Hq + 2 * Hkv) * per) return;
  const int h = i / per;
  const QkvUnit x =
      qkv_unit<PARTS>(rows, t, h, i % per, h < Hq + Hkv, Hq + 2 * Hkv, D);
  __hip_bfloat16 *dst;
  if (h < Hq) dst = q_out + (t * Hq + h) * D;
  else if (h < Hq + Hkv) dst = k_cache + (slot * Hkv + (h - Hq)) * D;
  else dst = v_cache + (slot * Hkv + (h - Hq - Hkv)) * D;
  *reinterpret_cast<shortx4 *>(dst + x.d1) = x.o1;
  *reinterpret_cast<shortx4 *>(dst + x.d2) = x.o2;
}

// The same of bf16 rows with an RMS norm per query and key head (D at most 128):
// 16 lanes a head, eight columns each; the norm is rounded before the rotation,
// as where it was a kernel of its own. It stands for two copies, two norms, a
// rotation and a scatter: 4096 x 20 heads of 128 38 us by those, 14 so.
template <typename TW>
__global__ __launch_bounds__(256) void qkv_norm_kernel(
    __hip_bfloat16 *__restrict__ q_out, __hip_bfloat16 *__restrict__ k_cache,
    __hip_bfloat16 *__restrict__ v_cache,
    const __hip_bfloat16 *__restrict__ src, long stride,
    const TW *__restrict__ q_w, const TW *__restrict__ k_w, float eps,
    const long *__restrict__ positions, const float *__restrict__ cos_sin,
    int rot, const long *__restrict__ slots, int Hq, int Hkv, int D) {
  const long t = blockIdx.x;
  const int h = blockIdx.y * 16 + threadIdx.x / 16, i = threadIdx.x & 15;
  const bool used = h < Hq + 2 * Hkv && i * 8 < D;
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  shortx8 row = {};
  if (used)
    row = *reinterpret_cast<const shortx8 *>(src + t * stride + h * D + i * 8);
  const bool turned = h < Hq + Hkv;
  if (turned) {  // (the same for a head's 16 lanes)
    unpack8<__hip_bfloat16>(row, v);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += v[j] * v[j];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float inv = rsqrtf(ss / D + eps);
    float w[8] = {0, 0, 0, 0, 0, 0, 0, 0}, other[8];
    if (used) ld8<TW>((h < Hq ? q_w : k_w) + i * 8, w);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf16_value(v[j] * inv * w[j]);
    const int half = rot / 16;  // in lanes
    const int mate = i < half ? i + half : i < 2 * half ? i - half : i;
#pragma unroll
    for (int j = 0; j < 8; ++j) other[j] = __shfl(v[j], mate, 16);
    if (i < 2 * half) {
      const float *cs = cos_sin + positions[t] * rot + min(i, mate) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = cs[j], s = cs[rot / 2 + j];
        const float x1 = i < half ? v[j] : other[j];
        const float x2 = i < half ? other[j] : v[j];
        v[j] = i < half ? x1 * c - x2 * s : x2 * c + x1 * s;
      }
    }
    row = pack8<__hip_bfloat16>(v);
  }
  if (!used) return;
  __hip_bfloat16 *dst;
  if (h < Hq) dst = q_out + (t * Hq + h) * D;
  else if (turned) dst = k_cache + (slots[t] * Hkv + (h - Hq)) * D;
  else dst = v_cache + (slots[t] * Hkv + (h - Hq - Hkv)) * D;
  *reinterpret_cast<shortx8 *>(dst + i * 8) = row;
}

bool aligned16(const torch::Tensor &t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct Plan {
  int bm, bn, nbm, nbn, splits, k_slice;
};

// How full `slots` workgroups are with `tiles`, each split where they fit
// more than once.
double fill_of(int tiles, int slots) {
  const int rounds = (tiles + slots - 1) / slots;
  return tiles <= slots ? (double)(slots / tiles * tiles) / slots
                        : (double)tiles / (rounds * slots);
}

int compute_units() {
  return at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
}

Plan finish(Plan p, int M, int N, int K, int splits) {
  const int stages = K / BK, per = (stages + splits - 1) / splits;
  p.nbm = (M + p.bm - 1) / p.bm;
  p.nbn = (N + p.bn - 1) / p.bn;
  p.k_slice = per * BK;
  p.splits = (stages + per - 1) / per;
  return p;
}

// Rows 4 KB apart, and parts whose shares are, meet in the same channels of
// memory: there fewer and narrower streams are the faster ones (us, four parts
// of K 8192 / three: 64 x 8192 x 8192 39.9 / 33.6, 64 x 7168 x 8192 35.2 /
// 32.5; two 64-column tiles a CU against one of 128, rows 8 KB apart: 48 x
// 28672 x 4096 gated 46 / 49, 10 KB apart 66 / 57).
bool far_apart(int values) { return values % 2048 == 0; }

// From here on 64-column tiles of up to 64 rows are not left whole (17 x 16384
// x 14336 92, in two parts 76; 32 x 14336 x 11008 whole 65, 72).
constexpr int DEEP = 12288;

// Gated products are not split: the width whose tiles fill whole rounds of
// workgroups (us). 64 columns with a tile a CU and no more (64 x 16384 x 3584
// 23, 128 columns 33; 128 x 16384 x 2048 20, 25), then 128 until 64 nearly fill
// two (64 x 22016 x 4096 44.5, 128 columns 38.2; 128 x 28672 x 4096 60, 50; 33
// x 28672 x 4096 44, 48), 256 from 36000 columns on. Up to 16 rows 128 there,
// 256 from 48000 unless rows are 4 KB apart (1 x 55296 x 5120 100 / 95, 1 x
// 43008 x 4096 70 / 74, 1 x 57344 x 4096 81 / 97, 64 columns 87).
Plan gated_plan(int M, int N, int K) {
  const int cus = compute_units(), tiles64 = (N + 63) / 64;
  const double fill = fill_of(tiles64, 2 * cus);
  const bool far = far_apart(K);
  Plan p;
  p.bm = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
  p.bn = 64;
  if (M <= 64) {
    const double full = p.bm == 64 ? (far ? 0.85 : 0.9) : far ? 0.74 : 0.8;
    const bool even =
        fill >= full || (M <= 16 && tiles64 <= 2 * cus && K < 4096);
    if (N >= 36000)
      p.bn = p.bm > 16 || (N >= 48000 && !far) ? 256 : 128;
    else if (tiles64 >= cus && tiles64 <= 2 * cus && !even)
      p.bn = 128;
  } else if (M <= 128) {
    p.bm = N >= 8192 ? 128 : 64;
    p.bn = N >= 36000 ? 256
           : tiles64 > cus && tiles64 <= 2 * cus ? 128 : 64;
  } else {
    p.bm = K >= 2 * N || N >= 16384 ? 256 : 128;
    p.bn = p.bm == 128 ? 64 : N >= 36000 ? 256 : 128;
  }
  return finish(p, M, N, K, 1);
}

// Products that may be split: in one round of a workgroup a CU, all there from
// the start, along K into as many parts as fit that round. Rounding up instead
// (to about 384 workgroups of 64 columns) left a second round nearly empty or
// half the CUs with twice the work, and a second workgroup a CU doubles the
// parts and brings no weight sooner. us in turn over weights that no cache
// holds, with the norm or the bias behind them:
//  * parts, rounded up / two a CU / one a CU: 1 x 5120 x 5120 17.1 / 15.8 /
//    14.4, 16 x 2560 x 8192 16.2 / 16.4 / 14.0, 1 x 4608 x 14336 29.5 / 28.0 /
//    26.3. Up to 16 rows take two where one leaves three tenths of the CUs
//    idle (16 x 18432 x 14336 in one part 118, in three 97).
//  * up to 64 rows: 64 columns below 20 M values (6 M for 16 rows; 64 x 4096 x
//    4096 16.7 / 13.6, 32 x 3648 x 2048 9.3 / 8.0, 64 x 2560 x 2560 13.3 /
//    10.9), where the most parts of 128 would leave a quarter of the CUs idle
//    (32 x 768 x 27648 128 columns 19.3, 64 14.4), and where they fill a round
//    of two a CU unsplit (32064 x 4096). Else 128 (1 x 6144 x 4096 11.8 / 10.0,
//    64 x 5120 x 5120 23.2 / 20.2, 64 x 4096 x 14336 36.5 / 28.7), or 256 where
//    they fill the chip better by a tenth (64 x 19008 x 5120 60 / 44). Beyond a
//    round of two a CU 64 up to 16 rows (1 x 38016 x 4096 128 columns 71, 64
//    59), else 256 (64 x 64128 x 5120 64 columns 140, 256 105).
//  * up to 128 rows 128 x 128 from 20 M values on, one row block in place of
//    two of 64: 128 x 6144 x 4096 21.6 / 16.4. Below, two row blocks of 64 x
//    64 where they fill six tenths of the CUs (128 x 2048 x 2048 12.9 / 10.4,
//    128 x 5120 x 2048 15.2 / 12.1, 128 x 3648 x 2048 13.8 / 11.5), else 128 x
//    64: 128 x 4608 x 3584 at 144 tiles 13.7, 64 x 64 over 15.
//  * up to 256 rows, narrow: below 12 M values 64 x 64 where they fill two
//    thirds of the CUs (256 x 2048 x 2048 14.3 / 12.4, 160 x 3648 x 2048 15.1 /
//    11.9), else 128 x 64 (256 x 2560 x 2048 9.8 / 8.9); above 128 x 128, but
//    256 x 128 for few columns and long K (136 x 1536 x 14336 29.0 / 24.2).
//    Rounding up stays for 256 x 128 tiles (160 x 19008 x 5120 58; unsplit 74).
// From 16384 columns on the router has the library for more than 64 rows; only
// a caller of the kernel itself gets there. A part has four stages at least on
// average; the last may be shorter (17 stages: 5, 5, 5, 2).
Plan parts_plan(int M, int N, int K) {
  const int cus = compute_units(), stages = K / BK;
  const long weights = (long)N * K;
  const int tiles64 = (N + 63) / 64, tiles128 = (N + 127) / 128;
  Plan p;
  p.bm = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
  p.bn = 64;
  if (M <= 64) {
    const bool even = tiles64 >= cus && tiles64 <= 2 * cus && K < DEEP &&
                      (fill_of(tiles64, 2 * cus) >=
                           (far_apart(K) ? 0.74 : 0.9) ||
                       (M <= 16 && K < 4096));
    const bool small = weights < (p.bm == 16 ? 6L << 20 : 20L << 20) ||
                       tiles128 * MAX_SPLIT < cus * 3 / 4;
    if (tiles64 > 2 * cus) {
      p.bn = p.bm == 16 ? 64 : 256;
    } else if (!small && !even) {
      p.bn = 128;
      if (p.bm > 16 && N >= 8192 &&
          fill_of((N + 255) / 256, cus) > fill_of(tiles128, cus) + 0.1)
        p.bn = 256;
    }
  } else if (M <= 128) {
    p.bn = N >= 36000 ? 256 : weights >= (20L << 20) ? 128 : 64;
    if (p.bn == 64 && tiles64 <= cus / 2 && fill_of(2 * tiles64, cus) >= 0.6)
      p.bm = 64;
  } else if (N >= 16384 || (K >= 2 * N && N >= 5120) ||
             (M <= 192 && K >= 5 * N && N > 1024 && N <= 2048)) {
    p.bm = 256;
    p.bn = 128;
  } else if (N < 5120) {
    const int tiles = (M + 63) / 64 * tiles64;
    if (weights >= (12L << 20)) p.bn = 128;
    else if (tiles <= cus && fill_of(tiles, cus) >= 0.65) p.bm = 64;
  }
  const int tiles = (M + p.bm - 1) / p.bm * ((N + p.bn - 1) / p.bn);
  int s = cus / tiles;
  if (M <= 16 && s > 0 && fill_of(tiles, cus) < 0.7) s = 2 * cus / tiles;
  if (p.bm == 256 && tiles < 160) s = (384 + tiles - 1) / tiles;
  s = std::max(1, std::min(std::min(s, MAX_SPLIT), stages / 4));
  if (M <= 64 && s > 2 && far_apart((stages + s - 1) / s * BK)) --s;
  return finish(p, M, N, K, s);
}

// The plain product in one launch, 64 columns a tile, where that is quicker
// than the parts and the launch that sums them; else no splits. Both sides from
// what a stage, the weight's bytes and the parts' take (us, parts / one launch:
// 64 x 12288 x 4096 29.6 / 25.0, 64 x 12288 x 2048 22.4 / 14.3, 16 x 16384 x
// 1024 12.1 / 7.7, 128 x 7168 x 4096 25.8 / 22.4; the other way, 128 x 64 tiles
// unsplit against parts of tile_gemm.hip: 192 x 8192 x 14336 112 / 68, 256 x
// 7168 x 11008 81 / 66). Over 3682 sizes (up to 256 rows, 512 to 38016 columns,
// K of 512 to 27648) it takes 0.89 of what rounding up took, which left 160
// tiles of 64 columns and more whole, and is behind it by more than 8 % in
// nine.
Plan plain_plan(int M, int N, int K, int parts, bool tiled) {
  const int cus = compute_units();
  const double bytes = 2e-6 * N * K, sums = 8e-6 * parts * M * N;  // MB
  // us beside what both take
  const double split = tiled ? bytes / 5.5 + sums / 6 + 8
                             : bytes / 6 + sums / (M <= 64 ? 4 : 3) + 2.5;
  Plan p;
  p.bm = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 || (M <= 128 && N < 8192) ? 64
                                                                       : 128;
  p.bn = 64;
  p = finish(p, M, N, K, 1);
  // a stage with a tile a CU, and with two
  const int tiles = p.nbm * p.nbn;
  const double few = p.bm == 16 ? 0.2 : p.bm == 32 ? 0.24 : 0.27;
  const double one = M <= 64 ? few + 0.1 * tiles / cus
                     : p.bm == 64 ? 0.31 : tiled && M <= 128 ? 0.52 : 0.46;
  const double two = p.bm == 16 ? 0.6 : p.bm == 32 ? 0.65
                     : p.bm == 64 ? 0.68 : M > 128 ? 0.8 : 0.92;
  const double stage =
      tiles <= cus ? one : two * std::max(1.0, tiles / (2.0 * cus));
  if ((M <= 64 && K >= DEEP) || K / BK * stage >= split) p.splits = 0;
  return p;
}

void check_operands(const torch::Tensor &x, const torch::Tensor &w) {
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16 && x.dim() == 2 &&
              w.dim() == 2 && x.size(1) == w.size(1));
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
              w.is_contiguous() && aligned16(x) && aligned16(w),
              "stream_gemm: 16 B aligned rows");
  TORCH_CHECK(w.size(1) % BK == 0 && w.size(1) > 0 && w.size(0) % 8 == 0,
              "stream_gemm: K a multiple of 64, N of 8");
  TORCH_CHECK(x.size(0) <= 256, "stream_gemm: at most 256 rows");
}

template <int FORM>
void launch(const Plan &p, void *C, const torch::Tensor &x,
            const torch::Tensor &w, const void *bias) {
  const int M = x.size(0), N = w.size(0), K = w.size(1);
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(BM, BN, WM, WN, ST)                                              \
  hipLaunchKernelGGL((stream_gemm_kernel<BM, BN, WM, WN, ST, FORM>),         \
                     dim3(p.nbm * p.nbn, p.splits), dim3((WM) * (WN) * 64),  \
                     0, stream, C, (const __hip_bfloat16 *)x.data_ptr(),     \
                     x.size(0) > 1 ? (long)x.stride(0) : 0L,                 \
                     (const __hip_bfloat16 *)w.data_ptr(),                   \
                     (const __hip_bfloat16 *)bias, M, N, K, p.k_slice,       \
                     p.nbm, p.nbn)
  // (a wave needs a gate and an up tile, so 16 columns are too few; the last
  // figure is the ring, as deep as one or two workgroups a CU leave room for)
  if (p.bm == 16 && p.bn == 64) RUN(16, 64, 1, FORM == GATED ? 2 : 4, 8);
  else if (p.bm == 16 && p.bn == 128) RUN(16, 128, 1, 4, 4);
  else if (p.bm == 32 && p.bn == 64) RUN(32, 64, 1, 2, 6);
  else if (p.bm == 32 && p.bn == 128 && FORM == GATED) RUN(32, 128, 1, 4, 4);
  else if (p.bm == 32 && p.bn == 128) RUN(32, 128, 1, 4, 7);
  else if (p.bm == 32) RUN(32, 256, 1, 8, 4);
  else if (p.bm == 64 && p.bn == 64) RUN(64, 64, 2, 2, 5);
  else if (p.bm == 64 && p.bn == 128) RUN(64, 128, 2, 4, 6);
  else if (p.bm == 64) RUN(64, 256, 2, 4, 4);
  else if (p.bm == 128 && p.bn == 64 && (FORM == GATED || x.size(0) > 128))
    RUN(128, 64, 2, 2, 3);
  else if (p.bm == 128 && p.bn == 64) {
    if constexpr (FORM != GATED) RUN(128, 64, 2, 4, 6);
  } else if (p.bm == 128 && p.bn == 128) RUN(128, 128, 2, 4, 5);
  else if (p.bm == 128) RUN(128, 256, 2, 4, 3);
  else if (p.bm == 256 && p.bn == 128) RUN(256, 128, 4, 2, 3);
  else if constexpr (FORM == GATED) {
    if (p.bm == 16) RUN(16, 256, 1, 8, 4);
    else RUN(256, 256, 2, 4, 2);
  }
  else TORCH_CHECK(false, "stream_gemm: no such tile");
#undef RUN
  HIP_CHECK_KERNEL();
}

const void *bias_ptr(const c10::optional<torch::Tensor> &bias, long N) {
  if (!bias.has_value()) return nullptr;
  TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() &&
              bias->numel() == N, "bias: bf16 [N]");
  return bias->data_ptr();
}

}  // namespace

// the fp32 parts [S, M, N] of x w^T
torch::Tensor stream_parts(torch::Tensor x, torch::Tensor w) {
  check_operands(x, w);
  const long M = x.size(0), N = w.size(0);
  TORCH_CHECK(M > 0);
  int bm, splits;
  tile_parts_plan(M, N, w.size(1), &bm, &splits);
  if (splits > 0 && x.is_contiguous()) {
    auto part = torch::empty({(long)splits, M, N},
                             x.options().dtype(at::kFloat));
    tile_parts(part.data_ptr<float>(), x.data_ptr(), w.data_ptr(), M, N,
               w.size(1), bm, splits);
    return part;
  }
  const Plan p = parts_plan(M, N, w.size(1));
  auto part = torch::empty({(long)p.splits, M, N},
                           x.options().dtype(at::kFloat));
  launch<PART>(p, part.data_ptr(), x, w, nullptr);
  return part;
}

// bf16 sum of fp32 parts [S, M, N] (N a multiple of 8) and a bias (bf16 or
// fp32)
torch::Tensor parts_sum(torch::Tensor part,
                        c10::optional<torch::Tensor> bias) {
  TORCH_CHECK(part.is_cuda() && part.dim() == 3 && part.is_contiguous() &&
              part.scalar_type() == at::kFloat && part.size(2) % 8 == 0 &&
              aligned16(part));
  const int S = part.size(0);
  const long M = part.size(1), N = part.size(2);
  auto out = torch::empty({M, N}, part.options().dtype(at::kBFloat16));
  if (M * N == 0) return out;
  const bool wide = bias.has_value() && bias->scalar_type() == at::kFloat;
  TORCH_CHECK(!wide || (bias->is_contiguous() && bias->numel() == N));
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(TB, BP)                                                          \
  hipLaunchKernelGGL((stream_sum_kernel<TB>), dim3((M * N / 4 + 255) / 256), \
                     dim3(256), 0, stream, (__hip_bfloat16 *)out.data_ptr(), \
                     part.data_ptr<float>(), (const TB *)(BP), M * N,        \
                     (int)N, S)
  if (wide) RUN(float, bias->data_ptr());
  else RUN(__hip_bfloat16, bias_ptr(bias, N));
#undef RUN
  HIP_CHECK_KERNEL();
  return out;
}

// How the plain product is formed: -1 by one launch of plan p, else by parts, of
// tile_gemm.hip (their number) or of p (0).
static int in_parts(int M, int N, int K, bool contiguous, Plan *p) {
  int bm, tiled = 0;
  *p = parts_plan(M, N, K);
  if (contiguous) tile_parts_plan(M, N, K, &bm, &tiled);
  if (tiled > 0 || p->splits > 1) {
    const Plan one =
        plain_plan(M, N, K, tiled > 0 ? tiled : p->splits, tiled > 0);
    if (one.splits == 0) return tiled;
    *p = one;
  }
  return -1;
}

long stream_slice(long M, long N, long K) {
  TORCH_CHECK(M > 0 && M <= 256 && N > 0 && N < 1L << 20 && K > 0 &&
              K % BK == 0 && K < 1L << 31, "stream_slice: no such product");
  Plan p;
  const int parts = in_parts(M, N, K, true, &p);
  return parts < 0 ? K : parts > 0 ? 0 : p.k_slice;
}

torch::Tensor stream_gemm(torch::Tensor x, torch::Tensor w,
                          c10::optional<torch::Tensor> bias) {
  check_operands(x, w);
  const long M = x.size(0), N = w.size(0);
  const void *bp = bias_ptr(bias, N);
  auto out = torch::empty({M, N}, x.options());
  if (M == 0) return out;
  Plan p;
  if (in_parts(M, N, w.size(1), x.is_contiguous(), &p) >= 0)
    return parts_sum(stream_parts(x, w), bias);
  launch<PLAIN>(p, out.data_ptr(), x, w, bp);
  return out;
}

// silu(x w_gate^T) * (x w_up^T), w = gate rows, up rows
torch::Tensor stream_gemm_gated(torch::Tensor x, torch::Tensor w) {
  check_operands(x, w);
  const long M = x.size(0), N = w.size(0);
  TORCH_CHECK(N % 16 == 0);
  auto out = torch::empty({M, N / 2}, x.options());
  if (M == 0) return out;
  launch<GATED>(gated_plan(M, N, w.size(1)), out.data_ptr(), x, w,
                nullptr);
  return out;
}

// residual (bf16 [M, N], in place) += the sum of the fp32 parts [S, M, N]
// (rounded: rounded to bf16 first); returns its RMS norm
static torch::Tensor add_norm(torch::Tensor part, torch::Tensor residual,
                              torch::Tensor norm_w, double eps, bool rounded,
                              const Fp8Out &fp8) {
  TORCH_CHECK(part.is_cuda() && part.dim() == 3 && part.is_contiguous() &&
              part.scalar_type() == at::kFloat && part.size(2) % 8 == 0 &&
              aligned16(part));
  const int S = part.size(0), M = part.size(1), N = part.size(2);
  TORCH_CHECK(residual.scalar_type() == at::kBFloat16 &&
              residual.is_contiguous() && residual.numel() == (long)M * N &&
              aligned16(residual));
  TORCH_CHECK(norm_w.is_contiguous() && norm_w.numel() == N &&
              N <= 512 * 4 * 4, "stream_add_norm: at most 8192 columns");
  auto out = torch::empty({(long)M, (long)N}, residual.options());
  if (M == 0) return out;
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(V, TW, FP8)                                                      \
  hipLaunchKernelGGL((stream_add_norm_kernel<V, TW, FP8>), dim3(M),          \
                     dim3(512), 0, stream, (__hip_bfloat16 *)out.data_ptr(), \
                     (__hip_bfloat16 *)residual.data_ptr(),                  \
                     part.data_ptr<float>(), (const TW *)norm_w.data_ptr(),  \
                     (float)eps, M, N, S, (int)rounded, fp8)
#define COLS(TW, FP8)                                                        \
  do {                                                                       \
    if (N <= 2048) RUN(1, TW, FP8);                                          \
    else if (N <= 4096) RUN(2, TW, FP8);                                     \
    else if (N <= 6144) RUN(3, TW, FP8);                                     \
    else RUN(4, TW, FP8);                                                    \
  } while (0)
#define WEIGHTS(TW)                                                          \
  do {                                                                       \
    if (fp8.q) COLS(TW, true);                                               \
    else COLS(TW, false);                                                    \
  } while (0)
  if (norm_w.scalar_type() == at::kFloat) WEIGHTS(float);
  else if (norm_w.scalar_type() == at::kBFloat16) WEIGHTS(__hip_bfloat16);
  else TORCH_CHECK(false, "norm_w: fp32 or bf16");
#undef WEIGHTS
#undef COLS
#undef RUN
  HIP_CHECK_KERNEL();
  return out;
}

torch::Tensor parts_add_norm(torch::Tensor part, torch::Tensor residual,
                             torch::Tensor norm_w, double eps,
                             bool rounded) {
  return add_norm(part, residual, norm_w, eps, rounded, Fp8Out{});
}

// ... with its e4m3 rows (N a multiple of 128): {bf16, bytes, scales}
std::vector<torch::Tensor> parts_add_norm_fp8(torch::Tensor part,
                                              torch::Tensor residual,
                                              torch::Tensor norm_w,
                                              double eps, bool rounded) {
  TORCH_CHECK(part.is_cuda() && part.dim() == 3 && part.size(2) % 128 == 0,
              "parts_add_norm_fp8: columns a multiple of 128");
  const long M = part.size(1), N = part.size(2);
  auto q = torch::empty({M, N}, part.options().dtype(at::kByte));
  auto st = torch::empty({N / 128, M}, part.options());
  auto out = add_norm(part, residual, norm_w, eps, rounded,
                      Fp8Out{q.data_ptr<unsigned char>(),
                             st.data_ptr<float>()});
  return {out, q, st};
}

// residual (bf16 [M, N], in place) += x w^T; returns its RMS norm
torch::Tensor stream_add_norm(torch::Tensor x, torch::Tensor w,
                              torch::Tensor residual, torch::Tensor norm_w,
                              double eps) {
  return parts_add_norm(stream_parts(x, w), residual, norm_w, eps, false);
}

// src: bf16 rows [M, (Hq + 2 Hkv) D] (a row view is fine) or the fp32 parts
// of the same (rounded: rounded to bf16, with the bias, first). Rotates (rotate-half on the first `rot` dims) queries and
// keys, writes keys and values to their slots, returns the queries.
torch::Tensor qkv_finish(torch::Tensor src, c10::optional<torch::Tensor> bias,
                         torch::Tensor positions, torch::Tensor cos_sin,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor slots, long Hq, bool rounded) {
  const bool parts = src.dim() == 3;
  const long M = src.size(parts ? 1 : 0), N = src.size(parts ? 2 : 1);
  const int Hkv = k_cache.size(2), D = k_cache.size(3);
  const int rot = cos_sin.size(-1);
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.is_contiguous() &&
              v_cache.is_contiguous() && v_cache.sizes() == k_cache.sizes() &&
              k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16 && aligned16(k_cache) &&
              aligned16(v_cache));
  TORCH_CHECK(N == (Hq + 2L * Hkv) * D && D % 8 == 0 && rot % 8 == 0 &&
              rot <= D && Hq > 0);
  TORCH_CHECK(src.is_cuda() && aligned16(src) &&
              (parts ? src.is_contiguous() &&
                           src.scalar_type() == at::kFloat
                     : src.scalar_type() == at::kBFloat16 &&
                           src.stride(1) == 1 && src.stride(0) % 8 == 0));
  TORCH_CHECK(positions.scalar_type() == at::kLong &&
              positions.is_contiguous() && positions.numel() == M &&
              slots.scalar_type() == at::kLong && slots.is_contiguous() &&
              slots.numel() == M);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat &&
              cos_sin.is_contiguous());
  const void *bp = bias_ptr(bias, N);
  auto q = torch::empty({M, Hq * D}, k_cache.options());
  if (M == 0) return q;
  auto stream = at::cuda::getCurrentCUDAStream();
  const QkvRows rows{src.data_ptr(),
                     parts ? 0L : (long)src.stride(0),
                     (const __hip_bfloat16 *)bp,
                     positions.data_ptr<long>(),
                     cos_sin.data_ptr<float>(),
                     (int)M,
                     parts ? (int)src.size(0) : 1,
                     rot,
                     (int)rounded};
#define RUN(P)                                                               \
  hipLaunchKernelGGL((qkv_finish_kernel<P>),                                 \
                     dim3(M, (N / 8 + 255) / 256), dim3(256), 0, stream,     \
                     (__hip_bfloat16 *)q.data_ptr(),                         \
                     (__hip_bfloat16 *)k_cache.data_ptr(),                   \
                     (__hip_bfloat16 *)v_cache.data_ptr(), rows,             \
                     slots.data_ptr<long>(), (int)Hq, Hkv, D)
  if (parts) RUN(true); else RUN(false);
#undef RUN
  HIP_CHECK_KERNEL();
  return q;
}

// qkv_finish of bf16 rows, which hold the bias already, with an RMS norm of each
// query and key head in front of the rotation
torch::Tensor qkv_norm_finish(torch::Tensor src, torch::Tensor q_w,
                              torch::Tensor k_w, double eps,
                              torch::Tensor positions, torch::Tensor cos_sin,
                              torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor slots, long Hq) {
  const long M = src.size(0);
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.is_contiguous() &&
              v_cache.is_contiguous() && v_cache.sizes() == k_cache.sizes() &&
              k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16 && aligned16(k_cache) &&
              aligned16(v_cache));
  const int Hkv = k_cache.size(2), D = k_cache.size(3);
  const int rot = cos_sin.size(-1);
  TORCH_CHECK(src.is_cuda() && src.dim() == 2 && aligned16(src) &&
              src.scalar_type() == at::kBFloat16 && src.stride(1) == 1 &&
              src.stride(0) % 8 == 0 && src.size(1) == (Hq + 2L * Hkv) * D &&
              Hq > 0 && M < 1L << 31);
  TORCH_CHECK(D % 8 == 0 && D <= 128 && rot % 16 == 0 && rot <= D,
              "qkv_norm_finish: heads of at most 128, turned by 16s");
  for (const auto *w : {&q_w, &k_w})
    TORCH_CHECK(w->is_contiguous() && w->numel() == D && aligned16(*w) &&
                w->scalar_type() == q_w.scalar_type());
  TORCH_CHECK(positions.scalar_type() == at::kLong &&
              positions.is_contiguous() && positions.numel() == M &&
              slots.scalar_type() == at::kLong && slots.is_contiguous() &&
              slots.numel() == M);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat &&
              cos_sin.is_contiguous());
  auto q = torch::empty({M, Hq * D}, k_cache.options());
  if (M == 0) return q;
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(TW)                                                              \
  hipLaunchKernelGGL((qkv_norm_kernel<TW>),                                  \
                     dim3(M, (Hq + 2 * Hkv + 15) / 16), dim3(256), 0, stream, \
                     (__hip_bfloat16 *)q.data_ptr(),                         \
                     (__hip_bfloat16 *)k_cache.data_ptr(),                   \
                     (__hip_bfloat16 *)v_cache.data_ptr(),                   \
                     (const __hip_bfloat16 *)src.data_ptr(),                 \
                     (long)src.stride(0), (const TW *)q_w.data_ptr(),        \
                     (const TW *)k_w.data_ptr(), (float)eps,                 \
                     positions.data_ptr<long>(), cos_sin.data_ptr<float>(),  \
                     rot, slots.data_ptr<long>(), (int)Hq, Hkv, D)
  if (q_w.scalar_type() == at::kFloat) RUN(float);
  else if (q_w.scalar_type() == at::kBFloat16) RUN(__hip_bfloat16);
  else TORCH_CHECK(false, "norms: fp32 or bf16");
#undef RUN
  HIP_CHECK_KERNEL();
  return q;
}
