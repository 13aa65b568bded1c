// Absorbed-MLA paged attention for gfx950 (DeepSeek V2/V3/V3.2 family).
//
// Semantics parity: the reference's MLA decode backends + chunked-context
// prefill (reference layers/attention.py:366-446,653-925) collapse into
// ONE varlen kernel here. The absorbed latent cache holds a single
// shared row per token [c_kv (512) | k_pe (64)] = 576 dims; attention is
// MQA: every q head attends the same K row, and V is the first 512 dims
// of that row (zero-copy view — each KV byte is read exactly once for
// ALL heads, and the PV B-fragments read straight out of the K tile).
//
// MI355X-native design: a (token, head) pair is a GEMM row; the causal mask
// depends only on the row's token, so one kernel serves decode, chunked
// prefill, prefix hits and mixed batches. Decode splits the keys over
// blockIdx.z with an fp32 LSE merge.
//
// A key tile sits in LDS once, as nine column blocks of [keys][128 B] whose 16
// B units are permuted by key & 7 (the layout both reads below want), in a
// ring of two filled by global_load_lds while the other tile is worked on.
// Scores are K Q^T and the output is O^T = V^T P^T, so a lane holds keys, then
// dims, of ONE row; V is read transposed out of the key tile
// (ds_read_tr16_b64).
//  * up to 16 rows and more workgroups than CUs (decode): mla_decode_kernel,
//    bound by memory.
//  * else a workgroup of four waves takes R row tiles of 16 and walks tiles of
//    64 keys (147 KB: one workgroup per CU). R = 1 (up to 16 rows): wave w
//    scores keys 16 w .. + 15, the row maxima and the weights pass through LDS,
//    then wave w owns dims 128 w .. + 127 of the output. R = 4 (prompts, more
//    heads): wave w scores row tile w against all 64 keys; the output is split
//    by dims as well, so V is read once for 64 rows instead of once per row
//    tile. Bound by LDS reads (K 295 KB + V 64 KB + P 32 KB a tile against 2176
//    cycles of products).
// 128 requests of 16 heads at 512 to 1536 keys (151 MB), us: element by
// element and in one split 282; in tiles of 64 keys, one workgroup per CU, 52
// + 6; of 32 keys, two per CU, 37 + 6. Prompts of 4096 tokens in four, 16
// heads: 257 (535 element by element).
// 512 workgroups as the aim of the splits: twice the CUs, so that all are on
// the chip at once.

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mfma_bf8;
typedef __attribute__((ext_vector_type(4))) float mfma_f4;

namespace {

typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int BLOCK = 256;    // 4 waves
constexpr int BKV = 64;       // keys of a tile
constexpr int DK = 576;       // latent dims (kv_lora 512 + rope 64)
constexpr int DV = 512;
constexpr int KT = DK / 32;   // score k-steps (18)
constexpr int NT = DV / 4 / 16;  // 16-dim output tiles of a wave (8)
constexpr int ROW_B = DK * 2;
constexpr int CB = ROW_B / 128;  // column blocks (9)
constexpr int CB_B = BKV * 128;
constexpr int TILE_B = CB * CB_B;
constexpr int P_ROW = BKV * 2 + 16;  // bytes of a weight row
constexpr float LOG2E = 1.4426950408889634f;
constexpr int SPLIT_TARGET = 512;  // workgroups that a decode batch aims at

union MlaFrag {
  mfma_bf8 v;
  shortx4 h[2];
};

DEV_INLINE short bf16_bits(float v) {
  return __builtin_bit_cast(short, __float2bfloat16(v));
}

// LDS writes of all waves are visible; loads to LDS stay in flight
DEV_INLINE void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int R, bool SPLIT>
__global__ __launch_bounds__(BLOCK, 1) void mla_attention_kernel(
    __hip_bfloat16 *__restrict__ out,      // [T, H, DV] (SPLIT: unused)
    float *__restrict__ partial_out,       // [S, TH, DV] (SPLIT only)
    float *__restrict__ partial_lse,       // [S, TH]
    const __hip_bfloat16 *__restrict__ q,  // [T, H, DK] contiguous
    const __hip_bfloat16 *__restrict__ kc, // [P, ps, 1, DK]
    const int *__restrict__ block_table,   // [B, max_pages]
    const int *__restrict__ seq_lens,      // [B]
    const int *__restrict__ qsl,           // [B+1]
    int max_pages, int page_size, int H, float scale, int num_splits,
    long th_total) {
  constexpr int BQ = R * 16;
  constexpr int NF = R == 1 ? 1 : 4;  // score fragments of a wave
  // the last row tiles see the most keys: they start first
  const int tile = gridDim.x - 1 - blockIdx.x;
  const int b = blockIdx.y;
  const int split = blockIdx.z;
  const int q_start = qsl[b];
  const int q_len = qsl[b + 1] - q_start;
  const int rows = q_len * H;
  if (tile * BQ >= rows) return;
  const int seq_len = seq_lens[b];
  const int past = seq_len - q_len;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lhi = lane >> 4;

  // causal bound of this row tile, then the split's share of it
  const int last_tok = min(rows - 1, (tile + 1) * BQ - 1) / H;
  const int kv_hi_all = min(seq_len, past + last_tok + 1);
  const int split_len =
      ((kv_hi_all + BKV - 1) / BKV + num_splits - 1) / num_splits * BKV;
  const int kv_lo = split * split_len;
  const int kv_hi = min(kv_lo + split_len, kv_hi_all);
  const long row0 = (long)q_start * H + (long)tile * BQ;
  const int rows_here = min(BQ, rows - tile * BQ);
  if (kv_lo >= kv_hi) {  // an empty split: the merge skips it
    if (SPLIT && tid < rows_here)
      partial_lse[(long)split * th_total + row0 + tid] = -INFINITY;
    return;
  }

  __shared__ __attribute__((aligned(16))) char ring[2 * TILE_B];
  __shared__ __attribute__((aligned(16))) char p_tile[BQ * P_ROW];
  __shared__ float s_a[4][16], s_b[4][16], s_m[4][16];

  // query fragments: column l16 = row, dims kt * 32 + lhi * 8
  const int my_tile = R == 1 ? 0 : wave;
  const int my_row = my_tile * 16 + l16;
  mfma_bf8 qf[KT];
  {
    const __hip_bfloat16 *qp =
        q + (row0 + min(my_row, rows_here - 1)) * DK + lhi * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      qf[kt] = *reinterpret_cast<const mfma_bf8 *>(qp + kt * 32);
  }
  // keys this lane's row sees: below vis (none for a row past the end)
  const int vis = my_row < rows_here
                      ? min(seq_len, past + (tile * BQ + my_row) / H + 1)
                      : 0;
  const float qscale = scale * LOG2E;

  // ---- staging: wave w brings keys 16 w .. + 15 as 2 x 9 units of
  // [8 keys][128 B]; rows of the next tile are looked up a tile ahead
  const int *bt = block_table + (long)b * max_pages;
  const int s_key = wave * 16 + (lane >> 3);
  const int s_col = ((lane & 7) ^ (lane >> 3)) * 16;
  int page[2];
  auto key_of = [&](int k0, int g) {
    return min(k0 + s_key + g * 8, seq_len - 1);
  };
  auto look_up = [&](int k0) {
#pragma unroll
    for (int g = 0; g < 2; ++g) page[g] = bt[key_of(k0, g) / page_size];
  };
  auto stage = [&](int k0, int slot) {
    const char *src[2];
#pragma unroll
    for (int g = 0; g < 2; ++g)
      src[g] = reinterpret_cast<const char *>(kc) +
               ((long)page[g] * page_size + key_of(k0, g) % page_size) *
                   ROW_B + s_col;
    char *dst = ring + slot * TILE_B + wave * 2048;
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int g = 0; g < 2; ++g)
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const unsigned int *>(src[g] + c * 128),
            reinterpret_cast<unsigned int *>(dst + c * CB_B + g * 1024), 16,
            0, R == 1 ? 2 : 0);
  };

  float m_run = -INFINITY, l_run = 0.f;
  mfma_f4 o[R][NT];
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o[rt][nt] = mfma_f4{0, 0, 0, 0};
  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;

  look_up(kv_lo);
  stage(kv_lo, 0);
  if (kv_lo + BKV < kv_hi) look_up(kv_lo + BKV);
  int slot = 0;
  for (int k0 = kv_lo; k0 < kv_hi; k0 += BKV, slot ^= 1) {
    // the tile is there; the other slot and P are free
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (k0 + BKV < kv_hi) {
      stage(k0 + BKV, slot ^ 1);
      if (k0 + 2 * BKV < kv_hi) look_up(k0 + 2 * BKV);
    }
    const char *kt_base = ring + slot * TILE_B;

    // ---- scores: fragment f = keys (R == 1 ? wave : f) * 16 + lhi * 4 + r
    mfma_f4 s[NF][2];
#pragma unroll
    for (int f = 0; f < NF; ++f)
      s[f][0] = s[f][1] = mfma_f4{0, 0, 0, 0};
    const int krow = (R == 1 ? wave * 16 : 0) + l16;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const mfma_bf8 kf = *reinterpret_cast<const mfma_bf8 *>(
            kt_base + (kt >> 1) * CB_B + (krow + f * 16) * 128 +
            (((kt & 1) * 64 + lhi * 16) ^ ((krow & 7) << 4)));
        // (one fragment: two chains)
        s[f][NF == 1 ? kt & 1 : 0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            kf, qf[kt], s[f][NF == 1 ? kt & 1 : 0], 0, 0, 0);
      }
    float mx = -INFINITY;
    float sv[NF][4];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = k0 + (R == 1 ? wave : f) * 16 + lhi * 4 + r;
        const float x = (s[f][0][r] + s[f][1][r]) * qscale;
        sv[f][r] = key < vis ? x : -INFINITY;
        mx = fmaxf(mx, sv[f][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (R == 1) {
      if (lhi == 0) s_a[wave][l16] = mx;
      lds_barrier();
#pragma unroll
      for (int w = 0; w < 4; ++w) mx = fmaxf(mx, s_a[w][l16]);
    }
    // (a row may see nothing yet: a finite maximum keeps its weights at 0)
    const float m_new = fmaxf(fmaxf(m_run, mx), -1e30f);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float sum = 0.f;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      shortx4 p;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(sv[f][r] - m_new);
        sum += e;
        p[r] = bf16_bits(e);
      }
      *reinterpret_cast<shortx4 *>(
          p_tile + my_row * P_ROW +
          ((R == 1 ? wave : f) * 16 + lhi * 4) * 2) = p;
    }
    l_run = l_run * alpha + sum;  // this lane's keys
    if (R > 1 && lhi == 0) s_a[wave][l16] = alpha;
    lds_barrier();

    // ---- output dims wave * 128 + nt * 16 .. of every row tile
    float al[R];
#pragma unroll
    for (int rt = 0; rt < R; ++rt) al[rt] = R == 1 ? alpha : s_a[rt][l16];
#pragma unroll
    for (int rt = 0; rt < R; ++rt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[rt][nt][r] *= al[rt];
#pragma unroll
    for (int kk = 0; kk < BKV / 32; ++kk) {
      MlaFrag pf[R];
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int half = 0; half < 2; ++half)
          pf[rt].h[half] = *reinterpret_cast<const shortx4 *>(
              p_tile + (rt * 16 + l16) * P_ROW +
              (kk * 32 + half * 16 + lhi * 4) * 2);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        MlaFrag vf;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int row = kk * 32 + half * 16 + tr_row;
          vf.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_shortx4 *)(kt_base + (wave * 2 + (nt >> 2)) * CB_B +
                              row * 128 +
                              (((nt & 3) * 32 + tr_col) ^
                               ((row & 7) << 4))));
        }
#pragma unroll
        for (int rt = 0; rt < R; ++rt)
          o[rt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf.v, pf[rt].v, o[rt][nt], 0, 0, 0);
      }
    }
  }

  // ---- join the sums, write (lane: row l16, four neighbouring dims)
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (lhi == 0) {
    s_b[wave][l16] = l_run;
    s_m[wave][l16] = m_run;
  }
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < R; ++rt) {
    const int row = rt * 16 + l16;
    if (row >= rows_here) continue;
    const float l = R == 1 ? s_b[0][l16] + s_b[1][l16] + s_b[2][l16] +
                                 s_b[3][l16]
                           : s_b[rt][l16];
    const float m = s_m[rt][l16];
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const long at = row0 + row;
    if (SPLIT) {
      float *op = partial_out + ((long)split * th_total + at) * DV +
                  wave * 128 + lhi * 4;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        *reinterpret_cast<floatx4 *>(op + nt * 16) =
            floatx4{o[rt][nt][0] * inv, o[rt][nt][1] * inv,
                    o[rt][nt][2] * inv, o[rt][nt][3] * inv};
      if (wave == 0 && lhi == 0)
        partial_lse[(long)split * th_total + at] =
            l > 0.f ? m / LOG2E + __logf(l) : -INFINITY;
    } else {
      __hip_bfloat16 *op = out + at * DV + wave * 128 + lhi * 4;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        shortx4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = bf16_bits(o[rt][nt][r] * inv);
        *reinterpret_cast<shortx4 *>(op + nt * 16) = v;
      }
    }
  }
}

// Up to 16 rows, decode: tiles of 32 keys in a ring of two, 78 KB, so that a
// CU holds two workgroups and one's latencies are the other's work. Waves w
// and w + 2 score keys 16 (w & 1) .. + 15, half of the dims each; the partial
// scores pass through LDS, behind which every wave has all 32 keys' scores in
// the layout that the second product takes: maxima, weights and sums stay in
// registers. Wave w then owns dims 128 w .. + 127 of the output.
template <bool SPLIT>
__global__ __launch_bounds__(BLOCK, 2) void mla_decode_kernel(
    __hip_bfloat16 *__restrict__ out, float *__restrict__ partial_out,
    float *__restrict__ partial_lse, const __hip_bfloat16 *__restrict__ q,
    const __hip_bfloat16 *__restrict__ kc,
    const int *__restrict__ block_table, const int *__restrict__ seq_lens,
    const int *__restrict__ qsl, int max_pages, int page_size, int H,
    float scale, int num_splits, long th_total) {
  constexpr int TK = 32, BLK_B = TK * 128, T_B = CB * BLK_B, HT = KT / 2;
  const int b = blockIdx.y, split = blockIdx.z;
  const int q_start = qsl[b];
  const int q_len = qsl[b + 1] - q_start;
  const int rows = min(q_len * H, 16);
  if (rows <= 0) return;
  const int seq_len = seq_lens[b], past = seq_len - q_len;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4;
  // (shares of whole 64-key tiles)
  const int split_len =
      ((seq_len + BKV - 1) / BKV + num_splits - 1) / num_splits * BKV;
  const int kv_lo = split * split_len;
  const int kv_hi = min(kv_lo + split_len, seq_len);
  const long row0 = (long)q_start * H;
  if (kv_lo >= kv_hi) {  // an empty split: the merge skips it
    if (SPLIT && tid < rows)
      partial_lse[(long)split * th_total + row0 + tid] = -INFINITY;
    return;
  }
  __shared__ __attribute__((aligned(16))) char ring[2 * T_B];
  __shared__ mfma_f4 part[4][64];

  // staging: wave w brings keys 8 w .. + 7 as nine units of [8 keys][128 B]
  const int *bt = block_table + (long)b * max_pages;
  const int s_key = wave * 8 + (lane >> 3);
  const int s_col = ((lane & 7) ^ (lane >> 3)) * 16;
  int page = 0;
  auto key_of = [&](int k0) { return min(k0 + s_key, seq_len - 1); };
  auto look_up = [&](int k0) { page = bt[key_of(k0) / page_size]; };
  auto stage = [&](int k0, int slot) {
    const char *src =
        reinterpret_cast<const char *>(kc) +
        ((long)page * page_size + key_of(k0) % page_size) * ROW_B + s_col;
    char *dst = ring + slot * T_B + wave * 1024;
#pragma unroll
    for (int c = 0; c < CB; ++c)
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const unsigned int *>(src + c * 128),
          reinterpret_cast<unsigned int *>(dst + c * BLK_B), 16, 0, 2);
  };
  look_up(kv_lo);
  stage(kv_lo, 0);
  if (kv_lo + TK < kv_hi) look_up(kv_lo + TK);

  // query fragments of this wave's half of the dims: column l16 = row
  const int my_half = wave >> 1, my_keys = (wave & 1) * 16;
  mfma_bf8 qf[HT];
  {
    const __hip_bfloat16 *qp =
        q + (row0 + min(l16, rows - 1)) * DK + my_half * HT * 32 + lhi * 8;
#pragma unroll
    for (int i = 0; i < HT; ++i)
      qf[i] = *reinterpret_cast<const mfma_bf8 *>(qp + i * 32);
  }
  const int vis = l16 < rows ? min(seq_len, past + l16 / H + 1) : 0;
  const float qscale = scale * LOG2E;

  float m_run = -INFINITY, l_run = 0.f;
  mfma_f4 o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) o[nt] = mfma_f4{0, 0, 0, 0};
  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;
  int slot = 0;
  for (int k0 = kv_lo; k0 < kv_hi; k0 += TK, slot ^= 1) {
    // the tile is there; the other slot and the scores are free
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (k0 + TK < kv_hi) {
      stage(k0 + TK, slot ^ 1);
      if (k0 + 2 * TK < kv_hi) look_up(k0 + 2 * TK);
    }
    const char *base = ring + slot * T_B;
    mfma_f4 s[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};  // two chains
    const int krow = my_keys + l16;
#pragma unroll
    for (int i = 0; i < HT; ++i) {
      const int kt = my_half * HT + i;
      const mfma_bf8 kf = *reinterpret_cast<const mfma_bf8 *>(
          base + (kt >> 1) * BLK_B + krow * 128 +
          (((kt & 1) * 64 + lhi * 16) ^ ((krow & 7) << 4)));
      s[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[i], s[i & 1],
                                                         0, 0, 0);
    }
    part[wave][lane] = s[0] + s[1];
    lds_barrier();
    // keys f * 16 + lhi * 4 + r of row l16
    float sv[2][4], mx = -INFINITY;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const mfma_f4 x = part[f][lane] + part[f + 2][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sv[f][r] = k0 + f * 16 + lhi * 4 + r < vis ? x[r] * qscale
                                                   : -INFINITY;
        mx = fmaxf(mx, sv[f][r]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // (a row may see nothing yet: a finite maximum keeps its weights at 0)
    const float m_new = fmaxf(fmaxf(m_run, mx), -1e30f);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float sum = 0.f;
    MlaFrag pf;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(sv[f][r] - m_new);
        sum += e;
        pf.h[f][r] = bf16_bits(e);
      }
    l_run = l_run * alpha + sum;  // this lane's keys
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      MlaFrag vf;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int row = half * 16 + tr_row;
        vf.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_shortx4 *)(base + (wave * 2 + (nt >> 2)) * BLK_B + row * 128 +
                            (((nt & 3) * 32 + tr_col) ^ ((row & 7) << 4))));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) o[nt][r] *= alpha;
      o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf.v, o[nt], 0, 0,
                                                      0);
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (l16 >= rows) return;
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  const long at = row0 + l16;
  if (SPLIT) {
    float *op = partial_out + ((long)split * th_total + at) * DV + wave * 128 +
                lhi * 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<floatx4 *>(op + nt * 16) =
          floatx4{o[nt][0] * inv, o[nt][1] * inv, o[nt][2] * inv,
                  o[nt][3] * inv};
    if (wave == 0 && lhi == 0)
      partial_lse[(long)split * th_total + at] =
          l_run > 0.f ? m_run / LOG2E + __logf(l_run) : -INFINITY;
  } else {
    __hip_bfloat16 *op = out + at * DV + wave * 128 + lhi * 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      shortx4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = bf16_bits(o[nt][r] * inv);
      *reinterpret_cast<shortx4 *>(op + nt * 16) = v;
    }
  }
}

// Merge split partials: out[row, :] = sum_s w_s * partial[s, row, :]
__global__ void mla_merge_kernel(__hip_bfloat16 *__restrict__ out,
                                 const float *__restrict__ partial_out,
                                 const float *__restrict__ partial_lse,
                                 int num_splits, long th_total) {
  const long row = blockIdx.x;
  const int d = threadIdx.x;  // 256 threads, 2 dims each
  float mx = -INFINITY;
  for (int s = 0; s < num_splits; ++s)
    mx = fmaxf(mx, partial_lse[(long)s * th_total + row]);
  float denom = 0.f, o0 = 0.f, o1 = 0.f;
  for (int s = 0; s < num_splits; ++s) {
    const float lse = partial_lse[(long)s * th_total + row];
    if (lse == -INFINITY) continue;
    const float w = __expf(lse - mx);
    denom += w;
    const float *p = partial_out + ((long)s * th_total + row) * DV;
    o0 += w * p[d];
    o1 += w * p[d + 256];
  }
  const float inv = (denom > 0.f) ? 1.f / denom : 0.f;
  out[row * DV + d] = __float2bfloat16(o0 * inv);
  out[row * DV + d + 256] = __float2bfloat16(o1 * inv);
}

// Scatter the per-token latent row [T, 1, DK] into the paged cache
// (reference concat_and_cache_mla, cache_kernels.py:161 — the caller
// has already concatenated [c_kv | k_pe]; the v cache is a view of the
// first 512 dims so one write covers both).
__global__ void cache_latent_kernel(const __hip_bfloat16 *__restrict__ k,
                                    __hip_bfloat16 *__restrict__ k_cache,
                                    const long *__restrict__ slot_mapping,
                                    int page_size, long k_stride) {
  const long t = blockIdx.x;
  const long slot = slot_mapping[t];
  const long row = (slot / page_size) * page_size + slot % page_size;
  const shortx8 *src = reinterpret_cast<const shortx8 *>(k + t * k_stride);
  shortx8 *dst = reinterpret_cast<shortx8 *>(k_cache + row * DK);
  for (int i = threadIdx.x; i < DK / 8; i += blockDim.x) dst[i] = src[i];
}

}  // namespace

void mla_paged_attention(torch::Tensor out, torch::Tensor q,
                         torch::Tensor k_cache, torch::Tensor block_table,
                         torch::Tensor seq_lens,
                         torch::Tensor query_start_loc, long max_query_len,
                         double scale) {
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "mla attn: bf16 only");
  TORCH_CHECK(q.is_contiguous() && out.is_contiguous());
  TORCH_CHECK(q.size(2) == DK, "mla attn: latent dim must be ", DK);
  TORCH_CHECK(out.size(2) == DV);
  TORCH_CHECK(k_cache.size(2) == 1 && k_cache.size(3) == DK,
              "mla attn: cache must be the shared latent layout");
  TORCH_CHECK(block_table.scalar_type() == at::kInt);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  const long T = q.size(0);
  if (T == 0) return;
  const int H = q.size(1);
  const int B = seq_lens.size(0);
  TORCH_CHECK(block_table.stride(1) == 1 && block_table.size(0) >= B &&
              query_start_loc.scalar_type() == at::kInt &&
              query_start_loc.numel() >= B + 1);
  TORCH_CHECK(k_cache.is_contiguous() &&
              reinterpret_cast<uintptr_t>(k_cache.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 == 0);
  const int R = max_query_len * H <= 16 ? 1 : 4;
  const int BQ = R * 16;
  const int tiles = (int)((max_query_len * H + BQ - 1) / BQ);
  const long th_total = T * H;
  auto stream = at::cuda::getCurrentCUDAStream();

  // split-KV only for pure-decode batches (uniform kv ranges). The count
  // depends on the batch size and the pool only: a captured launch serves
  // every length, an empty split costs a few hundred cycles.
  int splits = 1;
  if (max_query_len == 1) {
    const long max_len = (long)k_cache.size(0) * k_cache.size(1);
    while (splits < 32 && (long)B * tiles * splits < SPLIT_TARGET &&
           splits * 2 <= (max_len + BKV - 1) / BKV)
      splits *= 2;
  }
  torch::Tensor partial, lse;
  float *po = nullptr, *pl = nullptr;
  if (splits > 1) {
    auto opts = q.options().dtype(at::kFloat);
    partial = torch::empty({splits, th_total, (long)DV}, opts);
    lse = torch::empty({splits, th_total}, opts);
    po = partial.data_ptr<float>();
    pl = lse.data_ptr<float>();
  }
  // Two workgroups a CU hide each other's latencies; by itself one walks 64
  // keys at a time (us: one sequence of 4000 keys and two rows 185, by 32 keys
  // 241, 64 of 1000 74 / 92; decode, 4 of 4000 in 32 splits 23 / 24, 64 of 1000
  // in eight 32 / 25).
  const bool paired =
      R == 1 && (long)B * splits > at::cuda::getCurrentDeviceProperties()
                                       ->multiProcessorCount;
#define RUN(...)                                                             \
  hipLaunchKernelGGL((__VA_ARGS__), dim3(tiles, B, splits), dim3(BLOCK), 0,  \
                     stream, (__hip_bfloat16 *)out.data_ptr(), po, pl,       \
                     (const __hip_bfloat16 *)q.data_ptr(),                   \
                     (const __hip_bfloat16 *)k_cache.data_ptr(),             \
                     block_table.data_ptr<int>(), seq_lens.data_ptr<int>(),  \
                     query_start_loc.data_ptr<int>(),                        \
                     (int)block_table.stride(0), (int)k_cache.size(1), H,    \
                     (float)scale, splits, th_total)
  if (splits == 1) {
    if (paired) RUN(mla_decode_kernel<false>);
    else if (R == 1) RUN(mla_attention_kernel<1, false>);
    else RUN(mla_attention_kernel<4, false>);
    HIP_CHECK_KERNEL();
    return;
  }
  if (paired) RUN(mla_decode_kernel<true>);
  else if (R == 1) RUN(mla_attention_kernel<1, true>);
  else RUN(mla_attention_kernel<4, true>);
#undef RUN
  HIP_CHECK_KERNEL();
  hipLaunchKernelGGL((mla_merge_kernel), dim3((unsigned)th_total),
                     dim3(256), 0, stream,
                     (__hip_bfloat16 *)out.data_ptr(), po, pl, splits,
                     th_total);
  HIP_CHECK_KERNEL();
}

void cache_latent(torch::Tensor k, torch::Tensor k_cache,
                  torch::Tensor slot_mapping) {
  const long T = k.size(0);
  if (T == 0) return;
  TORCH_CHECK(k.scalar_type() == at::kBFloat16);
  TORCH_CHECK(k.stride(-1) == 1);
  TORCH_CHECK(k.numel() / T == DK, "cache_latent: row must be ", DK);
  TORCH_CHECK(k_cache.is_contiguous() && k_cache.size(3) == DK);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL((cache_latent_kernel), dim3(T), dim3(64), 0, stream,
                     (const __hip_bfloat16 *)k.data_ptr(),
                     (__hip_bfloat16 *)k_cache.data_ptr(),
                     slot_mapping.data_ptr<long>(), (int)k_cache.size(1),
                     k.stride(0));
  HIP_CHECK_KERNEL();
}
