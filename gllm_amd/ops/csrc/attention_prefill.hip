// Varlen causal (chunked-)prefill attention over the paged KV cache,
// MFMA-based, for gfx950.
//
// Workgroup = 4 waves, BQ = 128 q rows (32 per wave, two groups of 16) of
// one (sequence, head); K/V tiles of 64 keys in two LDS slots, the next
// tile in flight (global -> LDS loads) while this one is worked on.
// Everything is computed transposed: scores are K Q^T, so a lane holds 16
// keys of ONE query and the softmax state is one number per lane and
// group (two cross-lane steps for the max, none for the sum until the
// end); the tile of weights is then already the right operand of
// O^T = V^T P^T, whose left operand is read from the V tile transposed by
// ds_read_tr16_b64. A contraction over keys may run in any order as long
// as both operands agree: key 32 s + 16 half + 4 lhi + r, the order in
// which the score tiles hold them. Each K and V element read from LDS
// serves 32 q rows. LDS rows are XOR-swizzled in 16 B units through the
// load's source address. Tiles that no row of a wave can see are skipped
// by that wave; tiles every row sees wholly skip the mask.
//
// Plain causal attention of 64 or 128 dims goes to attention_causal.hip: the
// options that this kernel can carry are selects in every tile, 60 % of its
// instructions.
//
// Capability parity: flash_attn_with_kvcache varlen semantics
// (reference layers/attention.py:77-141) — one kernel serves chunked
// prefill, mixed prefill+decode batches, prefix-cache hits and sliding
// windows.

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "attention_causal.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mfma_bf8;
typedef __attribute__((ext_vector_type(4))) float mfma_f4;
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

namespace {

constexpr int WAVES = 4;
constexpr int BLOCK = 64 * WAVES;
constexpr int RG = 2;        // groups of 16 q rows per wave
constexpr int BQ = 16 * RG * WAVES;
constexpr int BKV = 64;      // kv tokens per LDS slot
constexpr int NF = BKV / 16; // score tiles per group
constexpr int BIAS_LDS = 8192;  // longest distance table kept in LDS
// entries repeated at either end of it: the distances a wave's rows and one
// tile can differ by, so that reads need no clamping
constexpr int BIAS_PAD = BKV + 16 * RG;
constexpr float LOG2E = 1.4426950408889634f;

template <int D>
DEV_INLINE int kswz(int row, int byte_off) {
  constexpr int MASK = (D * 2 / 16 - 1) & 15;
  return byte_off ^ ((row & MASK) << 4);
}

union KeyFrag {
  mfma_bf8 v;
  shortx4 h[2];
  __hip_bfloat16 e[8];
};

// D, DV: key / value size of the tiles. EXT: the heads are Dr <= D and
// Dvr <= DV wide (multiples of 8; a tile's spare columns repeat real ones,
// the query fragment is zero there and spare output columns are dropped),
// and the scores may carry a bias by distance and a query temperature.
template <int D, int DV, bool EXT>
__global__ __launch_bounds__(BLOCK, 2) void paged_prefill_kernel(
    __hip_bfloat16 *__restrict__ out,            // [T, Hq, D] (row stride)
    long out_stride,
    const __hip_bfloat16 *__restrict__ q,        // [T, Hq, D] (row stride)
    const __hip_bfloat16 *__restrict__ k_cache,  // [P, ps, Hkv, D]
    const __hip_bfloat16 *__restrict__ v_cache,
    const int *__restrict__ block_table,         // [B, max_pages]
    const int *__restrict__ seq_lens,            // [B]
    const int *__restrict__ qsl,                 // [B+1]
    int max_pages, int page_size, int Hq, int num_kv_heads, float scale,
    long q_stride, int window,
    // windowed-sink extensions (0 / 0 / nullptr = plain causal softmax):
    // keys j < keep_first stay visible outside the window; sink adds a
    // score-0, value-less key to the softmax (denominator 1 + sum exp);
    // gate multiplies the output by sigmoid(gate[t, h*D + d])
    int keep_first, int sink, const __hip_bfloat16 *__restrict__ gate,
    long gate_stride,
    // per-head learned sink scores (in place of 0) and a tanh cap
    // cap * tanh(s / cap) on the scaled scores (0 = none)
    const float *__restrict__ sinks, float softcap,
    // EXT: head sizes; bias [Hq, bias_len] (nullptr: none), entry
    // min(i - j, bias_len - 1) added to the scaled score
    int Dr_, int Dvr_, const float *__restrict__ bias, int bias_len,
    float temp_coef, int temp_every, int vec_out,
    // sequences of fewer query rows are served elsewhere
    int min_rows) {
  const int Dr = EXT ? Dr_ : D, Dvr = EXT ? Dvr_ : DV;
  const int tile = blockIdx.x;
  const int b = blockIdx.y;
  const int h = blockIdx.z;
  const int kvh = h / (Hq / num_kv_heads);

  const int q_start = qsl[b];
  const int q_len = qsl[b + 1] - q_start;
  if (tile * BQ >= q_len || q_len < min_rows) return;
  const int seq_len = seq_lens[b];
  const int past = seq_len - q_len;

  constexpr int KT = D / 32;        // score k-steps
  constexpr int NT = DV / 16;       // value column tiles
  constexpr int KROW_B = D * 2;     // K row bytes
  constexpr int VROW_B = DV * 2;    // V row bytes
  constexpr int TILE_B = BKV * KROW_B;           // the K tile
  constexpr int SLOT_B = TILE_B + BKV * VROW_B;  // K tile | V tile
  constexpr int GLK = TILE_B / 1024 / WAVES;     // 1 KiB loads per wave
  constexpr int GLV = (SLOT_B - TILE_B) / 1024 / WAVES;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lhi = lane >> 4;

  __shared__ __attribute__((aligned(16))) char kv_ring[2 * SLOT_B];
  __shared__ int s_row[2][BKV];     // cache rows of a tile's keys
  // EXT with a bias: the head's row of the table times log2 e, while it
  // fits
  extern __shared__ float bias_lds[];
  const float *brow = nullptr;
  bool blds = false;
  if (EXT && bias) {
    brow = bias + (long)h * bias_len;
    blds = bias_len <= BIAS_LDS;
    if (blds)  // (published by the first barrier)
      for (int i = tid; i < bias_len + 2 * BIAS_PAD; i += BLOCK)
        bias_lds[i] =
            brow[min(max(i - BIAS_PAD, 0), bias_len - 1)] * LOG2E;
  }

  const int *bt = block_table + (long)b * max_pages;
  const int kv_max = min(seq_len, past + min(q_len, (tile + 1) * BQ));
  int kv_lo = 0;
  if (window > 0)
    kv_lo = max(0, past + tile * BQ - window + 1) / BKV * BKV;
  // kept-first tiles [0, min(keep_first, kv_lo)) come before the
  // window tiles; kv_lo is a BKV multiple, so the two never overlap
  const int n_keep =
      (keep_first > 0 && kv_lo > 0)
          ? (min(keep_first, kv_lo) + BKV - 1) / BKV : 0;
  const int nkt = n_keep + (kv_max - kv_lo + BKV - 1) / BKV;
  // (a key past the end: the last one again, its scores are masked)
  auto key_at = [&](int t, int n) {
    return min((t < n_keep ? t * BKV : kv_lo + (t - n_keep) * BKV) + n,
               seq_len - 1);
  };

  // Loads straight into LDS, 1 KiB per wave and load. Issued as inline
  // assembly: the loop orders them against the LDS reads itself (vmcnt,
  // then the barrier), and the compiler must not wait for the next tile
  // ahead of this tile's reads.
  const unsigned lds0 =
      (unsigned)(unsigned long)(__attribute__((address_space(3))) char *)
          kv_ring + wave * 1024;
  auto load_lds = [&](const char *src, unsigned dst) {
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off"
        :
        : "v"(src), "s"(__builtin_amdgcn_readfirstlane(dst))
        : "memory", "m0");
  };
  const char *kbase = reinterpret_cast<const char *>(k_cache + kvh * Dr);
  const char *vbase = reinterpret_cast<const char *>(v_cache + kvh * Dvr);
  const long krow_b = (long)num_kv_heads * Dr * 2;
  const long vrow_b = (long)num_kv_heads * Dvr * 2;
  auto stage = [&](int t) {
    const unsigned base = lds0 + (t & 1) * SLOT_B;
#pragma unroll
    for (int j = 0; j < GLK; ++j) {
      const int p = (j * WAVES + wave) * 1024 + lane * 16;
      const int row = p / KROW_B;
      int col = kswz<D>(row, p % KROW_B);
      if (EXT && col >= Dr * 2) col = 0;
      load_lds(kbase + s_row[t & 1][row] * krow_b + col,
               base + j * WAVES * 1024);
    }
#pragma unroll
    for (int j = 0; j < GLV; ++j) {
      const int p = (j * WAVES + wave) * 1024 + lane * 16;
      const int row = p / VROW_B;
      int col = kswz<DV>(row, p % VROW_B);
      if (EXT && col >= Dvr * 2) col = 0;
      load_lds(vbase + s_row[t & 1][row] * vrow_b + col,
               base + TILE_B + j * WAVES * 1024);
    }
  };

  int page_id = 0;  // block-table entry of this thread's key, next tile
  if (tid < BKV) {
    const int j = key_at(0, tid);
    s_row[0][tid] = bt[j / page_size] * page_size + j % page_size;
    if (nkt > 1) page_id = bt[key_at(1, tid) / page_size];
  }

  // this lane's query per group: row, fragments, softmax state (log2 units)
  const int row0 = tile * BQ + wave * 16 * RG;  // first row of the wave
  const bool busy = row0 < q_len;
  mfma_bf8 qf[RG][KT];
  float m_run[RG], l_run[RG], rscale[RG];
  mfma_f4 o_acc[RG][NT];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int qrow = row0 + g * 16 + l16;
    const __hip_bfloat16 *qp =
        q + (long)(q_start + qrow) * q_stride + h * Dr + lhi * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (qrow < q_len && (!EXT || kt * 32 + lhi * 8 < Dr))
        qf[g][kt] = *reinterpret_cast<const mfma_bf8 *>(qp + kt * 32);
      else
        qf[g][kt] = mfma_bf8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    // the sink enters as an already-seen key of score 0
    m_run[g] = sinks ? sinks[h] * LOG2E : (sink ? 0.f : -INFINITY);
    l_run[g] = (sink || sinks) && lhi == 0 ? 1.f : 0.f;
    rscale[g] = scale * (EXT ? query_temp(past + qrow, temp_coef, temp_every)
                             : 1.0f);
    // with a cap the exponent of tanh, else the score in log2 units
    rscale[g] *= softcap > 0.f ? 2.f * LOG2E / softcap : LOG2E;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o_acc[g][nt] = mfma_f4{0, 0, 0, 0};
  }
  const float cap2 = softcap * LOG2E;
  // what the loop reads from registers has arrived before it starts (a
  // load still pending here would make the loop wait for its own tiles)
#pragma unroll
  for (int g = 0; g < RG; ++g) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) asm volatile("" : "+v"(qf[g][kt]));
    asm volatile("" : "+v"(m_run[g]));
  }
  asm volatile("" : "+v"(page_id));
  __syncthreads();
  stage(0);

  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;
  const int pos_lo = past + row0;               // the wave's positions
  const int pos_hi = past + min(row0 + 16 * RG, q_len) - 1;
  for (int it = 0; it < nkt; ++it) {
    const int kv0 = it < n_keep ? it * BKV : kv_lo + (it - n_keep) * BKV;
    // every wave's loads of this tile have landed; and every wave is done
    // with the other slot, which the next tile goes to
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (tid < BKV && it + 1 < nkt)
      s_row[(it + 1) & 1][tid] =
          page_id * page_size + key_at(it + 1, tid) % page_size;
    __syncthreads();
    if (tid < BKV && it + 2 < nkt)
      page_id = bt[key_at(it + 2, tid) / page_size];
    if (it + 1 < nkt) stage(it + 1);
    // nothing in this tile that a row of this wave sees
    if (!busy || kv0 > pos_hi) continue;
    if (window > 0 && kv0 + BKV - 1 <= pos_lo - window && kv0 >= keep_first)
      continue;

    const char *ktile = kv_ring + (it & 1) * SLOT_B;
    const char *vtile = ktile + TILE_B;

    // ---------- scores: [64 keys x 16 queries] per group ----------
    mfma_f4 s[RG][NF];
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
      for (int f = 0; f < NF; ++f) s[g][f] = mfma_f4{0, 0, 0, 0};
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int krow = f * 16 + l16;
        const mfma_bf8 kf = *reinterpret_cast<const mfma_bf8 *>(
            ktile + krow * KROW_B + kswz<D>(krow, (kt * 32 + lhi * 8) * 2));
#pragma unroll
        for (int g = 0; g < RG; ++g)
          s[g][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[g][kt],
                                                            s[g][f], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);

    // ---------- mask + online softmax ----------
    // interior tiles (every key visible to every row of this wave, no
    // window cut) skip the mask
    const bool inside = it >= n_keep && row0 + 16 * RG <= q_len &&
                        kv0 + BKV - 1 <= pos_lo && kv0 + BKV <= seq_len &&
                        (window <= 0 || kv0 > pos_hi - window);
    // every key of the tile beyond the table's reach: one number
    const bool far = EXT && brow && pos_lo - (kv0 + BKV - 1) >= bias_len - 1;
    const float far_bias =
        far ? brow[bias_len - 1] * LOG2E : 0.f;
    KeyFrag pf[RG][BKV / 32];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      const int qpos = past + row0 + g * 16 + l16;
      const int dist0 = qpos - kv0 - lhi * 4;  // distance of f = 0, r = 0
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[g][f][r] *= rscale[g];
          if (softcap > 0.f)  // cap tanh(x / cap) from one exponential
            s[g][f][r] =
                cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(
                                        1.f + __builtin_amdgcn_exp2f(
                                                  s[g][f][r]));
        }
      if (EXT && brow) {
        if (far) {
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[g][f][r] += far_bias;
        } else if (blds) {
          // (not far: dist0 < bias_len + PAD; not skipped: it is > -PAD)
          const float *bl = bias_lds + BIAS_PAD + dist0;
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[g][f][r] += bl[-f * 16 - r];
        } else {
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              s[g][f][r] +=
                  brow[min(max(dist0 - f * 16 - r, 0), bias_len - 1)] * LOG2E;
        }
      }
      if (!inside) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int d = dist0 - f * 16 - r, kvp = qpos - d;
            const bool hide = d < 0 || kvp >= seq_len ||
                              (window > 0 && d >= window && kvp >= keep_first);
            s[g][f][r] = hide ? -INFINITY : s[g][f][r];
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[g][f][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m_run[g], mx);
      const float base = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run[g] - base);
      m_run[g] = m_new;
      float sum = 0.f;  // this lane's keys; lanes join at the end
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(s[g][f][r] - base);
          sum += p;
          pf[g][f >> 1].e[(f & 1) * 4 + r] = __float2bfloat16(p);
        }
      l_run[g] = l_run[g] * alpha + sum;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o_acc[g][nt][r] *= alpha;
      }
    }

    // ---------- O^T += V^T P^T ----------
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < BKV / 32; ++ks) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        KeyFrag vf;
#pragma unroll
        for (int half = 0; half < 2; ++half)
          vf.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_shortx4 *)const_cast<char *>(
                  vtile + (ks * 32 + half * 16 + tr_row) * VROW_B +
                  kswz<DV>(tr_row, nt * 32 + tr_col)));
#pragma unroll
        for (int g = 0; g < RG; ++g)
          o_acc[g][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf.v, pf[g][ks].v, o_acc[g][nt], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // ---------- epilogue: lane = one query, 4 columns of each tile ----------
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    float l = l_run[g];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int qrow = row0 + g * 16 + l16;
    if (qrow >= q_len) continue;
    const float inv_l = l > 0.f ? 1.f / l : 0.f;
    __hip_bfloat16 *op =
        out + (long)(q_start + qrow) * out_stride + (long)h * Dvr + lhi * 4;
    const __hip_bfloat16 *gp =
        gate ? gate + (long)(q_start + qrow) * gate_stride + (long)h * Dvr +
                   lhi * 4
             : nullptr;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (EXT && nt * 16 + lhi * 4 >= Dvr) continue;  // (multiples of 8)
      KeyFrag ov, gv;
      if (gp) {
        if (vec_out) {
          gv.h[0] = *reinterpret_cast<const shortx4 *>(gp + nt * 16);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) gv.e[r] = gp[nt * 16 + r];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = o_acc[g][nt][r] * inv_l;
        if (gp) v /= 1.f + __expf(-__bfloat162float(gv.e[r]));
        ov.e[r] = __float2bfloat16(v);
      }
      if (vec_out) {
        *reinterpret_cast<shortx4 *>(op + nt * 16) = ov.h[0];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) op[nt * 16 + r] = ov.e[r];
      }
    }
  }
}

}  // namespace

namespace {

void launch_prefill(torch::Tensor &out, torch::Tensor &q, int Hq,
                    long q_stride, torch::Tensor &k_cache,
                    torch::Tensor &v_cache, torch::Tensor &block_table,
                    torch::Tensor &seq_lens, torch::Tensor &query_start_loc,
                    long max_query_len, double scale, long window,
                    long keep_first, bool sink, const void *gate,
                    long gate_stride, const float *sinks = nullptr,
                    float softcap = 0.f, const float *bias = nullptr,
                    int bias_len = 0, float temp_coef = 0.f,
                    int temp_every = 0, int min_rows = 1) {
  const int Hkv = k_cache.size(2);
  const int D = k_cache.size(3), Dv = v_cache.size(3);
  const int B = seq_lens.size(0);
  const int q_tiles = (int)((max_query_len + BQ - 1) / BQ);
  // a 2-D out may be a column block of a wider buffer
  const long out_stride = out.dim() == 2 ? out.stride(0) : (long)Hq * Dv;
  const bool ext = bias || temp_every > 0 || D != Dv ||
                   (D != 64 && D != 128);
  // 4 columns per access where rows allow it
  const int vec_out =
      out_stride % 4 == 0 && Dv % 4 == 0 &&
      reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0 &&
      (!gate || (gate_stride % 4 == 0 &&
                 reinterpret_cast<uintptr_t>(gate) % 8 == 0)) ? 1 : 0;
  // nothing but causal softmax (us, here / there: see attention_causal.hip)
  if (!ext && vec_out && window <= 0 && !sink && !sinks && !gate &&
      softcap == 0.f && causal_prefill_ok(D, Dv, (float)scale)) {
    causal_prefill(out.data_ptr(), out_stride, q.data_ptr(), q_stride,
                   k_cache.data_ptr(), v_cache.data_ptr(),
                   block_table.data_ptr<int>(), block_table.stride(0),
                   k_cache.size(1), seq_lens.data_ptr<int>(),
                   query_start_loc.data_ptr<int>(), B, q.size(0),
                   max_query_len, Hq, Hkv, D, (float)scale, min_rows);
    return;
  }
  const size_t lds =
      bias && bias_len <= BIAS_LDS
          ? (bias_len + 2 * BIAS_PAD) * sizeof(float) : 0;
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(DT, DVT, EXT)                                                    \
  hipLaunchKernelGGL((paged_prefill_kernel<DT, DVT, EXT>),                   \
                     dim3(q_tiles, B, Hq), dim3(BLOCK), lds, stream,         \
                     (__hip_bfloat16 *)out.data_ptr(), out_stride,           \
                     (const __hip_bfloat16 *)q.data_ptr(),                   \
                     (const __hip_bfloat16 *)k_cache.data_ptr(),             \
                     (const __hip_bfloat16 *)v_cache.data_ptr(),             \
                     block_table.data_ptr<int>(), seq_lens.data_ptr<int>(),  \
                     query_start_loc.data_ptr<int>(),                        \
                     (int)block_table.stride(0), (int)k_cache.size(1), Hq,   \
                     Hkv, (float)scale, q_stride, (int)window,               \
                     (int)keep_first, sink ? 1 : 0,                          \
                     (const __hip_bfloat16 *)gate, gate_stride, sinks,       \
                     softcap, D, Dv, bias, bias_len, temp_coef, temp_every,  \
                     vec_out, min_rows)
  if (!ext && D == 128) RUN(128, 128, false);
  else if (!ext && D == 64) RUN(64, 64, false);
  else if (D % 8 == 0 && Dv % 8 == 0 && D <= 128 && Dv <= 128) {
    if (D <= 64) {
      if (Dv <= 64) RUN(64, 64, true); else RUN(64, 128, true);
    } else {
      if (Dv <= 64) RUN(128, 64, true); else RUN(128, 128, true);
    }
  } else TORCH_CHECK(false, "prefill attn: head_dim ", D, " unsupported");
#undef RUN
  HIP_CHECK_KERNEL();
}

}  // namespace

void paged_attention_prefill(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_table,
                             torch::Tensor seq_lens,
                             torch::Tensor query_start_loc,
                             long max_query_len, double scale,
                             long sliding_window, bool skip_single) {
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "prefill attn: bf16 only");
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2),
              "q per-token row must be contiguous");
  if (q.size(0) == 0) return;
  launch_prefill(out, q, q.size(1), q.stride(0), k_cache, v_cache,
                 block_table, seq_lens, query_start_loc, max_query_len,
                 scale, sliding_window, 0, false, nullptr, 0, nullptr, 0.f,
                 nullptr, 0, 0.f, 0, skip_single ? 2 : 1);
}

// Windowed-sink form of the same MFMA kernel: q [T, H*D] (row-strided
// view allowed), bf16, D and Dv multiples of 8 up to 128. Callers route
// every other shape / dtype to the generic window_attention kernel.
void window_attention_mfma(torch::Tensor out, torch::Tensor q,
                           c10::optional<torch::Tensor> gate,
                           torch::Tensor k_cache, torch::Tensor v_cache,
                           torch::Tensor block_table, torch::Tensor seq_lens,
                           torch::Tensor query_start_loc, long max_query_len,
                           double scale, long window, long keep_first,
                           bool sink, c10::optional<torch::Tensor> sinks,
                           double softcap, c10::optional<torch::Tensor> bias,
                           double temp_coef, long temp_every) {
  const long T = q.size(0);
  if (T == 0) return;
  const int D = k_cache.size(3), Dv = v_cache.size(3);
  TORCH_CHECK(q.scalar_type() == at::kBFloat16 &&
              k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16);
  TORCH_CHECK(D % 8 == 0 && Dv % 8 == 0 && D <= 128 && Dv <= 128,
              "window_attention_mfma: D, Dv multiples of 8 up to 128");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(k_cache.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(v_cache.data_ptr()) % 16 == 0,
              "window_attention_mfma: 16 B aligned cache rows");
  TORCH_CHECK(q.dim() == 2 && q.stride(1) == 1 && q.size(1) % D == 0);
  const int H = q.size(1) / D;
  TORCH_CHECK(H % k_cache.size(2) == 0);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(out.dim() == 2 && out.stride(1) == 1 && out.size(0) == T &&
              out.size(1) == (long)H * Dv &&
              out.scalar_type() == at::kBFloat16,
              "out: bf16 [T, H*Dv] rows (a column block is fine)");
  TORCH_CHECK(block_table.scalar_type() == at::kInt &&
              block_table.stride(1) == 1 &&
              seq_lens.scalar_type() == at::kInt &&
              query_start_loc.scalar_type() == at::kInt);
  TORCH_CHECK(query_start_loc.numel() >= seq_lens.numel() + 1 &&
              block_table.size(0) >= seq_lens.numel());
  const void *gp = nullptr;
  long gs = 0;
  if (gate.has_value()) {
    TORCH_CHECK(gate->dim() == 2 && gate->stride(1) == 1 &&
                gate->size(0) == T && gate->size(1) == (long)H * Dv &&
                gate->scalar_type() == at::kBFloat16);
    gp = gate->data_ptr();
    gs = gate->stride(0);
  }
  const float *sp = nullptr;
  if (sinks.has_value()) {
    TORCH_CHECK(sinks->scalar_type() == at::kFloat && sinks->is_contiguous() &&
                sinks->numel() == H, "sinks: fp32 [H]");
    sp = sinks->data_ptr<float>();
  }
  const float *bp = nullptr;
  int bias_len = 0;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->scalar_type() == at::kFloat &&
                bias->is_contiguous() && bias->dim() == 2 &&
                bias->size(0) == H && bias->size(1) >= 1,
                "bias: fp32 [H, distances]");
    bp = bias->data_ptr<float>();
    bias_len = bias->size(1);
  }
  launch_prefill(out, q, H, q.stride(0), k_cache, v_cache, block_table,
                 seq_lens, query_start_loc, max_query_len, scale, window,
                 keep_first, sink, gp, gs, sp, (float)softcap, bp, bias_len,
                 (float)temp_coef, (int)temp_every);
}
