// Causal softmax attention of prompt rows for gfx950, bf16 in, fp32 sums:
//   causal_prefill  q [T, Hq, D] over the paged cache, D 64 or 128 (portions
//                   of prompts, cached prefixes, mixed batches)
//   mla_prompts     whole prompts of latent attention in their per-head form:
//                   192-wide keys (128 of the head, 64 rotated ones that all
//                   heads share) and 128-wide values, as rows of the batch
// Windows, sinks, caps, biases and gates are attention_prefill.hip's.
//
// Bound by the vector instructions of the softmax and the LDS reads of K and
// V, about level with each other and with the products (1100, 1000 and 1000
// clocks of a tile's 64 keys x 128 rows, two workgroups per CU), so:
//  * a weight is one multiply-add, one exponential, one addition and half a
//    conversion; the masked tiles are a branch of their own (as selects the
//    mask and the cap that the general kernel can carry made 60 % of its
//    instructions);
//  * the weights' sum is that of the fp32 weights, a lane's four at a time (a
//    product of the rounded weights with ones is 0 to 2.5 % faster, 4096 rows
//    209.6 for 212.6 us, but drops 16 bits of each). Counting weights from a
//    maximum that may lag behind by 2^8 would save 3 % and round the largest
//    weight too (error against 64 bits 0.00203 for 0.00200);
//  * the row maximum joins lane groups by swapping lanes, not through LDS;
//  * heavy tiles start first: workgroups are numbered by tile from the last
//    one on, only over tiles that exist, heads fastest with the heads of a kv
//    head on one die. Batches of one tile a sequence come by number, which
//    takes no search and one launch (1000 prompts of 5 rows, 32 heads of 64:
//    116 us, 184 with the search, general kernel 169).
// The structure is the general kernel's: four waves of 32 rows, scores K Q^T
// so that a lane holds 16 keys of one query, O^T = V^T P^T with V read
// transposed, K and V in two LDS slots of 64 keys. (us, general kernel / this;
// 128 wide: 5 prompts of 4096 rows in all, 40 heads on 8, 145 / 77; 7 of 5000
// in all, 32 on 8, 145 / 65; 4 of 2048 441 / 178; one of 8192 1387 / 588, 935
// TFLOP/s; 512 rows after 8192 347 / 233; 40 heads, 32 of 128 rows 41 / 32; 64
// wide, 2 of 2048, 32 heads 164 / 58.)

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "attention_causal.h"

typedef __attribute__((ext_vector_type(8))) __bf16 ca_bf8;
typedef __attribute__((ext_vector_type(4))) float ca_f4;
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

namespace {

constexpr int WAVES = 4, BLOCK = 64 * WAVES;
constexpr int RG = 2;                // groups of 16 rows per wave
constexpr int BQ = 16 * RG * WAVES;  // rows of a workgroup
constexpr int BKV = 64, NF = BKV / 16;
constexpr int LISTED = 256;          // sequences of a launch at most
constexpr float LOG2E = 1.4426950408889634f;

struct Args {
  __hip_bfloat16 *out;
  long out_stride;
  const __hip_bfloat16 *q;
  long q_stride;
  const __hip_bfloat16 *k, *v;  // paged caches; else kv [T, Hq, 256] and
  const __hip_bfloat16 *pe;     // the shared key part [T, 64]
  const int *block_table;
  long max_pages;
  int page_size;
  const int *seq_lens, *qsl;
  int B, Hq, Hkv, min_rows;  // (min_rows: 1 or more)
  bool one_tile;  // no sequence has more rows: they come by number
  float scale;  // times log2 e
};

union CaFrag {
  ca_bf8 v;
  shortx4 h[2];
  __hip_bfloat16 e[8];
};

// 16 B units of a row are permuted so that 16 rows' units of one column fall
// on all banks
template <int ROW_B>
DEV_INLINE int swz(int row, int off) {
  if (ROW_B == 384) return off ^ (((row >> 1) & 7) << 4);
  constexpr int MASK = ROW_B / 16 - 1;
  return off ^ ((row & MASK) << 4);
}

// The `rank`th tile of 128 rows, last tiles of the longest sequences first;
// every wave finds it by itself. False past the end.
DEV_INLINE bool tile_at(int rank, const Args &P, int &b, int &tile) {
  const int lane = threadIdx.x & 63;
  constexpr int PER = LISTED / 64;
  int n[PER], most = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int s = i * 64 + lane;
    n[i] = 0;
    if (i * 64 < P.B && s < P.B) {
      const int rows = P.qsl[s + 1] - P.qsl[s];
      if (rows >= P.min_rows) n[i] = (rows + BQ - 1) / BQ;
    }
    most = max(most, n[i]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    most = max(most, __shfl_xor(most, off, 64));
  most = __builtin_amdgcn_readfirstlane(most);
  if (P.B == 1) {
    b = 0;
    tile = most - 1 - rank;
    return tile >= 0;
  }
  for (tile = most - 1; tile >= 0; --tile) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i * 64 >= P.B) break;
      const unsigned long long m = __ballot(n[i] > tile);
      const int c = __popcll(m);
      if (rank < c) {
        const int before = __builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        b = i * 64 + __ffsll(__ballot(n[i] > tile && before == rank)) - 1;
        return true;
      }
      rank -= c;
    }
  }
  return false;
}

// over the four lanes that hold a query's keys (lanes swap halves, then
// sixteens; two wait states after x is written)
DEV_INLINE float max_of_lanes(float x) {
  float y = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y));
  x = y = fmaxf(x, y);
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "+v"(y));
  return fmaxf(x, y);
}

template <int D, int DV, bool PAGED>
__global__ __launch_bounds__(BLOCK, 2) void causal_kernel(const Args P) {
  constexpr int KT = D / 32, NT = DV / 16;
  constexpr int KROW_B = D * 2, VROW_B = DV * 2;
  constexpr int TILE_B = BKV * KROW_B, SLOT_B = TILE_B + BKV * VROW_B;
  constexpr int GLK = TILE_B / 1024 / WAVES;  // 1 KB loads per wave
  constexpr int GLV = BKV * VROW_B / 1024 / WAVES;
  __shared__ __attribute__((aligned(16))) char ring[2 * SLOT_B];
  __shared__ int s_row[PAGED ? 2 * BKV : 1];  // cache rows of a tile's keys
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lhi = lane >> 4;

  const int Hq = P.Hq, G = Hq / P.Hkv;
  const int hx = blockIdx.x % Hq, kvh = hx % P.Hkv;
  const int h = kvh * G + hx / P.Hkv;
  int b = blockIdx.x / Hq, tile = 0;
  if (!P.one_tile) {
    if (!tile_at(blockIdx.x / Hq, P, b, tile)) return;
    b = __builtin_amdgcn_readfirstlane(b);
    tile = __builtin_amdgcn_readfirstlane(tile);
  }
  const int q_start = P.qsl[b], q_len = P.qsl[b + 1] - q_start;
  if (P.one_tile && q_len < P.min_rows) return;
  const int seq_len = PAGED ? P.seq_lens[b] : q_len;
  const int past = seq_len - q_len;
  const int kv_max = min(seq_len, past + (tile + 1) * BQ);
  const int nkt = (kv_max + BKV - 1) / BKV;

  // Loads straight into LDS, 1 KB per wave and load. Issued as inline
  // assembly: the loop orders them against the LDS reads itself (vmcnt, then
  // the barrier), and the compiler must not wait for the next tile ahead of
  // this tile's reads.
  const unsigned lds0 =
      (unsigned)(unsigned long)(__attribute__((address_space(3))) char *)
          ring + wave * 1024;
  auto load_lds = [&](const char *src, unsigned dst) {
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off"
        :
        : "v"(src), "s"(__builtin_amdgcn_readfirstlane(dst))
        : "memory", "m0");
  };
  // this lane's key of each load and its address in key 0 of the sequence
  int krow[GLK], kstep[GLK];
  const char *kbase[GLK];
#pragma unroll
  for (int j = 0; j < GLK; ++j) {
    const int p = (j * WAVES + wave) * 1024 + lane * 16;
    krow[j] = p / KROW_B;
    const int col = swz<KROW_B>(krow[j], p % KROW_B);
    if (PAGED) {
      kbase[j] = (const char *)(P.k + kvh * D) + col;
      kstep[j] = P.Hkv * KROW_B;
    } else if (col < 256) {
      kbase[j] = (const char *)(P.k + ((long)q_start * Hq + h) * 256) + col;
      kstep[j] = Hq * 512;
    } else {
      kbase[j] = (const char *)(P.pe + (long)q_start * 64) + col - 256;
      kstep[j] = 128;
    }
  }
  const int vrow0 = (wave * 1024 + lane * 16) / VROW_B;
  const int vcol = swz<VROW_B>(vrow0, lane * 16 % VROW_B);
  constexpr int VROWS = WAVES * 1024 / VROW_B;  // keys between two loads
  static_assert(VROWS % (VROW_B / 16) == 0, "one column for all loads");
  const char *vbase =
      PAGED ? (const char *)(P.v + kvh * DV) + vcol
            : (const char *)(P.v + ((long)q_start * Hq + h) * 256) + vcol;
  const int vstep = PAGED ? P.Hkv * VROW_B : Hq * 512;
  auto stage = [&](int t) {
    const unsigned base = lds0 + (t & 1) * SLOT_B;
    auto key = [&](int n) {
      // (a key past the end: the last one again, its scores are masked)
      return PAGED ? s_row[(t & 1) * BKV + n]
                   : min(t * BKV + n, seq_len - 1);
    };
#pragma unroll
    for (int j = 0; j < GLK; ++j)
      load_lds(kbase[j] + (long)key(krow[j]) * kstep[j],
               base + j * WAVES * 1024);
#pragma unroll
    for (int j = 0; j < GLV; ++j)
      load_lds(vbase + (long)key(vrow0 + j * VROWS) * vstep,
               base + TILE_B + j * WAVES * 1024);
  };

  const int *bt = PAGED ? P.block_table + b * P.max_pages : nullptr;
  const int page_size = P.page_size;
  int page_id = 0;  // block-table entry of this thread's key, next tile
  auto key_at = [&](int t) { return min(t * BKV + tid, seq_len - 1); };
  if (PAGED && tid < BKV) {
    const int j = key_at(0);
    s_row[tid] = bt[j / page_size] * page_size + j % page_size;
    if (nkt > 1) page_id = bt[key_at(1) / page_size];
  }

  // this lane's query per group: fragments, softmax state (log2 units)
  const int row0 = tile * BQ + wave * 16 * RG;  // first row of the wave
  const bool busy = row0 < q_len;
  ca_bf8 qf[RG][KT];
  float m_run[RG];
  ca_f4 l_run[RG];  // of this lane's keys; lanes join at the end
  ca_f4 o_acc[RG][NT];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int qrow = min(row0 + g * 16 + l16, q_len - 1);
    const __hip_bfloat16 *qp =
        P.q + (long)(q_start + qrow) * P.q_stride + h * D + lhi * 8;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      qf[g][kt] = *reinterpret_cast<const ca_bf8 *>(qp + kt * 32);
    m_run[g] = -INFINITY;
    l_run[g] = ca_f4{0, 0, 0, 0};
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o_acc[g][nt] = ca_f4{0, 0, 0, 0};
  }
  // what the loop reads from registers has arrived before it starts (a load
  // still pending here would make the loop wait for its own tiles)
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) asm volatile("" : "+v"(qf[g][kt]));
  asm volatile("" : "+v"(page_id));
  if (PAGED) __syncthreads();
  stage(0);

  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;
  const float scale = P.scale;
  for (int it = 0; it < nkt; ++it) {
    const int kv0 = it * BKV;
    // every wave's loads of this tile have landed; and every wave is done
    // with the other slot, which the next tile goes to
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (PAGED && tid < BKV && it + 1 < nkt)
      s_row[((it + 1) & 1) * BKV + tid] =
          page_id * page_size + key_at(it + 1) % page_size;
    __syncthreads();
    if (PAGED && tid < BKV && it + 2 < nkt)
      page_id = bt[key_at(it + 2) / page_size];
    if (it + 1 < nkt) stage(it + 1);
    // nothing in this tile that a row of this wave sees
    if (!busy || kv0 > past + row0 + 16 * RG - 1) continue;

    const char *ktile = ring + (it & 1) * SLOT_B;
    const char *vtile = ktile + TILE_B;
    // ---------- scores: [64 keys x 16 queries] per group ----------
    ca_f4 s[RG][NF];
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
      for (int f = 0; f < NF; ++f) s[g][f] = ca_f4{0, 0, 0, 0};
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int kr = f * 16 + l16;
        const ca_bf8 kf = *reinterpret_cast<const ca_bf8 *>(
            ktile + kr * KROW_B + swz<KROW_B>(kr, (kt * 32 + lhi * 8) * 2));
#pragma unroll
        for (int g = 0; g < RG; ++g)
          s[g][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[g][kt],
                                                            s[g][f], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);

    // ---------- mask: tiles at the diagonal ----------
    if (kv0 + BKV - 1 > past + row0) {
      asm volatile("");  // (a branch, not selects in every tile)
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        const int last = past + row0 + g * 16 + l16 - kv0 - lhi * 4;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            s[g][f][r] = f * 16 + r > last ? -INFINITY : s[g][f][r];
      }
    }
    // ---------- online softmax ----------
    CaFrag pf[RG][BKV / 32];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      float mx = s[g][0][0];
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[g][f][r]);
      mx = max_of_lanes(mx) * scale;
      if (__any(mx > m_run[g])) {
        const float m_new = fmaxf(m_run[g], mx);
        const float alpha = __builtin_amdgcn_exp2f(
            m_run[g] - (m_new == -INFINITY ? 0.f : m_new));
        m_run[g] = m_new;
#pragma unroll
        for (int r = 0; r < 4; ++r) l_run[g][r] *= alpha;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o_acc[g][nt][r] *= alpha;
      }
      const float base = m_run[g] == -INFINITY ? 0.f : m_run[g];
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(
              __builtin_fmaf(s[g][f][r], scale, -base));
          l_run[g][r] += p;
          pf[g][f >> 1].e[(f & 1) * 4 + r] = __float2bfloat16(p);
        }
    }

    // ---------- O^T += V^T P^T ----------
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < BKV / 32; ++ks) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        CaFrag vf;
#pragma unroll
        for (int half = 0; half < 2; ++half)
          vf.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_shortx4 *)const_cast<char *>(
                  vtile + (ks * 32 + half * 16 + tr_row) * VROW_B +
                  swz<VROW_B>(tr_row, nt * 32 + tr_col)));
#pragma unroll
        for (int g = 0; g < RG; ++g)
          o_acc[g][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf.v, pf[g][ks].v, o_acc[g][nt], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // ---------- lane = one query, 4 columns of each column tile ----------
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    float l = (l_run[g][0] + l_run[g][1]) + (l_run[g][2] + l_run[g][3]);
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int qrow = row0 + g * 16 + l16;
    if (qrow >= q_len) continue;
    const float inv_l = l > 0.f ? 1.f / l : 0.f;
    __hip_bfloat16 *op = P.out + (long)(q_start + qrow) * P.out_stride +
                         (long)h * DV + lhi * 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      CaFrag ov;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        ov.e[r] = __float2bfloat16(o_acc[g][nt][r] * inv_l);
      *reinterpret_cast<shortx4 *>(op + nt * 16) = ov.h[0];
    }
  }
}

template <int D, int DV, bool PAGED>
void launch(Args P, long T, long max_query_len) {
  const long q_tiles = (max_query_len + BQ - 1) / BQ;
  P.one_tile = q_tiles == 1;
  const int most = P.one_tile ? P.B : LISTED;
  auto stream = at::cuda::getCurrentCUDAStream();
  for (int left = P.B; left > 0; left -= most) {
    P.B = std::min(left, most);
    // tiles at most
    const long ranks = std::min(q_tiles * P.B, T / BQ + P.B);
    if (ranks <= 0) return;
    hipLaunchKernelGGL((causal_kernel<D, DV, PAGED>), dim3(ranks * P.Hq),
                       dim3(BLOCK), 0, stream, P);
    HIP_CHECK_KERNEL();
    P.qsl += P.B;
    if (PAGED) {
      P.seq_lens += P.B;
      P.block_table += P.B * P.max_pages;
    }
  }
}

}  // namespace

bool causal_prefill_ok(int D, int Dv, float scale) {
  return D == Dv && (D == 64 || D == 128) && scale > 0.f &&
         scale <= 1e30f;
}

// (operands checked by launch_prefill's callers)
void causal_prefill(void *out, long out_stride, const void *q, long q_stride,
                    const void *k_cache, const void *v_cache,
                    const int *block_table, long max_pages, int page_size,
                    const int *seq_lens, const int *qsl, int B, long T,
                    long max_query_len, int Hq, int Hkv, int D, float scale,
                    int min_rows) {
  Args P{};
  P.out = (__hip_bfloat16 *)out;
  P.out_stride = out_stride;
  P.q = (const __hip_bfloat16 *)q;
  P.q_stride = q_stride;
  P.k = (const __hip_bfloat16 *)k_cache;
  P.v = (const __hip_bfloat16 *)v_cache;
  P.block_table = block_table;
  P.max_pages = max_pages;
  P.page_size = page_size;
  P.seq_lens = seq_lens;
  P.qsl = qsl;
  P.B = B;
  P.Hq = Hq;
  P.Hkv = Hkv;
  P.scale = scale * LOG2E;
  P.min_rows = min_rows;
  if (D == 64) launch<64, 64, true>(P, T, max_query_len);
  else launch<128, 128, true>(P, T, max_query_len);
}

// Whole prompts: rows qsl[b] .. qsl[b + 1] of q [T, H * 192] (rotated), of kv
// [T, H * 256] (a head's 128 keys' and 128 values' columns) and of pe [T, 64]
// are the tokens of prompt b. Writes those rows of out [T, H * 128].
void mla_prompts(torch::Tensor out, torch::Tensor q, torch::Tensor kv,
                 torch::Tensor pe, torch::Tensor query_start_loc,
                 long max_query_len, double scale) {
  const long T = q.size(0), H = q.size(1) / 192;
  auto rows_ok = [&](const torch::Tensor &t, long cols) {
    return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 &&
           t.size(0) == T && t.size(1) == cols && t.stride(1) == 1 &&
           t.stride(0) % 8 == 0 &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  TORCH_CHECK(q.dim() == 2 && H > 0 && rows_ok(q, H * 192) &&
              rows_ok(out, H * 128) && rows_ok(kv, H * 256) &&
              kv.is_contiguous() && rows_ok(pe, 64) && pe.is_contiguous(),
              "mla_prompts: bf16 rows, 16 B aligned");
  TORCH_CHECK(query_start_loc.is_cuda() && query_start_loc.is_contiguous() &&
              query_start_loc.scalar_type() == at::kInt &&
              query_start_loc.numel() >= 2);
  TORCH_CHECK(scale > 0 && max_query_len <= T);
  if (T == 0) return;
  Args P{};
  P.out = (__hip_bfloat16 *)out.data_ptr();
  P.out_stride = out.stride(0);
  P.q = (const __hip_bfloat16 *)q.data_ptr();
  P.q_stride = q.stride(0);
  P.k = (const __hip_bfloat16 *)kv.data_ptr();
  P.v = P.k + 128;
  P.pe = (const __hip_bfloat16 *)pe.data_ptr();
  P.qsl = query_start_loc.data_ptr<int>();
  P.B = query_start_loc.numel() - 1;
  P.Hq = P.Hkv = H;
  P.scale = (float)scale * LOG2E;
  P.min_rows = 1;
  launch<192, 128, false>(P, T, max_query_len);
}
