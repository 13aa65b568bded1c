// Paged decode attention (single query token per sequence) for gfx950.
//
// Memory-bound: the job is to stream each sequence's K/V pages once at
// near-HBM rate. Structure:
//   grid = B * Hkv * splits, block = 256 threads (4 waves). A workgroup
//   serves the whole GQA group (up to 16 query heads) of one kv head over
//   a share of the keys, so K/V bytes are read once for all its heads.
//   From 257 workgroups to two rounds of them, if a sequence gives each of its
//   workgroups more than 1024 keys of 128 + 128 values (700 in a round of at
//   most 64 sequences) and lengths differ, heads are the fastest index (the
//   eight dies take workgroups in turn, so with 8 heads each die gets a share
//   of every sequence), then splits, and sequences come longest first
//   (sequence_at), so what starts last is short. More rounds even out by
//   themselves, and a workgroup per CU starts at once in any order. Finding
//   the sequence costs each workgroup 1 to 3 us, more than short shares give
//   back, and heads fastest is the slower one for equal lengths: there
//   sequences are the fastest index, as they come. (us, with the keys' own
//   step, 32 heads on 8 of 128, sequences fastest / this: 64 sequences of 512
//   to 1536 keys 58 / 55, 128 of 1024 to 3072 182 / 176, 24 of 2700 to 8100 in
//   four splits 116 / 106, 100 of 1 to 4000 149 / 143, 32 of 10 to 1500 in two
//   32.6 / 31.6; 40 heads, 24 of 2700 to 7900 114 / 102. What finding out costs
//   where it gives nothing: 24 of 5400 101.3 / 103.1, 128 of 520 to 1500 93.1 /
//   96.2, 64 of 1600 to 2048 87.2 / 88.9.)
//   Its waves work on their own: wave w takes the 32-key tiles w, w + 4,
//   ... of the share, with a softmax state of its own and no barrier in the
//   loop. K and V go straight to a patch of LDS that belongs to the wave, whole
//   rows at a time, their 16 B units permuted by the row. As soon as a tile's K
//   is in registers the next tile's takes its place, and so with V (read
//   transposed, ds_read_tr16_b64): 16 KB a wave are on their way, 128 KB a CU,
//   what two workgroups find room for. K by registers, in operand layout, costs
//   a quarter of a row a lane group and the copies: the loads alone took 50 us
//   so and 43 by whole rows (64 sequences of 1024 keys, 8 heads of 128; 41 at
//   6.5 TB/s), the kernel 55 and 49 now; 256 of 1024 175 / 164, 24 of 5400 in
//   four splits 104 / 96, 64 of 4096 201 / 178, 29 of 1024 in two 34 / 31.
//   Scores are K Q^T and the output is
//   O^T = V^T P^T, so a lane holds keys of ONE head: one softmax state per
//   lane, and the weights are the right operand of the second product as
//   they stand. At the end the waves join through LDS.
//   Split partials written fp32 + LSE; merge kernel combines splits and
//   converts to bf16 (reference semantics: merge_state / split-KV decode).
//   One split writes the result itself.
//   A mixed batch sends the sequences that bring one query row here: the
//   prefill kernel would spend a 128-row tile per head on each (37 such
//   rows of ~1024 keys, 40 heads, beside 4096 prompt tokens: 683 us a layer
//   there, 43 + 5 us here, and 193 for the prompts that remain).

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include <cstdlib>
#include "common.h"
#include "fp8_rows.h"
#include "qkv_rows.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 dec_bf8;
typedef __attribute__((ext_vector_type(4))) float dec_f4;
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int BLOCK = 256;
constexpr int WAVES = BLOCK / 64;
constexpr int TK = 32;            // keys per tile
constexpr float LOG2E = 1.4426950408889634f;

union DecFrag {
  dec_bf8 v;
  shortx4 h[2];
  __hip_bfloat16 e[8];
};

constexpr int ORDERED = 1024;  // workgroups at most: two rounds
constexpr int ALONE = 256;     // a CU each: all start at once, in any order
// Values of K and V a workgroup: up to here, order gives less than it takes.
// (FEW: a round of workgroups of at most 64 sequences, found the fastest)
constexpr int SHARE = 1024 * 256, SHARE_FEW = 700 * 256;

// The sequence whose visible keys come `rank`th, the most first, to within a
// sixteenth of the most (equal ones by number); -1 if half of them have more
// than seven eighths of the most: too alike to gain. Every wave finds it by
// itself. B <= ORDERED.
DEV_INLINE int sequence_at(int rank, int B, const int *seq_lens, int window,
                           const int *qsl) {
  const int lane = threadIdx.x & 63;
  constexpr int PER = ORDERED / 64;
  int keys[PER], most = 1;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int b = i * 64 + lane;
    keys[i] = -1;
    if (i * 64 < B && b < B) {
      keys[i] = max(seq_lens[b], 0);
      if (window > 0) keys[i] = min(keys[i], window);
      if (qsl && qsl[b + 1] - qsl[b] != 1) keys[i] = 0;
      most = max(most, keys[i]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    most = max(most, __shfl_xor(most, off, 64));
  int alike = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (i * 64 >= B) break;
    alike += __popcll(__ballot(keys[i] > most - (most >> 3)));
  }
  if (2 * alike >= B) return -1;
  const float unit = 15.999f / most;
#pragma unroll
  for (int i = 0; i < PER; ++i)
    keys[i] = keys[i] < 0 ? -1 : (int)(keys[i] * unit);
  for (int k = 15; k >= 0; --k) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i * 64 >= B) break;
      const unsigned long long m = __ballot(keys[i] == k);
      const int n = __popcll(m);
      if (rank < n) {
        const int before = __builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        return i * 64 +
               __ffsll(__ballot(keys[i] == k && before == rank)) - 1;
      }
      rank -= n;
    }
  }
  return 0;  // (not reached: every key is in 0 .. 15)
}

// global -> LDS, 16 B a lane, non-temporal (a cached row is read by one wave)
DEV_INLINE void fetch16(const char *src, char *dst) {
  __builtin_amdgcn_global_load_lds(
      reinterpret_cast<const unsigned int *>(src),
      reinterpret_cast<unsigned int *>(dst), 16, 0, 2);
}

DEV_INLINE void fetch4(const int *src, int *dst) {
  __builtin_amdgcn_global_load_lds(
      reinterpret_cast<const unsigned int *>(src),
      reinterpret_cast<unsigned int *>(dst), 4, 0, 0);
}

template <int LEFT>
DEV_INLINE void wait_loads() {  // until at most LEFT are on their way
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LEFT) : "memory");
}

// What an instance that starts from the projection takes beside the caches.
struct NewRows {
  QkvRows rows;                    // q | k | v of each sequence's new token
  __hip_bfloat16 *k_cache, *v_cache;
  const long *slots;               // [B] where its key and value go
  int *arrived;                    // [B, Hkv] zeros, left as zeros
  Fp8Out fp8;                      // the result's e4m3 rows (heads of 128)
  // tiles up to which a sequence is not split, and a split's at least
  int whole, least;
};

// partials pass from one workgroup to another within a launch: written
// through to where every die reads them
DEV_INLINE void publish(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum_s w_s o_s, w the softmax of the splits' scores (and of `sink`, which has
// no value); scores of -inf take no part. AGENT: published by this launch.
// MOST partials are read at once; more than that only where it is 16, the most
// that the launcher chooses beside a kept-first segment (code for sixteen
// where there are two costs a merge 1 us: 64 sequences of 64 heads 3.9, 4.9)
template <bool AGENT, int MOST = 16>
DEV_INLINE float merged(const float *o, long o_stride, const float *lse,
                        long lse_stride, int n, float sink) {
  auto at = [](const float *p) {
    return AGENT ? __hip_atomic_load(p, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT)
                 : *p;
  };
  float x[MOST], v[MOST], mx = sink;
#pragma unroll
  for (int s = 0; s < MOST; ++s)
    if (s < n) {
      x[s] = at(lse + s * lse_stride);
      v[s] = at(o + s * o_stride);
    }
#pragma unroll
  for (int s = 0; s < MOST; ++s)
    if (s < n) mx = fmaxf(mx, x[s]);
  if constexpr (MOST == 16)
    for (int s = 16; s < n; ++s) mx = fmaxf(mx, at(lse + s * lse_stride));
  float denom = sink == -INFINITY ? 0.f : __expf(sink - mx), sum = 0.f;
  auto join = [&](float score, float value) {
    if (score == -INFINITY) return;  // (its values are not written)
    const float w = __expf(score - mx);
    denom += w;
    sum += w * value;
  };
#pragma unroll
  for (int s = 0; s < MOST; ++s)
    if (s < n) join(x[s], v[s]);
  if constexpr (MOST == 16)
    for (int s = 16; s < n; ++s)
      join(at(lse + s * lse_stride), at(o + s * o_stride));
  return denom > 0.f ? sum / denom : 0.f;
}

// Head sizes Dr <= D, Dvr <= DV (multiples of 8; D, DV 64 or 128): columns
// beyond a head are zero. G query heads per kv head, rows of the products
// beyond G are zero. Optional bias by distance and query temperature.
// FRESH: the step from the projection's rows in one launch. Each workgroup
// forms its heads' queries and the new key and value (in LDS; the first
// split's workgroup stores them to the caches), and the last of a sequence's
// workgroups to end joins their partials. (No bias, cap, gate, sink or
// temperature; one query row per sequence.)
template <int D, int DV, bool FRESH = false>
__global__ __launch_bounds__(BLOCK, 2) void paged_decode_kernel(
    float *__restrict__ partial_out,  // [S, B, Hq, Dvr]
    float *__restrict__ partial_lse,  // [S, B, Hq]
    const __hip_bfloat16 *__restrict__ q,        // [B, Hq, Dr]
    const __hip_bfloat16 *__restrict__ k_cache,  // [P, ps, Hkv, Dr]
    const __hip_bfloat16 *__restrict__ v_cache,  // [P, ps, Hkv, Dvr]
    const int *__restrict__ block_table, const int *__restrict__ seq_lens,
    int max_pages, int page_size, int num_kv_heads, int G, int Dr, int Dvr,
    float scale, int num_splits, long q_stride, int window, int keep_first,
    float softcap, const float *__restrict__ bias, int bias_len,
    float temp_coef, int temp_every,
    // rows of a mixed batch: [B + 1]; sequences of other than one query row
    // are left alone
    const int *__restrict__ qsl,
    // one split: the result itself, bf16 [rows, Hq * Dvr]
    __hip_bfloat16 *__restrict__ out, long out_stride, int sink,
    const float *__restrict__ sinks, const __hip_bfloat16 *__restrict__ gate,
    long gate_stride, int B, int zdim,
    // keys from which on the order of sequences matters
    int order_above, const NewRows fresh) {
  constexpr int KT = D / 32, NT = DV / 16;
  // 16 B units per lane, LDS row bytes, the rows that permute them
  constexpr int KU = TK * (D / 8) / 64, VU = TK * (DV / 8) / 64;
  constexpr int KROW = D * 2, VROW = DV * 2;
  constexpr int KMASK = (D / 8 - 1) & 15, VMASK = (DV / 8 - 1) & 15;
  if constexpr (FRESH) {
    softcap = temp_coef = 0.f;
    bias = sinks = nullptr;
    gate = nullptr;
    qsl = nullptr;
    keep_first = sink = 0;
    zdim = num_splits;
  }
  // (zdim: splits, and the kept-first segment)
  const int rest = blockIdx.x / B;
  int b = blockIdx.x - rest * B, kvh = rest % num_kv_heads;
  int split = rest / num_kv_heads;
  int seq_len = seq_lens[b];
  if (B > 1 && gridDim.x > ALONE && gridDim.x <= ORDERED) {
    bool order = false;
    if (window <= 0 || window > order_above)
      for (int i = threadIdx.x & 63; i < B; i += 256) {  // loads in fours
        int n = seq_lens[i];
#pragma unroll
        for (int j = 1; j < 4; ++j)
          n = max(n, seq_lens[min(i + j * 64, B - 1)]);
        order |= n > order_above;
      }
    if (__any(order)) {
      const int of_heads = blockIdx.x / num_kv_heads;
      const int s = __builtin_amdgcn_readfirstlane(
          sequence_at(of_heads / zdim, B, seq_lens, window, qsl));
      if (s >= 0) {
        b = s;
        kvh = blockIdx.x - of_heads * num_kv_heads;
        split = of_heads % zdim;
        seq_len = seq_lens[b];
      }
    }
  }
  const int Hq = num_kv_heads * G;
  const int row = qsl ? qsl[b] : b;  // of q and of the result
  if (qsl && qsl[b + 1] - row != 1) return;
  const int w_begin = (window > 0) ? max(0, seq_len - window) : 0;
  // this split's share of the visible keys, whole tiles
  const int tiles = (seq_len - w_begin + TK - 1) / TK;
  const int even = (tiles + num_splits - 1) / num_splits;
  const int split_len =
      TK * (!FRESH ? even
                   : tiles <= fresh.whole ? tiles : max(even, fresh.least));
  // split == num_splits (launched only when keep_first > 0) is the
  // kept-first segment [0, min(keep_first, w_begin)): tokens that stay
  // visible outside the window; its partial merges like any other
  const bool kept = split == num_splits;
  const int t0 = kept ? 0 : w_begin + split * split_len;
  const int t1 = kept ? min(keep_first, w_begin)
                      : min(t0 + split_len, seq_len);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lhi = lane >> 4;
  const long lse0 = (long)split * B * Hq + (long)b * Hq + kvh * G;
  if (FRESH && t0 >= t1 && split > 0) return;
  if (!FRESH && t0 >= t1) {
    // empty split: publish -inf lse so the merge ignores it
    if (out) {
      for (int i = tid; i < G * Dvr; i += BLOCK)
        out[row * out_stride + (long)kvh * G * Dvr + i] =
            __float2bfloat16(0.f);
    } else if (tid < G) {
      partial_lse[lse0 + tid] = -INFINITY;
    }
    return;
  }
  // a patch per wave: its V tile (later its output, as many bytes), its K tile
  __shared__ __attribute__((aligned(16))) char
      patch[WAVES][TK * (VROW + KROW)];
  __shared__ float s_m[WAVES][16], s_l[WAVES][16];

  const int *bt = block_table + (long)b * max_pages;
  const float *brow =
      bias ? bias + (long)(kvh * G + min(l16, G - 1)) * bias_len : nullptr;
  char *mine = patch[wave], *mine_k = mine + TK * VROW;
  float bn[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Cache row of key lane & 31 of a tile, its page looked up a tile ahead, into
  // LDS like K and V: behind the next K and before the next V, so that the
  // waits below can count what was issued behind what they need.
  __shared__ int pages[WAVES][64];
  int in_page = 0, krow = 0, rows[KU];
  const unsigned k_bytes = num_kv_heads * Dr * 2;
  const unsigned v_bytes = num_kv_heads * Dvr * 2;
  const char *k_head = reinterpret_cast<const char *>(k_cache + kvh * Dr);
  const char *v_head = reinterpret_cast<const char *>(v_cache + kvh * Dvr);
  auto look_up = [&](int k0) {
    const int key = min(k0 + (lane & 31), t1 - 1), page = key / page_size;
    in_page = key - page * page_size;
    fetch4(bt + page, pages[wave]);
  };
  // (columns beyond a head repeat its last unit)
  auto next_row = [&]() { krow = pages[wave][lane] * page_size + in_page; };
  auto load_k = [&](int k0) {
    // a table entry per key of this lane
    if (brow) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        bn[e] = brow[min(max(seq_len - 1 - (k0 + (e >> 2) * 16 + lhi * 4 +
                                            (e & 3)), 0), bias_len - 1)];
    }
#pragma unroll
    for (int j = 0; j < KU; ++j)
      rows[j] = __shfl(krow, (j * 64 + lane) / (D / 8), 64);
#pragma unroll
    for (int j = 0; j < KU; ++j) {
      const int u = j * 64 + lane, r = u / (D / 8);
      const int c = ((u % (D / 8)) ^ (r & KMASK)) * 8;
      fetch16(k_head + (unsigned long)(unsigned)rows[j] * k_bytes +
                  min(c, Dr - 8) * 2,
              mine_k + j * 1024);
    }
  };
  auto load_v = [&]() {
#pragma unroll
    for (int j = 0; j < VU; ++j) {
      const int u = j * 64 + lane, r = u / (DV / 8);
      const int row = D == DV ? rows[j % KU] : __shfl(krow, r, 64);
      const int c = ((u % (DV / 8)) ^ (r & VMASK)) * 8;
      fetch16(v_head + (unsigned long)(unsigned)row * v_bytes +
                  min(c, Dvr - 8) * 2,
              mine + j * 1024);
    }
  };
  float qscale = scale * query_temp(seq_len - 1, temp_coef, temp_every);
  // with a cap the exponent of tanh, else the score in log2 units
  qscale *= softcap > 0.f ? 2.f * LOG2E / softcap : LOG2E;
  const float cap2 = softcap * LOG2E;
  float m_run = -INFINITY, l_run = 0.f;
  dec_f4 o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) o[nt] = dec_f4{0, 0, 0, 0};
  const int tr_row = lhi * 4 + (l16 >> 2), tr_col = (l16 & 3) * 8;

  // query fragments: column l16 = head, dims kt * 32 + lhi * 8
  dec_bf8 qf[KT];
  auto load_q = [&](const __hip_bfloat16 *heads, int stride) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      qf[kt] = dec_bf8{0, 0, 0, 0, 0, 0, 0, 0};
      if (l16 < G && kt * 32 + lhi * 8 < Dr)
        qf[kt] = *reinterpret_cast<const dec_bf8 *>(heads + l16 * stride +
                                                    kt * 32 + lhi * 8);
    }
  };
  if constexpr (!FRESH)
    load_q(q + (long)row * q_stride + (long)kvh * G * Dr, Dr);
  int k0 = t0 + wave * TK;
  if (k0 < t1) {
    const int key = min(k0 + (lane & 31), t1 - 1), page = key / page_size;
    krow = bt[page] * page_size + key - page * page_size;
    load_k(k0);
    if (k0 + WAVES * TK < t1) look_up(k0 + WAVES * TK);
    load_v();
  }
  // FRESH: the new rows are formed while the first tiles arrive
  __shared__ __attribute__((aligned(16))) short
      own[FRESH ? (16 + 2) * D : 8];  // G queries, the key, the value
  if constexpr (FRESH) {
    const int per = Dr / 8;
    for (int i = tid; i < (G + 2) * per; i += BLOCK) {
      const int h = i / per;
      const int col = h < G ? kvh * G + h : Hq + kvh + (h - G) * num_kv_heads;
      const QkvUnit x = qkv_unit<true>(fresh.rows, b, col, i - h * per,
                                       h <= G, Hq + 2 * num_kv_heads, Dr);
      *reinterpret_cast<shortx4 *>(own + h * D + x.d1) = x.o1;
      *reinterpret_cast<shortx4 *>(own + h * D + x.d2) = x.o2;
      if (h >= G && split == 0) {
        __hip_bfloat16 *dst =
            (h == G ? fresh.k_cache : fresh.v_cache) +
            (fresh.slots[b] * num_kv_heads + kvh) * Dr;
        *reinterpret_cast<shortx4 *>(dst + x.d1) = x.o1;
        *reinterpret_cast<shortx4 *>(dst + x.d2) = x.o2;
      }
    }
    __syncthreads();
    if (t0 >= t1) {  // (a sequence without keys)
      for (int i = tid; i < G * Dvr; i += BLOCK) {
        out[row * out_stride + (long)kvh * G * Dvr + i] =
            __float2bfloat16(0.f);
        if (fresh.fp8.q)
          fresh.fp8.q[row * (long)Hq * Dvr + kvh * G * Dvr + i] = 0;
        if (fresh.fp8.q && i % 128 == 0)
          fresh.fp8.scales[(long)(kvh * G + i / 128) * B + row] =
              fp8_scale(0.f);
      }
      return;
    }
  }
  if constexpr (FRESH) load_q(reinterpret_cast<const __hip_bfloat16 *>(own), D);
  // (here, or each pass of the loop would wait for all that is on its way)
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) asm volatile("" : "+v"(qf[kt]));
  for (; k0 < t1; k0 += WAVES * TK) {
    const bool more = k0 + WAVES * TK < t1;
    DecFrag kf[2][KT];
    float bv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bv[e] = bn[e] * LOG2E;
    wait_loads<VU>();
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        kf[f][kt].v = *reinterpret_cast<const dec_bf8 *>(
            mine_k + (f * 16 + l16) * KROW +
            ((kt * 64 + lhi * 16) ^ ((l16 & KMASK) << 4)));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) {
      next_row();
      load_k(k0 + WAVES * TK);
      look_up(k0 + 2 * WAVES * TK);
    }
    if (FRESH && k0 + TK >= seq_len) {
      // the new token's row comes from LDS, and so does what stands behind
      // it in the tile (the cache's row may not be written yet)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          if (k0 + f * 16 + l16 >= seq_len - 1 && kt * 32 + lhi * 8 < Dr)
            kf[f][kt].v = *reinterpret_cast<const dec_bf8 *>(
                own + G * D + kt * 32 + lhi * 8);
    }
    if (Dr < D) {
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          if (kt * 32 + lhi * 8 >= Dr)
            kf[f][kt].v = dec_bf8{0, 0, 0, 0, 0, 0, 0, 0};
    }

    dec_f4 s[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) s[f] = dec_f4{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int f = 0; f < 2; ++f)
        s[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[f][kt].v, qf[kt],
                                                       s[f], 0, 0, 0);
    // lane: head l16, keys k0 + f * 16 + lhi * 4 + r
    float mx = -INFINITY;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = k0 + f * 16 + lhi * 4 + r;
        float x = s[f][r] * qscale;
        if (softcap > 0.f)  // cap tanh(x / cap) from one exponential
          x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(
                                      1.f + __builtin_amdgcn_exp2f(x));
        if (brow) x += bv[f * 4 + r];
        s[f][r] = tok < t1 ? x : -INFINITY;
        mx = fmaxf(mx, s[f][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // (the tile's first key is visible: m_new is finite)
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    DecFrag pf;
    float sum = 0.f;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(s[f][r] - m_new);
        sum += p;
        pf.e[f * 4 + r] = __float2bfloat16(p);
      }
    l_run = l_run * alpha + sum;  // this lane's keys; joined at the end
    if (more)
      wait_loads<KU + 1>();
    else
      wait_loads<0>();
    if (FRESH && k0 + TK >= seq_len) {
#pragma unroll
      for (int j = 0; j < VU; ++j) {
        const int u = j * 64 + lane, r = u / (DV / 8), c = u % (DV / 8);
        if (k0 + r >= seq_len - 1 && c * 8 < Dvr)
          *reinterpret_cast<shortx8 *>(mine + r * VROW +
                                       ((c ^ (r & VMASK)) << 4)) =
              *reinterpret_cast<const shortx8 *>(own + (G + 1) * D + c * 8);
      }
    }
    DecFrag vf[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int half = 0; half < 2; ++half)
        vf[nt].h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_shortx4 *)(mine + (half * 16 + tr_row) * VROW +
                            ((nt * 32 + tr_col) ^
                             ((tr_row & VMASK) << 4))));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) load_v();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[nt][r] *= alpha;
      o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[nt].v, pf.v, o[nt],
                                                      0, 0, 0);
    }
  }

  // ---------- the waves join ----------
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (lhi == 0) {
    s_m[wave][l16] = m_run;
    s_l[wave][l16] = l_run;
  }
  float *mo = reinterpret_cast<float *>(mine);  // [column][lane]
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 4; ++r) mo[(nt * 4 + r) * 64 + lane] = o[nt][r];
  __syncthreads();
  // FRESH: what is written, in LDS for its e4m3 form (a head is a group)
  auto keep = [&](int idx, __hip_bfloat16 v) {
    if (FRESH && fresh.fp8.q) own[idx] = __builtin_bit_cast(short, v);
  };
  auto write_fp8 = [&]() {
    if constexpr (FRESH && DV == 128) {
      if (!fresh.fp8.q) return;
      __syncthreads();
      for (int h = wave; h < G; h += WAVES) {
        float v[2], amax = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          v[i] = __bfloat162float(
              __builtin_bit_cast(__hip_bfloat16, own[h * 128 + lane * 2 + i]));
          amax = fmaxf(amax, fabsf(v[i]));
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
          amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const float scale = fp8_scale(amax), inv = 1.f / scale;
        const long head = kvh * G + h;
        *reinterpret_cast<unsigned short *>(
            fresh.fp8.q + ((long)row * Hq + head) * 128 + lane * 2) =
            fp8_byte(v[0] * inv) | fp8_byte(v[1] * inv) << 8;
        if (lane == 0) fresh.fp8.scales[head * B + row] = scale;
      }
    }
  };
  // workgroups that have keys of this sequence (one: it writes the result)
  const int live = (tiles * TK + split_len - 1) / split_len;
  for (int idx = tid; idx < G * Dvr; idx += BLOCK) {
    const int h = idx / Dvr, d = idx % Dvr;
    const int at = ((d >> 4) * 4 + (d & 3)) * 64 + ((d >> 2) & 3) * 16 + h;
    float m = s_m[0][h];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = fmaxf(m, s_m[w][h]);
    float l = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float e = __builtin_amdgcn_exp2f(s_m[w][h] - m);  // idle wave: 0
      l += e * s_l[w][h];
      acc += e * reinterpret_cast<const float *>(patch[w])[at];
    }
    if (FRESH ? live == 1 : out != nullptr) {  // the only split
      if (sinks || sink)
        l += __builtin_amdgcn_exp2f(
            (sinks ? sinks[kvh * G + h] : 0.f) * LOG2E - m);
      const long col = (long)(kvh * G + h) * Dvr + d;
      float res = acc / l;
      if (gate)
        res *= 1.f / (1.f + __expf(-__bfloat162float(
                                 gate[row * gate_stride + col])));
      const __hip_bfloat16 r = __float2bfloat16(res);
      out[row * out_stride + col] = r;
      keep(idx, r);
      continue;
    }
    const float lse = m / LOG2E + __logf(l);
    if constexpr (FRESH) {
      publish(&partial_out[(lse0 + h) * Dvr + d], acc / l);
      if (d == 0) publish(&partial_lse[lse0 + h], lse);
    } else {
      partial_out[(lse0 + h) * Dvr + d] = acc / l;
      if (d == 0) partial_lse[lse0 + h] = lse;
    }
  }
  if constexpr (FRESH) {
    if (live == 1) {
      write_fp8();
      return;
    }
    // Every wave's partials are where all dies see them before the count
    // goes up, and they are read there (a fence here would empty the L2 that
    // the other workgroups' keys pass through: 24 of 5400 keys in four splits
    // 30 us a launch).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int *last = reinterpret_cast<int *>(&s_m[0][0]);
    if (tid == 0) {
      int *at = fresh.arrived + b * num_kv_heads + kvh;
      const int before = __hip_atomic_fetch_add(at, 1, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
      *last = before == live - 1;
      if (before == live - 1)
        __hip_atomic_store(at, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*last) return;
    const long of_split = (long)B * Hq;
    for (int idx = tid; idx < G * Dvr; idx += BLOCK) {
      const int h = idx / Dvr, d = idx % Dvr;
      const long at = (long)b * Hq + kvh * G + h;
      const __hip_bfloat16 r = __float2bfloat16(
          merged<true>(partial_out + at * Dvr + d, of_split * Dvr,
                       partial_lse + at, of_split, live, -INFINITY));
      out[row * out_stride + (long)(kvh * G + h) * Dvr + d] = r;
      keep(idx, r);
    }
    write_fp8();
  }
}

// Merge split partials: out[b,h,:] = sum_s w_s * partial[s,b,h,:];
// a thread per column of the head. MOST: see merged
template <int MOST>
__global__ void decode_merge_kernel(
    __hip_bfloat16 *__restrict__ out,       // [B, Hq, D] (row stride)
    long out_stride,
    const float *__restrict__ partial_out,  // [S, B, Hq, D]
    const float *__restrict__ partial_lse,  // [S, B, Hq]
    int num_splits, int Hq, int sink,
    const __hip_bfloat16 *__restrict__ gate, long gate_stride,
    const float *__restrict__ sinks, const int *__restrict__ qsl) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int row = qsl ? qsl[b] : b;
  if (qsl && qsl[b + 1] - row != 1) return;
  const int d = threadIdx.x, D = blockDim.x;
  const int B = gridDim.x;
  // sink: one more "partial" with lse 0 (or the head's learned score) and no
  // value
  const long at = (long)b * Hq + h, of_split = (long)B * Hq;
  float res = merged<false, MOST>(
      partial_out + at * D + d, of_split * D, partial_lse + at, of_split,
      num_splits, sinks ? sinks[h] : sink ? 0.f : -INFINITY);
  if (gate != nullptr) {
    const float z =
        __bfloat162float(gate[(long)row * gate_stride + (long)h * D + d]);
    res *= 1.f / (1.f + __expf(-z));
  }
  out[(long)row * out_stride + (long)h * D + d] = __float2bfloat16(res);
}

bool decode_shape_ok(const torch::Tensor &k_cache,
                     const torch::Tensor &v_cache, int G) {
  const int D = k_cache.size(3), Dv = v_cache.size(3);
  return D % 8 == 0 && Dv % 8 == 0 && D <= 128 && Dv <= 128 && G >= 1 &&
         G <= 16 && v_cache.size(0) == k_cache.size(0) &&
         v_cache.size(1) == k_cache.size(1) &&
         v_cache.size(2) == k_cache.size(2) &&
         reinterpret_cast<uintptr_t>(k_cache.data_ptr()) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(v_cache.data_ptr()) % 16 == 0;
}

// Workgroups that share the keys of one sequence and kv head.
int splits_for(const torch::Tensor &k_cache, long B) {
  const long Hkv = k_cache.size(2);
  // the longest sequence the pool can hold bounds the useful splits; the
  // count depends on the batch size only (a captured launch serves every
  // length)
  const long max_seq_len = (long)k_cache.size(0) * k_cache.size(1);
  static int splits_env = [] {
    const char *e = getenv("GLLM_DECODE_SPLITS");
    return e ? atoi(e) : 0;
  }();
  // Two workgroups fit a CU. Twice as many would even unequal requests out
  // a little better (24 of 2700 to 7900 keys, 8 heads: 100 us in eight splits,
  // 102 in four) and are as exact: error against 64 bits 2.13e-3 in one split, 2.09e-3 in
  // two; 2.15e-3 in four, 2.11e-3 in eight. But each split rounds its
  // probabilities to bf16 against its own maximum, so another count is
  // another result, and behind products that quantize their rows to e4m3 it
  // moves a two-layer model's outputs by 3 % (0.0355 off 64 bits with either
  // count): the count stays the smallest that fills the chip.
  int splits = 1;
  while (splits < 16 && B * Hkv * splits < 512 &&
         splits * 2 <= (max_seq_len + 127) / 128)
    splits *= 2;
  if (splits_env > 0) splits = splits_env;
  return splits;
}

void launch_decode(torch::Tensor &out, const torch::Tensor &q,
                   const torch::Tensor &k_cache, const torch::Tensor &v_cache,
                   const torch::Tensor &block_table,
                   const torch::Tensor &seq_lens, int G, float scale,
                   int window, int keep_first = 0, bool sink = false,
                   const void *gate = nullptr, long gate_stride = 0,
                   const float *sinks = nullptr, float softcap = 0.f,
                   const float *bias = nullptr, int bias_len = 0,
                   float temp_coef = 0.f, int temp_every = 0,
                   const int *qsl = nullptr,
                   const NewRows *fresh = nullptr) {
  // (lengths past a step's own rows are not looked at; q: the result's
  // tensor where the rows are fresh)
  const int B = qsl ? seq_lens.size(0) : q.size(0);
  const int Hkv = k_cache.size(2), Hq = Hkv * G;
  const int D = k_cache.size(3), Dv = v_cache.size(3);
  const int splits = splits_for(k_cache, B);
  auto opts = q.options().dtype(at::kFloat);
  // + 1: the kept-first segment of a windowed layer
  const int zdim = splits + ((keep_first > 0 && window > 0) ? 1 : 0);
  const long out_stride =
      out.dim() == 2 ? (long)out.stride(0) : (long)Hq * Dv;
  // one split writes the result itself
  torch::Tensor partial, lse;
  float *po = nullptr, *pl = nullptr;
  auto *direct = (__hip_bfloat16 *)out.data_ptr();
  if (zdim > 1) {
    partial = torch::empty({zdim, B, Hq, Dv}, opts);
    lse = torch::empty({zdim, B, Hq}, opts);
    po = partial.data_ptr<float>();
    pl = lse.data_ptr<float>();
    if (!fresh) direct = nullptr;
  }
  const bool few = B <= 64 && B * Hkv * zdim <= ORDERED / 2;
  const int order_above = (few ? SHARE_FEW : SHARE) / (D + Dv) * splits;
  auto stream = at::cuda::getCurrentCUDAStream();
#define RUN(...)                                                             \
  hipLaunchKernelGGL((paged_decode_kernel<__VA_ARGS__>),                     \
                     dim3(B * Hkv * zdim), dim3(BLOCK), 0, stream, po, pl,   \
                     (const __hip_bfloat16 *)q.data_ptr(),                   \
                     (const __hip_bfloat16 *)k_cache.data_ptr(),             \
                     (const __hip_bfloat16 *)v_cache.data_ptr(),             \
                     block_table.data_ptr<int>(), seq_lens.data_ptr<int>(),  \
                     (int)block_table.stride(0), (int)k_cache.size(1), Hkv,  \
                     G, D, Dv, scale, splits, (long)q.stride(0), window,     \
                     keep_first, softcap, bias, bias_len, temp_coef,         \
                     temp_every, qsl, direct, out_stride, sink ? 1 : 0,      \
                     sinks, (const __hip_bfloat16 *)gate, gate_stride, B,    \
                     zdim, order_above, rows)
  // A split's rows, partials and the join take 3 us, as long as a wave takes
  // for one or two tiles while most of the chip idles, for two to four in one
  // round of workgroups and for six beside others; a sequence stays whole up
  // to twice that in a round, and beyond up to eight tiles a wave, ten where
  // the sequences by themselves nearly fill a round (us, 40 heads on 8 of 128,
  // every sequence over all splits / so: 4 of 520 to 1500 keys 17.7 / 15.2, 16
  // of 150 to 450 15.8 / 12.8, 12 of them 22.6 / 12.6, 12 of 520 to 1500 28.4 /
  // 21.2, 24 of 60 to 180 21.1 / 10.2, 31 of 150 to 450 25.8 / 14.7, 60 of 600
  // 40.2 / 30.5, 9 of 5400 46.9 / 43.8; 24 of 2700 to 7900 102.5 / 102.8. 24
  // tiles in one round: 8 of 520 to 1500 20.4 for 18.8; 16 beyond: 60 of 600
  // 40.2. Whole up to 24 / 32 / 40 / 48 tiles beyond a round: 24 of 1000 27.5 /
  // 24.0 / 23.9 / 24.0, of 520 to 1500 31.5 / 31.5 / 34.0 / 28.0, 40 of 440 to
  // 1270 44.3 / 44.0 / 39.7 / 39.8, of 770 to 2240 66.7 / 64.2 / 69.2 / 70.8,
  // 60 of 520 to 1500 59.6 / 58.4 / 56.4 / 54.2, of 1150 to 3400 114.1 /
  // 115.0 / 115.1 / 119.1). Rounded rows stand behind e4m3 products: there the
  // count stays (splits_for).
  NewRows rows = fresh ? *fresh : NewRows{};
  if (fresh && !fresh->rows.rounded) {
    const long all = (long)B * Hkv * splits;
    rows.whole = all <= ALONE ? 8 : all <= 2 * ALONE ? 16
                 : 5L * B * Hkv >= 7 * ALONE ? 40 : 32;
    rows.least = all <= ALONE ? 4 : all <= 2 * ALONE ? 8 : 24;
  }
  if (fresh) { if (D <= 64) RUN(64, 64, true); else RUN(128, 128, true); }
  else if (D <= 64) { if (Dv <= 64) RUN(64, 64); else RUN(64, 128); }
  else { if (Dv <= 64) RUN(128, 64); else RUN(128, 128); }
#undef RUN
  HIP_CHECK_KERNEL();
  if (zdim == 1 || fresh) return;
#define RUN(MOST)                                                            \
  hipLaunchKernelGGL((decode_merge_kernel<MOST>), dim3(B, Hq), dim3(Dv), 0,  \
                     stream, (__hip_bfloat16 *)out.data_ptr(), out_stride,   \
                     po, pl, zdim, Hq, sink ? 1 : 0,                         \
                     (const __hip_bfloat16 *)gate, gate_stride, sinks, qsl)
  if (zdim <= 2) RUN(2);
  else if (zdim <= 4) RUN(4);
  else if (zdim <= 8) RUN(8);
  else RUN(16);
#undef RUN
  HIP_CHECK_KERNEL();
}

}  // namespace

void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_table, torch::Tensor seq_lens,
                            double scale, long sliding_window,
                            c10::optional<torch::Tensor> query_start_loc) {
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "decode attn: bf16 only");
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2),
              "q per-token row must be contiguous");
  TORCH_CHECK(block_table.scalar_type() == at::kInt);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  const int Hq = q.size(1), Hkv = k_cache.size(2);
  if (q.size(0) == 0) return;
  TORCH_CHECK(Hq % Hkv == 0 && q.size(2) == k_cache.size(3));
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              decode_shape_ok(k_cache, v_cache, Hq / Hkv),
              "paged_attention_decode: unsupported head_dim=", q.size(2),
              " group=", Hq / Hkv);
  const int *qsl = nullptr;
  if (query_start_loc.has_value()) {
    TORCH_CHECK(query_start_loc->scalar_type() == at::kInt &&
                query_start_loc->is_contiguous() &&
                query_start_loc->numel() == seq_lens.numel() + 1);
    qsl = query_start_loc->data_ptr<int>();
  } else {
    TORCH_CHECK(seq_lens.numel() >= q.size(0), "a length per query row");
  }
  TORCH_CHECK(block_table.size(0) >= (qsl ? seq_lens.numel() : q.size(0)));
  launch_decode(out, q, k_cache, v_cache, block_table, seq_lens, Hq / Hkv,
                (float)scale, (int)sliding_window, 0, false, nullptr, 0,
                nullptr, 0.f, nullptr, 0, 0.f, 0, qsl);
}

bool decode_rows_ok(torch::Tensor k_cache, torch::Tensor v_cache, long Hq);

// One decode token per sequence from the fp32 parts [S, B, (Hq + 2 Hkv) D] of
// the merged q | k | v projection: bias, rotation (rotate-half on the first
// rot columns), keys and values to their slots, which must be the last of
// their sequence's (block table, length), and attention, in one launch;
// bf16 [B, Hq * D]. rounded: the biased rows are rounded to bf16 first.
// arrived: int32 zeros, one per sequence and kv head, left as zeros; launches
// that may overlap need their own.
static torch::Tensor decode_rows(
    torch::Tensor parts, c10::optional<torch::Tensor> bias,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor k_cache,
    torch::Tensor v_cache, torch::Tensor slots, torch::Tensor block_table,
    torch::Tensor seq_lens, torch::Tensor arrived, long Hq, double scale,
    long sliding_window, bool rounded, const Fp8Out &fp8) {
  const long B = parts.size(1), Hkv = k_cache.size(2), D = k_cache.size(3);
  const int rot = cos_sin.size(-1);
  TORCH_CHECK(parts.is_cuda() && parts.dim() == 3 && parts.is_contiguous() &&
              parts.scalar_type() == at::kFloat &&
              reinterpret_cast<uintptr_t>(parts.data_ptr()) % 16 == 0 &&
              parts.size(2) == (Hq + 2 * Hkv) * D,
              "qkv_decode: fp32 parts [S, B, (Hq + 2 Hkv) D]");
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.is_contiguous() &&
              v_cache.is_contiguous() && v_cache.sizes() == k_cache.sizes() &&
              k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16 && Hq > 0 &&
              Hq % Hkv == 0 && decode_shape_ok(k_cache, v_cache, Hq / Hkv),
              "qkv_decode: unsupported head_dim=", D, " group=", Hq / Hkv);
  TORCH_CHECK(rot % 8 == 0 && rot <= D &&
              cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous());
  TORCH_CHECK(positions.scalar_type() == at::kLong &&
              positions.is_contiguous() && positions.numel() == B &&
              slots.scalar_type() == at::kLong && slots.is_contiguous() &&
              slots.numel() == B);
  TORCH_CHECK(block_table.scalar_type() == at::kInt &&
              block_table.size(0) >= B &&
              (block_table.size(1) <= 1 || block_table.stride(1) == 1) &&
              seq_lens.scalar_type() == at::kInt &&
              seq_lens.is_contiguous() && seq_lens.numel() >= B);
  TORCH_CHECK(arrived.is_cuda() && arrived.scalar_type() == at::kInt &&
              arrived.is_contiguous() && arrived.numel() >= B * Hkv,
              "qkv_decode: a zero per sequence and kv head");
  const __hip_bfloat16 *bp = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == parts.size(2));
    bp = (const __hip_bfloat16 *)bias->data_ptr();
  }
  auto out = torch::empty({B, Hq * D}, k_cache.options());
  if (B == 0) return out;
  const NewRows fresh{{parts.data_ptr(), 0L, bp, positions.data_ptr<long>(),
                       cos_sin.data_ptr<float>(), (int)B,
                       (int)parts.size(0), rot, (int)rounded},
                      (__hip_bfloat16 *)k_cache.data_ptr(),
                      (__hip_bfloat16 *)v_cache.data_ptr(),
                      slots.data_ptr<long>(), arrived.data_ptr<int>(), fp8, 0, 0};
  launch_decode(out, out, k_cache, v_cache, block_table, seq_lens, Hq / Hkv,
                (float)scale, (int)sliding_window, 0, false, nullptr, 0,
                nullptr, 0.f, nullptr, 0, 0.f, 0, nullptr, &fresh);
  return out;
}

torch::Tensor qkv_decode(torch::Tensor parts,
                         c10::optional<torch::Tensor> bias,
                         torch::Tensor positions, torch::Tensor cos_sin,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor slots, torch::Tensor block_table,
                         torch::Tensor seq_lens, torch::Tensor arrived,
                         long Hq, double scale, long sliding_window,
                         bool rounded) {
  return decode_rows(parts, bias, positions, cos_sin, k_cache, v_cache, slots,
                     block_table, seq_lens, arrived, Hq, scale,
                     sliding_window, rounded, Fp8Out{});
}

// ... with the result's e4m3 rows (heads of 128): {bf16, bytes, scales}
std::vector<torch::Tensor> qkv_decode_fp8(
    torch::Tensor parts, c10::optional<torch::Tensor> bias,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor k_cache,
    torch::Tensor v_cache, torch::Tensor slots, torch::Tensor block_table,
    torch::Tensor seq_lens, torch::Tensor arrived, long Hq, double scale,
    long sliding_window, bool rounded) {
  TORCH_CHECK(parts.dim() == 3 && k_cache.dim() == 4 && k_cache.size(3) == 128,
              "qkv_decode_fp8: heads of 128");
  const long B = parts.size(1);
  auto q = torch::empty({B, Hq * 128}, k_cache.options().dtype(at::kByte));
  auto st = torch::empty({Hq, B}, k_cache.options().dtype(at::kFloat));
  auto out = decode_rows(parts, bias, positions, cos_sin, k_cache, v_cache,
                         slots, block_table, seq_lens, arrived, Hq, scale,
                         sliding_window, rounded,
                         Fp8Out{q.data_ptr<unsigned char>(),
                                st.data_ptr<float>()});
  return {out, q, st};
}

// Whether qkv_decode takes heads of this geometry (caches of one shape), and
// is the faster form: its rows cost each workgroup a few us, which pays in up
// to two rounds of workgroups; rounded, with all sequences in all splits, in
// one if they are split. (us of an attention step, 40 heads on 8 of 128, two
// kernels or three / this one: 1 sequence of 600 keys 13.9 / 12.8, 2 of 2400
// 19.4 / 18.1, 16 of 340 to 880 19.4 / 18.9, 24 of 150 to 450 21.5 / 13.5, of
// 2700 to 7900 102.3 / 102.8, 32 of 520 to 1500 36.5 / 34.6, 60 of them 57.3 /
// 56.4, of 150 to 450 30.2 / 21.2, 64 of 520 to 1500 54.8 / 51.5, 128 96.2 /
// 92.3; 14 on 2 of 64, 64 of 520 to 1500 17.0 / 15.5. Long unequal sequences
// lose by the join what the rest gains: 60 of 1150 to 3400 112.8 / 115.1.
// Beyond: 256 of 150 to 450 65.2 / 67.1. Rounded: 24 of 150 to 450 in four
// splits 21.6 / 24.2.)
bool qkv_decode_ok(torch::Tensor k_cache, long Hq, long B, bool rounded) {
  const long Hkv = k_cache.size(2);
  const int cus = at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
  const int splits = splits_for(k_cache, B);
  return decode_rows_ok(k_cache, k_cache, Hq) &&
         B * Hkv * splits <= (rounded && splits > 1 ? 2L : 4L) * cus;
}

// whether the decode kernel takes heads of this geometry (a mixed batch
// sends its one-row sequences there)
bool decode_rows_ok(torch::Tensor k_cache, torch::Tensor v_cache, long Hq) {
  const long Hkv = k_cache.size(2);
  return k_cache.is_contiguous() && v_cache.is_contiguous() &&
         Hkv > 0 && Hq % Hkv == 0 &&
         decode_shape_ok(k_cache, v_cache, Hq / Hkv);
}

// Windowed-sink form of the split-KV decode kernels: one decode token per
// sequence, q [B, H*D] (row-strided view allowed), bf16, head sizes
// that are multiples of 8 up to 128, up to 16 query heads per kv head;
// optional bias by distance and query temperature. Returns false (nothing
// launched) for any other geometry so the caller can take the generic
// kernel.
bool window_attention_decode(torch::Tensor out, torch::Tensor q,
                             c10::optional<torch::Tensor> gate,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_table,
                             torch::Tensor seq_lens, double scale,
                             long window, long keep_first, bool sink,
                             c10::optional<torch::Tensor> sinks,
                             double softcap,
                             c10::optional<torch::Tensor> bias,
                             double temp_coef, long temp_every) {
  const int B = q.size(0);
  if (B == 0) return true;
  const int D = k_cache.size(3);
  const int Hkv = k_cache.size(2);
  const int Dv = v_cache.size(3);
  if (q.scalar_type() != at::kBFloat16 || q.dim() != 2 ||
      q.size(1) % (D * Hkv) != 0)
    return false;
  const int G = q.size(1) / D / Hkv;
  TORCH_CHECK(q.stride(1) == 1 && out.dim() == 2 && out.stride(1) == 1 &&
              out.size(0) == B && out.size(1) == (long)Hkv * G * Dv &&
              out.scalar_type() == at::kBFloat16,
              "out: bf16 [B, H*Dv] rows (a column block is fine)");
  TORCH_CHECK(k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16 &&
              k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(block_table.scalar_type() == at::kInt &&
              block_table.stride(1) == 1 && block_table.size(0) >= B);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt && seq_lens.numel() == B);
  const void *gp = nullptr;
  long gs = 0;
  if (gate.has_value()) {
    TORCH_CHECK(gate->dim() == 2 && gate->stride(1) == 1 &&
                gate->size(0) == B && gate->size(1) == (long)Hkv * G * Dv &&
                gate->scalar_type() == at::kBFloat16);
    gp = gate->data_ptr();
    gs = gate->stride(0);
  }
  const float *sp = nullptr;
  if (sinks.has_value()) {
    TORCH_CHECK(sinks->scalar_type() == at::kFloat && sinks->is_contiguous() &&
                sinks->numel() == (long)Hkv * G, "sinks: fp32 [H]");
    sp = sinks->data_ptr<float>();
  }
  if (!decode_shape_ok(k_cache, v_cache, G)) return false;
  const float *bp = nullptr;
  int bias_len = 0;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->scalar_type() == at::kFloat &&
                bias->is_contiguous() && bias->dim() == 2 &&
                bias->size(0) == (long)Hkv * G && bias->size(1) >= 1,
                "bias: fp32 [H, distances]");
    bp = bias->data_ptr<float>();
    bias_len = bias->size(1);
  }
  launch_decode(out, q, k_cache, v_cache, block_table, seq_lens, G,
                (float)scale, (int)window, (int)keep_first, sink, gp, gs, sp,
                (float)softcap, bp, bias_len, (float)temp_coef,
                (int)temp_every);
  return true;
}
