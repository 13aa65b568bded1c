// Products of many rows for gfx950 (bf16 in, fp32 sums, K a multiple of 64):
// x [M, K] W[N, K]^T of a linear layer, and the grouped products of experts
// with 256-row blocks (tables as in moe.hip).
//   plain    out = x W^T (+ bias)
//   gated    out = f(x W_gate^T)(x W_up^T), W = gate rows over up rows: the
//            [M, N] product is never written
//   scatter  out[pair] = w[pair] * act W^T (grouped)
//   parts    fp32 [S, M, N] of at most 256 rows, each part over a share of K
//
// Bound by the matrix cores' power and clock where it is fed well: 4096 x
// 4096 x 16384 runs at 1550 TFLOP/s on normal data and 1830 on zeros. What
// costs is what keeps the cores waiting, so:
//  * four waves, one per SIMD, of 128 x 128 results each: the fragments of
//    64 columns are 128 KB of LDS reads per 256 x 256 tile where eight waves
//    of 128 x 64 read 192 KB. The sums fill the accumulation registers, the
//    other half holds two sets of fragments: while the products of one set
//    run, the other is read, one read per four products. (With every
//    accumulation register in use the compiler's allocator shuffles sums
//    between products or through scratch: they are named in asm, see Sum.)
//  * one barrier per 64 columns, in the middle: by then the second half's
//    fragments are in registers and the next stage has landed.
//  * LDS (160 KB) holds two stages of x and three of W: W is loaded in the
//    first half of a step and x in the second, one load per six products. The
//    same loads bunched in one half stall the issue of products (1310
//    against 1550 TFLOP/s), and W, which often comes from HBM, gets
//    more than a step to arrive. Rows of 32 columns with five stages lose to
//    64 B accesses (1110).
//  * a workgroup per CU walks over tiles: loads run two stages ahead across
//    the end of a tile, results are stored while the next tile's operands
//    arrive. 8192 x 8192 x 1024: 107 us, 126 with a workgroup per tile.
//  * results are W x^T: a lane holds eight neighbouring columns of a row in
//    two fragments (the rows of W are staged in that order), so stores are
//    16 B.
//  * what a tile costs beside its products is kept off the waves: division
//    by multiplying, no branch that lanes take differently, stores that the
//    descriptor's bounds cut off, and a tile's first wait leaves the stores
//    of the one before on their way (4 steps a tile before, 2.5 now).
// A block of at most 128 rows runs half the products (waves of 64 x 128).
// Beside a grouped product a plain one of the same form can take part in its
// rounds (SHARED: a shared expert, rows in order): its tiles come first, spread
// over the dies, and workgroups without one of the last of them take routed
// tiles meanwhile. 4096 rows of 2048, 64 experts of 1408 and a shared one of
// 2816: 661 us with sum and norm by launches of their own (352 and 128 tiles on
// 256 CUs), 624 so.
// Tiles of the last round are split along K when most CUs would idle
// (plan_for); the fp32 parts are then joined by tile_sum_kernel in the order
// of K. (us, before / now:) 4133 x 5120 x 27648 1448 (hipBLASLt) / 810; 4133
// x 55296 x 5120 gated 1825 + 120 / 1700; 8 experts of 4096 x 14336 with
// 10000 rows 2289 + 1259 (eight waves of 128 x 64, a workgroup per tile, one
// wait and barrier ahead of a step's reads) / 1910 + 990.
// Workgroups go to the eight dies in turn; each die gets a contiguous run of
// tiles, row blocks fastest within groups, so that a die's 32 tiles share
// operands in its L2.

#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "tile_gemm.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tg_bf8;
typedef __attribute__((ext_vector_type(4))) float tg_f4;
typedef __attribute__((ext_vector_type(4))) unsigned tg_u4;
typedef __attribute__((address_space(3))) void lds_void;

namespace {

constexpr int BK = 64;
constexpr int ROW_B = BK * 2;      // LDS row bytes
constexpr int SLOT = 256 * ROW_B;  // a stage of one operand

enum Form { PLAIN = 0, GATED = 1, SCATTER = 2, PARTS = 3 };
enum Act { NONE = 0, SILU = 1, CLAMP = 2, RELU2 = 3 };

struct Args {
  __hip_bfloat16 *C;
  const __hip_bfloat16 *A, *W, *bias;
  float *part;  // split tiles: [R * splits, 256, 256]
  int M, N, K, bm, nbm, nbn, group;
  unsigned group_inv, run_inv;  // ceil(2^32 / d) of group and group * nbn
  int whole, splits;  // the first `whole` tiles are not split
  // grouped
  const int *sorted_ids, *expert_blocks, *n_post_pad;
  const float *topk_w;
  int n_pairs, topk, a_bytes;
  float limit, alpha;
  // grouped, with a product [s_rows, s_K] [s_N, s_K]^T beside it, a tile of
  // which takes about s_slots times as long
  __hip_bfloat16 *s_C;
  const __hip_bfloat16 *s_A, *s_W;
  int s_rows, s_K, s_N, s_nbm, s_nbn, s_group, s_slots;
};

#define RFL(x) __builtin_amdgcn_readfirstlane(x)
#define ORDER __builtin_amdgcn_sched_barrier(0)

DEV_INLINE short to_bf16(float v) {
  return __builtin_bit_cast(short, __float2bfloat16(v));
}

// Sum I of the 64 of a wave: 16 x 16 results in accumulation registers 4 I
// to 4 I + 3, which nothing else uses. Products of one sum are 32 or more
// apart; what else needs waits: a sum's first product after zero(), get()
// after its last one (settle() between both).
template <int I> struct Sum;
#define SUM(I, R0, R1, R2, R3)                                               \
  template <> struct Sum<I> {                                                \
    static DEV_INLINE void add(const tg_bf8 &a, const tg_bf8 &b) {           \
      asm volatile("v_mfma_f32_16x16x32_bf16 a[" #R0 ":" #R3                 \
                   "], %0, %1, a[" #R0 ":" #R3 "]"                           \
                   ::"v"(a), "v"(b)                                          \
                   : "a" #R0, "a" #R1, "a" #R2, "a" #R3);                    \
    }                                                                        \
    static DEV_INLINE void zero() {                                          \
      asm volatile("v_accvgpr_write_b32 a" #R0 ", 0\n\t"                     \
                   "v_accvgpr_write_b32 a" #R1 ", 0\n\t"                     \
                   "v_accvgpr_write_b32 a" #R2 ", 0\n\t"                     \
                   "v_accvgpr_write_b32 a" #R3 ", 0" ::                      \
                   : "a" #R0, "a" #R1, "a" #R2, "a" #R3);                    \
    }                                                                        \
    static DEV_INLINE tg_f4 get() {                                          \
      float x, y, z, w;                                                      \
      asm volatile("v_accvgpr_read_b32 %0, a" #R0 "\n\t"                     \
                   "v_accvgpr_read_b32 %1, a" #R1 "\n\t"                     \
                   "v_accvgpr_read_b32 %2, a" #R2 "\n\t"                     \
                   "v_accvgpr_read_b32 %3, a" #R3                            \
                   : "=&v"(x), "=&v"(y), "=&v"(z), "=&v"(w));                \
      return tg_f4{x, y, z, w};                                              \
    }                                                                        \
  };
SUM(0, 0, 1, 2, 3)
SUM(1, 4, 5, 6, 7)
SUM(2, 8, 9, 10, 11)
SUM(3, 12, 13, 14, 15)
SUM(4, 16, 17, 18, 19)
SUM(5, 20, 21, 22, 23)
SUM(6, 24, 25, 26, 27)
SUM(7, 28, 29, 30, 31)
SUM(8, 32, 33, 34, 35)
SUM(9, 36, 37, 38, 39)
SUM(10, 40, 41, 42, 43)
SUM(11, 44, 45, 46, 47)
SUM(12, 48, 49, 50, 51)
SUM(13, 52, 53, 54, 55)
SUM(14, 56, 57, 58, 59)
SUM(15, 60, 61, 62, 63)
SUM(16, 64, 65, 66, 67)
SUM(17, 68, 69, 70, 71)
SUM(18, 72, 73, 74, 75)
SUM(19, 76, 77, 78, 79)
SUM(20, 80, 81, 82, 83)
SUM(21, 84, 85, 86, 87)
SUM(22, 88, 89, 90, 91)
SUM(23, 92, 93, 94, 95)
SUM(24, 96, 97, 98, 99)
SUM(25, 100, 101, 102, 103)
SUM(26, 104, 105, 106, 107)
SUM(27, 108, 109, 110, 111)
SUM(28, 112, 113, 114, 115)
SUM(29, 116, 117, 118, 119)
SUM(30, 120, 121, 122, 123)
SUM(31, 124, 125, 126, 127)
SUM(32, 128, 129, 130, 131)
SUM(33, 132, 133, 134, 135)
SUM(34, 136, 137, 138, 139)
SUM(35, 140, 141, 142, 143)
SUM(36, 144, 145, 146, 147)
SUM(37, 148, 149, 150, 151)
SUM(38, 152, 153, 154, 155)
SUM(39, 156, 157, 158, 159)
SUM(40, 160, 161, 162, 163)
SUM(41, 164, 165, 166, 167)
SUM(42, 168, 169, 170, 171)
SUM(43, 172, 173, 174, 175)
SUM(44, 176, 177, 178, 179)
SUM(45, 180, 181, 182, 183)
SUM(46, 184, 185, 186, 187)
SUM(47, 188, 189, 190, 191)
SUM(48, 192, 193, 194, 195)
SUM(49, 196, 197, 198, 199)
SUM(50, 200, 201, 202, 203)
SUM(51, 204, 205, 206, 207)
SUM(52, 208, 209, 210, 211)
SUM(53, 212, 213, 214, 215)
SUM(54, 216, 217, 218, 219)
SUM(55, 220, 221, 222, 223)
SUM(56, 224, 225, 226, 227)
SUM(57, 228, 229, 230, 231)
SUM(58, 232, 233, 234, 235)
SUM(59, 236, 237, 238, 239)
SUM(60, 240, 241, 242, 243)
SUM(61, 244, 245, 246, 247)
SUM(62, 248, 249, 250, 251)
SUM(63, 252, 253, 254, 255)
#undef SUM

DEV_INLINE void settle() {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
}

// bytes from p on. (What decides them, and every branch of the kernel, is the
// same in all lanes: a descriptor that the compiler holds in vector registers
// makes each load a loop over lanes.)
DEV_INLINE __amdgpu_buffer_rsrc_t rows_of(const __hip_bfloat16 *p,
                                          int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, bytes, 0x00020000);
}

// a table entry that all lanes want, by the scalar path: waiting for it does
// not wait for the loads to LDS
DEV_INLINE int table_at(const int *p, int i) {
  return ((const __attribute__((address_space(4))) int *)p)[i];
}

DEV_INLINE __amdgpu_buffer_rsrc_t bytes_of(float *p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, bytes, 0x00020000);
}

template <int V> struct Int { static constexpr int value = V; };

// f(Int<0>), f(Int<1>), ... f(Int<N - 1>)
template <int N, class F> DEV_INLINE void repeat(F &&f) {
  if constexpr (N > 0) {
    repeat<N - 1>(f);
    f(Int<N - 1>());
  }
}

// n / d from inv = ceil(2^32 / d) (one too many at most), d > 1
DEV_INLINE int quotient(int n, int d, unsigned inv) {
  const int q = __umulhi(n, inv);
  return q * d > n ? q - 1 : q;
}

// tile t of row blocks and column blocks: groups of `group` row blocks
DEV_INLINE void tile_at(int t, int nbm, const Args &P, int &mb, int &nb) {
  const int run = P.group * P.nbn;
  const int g = run > 1 ? quotient(t, run, P.run_inv) : t;
  const int in_g = t - g * run, rows = min(P.group, nbm - g * P.group);
  int q = in_g;
  if (rows == P.group && rows > 1) q = quotient(in_g, rows, P.group_inv);
  else if (rows > 1) q = in_g / rows;
  mb = RFL(g * P.group + in_g - q * rows);
  nb = RFL(q);
}

// 8 results from their sums; gated: four gate and four up columns each in
// `g`, `u` (g: all eight columns otherwise)
template <int FORM, int ACT>
DEV_INLINE shortx8 results(const float *g, const float *u, float scale,
                           float limit, float alpha) {
  shortx8 o;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    float x = g[r];
    if (FORM == GATED && ACT == CLAMP) {
      x = fminf(x, limit);
      const float up = fminf(fmaxf(u[r], -limit), limit) + 1.f;
      x = x / (1.f + __expf(-alpha * x)) * up;
    } else if (FORM == GATED) {
      x = x / (1.f + __expf(-x)) * u[r];
    } else if (ACT == RELU2) {
      x = fmaxf(x, 0.f);
      x = x * x;
    } else {
      x *= scale;
    }
    o[r] = to_bf16(x);
  }
  return o;
}

// ONCE: a weight row is read by one workgroup (non-temporal loads leave the
// L2 to x). SHARED (grouped, gated or scatter): the product beside
template <int FORM, int ACT, bool GROUPED, bool BIAS, bool ONCE = false,
          bool SHARED = false>
__global__ __launch_bounds__(256, 1) void tile_gemm_kernel(const Args P) {
  // two stages of x, then three of W
  __shared__ __attribute__((aligned(16))) char smem[5 * SLOT];
  char *const sw = smem + 2 * SLOT;
  const int tid = threadIdx.x, wave = RFL(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, lhi = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int K = P.K, nkt = K / BK;
  const int NC = FORM == GATED ? P.N >> 1 : P.N;   // columns of C
  constexpr int BC = FORM == GATED ? 128 : 256;    // of a tile
  constexpr bool GATHER = GROUPED && FORM != SCATTER;

  // this workgroup's items: whole tiles, then parts of split ones
  const int nbm = GROUPED ? table_at(P.n_post_pad, 0) / 256 : P.nbm;
  const int tiles = nbm * P.nbn;
  const int whole = GROUPED ? tiles : P.whole;
  const int R = tiles - whole, parts = R * P.splits;
  // (the grid is a multiple of eight)
  const int die = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int step = gridDim.x >> 3;  // workgroups of a die
  const int w0 = (die * whole >> 3) + idx, w1 = (die + 1) * whole >> 3;
  const int p0 = (die * parts >> 3) + idx, p1 = (die + 1) * parts >> 3;
  int n_whole = RFL(max(0, (w1 - w0 + step - 1) / step));
  // SHARED: a die's tiles of the product beside are dealt out first; of the
  // others a workgroup without one of the last `b` of these takes `lead` while
  // those take theirs (`width` such workgroups a turn), then all take turns
  int n_sh = 0, sh0 = 0, lead = 0, width = 0, b = 0, behind = 0;
  if (SHARED) {
    const int all = P.s_nbm * P.s_nbn;
    sh0 = (die * all >> 3) + idx;
    const int mine = ((die + 1) * all >> 3) - (die * all >> 3);
    n_sh = RFL(max(0, (mine - idx + step - 1) / step));
    b = mine % step;
    if (b > 0) {
      width = step - b;
      behind = P.s_slots * width;
      lead = idx >= b ? P.s_slots : 0;
    }
    const int n = w1 - (w0 - idx);  // the die's others
    int first = 0;
    if (lead > 0)
      first = min(lead, max(0, (n - (idx - b) + width - 1) / width));
    n_whole = RFL(first);
    if (first == lead)
      n_whole = RFL(first + max(0, (n - behind - idx + step - 1) / step));
  }
  const int items =
      RFL(n_sh + n_whole + max(0, (p1 - p0 + step - 1) / step));
  if (items == 0) return;
  struct Item {
    int mb, nb, k0, nk, part, sh;
  };
  auto item_at = [&](int i) __attribute__((always_inline)) {
    Item it;
    int t;
    it.sh = SHARED && i < n_sh;
    if (SHARED) {
      it.k0 = 0;
      it.part = -1;
      if (it.sh) {
        t = sh0 + i * step;
        it.nk = P.s_K / BK;
        const int g = t / (P.s_group * P.s_nbn), r0 = g * P.s_group;
        const int in_g = t - r0 * P.s_nbn;
        const int rows = min(P.s_group, P.s_nbm - r0);
        it.nb = RFL(in_g / rows);
        it.mb = RFL(r0 + in_g - it.nb * rows);
        return it;
      }
      const int j = i - n_sh;
      t = w0 - idx + (j < lead ? j * width + idx - b
                               : behind + (j - lead) * step + idx);
      it.nk = nkt;
    } else if (i < n_whole) {
      t = w0 + i * step;
      it.k0 = 0;
      it.nk = nkt;
      it.part = -1;
    } else {
      const int q = p0 + (i - n_whole) * step, s = q / R;
      t = whole + q - s * R;
      it.k0 = RFL(s * nkt / P.splits);
      it.nk = RFL((s + 1) * nkt / P.splits) - it.k0;
      it.part = RFL(q);
    }
    tile_at(t, nbm, P, it.mb, it.nb);
    return it;
  };
  // at most 128 rows of the block are in use
  auto is_half = [&](const Item &it) __attribute__((always_inline)) {
    if (SHARED && it.sh) return (int)(P.s_rows - it.mb * 256 <= 128);
    if (GROUPED)
      return (int)(table_at(P.sorted_ids, it.mb * 256 + 128) >= P.n_pairs);
    return (int)(min(P.bm, P.M - it.mb * P.bm) <= 128);
  };

  // sources of this lane: LDS rows j * 32 + wave * 8 + sub, 16 B units
  // permuted by row & 7
  const int sub = lane >> 3, unit = ((lane & 7) ^ sub) * 16;
  int va[8], vw[8], ids[8];
  auto a_rows = [&](int K) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      va[j] = (j * 32 + wave * 8 + sub) * K * 2 + unit;
  };
  auto w_rows = [&](int K, int NC) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = j * 32 + wave * 8 + sub, i = r & 15, n = r >> 4;
      // row i of fragment n: lane group i >> 2 holds its columns i & 3
      int c;
      if (FORM == GATED)
        c = (n >> 2) * 32 + (i >> 2) * 8 + ((n >> 1) & 1) * 4 + (i & 3) +
            (n & 1) * NC;
      else
        c = (n >> 1) * 32 + (i >> 2) * 8 + (n & 1) * 4 + (i & 3);
      vw[j] = c * K * 2 + unit;
    }
  };
  a_rows(K);
  w_rows(K, NC);
  auto fetch_ids = [&](int i) __attribute__((always_inline)) {
    if (i >= items) return;
    const Item it = item_at(i);
    if (SHARED && it.sh) return;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      ids[j] = P.sorted_ids[it.mb * 256 + j * 32 + wave * 8 + sub];
  };
  // the loads' position, two stages ahead of the products; past the last
  // item they read nothing
  __amdgpu_buffer_rsrc_t ra, rw;
  int li = -1, lleft = 0, lso = 0;
  auto advance = [&]() __attribute__((always_inline)) {
    if (lleft == 0) {
      ++li;
      if (li < items) {
        const Item it = item_at(li);
        lleft = it.nk;
        lso = it.k0 * ROW_B;
        if (SHARED) {
          if (it.sh) {
            const int sk = P.s_K, at = it.nb * BC;
            rw = rows_of(P.s_W + (long)at * sk,
                         (FORM == GATED ? P.s_N - at : min(256, P.s_N - at)) *
                             sk * 2);
            ra = rows_of(P.s_A + (long)it.mb * 256 * sk,
                         min(256, P.s_rows - it.mb * 256) * sk * 2);
            a_rows(sk);
            w_rows(sk, P.s_N >> 1);
            if (GATHER) fetch_ids(li + 1);
            --lleft;
            return;
          }
          a_rows(K);
          w_rows(K, NC);
        }
        const __hip_bfloat16 *w = P.W;
        if (GROUPED) w += (long)table_at(P.expert_blocks, it.mb) * P.N * K;
        rw = rows_of(w + (long)it.nb * BC * K,
                     (FORM == GATED ? P.N - it.nb * BC
                                    : min(256, P.N - it.nb * BC)) * K * 2);
        if (GATHER) {
          ra = rows_of(P.A, P.a_bytes);
#pragma unroll
          for (int j = 0; j < 8; ++j)  // (rows that pad a block: none)
            va[j] = ids[j] < P.n_pairs ? ids[j] / P.topk * (K * 2) + unit
                                       : 0x7ffffff0;
          fetch_ids(li + 1);
        } else if (GROUPED) {
          ra = rows_of(P.A + (long)it.mb * 256 * K, 256 * K * 2);
        } else {
          ra = rows_of(P.A + (long)it.mb * P.bm * K,
                       min(P.bm, P.M - it.mb * P.bm) * K * 2);
        }
      } else {
        lleft = 1 << 30;
        lso = 0;
        ra = rows_of(P.A, 0);
        rw = rows_of(P.W, 0);
      }
    } else {
      lso += ROW_B;
    }
    --lleft;
  };
  auto load = [&](__amdgpu_buffer_rsrc_t r, char *slot, int v, int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        r, (lds_void *)(slot + wave * 1024 + j * 4096), 16, v, lso, 0, 0);
  };
  auto load_w = [&](char *slot, int v, int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rw, (lds_void *)(slot + wave * 1024 + j * 4096), 16, v, lso, 0,
        ONCE ? 2 : 0);
  };

  tg_bf8 fa[2][8], fb[2][8];  // fragments of 32 columns
  const int off = (lhi ^ (l16 & 7)) << 4;
  const int bb = (wn * 128 + l16) * ROW_B + off;
  auto a_base = [&](int half) {
    return (wm * (half ? 64 : 128) + l16) * ROW_B + off;
  };
  auto read_a = [&](int base, int slot, int ks, int m) {
    fa[ks][m] = *reinterpret_cast<const tg_bf8 *>(
        smem + slot + (base ^ (ks * 64)) + m * 16 * ROW_B);
  };
  auto read_b = [&](int slot, int ks, int n) {
    fb[ks][n] = *reinterpret_cast<const tg_bf8 *>(
        sw + slot + (bb ^ (ks * 64)) + n * 16 * ROW_B);
  };

  if (GATHER) fetch_ids(0);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    advance();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      load_w(sw + s * SLOT, vw[j], j);
      load(ra, smem + s * SLOT, va[j], j);
    }
  }
  // stage 0 has landed (one stage is younger, and the row ids of a later
  // item may be)
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  __builtin_amdgcn_s_barrier();

  Item it = item_at(0);
  int half = is_half(it);
  int ab = a_base(half);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    read_b(0, 0, j);
    read_a(ab, 0, 0, j);
  }
  int xs = 0, ws = 0;  // slots of the current stage
  int stores = 0;      // of the tile before, if this is a tile's first step
  for (int ci = 0; ci < items; ++ci) {
    const Item nx = item_at(min(ci + 1, items - 1));
    const int next_half = is_half(nx);
    const int next_ab = a_base(next_half);
    int row_id[8];
    if (GROUPED && !(SHARED && it.sh)) {
#pragma unroll
      for (int m = 0; m < 8; ++m)
        row_id[m] = P.sorted_ids[it.mb * 256 +
                                 (half ? wm * 64 + (m & 3) * 16
                                       : wm * 128 + m * 16) + l16];
    }
    int left = it.nk;
    auto run = [&](auto mt) {
      constexpr int MT = decltype(mt)::value, P1 = MT * 8;
      repeat<P1>([](auto i) { Sum<decltype(i)::value>::zero(); });
      settle();
      do {
        const int xn = xs ^ SLOT, wn1 = ws == 2 * SLOT ? 0 : ws + SLOT,
                  wn2 = wn1 == 2 * SLOT ? 0 : wn1 + SLOT;
        const int nb_ = left == 1 ? next_ab : ab;
        advance();
            ORDER;
        // first 32 columns; fragments of the others; W two stages on, into
        // the slot of the stage before
        repeat<P1>([&](auto at) {
          constexpr int i = decltype(at)::value;
          constexpr int RD = MT == 8 ? 4 : 2, LD = MT == 8 ? 6 : 3;
          if (i % RD == 0) {
            const int r = i / RD;
            ORDER;
            if (r < 8) read_b(ws, 1, r);
            else if (r - 8 < MT) read_a(ab, xs, 1, r - 8);
            ORDER;
          }
          if (i % LD == LD / 2 && i / LD < 8) {
            ORDER;
            load_w(sw + wn2, vw[i / LD], i / LD);
            ORDER;
          }
          Sum<i>::add(fb[0][i & 7], fa[0][i >> 3]);
        });
        ORDER;
        // the next stage is there (eight loads are younger, and the stores
        // of a tile that ended a step ago), this one's fragments are in
        // registers
        if (stores >= 55)
          asm volatile("s_waitcnt vmcnt(63) lgkmcnt(0)" ::: "memory");
        else if (stores >= 32)
          asm volatile("s_waitcnt vmcnt(40) lgkmcnt(0)" ::: "memory");
        else if (stores >= 16)
          asm volatile("s_waitcnt vmcnt(24) lgkmcnt(0)" ::: "memory");
        else
          asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
        stores = 0;
        __builtin_amdgcn_s_barrier();
        ORDER;
        // other 32 columns; first fragments of the next stage; x two stages
        // on, into this one's slot
        repeat<P1>([&](auto at) {
          constexpr int i = decltype(at)::value;
          constexpr int RD = MT == 8 ? 4 : 2, LD = MT == 8 ? 6 : 3;
          if (i % RD == 0) {
            const int r = i / RD;
            ORDER;
            if (r < 8) read_b(wn1, 0, r);
            else read_a(nb_, xn, 0, r - 8);
            ORDER;
          }
          if (i % LD == LD / 2 && i / LD < 8) {
            ORDER;
            load(ra, smem + xs, va[i / LD], i / LD);
            ORDER;
          }
          Sum<i>::add(fb[1][i & 7], fa[1][i >> 3]);
        });
        ORDER;
        xs = xn;
        ws = wn1;
      } while (--left > 0);

      settle();
      int x16 = l16, xhi = lhi;  // addresses are formed here, not above
      asm volatile("" : "+v"(x16), "+v"(xhi));
      const int r0 = wm * MT * 16 + x16;  // row of the tile
      if (FORM == PARTS) {
        // (a row is N * 4 bytes; rows and columns outside are not stored)
        const int s = RFL(it.part / R);
        const int rows = RFL(min(P.bm, P.M - it.mb * P.bm));
        const auto rc = bytes_of(
            P.part + ((long)s * P.M + it.mb * P.bm) * P.N, rows * P.N * 4);
        const int c0 = it.nb * 256 + wn * 128 + xhi * 8;
        repeat<P1>([&](auto at) {
          constexpr int i = decltype(at)::value, n = i & 7, m = i >> 3;
          constexpr int dc = (n >> 1) * 32 + (n & 1) * 4;
          ORDER;
          const bool used = r0 + m * 16 < rows && c0 + dc < P.N;
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(tg_u4, Sum<i>::get()), rc,
              used ? ((r0 + m * 16) * P.N + c0 + dc) * 4 : 0x7ffffff0, 0, 0);
        });
        stores = P1;
        return;
      }
      if (!GROUPED && it.part >= 0) {
        float *p = P.part + (long)it.part * 65536 + r0 * 256 + wn * 128 +
                   xhi * 8;
        repeat<P1>([&](auto at) {
          constexpr int i = decltype(at)::value, n = i & 7, m = i >> 3;
          ORDER;
          *reinterpret_cast<tg_f4 *>(p + m * 4096 + (n >> 1) * 32 +
                                     (n & 1) * 4) = Sum<i>::get();
        });
        stores = P1;
        return;
      }
      // this lane's columns: 8 at c0 + 32 p
      constexpr int NP = BC / 64;
      const bool sh = SHARED && it.sh;
      const int NCi =
          sh ? (FORM == GATED ? P.s_N >> 1 : P.s_N) : NC;
      const int c0 = it.nb * BC + wn * (BC / 2) + xhi * 8;
      float bias[NP][8];
      if (BIAS) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
          ld8<__hip_bfloat16>(P.bias + min(c0 + p * 32, NC - 8), bias[p]);
      }
      float sc[MT];
      if (FORM == SCATTER) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
          sc[m] = P.topk_w && !sh ? P.topk_w[min(row_id[m], P.n_pairs - 1)]
                                  : 1.f;
      }
      auto result = [&](auto mt_, auto pt) {
        constexpr int m = decltype(mt_)::value, p = decltype(pt)::value;
        float g[8], u[8];
        if constexpr (FORM == GATED) {
          constexpr int i = m * 8 + p * 4;
          const tg_f4 g0 = Sum<i>::get(), u0 = Sum<i + 1>::get();
          const tg_f4 g1 = Sum<i + 2>::get(), u1 = Sum<i + 3>::get();
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            g[r] = g0[r]; g[r + 4] = g1[r];
            u[r] = u0[r]; u[r + 4] = u1[r];
          }
        } else {
          constexpr int i = m * 8 + p * 2;
          const tg_f4 g0 = Sum<i>::get(), g1 = Sum<i + 1>::get();
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            g[r] = g0[r];
            g[r + 4] = g1[r];
            if (BIAS) {
              g[r] += bias[p][r];
              g[r + 4] += bias[p][r + 4];
            }
          }
        }
        return results<FORM, ACT>(g, u, FORM == SCATTER ? sc[m] : 1.f,
                                  P.limit, P.alpha);
      };
      // stores count rows from the block's first (scatter: from C's); what
      // lies outside is not stored
      const int bm = GROUPED ? 256 : P.bm;
      const auto rc =
          sh ? rows_of(P.s_C + (long)it.mb * 256 * NCi,
                       min(256, P.s_rows - it.mb * 256) * NCi * 2)
          : FORM == SCATTER
              ? rows_of(P.C, P.n_pairs * NC * 2)
              : rows_of(P.C + (long)it.mb * bm * NC,
                        (GROUPED ? 256 : min(bm, P.M - it.mb * bm)) * NC * 2);
      repeat<MT>([&](auto mt_) {
        constexpr int m = decltype(mt_)::value;
        ORDER;
        const int row = FORM == SCATTER && !sh ? row_id[m] : r0 + m * 16;
        const bool used = !GROUPED || sh || row_id[m] < P.n_pairs;
        const int at = (row * NCi + c0) * 2;
        repeat<NP>([&](auto pt) {
          constexpr int p = decltype(pt)::value;
          const tg_u4 o = __builtin_bit_cast(tg_u4, result(mt_, pt));
          __builtin_amdgcn_raw_buffer_store_b128(
              o, rc, used && c0 + p * 32 < NCi ? at + p * 64 : 0x7ffffff0, 0,
              0);
        });
      });
      stores = MT * NP;
    };
    if (half) run(Int<4>());
    else run(Int<8>());
    it = nx;
    half = next_half;
    ab = next_ab;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// The split tiles from their parts: a workgroup per 8 rows of a tile (plain)
// or 16 (gated), 8 results per thread.
template <int FORM>
__global__ __launch_bounds__(256) void tile_sum_kernel(const Args P) {
  constexpr int BC = FORM == GATED ? 128 : 256, UNITS = BC / 8;
  const int NC = FORM == GATED ? P.N >> 1 : P.N;
  const int R = P.nbm * P.nbn - P.whole;
  constexpr int PER = UNITS;  // workgroups of a tile
  const int tl = blockIdx.x / PER;
  int mb, nb;
  tile_at(P.whole + tl, P.nbm, P, mb, nb);
  const int rr = blockIdx.x % PER * (256 / UNITS) + threadIdx.x / UNITS;
  const int cu = threadIdx.x % UNITS * 8, c = nb * BC + cu;
  const int row = mb * P.bm + rr;
  if (rr >= P.bm || row >= P.M || c >= NC) return;
  // first of the sums that this thread adds up: a gated tile holds, of 64
  // columns, 32 low halves and then 32 high halves
  const int at = FORM == GATED ? (cu >> 6) * 128 + ((cu >> 5) & 1) * 64 +
                                     (cu & 31)
                               : cu;
  constexpr int HI = FORM == GATED ? 32 : 4;  // second four results
  tg_f4 a[2], b[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) a[h] = b[h] = tg_f4{0, 0, 0, 0};
  for (int s = 0; s < P.splits; ++s) {
    const float *p =
        P.part + (((long)s * R + tl) * 256 + rr) * 256 + at;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      a[h] += *reinterpret_cast<const tg_f4 *>(p + h * HI);
      if (FORM == GATED)
        b[h] += *reinterpret_cast<const tg_f4 *>(p + h * HI + 4);
    }
  }
  float g[8], u[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    g[r] = a[r >> 2][r & 3];
    u[r] = b[r >> 2][r & 3];
    if (FORM == PLAIN && P.bias) g[r] += __bfloat162float(P.bias[c + r]);
  }
  *reinterpret_cast<shortx8 *>(P.C + (long)row * NC + c) =
      results<FORM, FORM == GATED ? SILU : NONE>(g, u, 1.f, 0.f, 0.f);
}

bool aligned16(const torch::Tensor &t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct Plan {
  int bm, nbm, nbn, whole, splits;
  double cost;  // in steps of a whole tile
};

// Row block and split of the last tiles. In steps of 64 columns of a 256-row
// tile (about 1.3 us): a tile of nk steps takes nk + 4, one of 128 rows 0.58
// nk + 3; a part's fp32 results 3 more, their sum about 4 and 0.02 per part.
Plan plan_for(int M, int N, int K, bool gated, int cus) {
  Plan best{};
  best.cost = 1e30;
  const int nkt = K / BK, cols = gated ? 128 : 256;
  const int nc = gated ? N / 2 : N;
  for (int bm : {256, 128}) {
    const double unit = bm == 256 ? 1.0 : 0.58, edge = bm == 256 ? 4 : 3;
    Plan p;
    p.bm = bm;
    p.nbm = (M + bm - 1) / bm;
    p.nbn = (nc + cols - 1) / cols;
    const int tiles = p.nbm * p.nbn, rounds = tiles / cus;
    const int rest = tiles - rounds * cus;
    for (int s = 1; s <= 8 && (s == 1 || nkt / s >= 4); ++s) {
      p.splits = s;
      p.whole = s == 1 ? tiles : rounds * cus;
      if (s > 1 && rest == 0) break;
      const int items = s == 1 ? 0 : rest * s;
      const int full = s == 1 ? (tiles + cus - 1) / cus : rounds;
      p.cost = full * (unit * nkt + edge);
      if (items)
        p.cost += (items + cus - 1) / cus * (unit * nkt / s + edge + 3) + 4 +
                  0.02 * items * (bm / 256.0);
      if (p.cost < best.cost * (s == 1 ? 1.0 : 0.98)) best = p;
    }
  }
  return best;
}

void set_divisors(Args &P) {
  auto inv = [](long d) {
    return (unsigned)(((1L << 32) + d - 1) / d);  // (not used for 1)
  };
  P.group_inv = inv(P.group);
  P.run_inv = inv((long)P.group * P.nbn);
}

int compute_units() {
  return at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
}

}  // namespace

// Steps of a whole tile (see plan_for) that the product would take here.
double tile_gemm_cost(long M, long N, long K, bool gated) {
  if (M <= 0 || N <= 0 || K < BK) return 0.0;
  return plan_for(M, N, K, gated, compute_units()).cost;
}

// x [M, K] w [N, K]^T (+ bias); gated: silu(x w_gate^T) * (x w_up^T), w =
// gate rows, up rows
torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w,
                        c10::optional<torch::Tensor> bias, bool gated) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 &&
              x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16 && x.size(1) == w.size(1) &&
              x.is_contiguous() && w.is_contiguous() && aligned16(x) &&
              aligned16(w), "tile_gemm: contiguous bf16, 16 B aligned");
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  const long cols = gated ? N / 2 : N;
  TORCH_CHECK(K > 0 && K % BK == 0 && cols > 0 && cols % 8 == 0 &&
              (!gated || N % 2 == 0),
              "tile_gemm: K a multiple of 64, columns of 8");
  // (offsets within a block of rows are 32 bits, tiles are counted in 24)
  TORCH_CHECK(N <= (1L << 20) && K <= (1L << 21) && M <= (1L << 24) &&
              (M + 127) / 128 * ((N + 255) / 256 + 1) < (1L << 24) &&
              (!gated || N * K < (1L << 30)), "tile_gemm: too large");
  TORCH_CHECK(!gated || !bias.has_value());
  Args P{};
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == N &&
                aligned16(*bias), "bias: bf16 [N]");
    P.bias = (const __hip_bfloat16 *)bias->data_ptr();
  }
  auto out = torch::empty({M, cols}, x.options());
  if (M == 0) return out;
  const int cus = compute_units();
  const Plan p = plan_for(M, N, K, gated, cus);
  P.C = (__hip_bfloat16 *)out.data_ptr();
  P.A = (const __hip_bfloat16 *)x.data_ptr();
  P.W = (const __hip_bfloat16 *)w.data_ptr();
  P.M = M;
  P.N = N;
  P.K = K;
  P.bm = p.bm;
  P.nbm = p.nbm;
  P.nbn = p.nbn;
  P.whole = p.whole;
  P.splits = p.splits;
  // row blocks in even groups of at most 8
  const int groups = (p.nbm + 7) / 8;
  P.group = (p.nbm + groups - 1) / groups;
  set_divisors(P);
  const int rest = p.nbm * p.nbn - p.whole, items = p.whole + rest * p.splits;
  torch::Tensor part;
  if (rest > 0) {
    part = torch::empty({(long)rest * p.splits, 256, 256},
                        x.options().dtype(at::kFloat));
    P.part = part.data_ptr<float>();
  }
  auto stream = at::cuda::getCurrentCUDAStream();
  // (whole multiples of eight: as many workgroups as tiles on each die)
  const dim3 grid(std::min((items + 7) / 8 * 8, cus)), block(256);
  if (gated && p.nbm == 1)  // (256 x 55296 x 5120 137 us, 151 without)
    hipLaunchKernelGGL((tile_gemm_kernel<GATED, SILU, false, false, true>),
                       grid, block, 0, stream, P);
  else if (gated)
    hipLaunchKernelGGL((tile_gemm_kernel<GATED, SILU, false, false>), grid,
                       block, 0, stream, P);
  else if (P.bias)
    hipLaunchKernelGGL((tile_gemm_kernel<PLAIN, NONE, false, true>), grid,
                       block, 0, stream, P);
  else
    hipLaunchKernelGGL((tile_gemm_kernel<PLAIN, NONE, false, false>), grid,
                       block, 0, stream, P);
  HIP_CHECK_KERNEL();
  if (rest > 0) {
    if (gated)
      hipLaunchKernelGGL((tile_sum_kernel<GATED>), dim3(rest * 16), block, 0,
                         stream, P);
    else
      hipLaunchKernelGGL((tile_sum_kernel<PLAIN>), dim3(rest * 32), block, 0,
                         stream, P);
    HIP_CHECK_KERNEL();
  }
  return out;
}

// Row block and splits of few rows (at most 256), 0 splits where the
// streaming kernel's ring is the better one. A round of workgroups at most.
// Rows beyond 128 are one block while the parts are at most 0.4 of the
// weight's bytes, else two of 128 rows with half the splits (us with the norm
// that sums the parts, one / two: 256 x 5120 x 27648 81 / 95, 256 x 5120 x
// 5120 44 / 36, 256 x 4096 x 14336 57 / 51, 136 x 7168 x 5120 37 / 38).
// Against the stream, with the norm (us, stream / this): 256 x 5120 x 27648
// 117 / 95, 256 x 7168 x 5120 44.8 / 41.1, 256 x 5120 x 5120 42.7 / 34.1, 160
// x 6144 x 4096 34.1 / 29.2, 192 x 5120 x 5120 40 / 32, 192 x 7168 x 5120 42.3
// / 38.7; level with few columns and long K (256 x 4096 x 14336 48.2 / 49.5,
// 256 x 2560 x 12800 36.1 / 37.6); below 24 M weights its short parts lose.
// The lines up to 128 rows (K from 4608 on; up to 64 rows from 8192 on and 72 M
// weights) were drawn where the stream of 64-column tiles fell behind; the
// stream of 128-column tiles is level or ahead there (128 x 5120 x 27648 65.4 /
// 64.0, 128 x 5120 x 5120 25.4 / 30.5, 128 x 7168 x 5120 29.7 / 33.7, 128 x
// 4096 x 14336 34.0 / 39.3, 96 x 3584 x 8192 22.9 / 25.9, 64 x 5120 x 27648
// 54.2 / 61.3, 40 x 8192 x 10240 35.5 / 41.8). Few columns leave CUs idle with
// 16 parts, the most: it takes 160 workgroups for a block of rows, 200 for half
// a one.
void tile_parts_plan(long M, long N, long K, int *bm, int *splits) {
  *splits = 0;
  *bm = M > 128 ? 256 : 128;
  const long weights = N * K, nbn = (N + 255) / 256;
  const int cus = compute_units(), nkt = K / BK;
  if (M <= 32 || M > 256 || nbn > cus || N > (1 << 20) || K > (1 << 21) ||
      weights < (M > 64 ? 24L : 72L) << 20 ||
      K < (M > 128 ? 0 : M > 64 ? 4608 : 8192))
    return;
  auto most = [&](int blocks) {
    return (int)std::min<long>(std::min<long>(cus / (nbn * blocks), nkt / 4),
                               16);
  };
  int s = most(1);
  if (nbn * s * 32 < cus * (M > 128 ? 20 : 25)) return;
  if (M > 128 && 5 * s * M > K && most(2) > 0) {
    *bm = 128;
    s = most(2);
  }
  *splits = s;
}

// The fp32 parts [S, M, N] of x w^T, each over a share of K (operands checked
// by stream_parts; sizes as tile_parts_plan takes them).
void tile_parts(float *part, const void *x, const void *w, long M, long N,
                long K, int bm, int splits) {
  Args P{};
  P.A = (const __hip_bfloat16 *)x;
  P.W = (const __hip_bfloat16 *)w;
  P.part = part;
  P.M = M;
  P.N = N;
  P.K = K;
  P.bm = bm;
  P.nbm = (M + bm - 1) / bm;
  P.nbn = (N + 255) / 256;
  P.whole = 0;
  P.splits = splits;
  P.group = P.nbm;
  set_divisors(P);
  const int items = P.nbm * P.nbn * splits;
  const dim3 grid(std::min((items + 7) / 8 * 8, compute_units())), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  if (P.nbm == 1)
    hipLaunchKernelGGL((tile_gemm_kernel<PARTS, NONE, false, false, true>),
                       grid, block, 0, stream, P);
  else
    hipLaunchKernelGGL((tile_gemm_kernel<PARTS, NONE, false, false>), grid,
                       block, 0, stream, P);
  HIP_CHECK_KERNEL();
}

// Offsets into A, into an expert's weights and, for scatter, into C are 32
// bits.
bool tile_gemm_grouped_ok(long a_numel, long n_pairs, long Nd, long K,
                          int act) {
  return a_numel < (1L << 30) && Nd * K < (1L << 30) &&
         (act != NONE || n_pairs * Nd < (1L << 30));
}

// The grouped forms over blocks of 256 rows (operands checked by
// moe_gemm_tiled, sizes by tile_gemm_grouped_ok; act as there).
void tile_gemm_grouped(void *C, const void *A, const void *W,
                       const int *sorted_ids, const int *expert_blocks,
                       const int *n_post_pad, const float *topk_w,
                       long max_blocks, long n_pairs, long topk, long Nd,
                       long K, long a_rows, int act, float limit,
                       float alpha, const TileShared &shared) {
  const bool gated = act == SILU || act == CLAMP;
  Args P{};
  P.C = (__hip_bfloat16 *)C;
  P.A = (const __hip_bfloat16 *)A;
  P.W = (const __hip_bfloat16 *)W;
  P.N = Nd;
  P.K = K;
  P.bm = 256;
  P.nbn = ((gated ? Nd / 2 : Nd) + (gated ? 127 : 255)) / (gated ? 128 : 256);
  P.group = 4;
  set_divisors(P);
  P.splits = 1;
  P.sorted_ids = sorted_ids;
  P.expert_blocks = expert_blocks;
  P.n_post_pad = n_post_pad;
  P.topk_w = topk_w;
  P.n_pairs = n_pairs;
  P.topk = topk;
  P.a_bytes = a_rows * K * 2;
  P.limit = limit;
  P.alpha = alpha;
  auto stream = at::cuda::getCurrentCUDAStream();
  if (shared.C) {
    P.s_C = (__hip_bfloat16 *)shared.C;
    P.s_A = (const __hip_bfloat16 *)shared.A;
    P.s_W = (const __hip_bfloat16 *)shared.W;
    P.s_rows = shared.rows;
    P.s_K = shared.K;
    P.s_N = shared.N;
    P.s_nbm = (shared.rows + 255) / 256;
    P.s_nbn = ((gated ? shared.N / 2 : shared.N) + (gated ? 127 : 255)) /
              (gated ? 128 : 256);
    const int groups = (P.s_nbm + 7) / 8;
    P.s_group = (P.s_nbm + groups - 1) / groups;
    P.s_slots = std::max<long>(1, (shared.K + K / 2) / K);
  }
  const dim3 grid(std::min<long>(
      (max_blocks * P.nbn + P.s_nbm * P.s_nbn + 7) / 8 * 8, compute_units()));
#define RUN(FORM, ACT, ...)                                                  \
  hipLaunchKernelGGL((tile_gemm_kernel<FORM, ACT, true, false                \
                                       __VA_OPT__(,) __VA_ARGS__>), grid,    \
                     dim3(256), 0, stream, P)
  if (shared.C) {
    if (act == NONE) RUN(SCATTER, NONE, false, true);
    else if (act == SILU) RUN(GATED, SILU, false, true);
    else TORCH_CHECK(false, "moe_gemm_tiled_shared: act ", act);
    HIP_CHECK_KERNEL();
    return;
  }
  if (act == NONE) RUN(SCATTER, NONE);
  else if (act == SILU) RUN(GATED, SILU);
  else if (act == CLAMP) RUN(GATED, CLAMP);
  else if (act == RELU2) RUN(PLAIN, RELU2);
  else TORCH_CHECK(false, "moe_gemm_tiled: act ", act);
#undef RUN
  HIP_CHECK_KERNEL();
}
