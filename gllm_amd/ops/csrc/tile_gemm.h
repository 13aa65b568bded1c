// tile_gemm.hip: grouped products on 256-row blocks, called by
// moe_gemm_tiled; split products of few rows, called by stream_parts.
#pragma once

bool tile_gemm_grouped_ok(long a_numel, long n_pairs, long Nd, long K,
                          int act);
// a product [rows, K] [N, K]^T of the same form beside the grouped one; C null:
// none. N * K below 2^30
struct TileShared {
  void *C;
  const void *A, *W;
  int rows, K, N;
};
void tile_gemm_grouped(void *C, const void *A, const void *W,
                       const int *sorted_ids, const int *expert_blocks,
                       const int *n_post_pad, const float *topk_w,
                       long max_blocks, long n_pairs, long topk, long Nd,
                       long K, long a_rows, int act, float limit,
                       float alpha, const TileShared &shared);

// x [M, K] w [N, K]^T of at most 256 rows as fp32 parts [splits, M, N]
void tile_parts_plan(long M, long N, long K, int *bm, int *splits);
void tile_parts(float *part, const void *x, const void *w, long M, long N,
                long K, int bm, int splits);

// stream_gemm.hip: the columns of K that one fp32 sum of stream_gemm's covers
// (the sums are added in the order of K), 0 where it takes tile_parts'
long stream_slice(long M, long N, long K);
