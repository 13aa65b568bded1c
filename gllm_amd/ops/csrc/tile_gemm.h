// Grouped products on 256-row blocks (tile_gemm.hip), called by
// moe_gemm_tiled.
#pragma once

void tile_gemm_grouped(void *C, const void *A, const void *W,
                       const int *sorted_ids, const int *expert_blocks,
                       const int *n_post_pad, const float *topk_w,
                       long max_blocks, long n_pairs, long topk, long Nd,
                       long K, long a_rows, int act, float limit,
                       float alpha);
