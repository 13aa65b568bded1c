// attention_causal.hip: plain causal softmax attention of prompt rows, called
// by launch_prefill where nothing else is asked for.
#pragma once

bool causal_prefill_ok(int D, int Dv, float scale);
void causal_prefill(void *out, long out_stride, const void *q, long q_stride,
                    const void *k_cache, const void *v_cache,
                    const int *block_table, long max_pages, int page_size,
                    const int *seq_lens, const int *qsl, int B, long T,
                    long max_query_len, int Hq, int Hkv, int D, float scale,
                    int min_rows);
