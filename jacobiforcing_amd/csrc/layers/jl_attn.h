// jl_attn.h — what the attention sources share.
#ifndef JL_ATTN_H
#define JL_ATTN_H

#include "jl_common.h"

constexpr int AR_ROWS = 128;          // (query, head) rows of a tile of the wide form

// the wide form's launch (jl_attn_rows.hip); sizes as jl_attn_sweep has checked them, ``hf`` heads of a.TQ queries per tile, ``hb`` tiles per group
int jl_attn_rows_launch(const jl_attn_args &a, int hf, int hb, bool v_in_k, hipStream_t st);

#endif
