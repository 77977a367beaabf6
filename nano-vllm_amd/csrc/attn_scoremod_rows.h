// The 32 x 32 tile launch for prompt portions of the score-modified attention (attn_scoremod_rows.hip).
#pragma once
#include "launch_order.h"
#include "nv_common.h"

namespace nv {

struct ScoremodRowsParams {
    const __bf16 *q, *k_cache, *v_cache;
    __bf16* out;
    const int *cu_q, *cu_k, *block_tables;
    const float *sink, *dist_bias;
    float* part;                               // [T, H, nsplit, Dv + 2] when nsplit > 1
    int64_t q_stride, out_stride;
    int v_ld, n_dist, H, G, block_size, max_blocks, max_block;
    float softcap, scale_log2, cap_in;         // cap_in: a raw score's factor to the exponent of tanh
    int hpw, n_qtiles, wg_per_pair, n_pairs, xs_shift, slots_per_pair, grid_base, nsplit, tiles_per_split;
    PairSets sets;                             // of an XCD's pairs
    int even, there_and_back;                  // the pairs of a set are about as long (1, 0, or -1: see cu_k); all workgroups run at a time
};
struct ScoremodRowsPlan {
    int hpw;                                   // heads of a kv head's group that a workgroup takes (1, 2 or 4)
    int n_qtiles, wg_per_pair, n_pairs, xs_shift, slots_per_pair, nsplit, tiles_per_split;
    int64_t grid_base, ws_bytes;
};

bool scoremod_rows_built(int D, int Dv, int block_size);
ScoremodRowsPlan scoremod_rows_plan(int num_seqs, int64_t T, int H, int G, int Dv, int max_seqlen_q, int max_seqlen_k);
int launch_scoremod_rows(ScoremodRowsParams p, const ScoremodRowsPlan& f, int D, int Dv, int num_seqs, int64_t total_q, int max_seqlen_q, int max_seqlen_k, float scale,
                         hipStream_t s);

}  // namespace nv
