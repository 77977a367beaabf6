// Launchers of the recurrences with a decay per head and key channel, [D, Dv] states in fp32 per sequence and head:
// portions in chunks of 16 or 8 tokens on the matrix cores, single tokens as one pass over the state (chunk_recurrence.hip,
// chunk_recurrence_short.hip).
#pragma once
#include "nv_common.h"

namespace nv {

enum { kCrGated = 0, kCrGeneral = 1, kCrWrite = 2 };

// Raw projections as the entry points take them; which of them a form reads is written beside the form in chunk_recurrence.hip.
struct ChunkRecurrenceArgs {
    const void *x0, *x1, *x2, *x3, *v;         // [T, heads * D] each (x0, x1: heads / group heads), v: [T, H * Dv]
    int64_t s0, s1, s2, s3, sv;                // row strides in elements
    const void* b_raw;                         // gated: [T, H]
    int64_t b_stride;
    const float *c0, *c1;                      // constants per head and key channel (gated: c0 per head)
    const void* gate_raw;                      // [T, H * Dv] or NULL
    int64_t gate_stride;
    const float* norm_w;                       // [H * Dv] (norm_head_stride = Dv) or [Dv] (0)
    int norm_head_stride;
    float* state;                              // [slots, H, D, Dv]
    void* out;                                 // [T, H * Dv]
    int64_t out_stride;
    float* chunks;                             // the chunks' operands: [H, records, ..]
    void* columns;                             // their rows of V: [H, records, tokens of a chunk, Dv]
    float* raw;                                // [H, T, Dv]: read-outs in front of their norm
    uint32_t* odd;                             // [H, records]: some value of the chunk is not finite
    int64_t records;
    const int *cu_q, *cu_k, *slots;
    int num_seqs, H, group, D, Dv;             // group: heads that share a row of x0 and x1
    int64_t T;
    float eps, p0, p1;                         // gated: -, key_eps; general: decay_rate, key_eps
};

// Chunks of 8 tokens (chunk_recurrence_short.hip): records of `rows` rows in `seqs` sequences, words of a record, and both launches
// for the sequences first_seq .. with at least two rows (vec: two channels by one load; waves: for a state's 16 columns).
int64_t short_recurrence_records(int64_t rows, int seqs);
int short_recurrence_words(int form, int D);
void launch_short_recurrence(int form, const ChunkRecurrenceArgs& a, int first_seq, bool vec, int waves, int dtype, hipStream_t s);

// The launches of a step by what is known of its portions; false, with *rc NV_OK and nothing launched, when the sizes, the rows, a
// missing workspace or an unknown number of rows (T = 0) leave a step that may hold longer portions to the token-by-token launch.
bool run_recurrence_portions(int form, ChunkRecurrenceArgs a, int leading_singles, int portions, int dtype, void* workspace,
                             int64_t workspace_bytes, hipStream_t s, int* rc);

}  // namespace nv
