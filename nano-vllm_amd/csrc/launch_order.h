// Rules and index arithmetic of launches as plain functions of integers, so that a host compiler can check them over every launch shape.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define NV_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define NV_HD inline
#endif

namespace nv {

// Latent attention, several tokens, with ranges sized on the device: key tiles of a range of a launch with room for `slots` workgroups at a time.
NV_HD int latent_share(int64_t total_tiles, int slots, int fewest) {
    const int64_t share = (total_tiles + slots - 1) / slots, most = (int64_t)1 << 24;
    return (int)(share < fewest ? fewest : share > most ? most : share);
}
// Chunks behind at least three quarters of the longest sequence: all row tiles are about as long, so equal ranges of each, as the host plans them, are
// even already, and a share for every slot may leave whole row tiles over for a second round.  Share / equal ranges, us, 16 heads: rows of 256, 7 chunks of 290
// rows on 2966 .. 3257 keys 156 / 152, 6 of 183 on 5003 .. 5427 141 / 124, 5 of 194 on 6422 .. 7383 126 / 131;  rows of 320, 8 of 136 on 2808 .. 3466
// 177 / 159;  rows of 160, 9 of 161 on 3708 .. 3828 89 / 91.  With less in front: rows of 256, 8 of 256 on 3053 .. 4036 125 / 144.  The line dates
// from a slower loop over the tiles: of 40 such launches now, those of few row tiles were mostly faster with a share (3 chunks of 25 rows on 6717 .. 7748,
// rows of 320, 54 / 82), larger ones about even; 1.08 times as fast over all.
NV_HD bool latent_alike(int least_in_front, int longest) { return (int64_t)least_in_front * 4 >= (int64_t)longest * 3; }
// Launches of more than one round without key ranges: whether the order of workgroups is turned.  Their sequences come in turn, so each of 2, 4, 8 ..
// keeps to some of the XCDs and shader engines, and those of the longest are what the launch waits for; any other number, and sequences
// of about the same length, spread by themselves.  16 heads, us, as they come / turned: rows of 320, 4 prompts of 446 .. 931 70.6 / 53.9,
// 13 of 103 .. 164 20.7 / 26.1, 9 of 616 .. 805 110 / 116;  256: 2 of 1000 .. 2048 62.6 / 54.9, 8 of 318 .. 670 46.1 / 33.4, 16 of 200 .. 500 55.6 / 42.8,
// 8 of 1000 .. 1024 83.1 / 86.2, 7 of 309 .. 542 25.9 / 28.1;  160: 4 of 1000 .. 2048 69.5 / 60.8;  96: 8 of 600 .. 1024 30.1 / 28.7.
NV_HD bool latent_turns(int num_seqs, int64_t total_q, int max_q, int max_k) {
    return num_seqs > 1 && (num_seqs & (num_seqs - 1)) == 0 && (max_q != max_k || total_q * 9 < (int64_t)num_seqs * max_q * 8);
}
// Key tiles of a row tile whose last row sees `last_key`.  Workspace and block tables hold what the caller's longest length has room for,
// nsplit ranges of `fewest` tiles; keys beyond it, where that length was stated too small, are left out.
NV_HD int latent_tiles(int last_key, int tile_keys, int nsplit, int fewest) {
    const int tiles = last_key / tile_keys + 1, room = nsplit * fewest;
    return tiles < room ? tiles : room;
}
// Its ranges: at most nsplit, since a share is never below `fewest`.
NV_HD int latent_ranges(int tiles, int share) { return tiles <= share ? 1 : (tiles - 1) / share + 1; }

// An XCD's pairs in sets that differ by one at most: the first `more` pairs in sets of least + 1, the others in sets of `least`.
struct PairSets {
    int least, more;
};
NV_HD PairSets pair_sets(int pairs, int sets) { return {pairs / sets, pairs % sets * (pairs / sets + 1)}; }
// A workgroup's slot on its XCD -> its set's first pair, how many there are, and its place among their workgroups.  (One division on the device.)
struct SetPlace {
    int first, n, at;
};
NV_HD SetPlace set_place(int slot, int slots_per_pair, const PairSets& s) {
    const int front = s.more * slots_per_pair, n = slot < front ? s.least + 1 : s.least, rest = slot < front ? slot : slot - front;
    const int set = rest / (n * slots_per_pair);
    return {(slot < front ? 0 : s.more) + set * n, n, rest - set * n * slots_per_pair};
}

// Prompt attention, single query tiles a workgroup: how many pairs of sequence and kv head an XCD takes together, the heaviest tiles of all first.  For
// sequences of about the same length and about two rounds of workgroups, as long as the pairs' keys and values stay within half its L2 (those of a larger set, below, within all of it).  4 prompts of 2000 ..
// 2048 tokens, 16 / 8 heads: 101 -> 86 us, 8 of 900 .. 1024 68 -> 57, 6 of 1000 .. 1365 72 -> 64; 2 of 600 and 2048, 32 / 8 heads, 61 -> 66, and with
// more rounds the order counts for less than the L2 (32 / 8 heads, 7 of 600 .. 1100: 76 -> 81, 4 of 1000 new tokens on 3000: 107 -> 130).
NV_HD int prefill_together(int64_t workgroups, int64_t total_q, int num_seqs, int max_q, int max_k) {
    if (workgroups > 576 || total_q * 4 < (int64_t)num_seqs * max_q * 3) return 1;
    const int fit = 4096 / (max_k > 1 ? max_k : 1);
    return fit < 1 ? 1 : fit < 4 ? fit : 4;
}
// An XCD's `rounds` pairs in sets of as many as that, or a few more: sets differ by a pair at most, because what is left over for a short last one begins with
// its heaviest tile when the others end.  One after the other / in sets of four with the rest last / so: 9 prompts of 545 .. 793, 16 / 8 heads,
// 48.8 / 51.8 / 44.7 us, 10 of 627 .. 654, 16 / 4, 45.0 / 46.4 / 39.7, 5 of 771 .. 1206, 16 / 16, 58.7 / 63.1 / 58.9; 90 launches of 257 to 576
// workgroups 1 / 0.960 / 0.938 on average, 1.06 at most (1.07 with the rest last).
NV_HD PairSets prefill_sets(int rounds, int together) { return pair_sets(rounds, rounds > together ? rounds / together : 1); }
// A workgroup's slot on its XCD -> round of pairs and place in the pair: the rounds of a set place by place, turning by one every time.
struct RoundPlace {
    int round, place;
};
NV_HD RoundPlace prefill_order(int slot, int slots_per_pair, const PairSets& sets) {
    const SetPlace s = set_place(slot, slots_per_pair, sets);
    if (s.n == 1) return {s.first, s.at};
    const int place = s.at / s.n;
    return {s.first + (s.at + place) % s.n, place};
}

// Score-modified attention, prompt portions: workgroup (of a key range) -> its pair of sequence and kv head and its place in the pair, heaviest query
// tile first.  Workgroups go to the eight XCDs in turn; an XCD has `rounds` pairs (8 >> xs_shift of them a round over all XCDs) in sets of three to
// five: what four at a time leave over begins with its heaviest tile when the others end.  One after the other /
// so, the launch alone: 3 prompts of 1893 .. 2197, 16 heads of 128 each, 97 / 86 us, 12 of 444 .. 676, 16 / 4 of 64, 29.8 / 28.3.  With an earlier loop
// over the tiles, 70 launches of a number of pairs that fours do not divide, one after the other / fours and the rest last / so: 1 / 0.991 / 0.975 on
// average, 1.05 at most (1.08 with the rest last).
// grid: 8 * rounds * slots_per_pair; places past a pair's workgroups and pairs past the last one are for the caller to leave out.
NV_HD PairSets scoremod_sets(int rounds) { return pair_sets(rounds, rounds < 6 ? 1 : (rounds + 2) / 4); }
struct PairGroup {
    int pair, step, n;          // the group's first pair, from one pair to the next, how many there are
    int at;                     // the workgroup's place in the group
};
struct PairPlace {
    int pair, place;
};
NV_HD PairGroup scoremod_group(int index, const PairSets& sets, int slots_per_pair, int xs_shift) {
    const SetPlace at = set_place(index >> 3, slots_per_pair, sets);
    return {at.first * (8 >> xs_shift) + ((index & 7) >> xs_shift), 8 >> xs_shift, at.n, at.at};
}
// Whether pairs are of about the same length: `n` of them (of a group of chunks; the sequences of a step of whole prompts) with `keys` keys in all.  In 170 steps of 2 to 16 sequences whole prompts gained from
// an average of three quarters of the longest on, chunks, whose tiles are all about as heavy as their sequence is long, from eight ninths on.
NV_HD bool scoremod_even(int64_t keys, int64_t longest, int n, int whole_prompts) {
    return whole_prompts ? keys * 4 >= longest * n * 3 : keys * 9 >= longest * n * 8;
}
// What a launch knows of that: 1 and 0, or -1 where a group of chunks is to look at its own lengths.  Chunks of no more workgroups of a key range than CUs
// do not look, which takes half a microsecond of 13 to 21, and go one after the other: with several key ranges the order is not without
// effect there, 5 of 230 rows on 2194 .. 3955 keys, 16 / 8 heads of 128, 73 us so and 91 together, 2 of 431 on 3229 .. 4093 64 and 75; with an earlier loop 80 such
// steps, from 0.90 to 1.14 of the time and 1.005 on average together, 0.997 looking first (7 of them 2 to 4 % slower for it).
NV_HD int scoremod_pairs(int64_t grid_base, int num_seqs, int64_t total_q, int max_q, int max_k) {
    if (max_q == max_k) return scoremod_even(total_q, max_q, num_seqs, 1);
    return grid_base <= 256 ? 0 : -1;
}
// together: the pairs of the set place by place, turning by one every time, or one after the other.  there_and_back: 32 workgroups of the XCD there and the next 32 back instead.
NV_HD PairPlace scoremod_order(const PairGroup& g, int index, int slots_per_pair, int xs_shift, bool together, int there_and_back) {
    int at = g.at;
    if (together && there_and_back && (at & 32) && (at | 31) < g.n * slots_per_pair) at ^= 31;
    const int rank = together ? at / g.n : at % slots_per_pair;
    const int one = together ? (at - rank * g.n + (there_and_back ? 0 : rank)) % g.n : at / slots_per_pair;
    return {g.pair + one * g.step, (rank << xs_shift) + (index & ((1 << xs_shift) - 1))};
}

// Score-modified attention, prompt portions: the loop for launches of several tiles, from four on and wherever a bias is added.  Shorter ones have few steps to
// gain in and more in front of the first.  Short loop / long, us, the call with its preparation, 16 heads, soft cap: rows of 128, one prompt of 64 tokens
// 10.55 / 10.76, 13 of 20 .. 64 13.0 / 13.3, 8 of 100 .. 190 18.1 / 18.2, 3 of 200 .. 256 19.1 / 18.9, 2 of 385 .. 762 32.9 / 31.9;  rows of 64, one of 54 8.75 / 8.88,
// 2 of 121 .. 395 16.81 / 16.85, 3 of 900 .. 2000 71.1 / 69.7.  With a bias, the launch alone: one prompt of 54 tokens, rows of 128, 7.2 / 6.7, 3 of 700 .. 1900 86 / 63.
NV_HD bool scoremod_long(int max_k, bool biased) { return biased || max_k > 192; }

// Tiles of 128 rows, no more blocks than CUs: slices 32 deep, since nothing else runs on a CU while its one workgroup waits for a slice.  Tiles of an
// expert: one, from 100 pairs on as many as its pairs fill and a half.  First / second product of 16 or 32 experts, us, 64 and 32 deep:
//   128 blocks   width 2048, ff 1024: 41.5 and 36.7 / 23.9 and 21.8;  width 1024, ff 512: 25.7 and 23.0 / 15.7 and 15.3
//   256          2048, 1024: 50.5 and 46.8 / 30.2 and 27.3;  1024, 1024: 31.9 and 27.8 / (128) 24.3 and 22.1
//   192, 256     2048, 1024, 128 and 192 pairs an expert: 46.6 and 38.9 / 27.2 and 23.9, 42.9 and 41.0 / 25.5 and 25.4
//   320, 384     2048, 1024: 50.7 and 68.5 / 32.0 and 39.7, 68.0 and 83.0 / 34.6 and 42.1
// (the same order with weights that come from memory instead of the last cache: 51.9 and 47.0 / 27.4 and 25.1 for the first)
NV_HD bool moe_few_blocks(int64_t pairs, int E, int n_cols) {
    return (pairs <= 100 * (int64_t)E ? E : pairs / 128 + E / 2) * n_cols <= 256;
}

// Tiles of up to 64 rows past LDS, an expert's weights once for each of its tiles, or through it.  What pays depends on how many tiles read
// the same weights, and where a whole tile an expert does, on how many blocks of 128 x 128 the first product has.  Both products, us, past / through LDS:
//   tiles of 16: 32 experts, 2048, 1024: 8 pairs an expert 69 / 65 (weights from memory: 76 / 91), 12: 75 / 67 (83 / 92), 20: 108 / 71 (113 / 96);
//     16 of 2048, 1024: 12: 49 / 45 (54 / 62), 16: 48 / 46 (52 / 64), 20: 59 / 46 (62 / 64)
//   tiles of 64, 256 blocks: 32 of 2048, 1024: 32: 92 / 82 (98 / 100), 40: 99 / 85 (105 / 104), 64: 142 / 102, 1024: 1477 / 713
//     128 blocks: 16 of 2048, 1024: 48: 54 / 74, 56: 73 / 75 (77 / 88), 64: 86 / 76;  32 of 1024, 512: 56: 44 / 47, 64: 54 / 47
//     64 blocks: 16 of 1024, 512: 64: 32 / 44, 96: 33 / 44, 160: 53 / 46
NV_HD bool moe_streams(int tile_rows, int64_t pairs, int E, int ff) {
    const int64_t blocks = (int64_t)E * ((ff + 127) / 128);
    const int line = tile_rows == 16 ? 16 : tile_rows == 32 ? 28 : tile_rows == 64 ? (blocks >= 256 ? 40 : blocks >= 128 ? 64 : 128) : 0;
    return pairs < line * (int64_t)E;
}

// Recurrences, single tokens: sequences known to be of one token in a launch over those in front (`lead`) and, among longer portions (`rest`), behind
// them.  Only their states are read and written by it.
NV_HD int recurrence_singles(int num_seqs, int lead, bool rest) { return rest ? lead : num_seqs; }
// Whether their states pass by the caches (loads and stores).  What pays depends on whether the last cache (256 MB) keeps a layer's states until its next step,
// so on what the step touches in between, which a launch does not know.  Through / past, us, 16 heads 128 x 128, gated, states of as many layers in turn:
//                         1              3              6 and 12             1, written just before   a state's first pass
//   32 seqs (34 MB)   13.9 / 13.2    16.6 / 14.7    16.4 / 15.2, 20.1 / 15.5
//   64 (67 MB)        25.0 / 27.6    24.7 / 29.5    39.2 / 30.0, 39.3 / 30.0
//   80 (84 MB)        31.1 / 33.1    31.3 / 35.5    44.0 / 35.4, 43.9 / 36.3
//   92 (96 MB)        33.8 / 38.5    40.6 / 40.5    49.4 / 40.7, 49.5 / 40.8
//   128 (134 MB)      44.1 / 49.4    60.5 / 50.5    60.9 / 50.8, 60.6 / 50.9       46.0 / 46.7               83 / 88
//   256 (268 MB)      100 / 98       113 / 99       112 / 99, 112 / 99             95.6 / 92.6              129 / 145
//   64 x 64, 256 (67 MB)  37.2 / 45.0, 36.9 / 45.2, 51.1 / 45.2, 51.1 / 45.2;  384 (101 MB)  51.7 / 66.4, 71.8 / 66.7, 73.2 / 66.7, 73.2 / 66.8
// The line is where three layers' states stop fitting.  A model of more layers would gain from less on and loses nothing at it; one whose
// states all stay loses up to 28 % between 96 and 200 MB.  General and write as gated.  Only loads or only stores past the caches: 106 and 114 for 256.
NV_HD bool recurrence_streams(int singles, int H, int D, int Dv) { return (int64_t)singles * H * D * Dv * 4 >= 92LL << 20; }

// Outputs of the second product (fp32, a row a pair) past the caches, where they and the experts' weights (three matrices of ff x width each) together do not
// stay in the last cache (256 MB, beside rows and activations): they drive out what other blocks read, and themselves before the caller adds a token's
// rows up.  The call with that sum, through / past, us, weights of one layer, of six layers in turn (MiB of outputs + weights; experts, top, width, ff):
//   64 + 384 (32, 4, 2048, 1024)   215 / 208, 221 / 215        64 + 192 (16, 2, 2048, 1024)   190 / 190, 195 / 197
//   256 + 384                      560 / 550, 541 / 527        128 + 192                      303 / 295, 310 / 300
//   64 + 192 (32, 2, 2048, 512)    139 / 139, 142 / 144        128 + 192                      219 / 214, 226 / 221
//   128 + 96 (16, 4, 2048, 512)    190 / 188, 193 / 197        256 + 96                       342 / 318, 339 / 321
// and below the line:
//   64 + 96 (16, 4, 2048, 512)     107 / 109, 120 / 121        93 + 96                        124 / 127, 133 / 135
//   64 + 96 (16, 2, 1024, 1024)    168 / 170, 180 / 182        128 + 48 (16, 4, 1024, 512)    180 / 181, 181 / 186
// Without the sum they pay from less on (64 + 192 of 32 experts, 115 / 95); outputs of less than 64 MiB made no difference to the call with it.
NV_HD bool moe_streams_out(int64_t pairs, int width, int E, int ff) {
    const int64_t out = pairs * width * 4, weights = (int64_t)E * ff * width * 6;
    return out >= 64LL << 20 && out + weights >= 224LL << 20;
}

}  // namespace nv
