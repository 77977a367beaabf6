// Prompt portions of the score-modified attention on 32 x 32 matrix-core tiles (nv_attn_scoremod_paged: scores scaled, soft-capped,
// distance-biased; a sink in the denominator).
//
// A wave owns 32 query rows of one head; the four waves of a workgroup share a kv head: up to four heads of its group times
// consecutive row blocks, so a key tile serves them all.  Tiles of 64 keys go through the block table straight into LDS (LDS-DMA,
// double-buffered, swizzled in 8-row x 32-column subtiles), and
//     S^T (keys x rows) = K Q^T        v_mfma_f32_32x32x16_bf16: A = K rows from LDS, B = Q^T in registers
//     O^T (columns x rows) += V^T P^T  A = V rows read transposed (ds_read_b64_tr_b16), B = P^T, the registers of S^T as bf16
// A row's scores live in two lanes, so a maximum is one exchange a tile.  It is the row's true running maximum (a tile that does not
// raise it in any row skips the rescale), so that its largest weight is an exact 1, and the denominator sums the weights in front of
// their rounding to bf16, both as on the 16 x 16 tiles: outputs of the call below differ from theirs by 9e-5 and are 0.00258 from
// the same in 64 bits (2-norms relative to the output rows, bf16), on either.  Exponentials relative to the soft cap, without any
// maximum: 0.0028 and 119 us; the same with probabilities as the sum of two bf16 numbers: 0.0022 and 148 us.
//
// What bounds it: the instructions of the scores.  64 soft-capped scores are nine vector instructions and three at quarter rate (two exponentials, a
// reciprocal) for a row beside 32 cycles of matrix products, which are 34 % of the busy cycles of the call below.  So, in launches
// of several tiles, tiles come by loads that the compiler does not know (it would wait for the next tile in front of the first transposed read), and with
// rows of 128 columns, two waves a SIMD, the weights of a tile are made beside the scores of the next one, which are capped beside the values of this one.
// With rows of 64 columns more waves take turns, and the registers of the next scores would cost one or two of them: 8 prompts of 1024, 16 / 4 heads of 64, 51 us, so with two waves 56.
// 4 prompts of 1777 .. 2048 tokens, 16 / 8 heads of 128, soft cap and sink, the call with its preparation of 21 us: 112 us on a card where a tile's work one
// after the other takes 114; 3 prompts of 700 .. 1900 71 and 75, 2 portions of 1000 on 3000 .. 4000 117 and 121.  On another card 117 for that order, 127 with an
// XCD's pairs one after the other (see there) and 129 with the denominator as a product of rounded weights with ones; with the launch on 16 x 16
// tiles, values transposed through registers, which other sizes still take, 496 us (44 of them preparation).
// Not taken: an odd polynomial of tanh where a tile's products are within 0.4 caps (the same call 112; 8 prompts of 300 .. 800, 16 / 4 heads of 64, 39 us instead
// of 42).  Whether a tile takes it depends on the portion a row comes in, and with it the row's bits; its coefficients
// overflow with caps below about 1e-8, its squares with products above 1.8e19.
#include <algorithm>
#include <type_traits>

#include "attn_scoremod_rows.h"

namespace nv {

constexpr int kSrTile = 64;
constexpr float kSrLog2e = 1.4426950408889634f;
constexpr float kSrInit = -1.0e30f;

typedef __attribute__((address_space(3))) s16x4 sr_lds_s16x4;

enum { kSrPlain = 0, kSrCap = 1, kSrGeneral = 2 };    // scale only | soft cap alone | bias, with a cap or without

// byte offset of 16-byte chunk `ch` of row `row` in the image of a tile whose rows are 32 * C32 columns wide
template <int C32>
__device__ __forceinline__ int sr_off(int row, int ch) {
    return 512 * C32 * (row >> 3) + 512 * (ch >> 2) + 64 * (row & 7) + 16 * ((ch & 3) ^ ((row >> 2) & 3));
}
__device__ __forceinline__ float sr_max_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sr_sum_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// LONG: the loop for launches of several tiles (see scoremod_long).
template <int D32, int V32, int MOD, bool LONG>
__global__ __launch_bounds__(256, !LONG ? 2 : D32 + V32 == 4 ? (MOD == kSrGeneral ? 3 : 4) : D32 + V32 == 6 && MOD != kSrGeneral ? 3 : 2) void scoremod_rows_kernel(const ScoremodRowsParams p) {
    constexpr int KB = 4096 * D32, VB = 4096 * V32, BUF = KB + VB;          // bytes of a K tile, a V tile, both
    constexpr int STG = 64 * V32 + 16;                                      // bytes of an output row on its way through LDS
    constexpr int LDS = 2 * BUF > 4 * 32 * STG ? 2 * BUF : 4 * 32 * STG;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, hh = lane >> 5;

    // Workgroup -> (sequence, kv head, head group, query tile): workgroups that read the same keys share an XCD.  An XCD takes its pairs
    // (of sequence and kv head) about four together, the heaviest query tiles of all first; pair after pair, a CU's workgroups were heavy or light
    // together and the last pair's heaviest tile began half way.  Workgroups one after the other run on the XCD's four shader engines, so
    // the pairs turn by one every time.  Where all workgroups are there from the start, 32 (one for each CU) go there and the next 32
    // back instead, so that a CU that has a heavy one gets a light one with it (one heavy after the other is better where
    // CUs that have ended take the next).  Pairs of very different lengths are no order of weight that way and go one after the other:
    // 16 / 4 heads of 64, the launch alone, 16 chunks of 300 rows on 600 .. 4000 keys 106 us, together 133, 6 prompts of 300 .. 1300 36 and 44, 6 of 466 .. 862
    // 36 and 23.
    const int split = blockIdx.x / p.grid_base, bid = blockIdx.x - split * p.grid_base;
    const PairGroup group = scoremod_group(bid, p.sets, p.slots_per_pair, p.xs_shift);
    bool even = p.even > 0;
    if (p.even < 0) {                                 // (keys in front of the rows: the host does not know their number)
        int longest = 0, keys = 0, n = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int pair = group.pair + i * group.step;
            if (i < group.n && pair < p.n_pairs) {
                const int b = pair / p.G, rows = p.cu_q[b + 1] - p.cu_q[b], n_k = rows > 1 ? p.cu_k[b + 1] - p.cu_k[b] : 0;
                longest = max(longest, n_k);
                keys += n_k;
                n += rows > 1;
            }
        }
        even = scoremod_even(keys, longest, n, 0);
    }
    const PairPlace at = scoremod_order(group, bid, p.slots_per_pair, p.xs_shift, even, p.there_and_back);
    const int pair = at.pair, widx = at.place;
    if (pair >= p.n_pairs || widx >= p.wg_per_pair) return;
    const int groups = p.wg_per_pair / p.n_qtiles, hg = widx % groups, qt = p.n_qtiles - 1 - widx / groups;   // heaviest first
    const int b = pair / p.G, g = pair - b * p.G;
    const int hq = g * (p.H / p.G) + hg * p.hpw + wave % p.hpw;
    const int q_begin = p.cu_q[b], n_q = p.cu_q[b + 1] - q_begin, n_k = p.cu_k[b + 1] - p.cu_k[b];
    const int rows_per_wg = 32 * (4 / p.hpw), q0 = qt * rows_per_wg;
    if (n_q <= 1 || q0 >= n_q) return;                // single rows belong to another launch
    const int shift = n_k - n_q, rw0 = q0 + (wave / p.hpw) * 32;            // row i sees keys <= i + shift
    const bool wave_live = rw0 < n_q;
    const int max_key = min(min(q0 + rows_per_wg, n_q) - 1 + shift, n_k - 1);
    // (no key at all, e.g. a sequence that has none: no tile, or its rows' clamp to the last key would leave the cache)
    const int t_begin = split * p.tiles_per_split, nt = min(max_key < 0 ? 0 : max_key / kSrTile + 1, t_begin + p.tiles_per_split);

    bf16x8 qf[2 * D32];                               // lane (r, hh): Q[row r][16 s + 8 hh ..]
    {
        const __bf16* qp = p.q + (int64_t)(q_begin + min(rw0 + r, n_q - 1)) * p.q_stride + (int64_t)hq * (32 * D32) + 8 * hh;
#pragma unroll
        for (int s = 0; s < 2 * D32; ++s) qf[s] = *(const bf16x8*)(qp + 16 * s);
    }
    f32x16 oacc[V32];
#pragma unroll
    for (int d = 0; d < V32; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[d][i] = 0.f;
    const float cap2 = p.softcap * kSrLog2e;
    float m_run = kSrInit;                            // the row's maximum so far, log2 units
    // The denominator, this lane's keys: a sum of the weights as computed (of the rounded ones it would be off by up to 2^-9).
    float l_run = 0.f;
    const float* bias = MOD == kSrGeneral ? p.dist_bias + (int64_t)hq * p.n_dist : nullptr;

    // staging: one DMA instruction fills 1 KiB of LDS linearly (lane l: bytes 16 l ..), two subtiles; a lane picks the (row, chunk)
    // that the image has there.  Wave w takes pieces w, w + 4, .. of K and of V.
    const int* bt = p.block_tables + (int64_t)b * p.max_blocks;
    const int tpb = p.block_size / kSrTile;
    const uint32_t k_row = (uint32_t)p.G * 64u * D32, v_row = (uint32_t)(p.G * p.v_ld * 2);            // bytes between cache rows
    int dk_row[D32], dv_row[V32];
    uint32_t dk_off[D32], dv_off[V32];
#pragma unroll
    for (int i = 0; i < D32; ++i) {
        const int sub = 2 * (wave + 4 * i) + (lane >> 5);
        dk_row[i] = 8 * (sub / D32) + ((lane & 31) >> 2);
        dk_off[i] = dk_row[i] * k_row + (4 * (sub % D32) + ((lane & 3) ^ ((dk_row[i] >> 2) & 3))) * 16u;
    }
#pragma unroll
    for (int i = 0; i < V32; ++i) {
        const int sub = 2 * (wave + 4 * i) + (lane >> 5);
        dv_row[i] = 8 * (sub / V32) + ((lane & 31) >> 2);
        dv_off[i] = dv_row[i] * v_row + (4 * (sub % V32) + ((lane & 3) ^ ((dv_row[i] >> 2) & 3))) * 16u;
    }
    const int i16 = lane & 15, g16 = (lane >> 4) & 1;
    const int qpos = rw0 + r + shift;                 // last key this lane's row sees
    const int wave_last = min(rw0 + 31, n_q - 1) + shift;
    // cap tanh(x / cap) = cap - 2 cap / (exp(2 x / cap) + 1), in log2 units, of a product x
    auto capped = [&](float x) { return cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * p.cap_in) + 1.0f); };
    if constexpr (LONG) {
        // Rows of 128 columns: the next tile's scores beside this tile's weights.  Rows of 64 columns leave room for three or four waves a SIMD,
        // which take turns: a tile's work one after the other, in the compiler's order.
        constexpr bool AHEAD = D32 + V32 == 8;
        // K tiles and V tiles have two buffers each; a K tile is asked for two steps before its scores' weights are needed, a V tile one.
        const uint32_t lds_at = lds_address(lds), lane_to = lds_at + wave * 1024;
        int st_block = t_begin / tpb, st_in = t_begin - st_block * tpb;         // where the K tile staged next lies
        auto entry_here = [&] { return bt[min(st_block, p.max_blocks - 1)]; };  // (a tile that there is has its entry; others' are not used)
        auto row_here = [&](int entry) {                  // its first cache row; then on to the next tile
            const int phys = min(max(__builtin_amdgcn_readfirstlane(entry), 0), p.max_block);
            const int64_t row = ((int64_t)phys * p.block_size + st_in * kSrTile) * p.G + g;
            const int wrap = ++st_in == tpb;
            st_in = wrap ? 0 : st_in;
            st_block += wrap;
            return row;
        };
        auto stage_k = [&](int t, int64_t row) {
            const char* kb = (const char*)p.k_cache + row * (64 * D32);
            const int last = n_k - 1 - t * kSrTile;       // (rows past the sequence re-read the last one: finite, and hidden by the mask)
            const uint32_t to = lane_to + (t & 1) * KB;
            if (last >= kSrTile - 1) {
#pragma unroll
                for (int i = 0; i < D32; ++i) lds_load16(kb, dk_off[i], to + i * 4096);
            } else {
#pragma unroll
                for (int i = 0; i < D32; ++i) lds_load16(kb, dk_off[i] - (uint32_t)max(dk_row[i] - last, 0) * k_row, to + i * 4096);
            }
        };
        auto stage_v = [&](int t, int64_t row) {
            const char* vb = (const char*)p.v_cache + row * (p.v_ld * 2);
            const int last = n_k - 1 - t * kSrTile;
            const uint32_t to = lane_to + 2 * KB + (t & 1) * VB;
            if (last >= kSrTile - 1) {
#pragma unroll
                for (int i = 0; i < V32; ++i) lds_load16(vb, dv_off[i], to + i * 4096);
            } else {
#pragma unroll
                for (int i = 0; i < V32; ++i) lds_load16(vb, dv_off[i] - (uint32_t)max(dv_row[i] - last, 0) * v_row, to + i * 4096);
            }
        };
        const int w_end = wave_live && wave_last >= 0 ? min(nt, wave_last / kSrTile + 1) : t_begin;       // behind the wave's last tile

        // operands: lane's places in a tile; the others lie at constant distances
        uint32_t key_at[2], value_at[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            key_at[i] = lds_at + sr_off<D32>(r, 2 * i + hh);
            value_at[i] = lds_at + 2 * KB + sr_off<V32>(8 * i + 4 * hh + (i16 >> 2), 2 * g16 + ((i16 & 3) >> 1)) + 8 * (i16 & 1);
        }
        constexpr int KSTEPS = 2 * D32, VSTEPS = 4 * V32, KA = 2, VA = 4;       // products a key block and tile; operands ahead
        typedef __attribute__((address_space(3))) const bf16x8* KeyPtr;
        struct Tile {
            const lds_byte* at[2];
        };
        auto key = [&](const Tile& t, int c, int kb) { return *(KeyPtr)(t.at[c & 1] + 2048 * D32 * kb + 512 * (c >> 1)); };
        auto value = [&](const Tile& t, int n) {          // 16 keys (n / V32) x 32 columns (n % V32), transposed on their way
            const int off = 1024 * V32 * (n / V32) + 512 * (n % V32);
            const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((sr_lds_s16x4*)(t.at[0] + off));
            const s16x4 v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((sr_lds_s16x4*)(t.at[1] + off));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(v1, v2, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        float s[32];                                      // a tile's scores, then weights: 16 kb + i is key kt + 32 kb + (i & 3) + 8 (i >> 2) + 4 hh; row rw0 + r
        f32x16 n[2];                                      // the next tile's as they are multiplied
        auto scores = [&](int t, auto beside) __attribute__((always_inline)) {
            const Tile tile = {{lds_pointer(key_at[0] + (t & 1) * KB), lds_pointer(key_at[1] + (t & 1) * KB)}};
            constexpr f32x16 zero = {};
            if constexpr (!AHEAD) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int c = 0; c < KSTEPS; ++c) n[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(key(tile, c, kb), qf[c], c ? n[kb] : zero, 0, 0, 0);
                return;
            }
            bf16x8 a[KA][2];
#pragma unroll
            for (int c = 0; c < KA; ++c) {
                a[c][0] = key(tile, c, 0);
                a[c][1] = key(tile, c, 1);
            }
#pragma unroll
            for (int c = 0; c < KSTEPS; ++c) {
                __builtin_amdgcn_sched_barrier(0);        // (left alone, a product waits for the read just before it)
                n[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c % KA][0], qf[c], c ? n[0] : zero, 0, 0, 0);
                n[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c % KA][1], qf[c], c ? n[1] : zero, 0, 0, 0);
                if (c + KA < KSTEPS) {
                    a[c % KA][0] = key(tile, c + KA, 0);
                    a[c % KA][1] = key(tile, c + KA, 1);
                }
                beside(c);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto values = [&](int t, const bf16x8 (&pb)[4], auto beside) __attribute__((always_inline)) {
            const Tile tile = {{lds_pointer(value_at[0] + (t & 1) * VB), lds_pointer(value_at[1] + (t & 1) * VB)}};
            if constexpr (!AHEAD) {
#pragma unroll
                for (int c = 0; c < VSTEPS; ++c) oacc[c % V32] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(value(tile, c), pb[c / V32], oacc[c % V32], 0, 0, 0);
                return;
            }
            bf16x8 a[VA];
#pragma unroll
            for (int i = 0; i < VA; ++i) a[i] = value(tile, i);
#pragma unroll
            for (int c = 0; c < VSTEPS; ++c) {
                __builtin_amdgcn_sched_barrier(0);
                oacc[c % V32] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c % VA], pb[c / V32], oacc[c % V32], 0, 0, 0);
                if (c + VA < VSTEPS) a[c % VA] = value(tile, c + VA);
                beside(c);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // A score from its product to log2 units: capped, scaled or, elsewhere, with a bias on top.
        constexpr bool BESIDE = MOD != kSrGeneral;        // (a bias comes from memory: all of them together)
        auto modify = [&](int i, float& top) __attribute__((always_inline)) {
            const float x = n[i >> 4][i & 15];
            s[i] = MOD == kSrCap ? capped(x) : x * p.scale_log2;
            top = fmaxf(top, s[i]);
        };
        // (One branch for all of them: one a score left the reads of the bias one after the other.  3 prompts of 700 .. 1900, 16 / 8 heads of 128: 82 -> 63 us.)
        auto all_general = [&](int kt) __attribute__((always_inline)) {
            if (p.softcap > 0.f) {
#pragma unroll
                for (int i = 0; i < 32; ++i) s[i] = capped(n[i >> 4][i & 15]);
            } else {
#pragma unroll
                for (int i = 0; i < 32; ++i) s[i] = n[i >> 4][i & 15] * p.scale_log2;
            }
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const int j = kt + (i >> 4) * 32 + (i & 3) + 8 * ((i & 15) >> 2) + 4 * hh;
                s[i] += kSrLog2e * bias[min(max(qpos - j, 0), p.n_dist - 1)];
            }
        };
        // Hides what a row does not see of the tile at key kt, where some row of the wave does not see all of it, and raises the running maximum.
        // top: the largest of this lane's scores.
        auto settle = [&](int kt, float top) __attribute__((always_inline)) {
            const bool edge = kt + kSrTile - 1 > rw0 + shift;
            if (edge) {
                asm volatile("");                         // (a branch around it, not 32 selections in every tile)
                top = -INFINITY;
#pragma unroll
                for (int i = 0; i < 32; ++i) {
                    s[i] = kt + (i >> 4) * 32 + (i & 3) + 8 * ((i & 15) >> 2) + 4 * hh <= qpos ? s[i] : -INFINITY;
                    top = fmaxf(top, s[i]);
                }
            }
            const float tmax = sr_max_xor32(top);
            if (!__all(tmax <= m_run)) {                  // rare after the first tiles
                const float m_new = fmaxf(m_run, tmax), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < V32; ++d) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) oacc[d][i] *= alpha;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        float l_part[4];
        auto weigh = [&](int i, int step, bf16x8 (&pb)[4]) __attribute__((always_inline)) {
            if (step == 0) s[i] -= m_run;
            if (step == 1) s[i] = __builtin_amdgcn_exp2f(s[i]);
            if (step == 2) {
                l_part[i & 3] += s[i];
                if ((i & 7) == 7) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) pb[i >> 3][j] = (__bf16)s[i - 7 + j];
                    if constexpr (AHEAD) asm volatile("" : "+v"(pb[i >> 3]));        // (here and not where it is needed)
                }
            }
        };
        // The weights of tile t, and beside them the scores of tile t + 1 (MORE).
        auto weights = [&](int t, auto more, bf16x8 (&pb)[4]) __attribute__((always_inline)) {
            constexpr bool MORE = decltype(more)::value;
            constexpr int W = KSTEPS > 4 ? KSTEPS - 2 : KSTEPS, PER = (32 + W - 1) / W;
            l_part[0] = l_part[1] = l_part[2] = l_part[3] = 0.f;
            auto weighs = [&](int c) {
#pragma unroll
                for (int i = 0; i < 32; ++i)
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        if (i / PER == c - k) weigh(i, k, pb);
            };
            if constexpr (MORE) scores(t + 1, weighs);
#pragma unroll
            for (int c = MORE ? KSTEPS : 0; c <= 31 / PER + 2; ++c) weighs(c);
            l_run += (l_part[0] + l_part[1]) + (l_part[2] + l_part[3]);
            if constexpr (AHEAD) asm volatile("" : "+v"(l_run));
        };
        auto first_scores = [&](int t) __attribute__((always_inline)) {
            float top = -INFINITY;
            scores(t, [](int) {});
            if constexpr (!BESIDE) all_general(t * kSrTile);
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                if constexpr (BESIDE) modify(i, top);
                else top = fmaxf(top, s[i]);
            }
            settle(t * kSrTile, top);
        };
        // A step: the weights of tile t beside the scores of tile t + 1 (MORE), then the values of tile t.
        auto step = [&](int t, auto more) __attribute__((always_inline)) {
            constexpr bool MORE = decltype(more)::value;
            bf16x8 pb[4];
            weights(t, more, pb);
            float top[2] = {-INFINITY, -INFINITY};
            constexpr int EACH = (32 + VSTEPS - 2) / (VSTEPS - 1);
            values(t, pb, [&](int c) {
                if constexpr (MORE && BESIDE) {
#pragma unroll
                    for (int i = 0; i < 32; ++i)
                        if (i / EACH == c - 1) modify(i, top[i & 1]);
                }
            });
            if constexpr (MORE) {
                if constexpr (!BESIDE) {
                    all_general((t + 1) * kSrTile);
#pragma unroll
                    for (int i = 0; i < 32; ++i) top[i & 1] = fmaxf(top[i & 1], s[i]);
                }
                settle((t + 1) * kSrTile, fmaxf(top[0], top[1]));
            }
        };

        int t = t_begin;
        auto arrived = [&] {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        };
        auto queries = [&] {                              // (the compiler would wait for them, and for tiles with them, in the loop)
#pragma unroll
            for (int c = 0; c < 2 * D32; ++c) asm volatile("" : "+v"(qf[c]));
        };
        if constexpr (!AHEAD) {
            int entry = 0;                                // block-table entry of the tile staged next, fetched a tile ahead
            auto stage = [&](int t) {
                const int64_t row = row_here(entry);
                if (t + 1 < nt) entry = entry_here();
                stage_k(t, row);
                stage_v(t, row);
            };
            if (t < nt) {
                entry = entry_here();
                stage(t);
            }
            queries();
            auto head = [&] {                             // past it tile t is there, tile t - 1 is done with
                arrived();
                if (t + 1 < nt) stage(t + 1);
            };
            for (; t < w_end; ++t) {
                bf16x8 pb[4];
                head();
                first_scores(t);
                weights(t, std::false_type{}, pb);
                values(t, pb, [](int) {});
            }
            for (; t < nt; ++t) head();                   // (loads for the waves that have more tiles)
        } else {
            int entry = 0;                                // block-table entry of the K tile staged next, fetched a step ahead
            int64_t row = 0;                              // first cache row of the V tile staged next
            if (t < nt) {
                const int e0 = entry_here();
                const int64_t row0 = row_here(e0);
                const int e1 = entry_here();
                stage_k(t, row0);
                stage_v(t, row0);
                if (t + 1 < nt) {
                    row = row_here(e1);
                    entry = entry_here();
                    stage_k(t + 1, row);
                }
            }
            auto head = [&] {                             // past it tile t's V and tile t + 1's K are there, their predecessors are done with
                arrived();
                const int64_t v_from = row;
                if (t + 2 < nt) {
                    row = row_here(entry);
                    entry = entry_here();
                }
                if (t + 1 < nt) stage_v(t + 1, v_from);
                if (t + 2 < nt) stage_k(t + 2, row);
            };
            if (t + 1 < nt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D32 + V32) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            queries();
            __syncthreads();
            if (t < w_end) first_scores(t);
            for (; t + 1 < w_end; ++t) {
                head();
                step(t, std::true_type{});
            }
            if (t < w_end) {
                head();
                step(t, std::false_type{});
                ++t;
            }
            for (; t < nt; ++t) head();                   // (loads for the waves that have more tiles)
        }
    } else {
        auto stage = [&](auto buf_tag, int t, int entry) {
            constexpr int AT = decltype(buf_tag)::value * BUF;
            const int phys = min(max(__builtin_amdgcn_readfirstlane(entry), 0), p.max_block);
            const int64_t row0 = ((int64_t)phys * p.block_size + (t % tpb) * kSrTile) * p.G + g;
            const char* kb = (const char*)p.k_cache + row0 * (64 * D32);
            const char* vb = (const char*)p.v_cache + row0 * (p.v_ld * 2);
            const int last = n_k - 1 - t * kSrTile;       // (rows past the sequence re-read the last one: finite, and hidden by the mask)
#pragma unroll
            for (int i = 0; i < D32; ++i) {
                const uint32_t o = dk_off[i] - (uint32_t)max(dk_row[i] - last, 0) * k_row;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(kb + o),
                                                 (__attribute__((address_space(3))) void*)(lds + AT + (wave + 4 * i) * 1024), 16, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < V32; ++i) {
                const uint32_t o = dv_off[i] - (uint32_t)max(dv_row[i] - last, 0) * v_row;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vb + o),
                                                 (__attribute__((address_space(3))) void*)(lds + AT + KB + (wave + 4 * i) * 1024), 16, 0, 0);
            }
        };
        auto entry_of = [&](int t) { return bt[min(t / tpb, p.max_blocks - 1)]; };
        int entry = 0;                                    // block-table entry of the tile staged next, fetched a tile ahead
        if (t_begin < nt) stage(std::integral_constant<int, 0>{}, t_begin, entry_of(t_begin));
        if (t_begin + 1 < nt) entry = entry_of(t_begin + 1);

        auto tile_step = [&](auto buf_tag, int t) {
            constexpr int B = decltype(buf_tag)::value;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this tile has landed, and everybody is done with the other buffer
            __syncthreads();
            const int use = entry;
            if (t + 2 < nt) entry = entry_of(t + 2);
            if (t + 1 < nt) stage(std::integral_constant<int, 1 - B>{}, t + 1, use);
            const unsigned char* ldsK = lds + B * BUF;
            const unsigned char* ldsV = ldsK + KB;
            const int kt = t * kSrTile;
            if (!(wave_live && kt <= wave_last)) return;
            f32x16 s[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
                for (int c = 0; c < 2 * D32; ++c)
                    s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(ldsK + sr_off<D32>(kb * 32 + r, 2 * c + hh)), qf[c], s[kb], 0, 0, 0);
            }
            // register i of block kb is key kt + 32 kb + (i & 3) + 8 (i >> 2) + 4 hh; row rw0 + r
            const bool edge = kt + kSrTile - 1 > rw0 + shift;     // some row of the wave does not see all of the tile
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float x = s[kb][i];
                    if (MOD == kSrCap || (MOD == kSrGeneral && p.softcap > 0.f))
                        x = capped(x);
                    else
                        x *= p.scale_log2;
                    if constexpr (MOD == kSrGeneral) {
                        const int j = kt + kb * 32 + (i & 3) + 8 * (i >> 2) + 4 * hh;
                        x += kSrLog2e * bias[min(max(qpos - j, 0), p.n_dist - 1)];
                    }
                    s[kb][i] = x;
                }
            if (edge) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[kb][i] = kt + kb * 32 + (i & 3) + 8 * (i >> 2) + 4 * hh <= qpos ? s[kb][i] : -INFINITY;
            }
            float tmax = s[0][0];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[kb][i]);
            tmax = sr_max_xor32(tmax);
            if (!__all(tmax <= m_run)) {   // rare after the first tiles
                const float m_new = fmaxf(m_run, tmax), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < V32; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) oacc[d][i] *= alpha;
            }
            float l_part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[kb][i] = __builtin_amdgcn_exp2f(s[kb][i] - m_run);
                    l_part[i & 3] += s[kb][i];
                }
            l_run += (l_part[0] + l_part[1]) + (l_part[2] + l_part[3]);
#pragma unroll
            for (int c = 0; c < 4; ++c) {                 // 16 keys each
                const int kb = c >> 1, s2 = c & 1;
                bf16x8 pb;
#pragma unroll
                for (int j = 0; j < 8; ++j) pb[j] = (__bf16)s[kb][8 * s2 + j];
                const int row1 = kb * 32 + 16 * s2 + 4 * hh + (i16 >> 2), row2 = row1 + 8;
#pragma unroll
                for (int d = 0; d < V32; ++d) {
                    const int ch = d * 4 + 2 * g16 + ((i16 & 3) >> 1), sub = 8 * (i16 & 1);
                    const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((sr_lds_s16x4*)(ldsV + sr_off<V32>(row1, ch) + sub));
                    const s16x4 v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((sr_lds_s16x4*)(ldsV + sr_off<V32>(row2, ch) + sub));
                    const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v1, v2, 0, 1, 2, 3, 4, 5, 6, 7));
                    oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pb, oacc[d], 0, 0, 0);
                }
            }
        };
        for (int t = t_begin; t < nt; t += 2) {
            tile_step(std::integral_constant<int, 0>{}, t);
            if (t + 1 < nt) tile_step(std::integral_constant<int, 1>{}, t + 1);
        }
    }

    // (the lane's number anew: kept over the loop it would cost it registers)
    const int lane_out = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), r_out = lane_out & 31, hh_out = lane_out >> 5;
    float l = sr_sum_xor32(l_run);
    __syncthreads();                                  // every wave is done with the tiles
    if (!wave_live) return;
    unsigned char* stg = lds + wave * (32 * STG);
    const int rows_here = min(32, n_q - rw0);
    // lane (r, hh): row rw0 + r_out, columns 32 d + 8 (i >> 2) + 4 hh_out + (i & 3)
    if (p.nsplit > 1) {                               // the state of this key range; an empty one leaves l = 0
        constexpr int PS = 32 * V32 + 2;
        float* dst = p.part + (((int64_t)(q_begin + rw0 + r_out) * p.H + hq) * p.nsplit + split) * PS;
        if (r_out < rows_here) {
            if (hh_out == 0) {
                dst[32 * V32] = m_run;
                dst[32 * V32 + 1] = l;
            }
            if (t_begin < nt) {
#pragma unroll
                for (int d = 0; d < V32; ++d)
#pragma unroll
                    for (int i = 0; i < 16; i += 2)
                        *(float2*)(dst + 32 * d + 8 * (i >> 2) + 4 * hh_out + (i & 3)) = make_float2(oacc[d][i], oacc[d][i + 1]);
            }
        }
        return;
    }
    if (p.sink != nullptr) {
        const float sk = p.sink[hq] * kSrLog2e, m2 = fmaxf(m_run, sk), f = __builtin_amdgcn_exp2f(m_run - m2);
        l = l * f + __builtin_amdgcn_exp2f(sk - m2);
        l = f > 0.f ? l / f : INFINITY;               // (accumulators stay relative to m_run)
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int d = 0; d < V32; ++d)
#pragma unroll
        for (int i = 0; i < 16; i += 4)
            *(uint2*)(stg + r_out * STG + (32 * d + 2 * i + 4 * hh_out) * 2) =
                make_uint2(pack_bf16(oacc[d][i] * inv, oacc[d][i + 1] * inv), pack_bf16(oacc[d][i + 2] * inv, oacc[d][i + 3] * inv));
    constexpr int LPR = 4 * V32, RPI = 64 / LPR;      // lanes a row (16 bytes each), rows an instruction
    unsigned char* out = (unsigned char*)(p.out + (int64_t)(q_begin + rw0) * p.out_stride + (int64_t)hq * (32 * V32));
#pragma unroll
    for (int it = 0; it < (32 + RPI - 1) / RPI; ++it) {
        const int rr = RPI * it + lane_out / LPR, c = lane_out % LPR;
        if (lane_out < RPI * LPR && rr < rows_here) *(uint4*)(out + rr * p.out_stride * 2 + c * 16) = *(const uint4*)(stg + rr * STG + c * 16);
    }
}

// Joins the key ranges of a row: a wave per (row, head).
__global__ __launch_bounds__(256) void scoremod_rows_merge_kernel(const ScoremodRowsParams p, const int Dv) {
    const int b = blockIdx.y, idx = blockIdx.x * 4 + (threadIdx.x >> 6), row = idx / p.H, hq = idx - row * p.H, lane = threadIdx.x & 63;
    const int q_begin = p.cu_q[b], n_q = p.cu_q[b + 1] - q_begin;
    if (n_q <= 1 || row >= n_q) return;
    const int ps = Dv + 2;
    const float* base = p.part + ((int64_t)(q_begin + row) * p.H + hq) * p.nsplit * ps;
    float mm = p.sink != nullptr ? p.sink[hq] * kSrLog2e : kSrInit;
    for (int s = 0; s < p.nsplit; ++s)
        if (base[s * ps + Dv + 1] != 0.f) mm = fmaxf(mm, base[s * ps + Dv]);
    float den = p.sink != nullptr ? __builtin_amdgcn_exp2f(p.sink[hq] * kSrLog2e - mm) : 0.f;
    float o[2] = {0.f, 0.f};                          // columns lane, lane + 64
    for (int s = 0; s < p.nsplit; ++s) {
        const float l = base[s * ps + Dv + 1];
        if (l == 0.f) continue;                       // an empty range (not one whose sum is not a number: it counts)
        const float f = __builtin_amdgcn_exp2f(base[s * ps + Dv] - mm);
        den += f * l;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (lane + 64 * i < Dv) o[i] += f * base[s * ps + lane + 64 * i];
    }
    const float inv = den > 0.f ? 1.0f / den : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (lane + 64 * i < Dv) p.out[(int64_t)(q_begin + row) * p.out_stride + (int64_t)hq * Dv + lane + 64 * i] = (__bf16)(o[i] * inv);
}

bool scoremod_rows_built(int D, int Dv, int block_size) {
    return (D == 64 || D == 128) && (Dv == 64 || Dv == 128) && block_size > 0 && block_size % kSrTile == 0;
}

ScoremodRowsPlan scoremod_rows_plan(int num_seqs, int64_t T, int H, int G, int Dv, int max_seqlen_q, int max_seqlen_k) {
    ScoremodRowsPlan f{};
    const int rep = H / G;
    f.hpw = rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1;
    const int rows = 32 * (4 / f.hpw);
    f.n_qtiles = (max_seqlen_q + rows - 1) / rows;
    f.wg_per_pair = (rep / f.hpw) * f.n_qtiles;
    f.n_pairs = num_seqs * G;
    while (f.xs_shift < 3 && f.n_pairs <= (8 >> (f.xs_shift + 1))) ++f.xs_shift;       // few pairs: each over several XCDs
    f.slots_per_pair = (f.wg_per_pair + (1 << f.xs_shift) - 1) >> f.xs_shift;
    const int per_round = 8 >> f.xs_shift;
    f.grid_base = (int64_t)((f.n_pairs + per_round - 1) / per_round) * f.slots_per_pair * 8;
    // Key ranges so that a launch has about two workgroups per CU, at least 8 tiles each.  The sequences that count are the long
    // ones: T rows make at most that many portions of the longest one's length.
    const int64_t portions = std::max<int64_t>(1, std::min<int64_t>(num_seqs, (T + max_seqlen_q - 1) / max_seqlen_q));
    const int64_t groups = portions * G * f.wg_per_pair;
    const int tiles = (max_seqlen_k + kSrTile - 1) / kSrTile;
    f.nsplit = 1;
    if (max_seqlen_k > 0 && groups < 512) f.nsplit = (int)std::max<int64_t>(1, std::min<int64_t>((512 + groups - 1) / groups, tiles / 8));
    f.tiles_per_split = f.nsplit > 1 ? (tiles + f.nsplit - 1) / f.nsplit : 1 << 24;
    f.ws_bytes = f.nsplit > 1 ? T * H * f.nsplit * (int64_t)(Dv + 2) * 4 : 0;
    return f;
}

template <int D32, int V32, bool LONG>
static void rows_by_mod(const ScoremodRowsParams& p, hipStream_t s) {
    const dim3 grid((unsigned)(p.grid_base * p.nsplit));
    if (p.dist_bias != nullptr) hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrGeneral, LONG>), grid, dim3(256), 0, s, p);
    else if (p.softcap > 0.f) hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrCap, LONG>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrPlain, LONG>), grid, dim3(256), 0, s, p);
}

int launch_scoremod_rows(ScoremodRowsParams p, const ScoremodRowsPlan& f, int D, int Dv, int num_seqs, int64_t total_q, int max_seqlen_q, int max_seqlen_k, float scale,
                         hipStream_t s) {
    p.hpw = f.hpw;
    p.n_qtiles = f.n_qtiles;
    p.wg_per_pair = f.wg_per_pair;
    p.n_pairs = f.n_pairs;
    p.xs_shift = f.xs_shift;
    p.slots_per_pair = f.slots_per_pair;
    p.sets = scoremod_sets((int)(f.grid_base / (8 * (int64_t)f.slots_per_pair)));
    p.even = scoremod_pairs(f.grid_base, num_seqs, total_q, max_seqlen_q, max_seqlen_k);
    p.there_and_back = f.grid_base * f.nsplit <= 256 * (D + Dv == 128 ? 4 : D + Dv == 192 ? 3 : 2);       // (workgroups that a CU holds)
    p.grid_base = (int)f.grid_base;
    p.nsplit = f.nsplit;
    p.tiles_per_split = f.tiles_per_split;
    p.scale_log2 = scale * kSrLog2e;
    p.cap_in = p.softcap > 0.f ? 2.f * kSrLog2e * scale / p.softcap : 0.f;
    const auto launch = [&](auto tag) {
        constexpr bool LONG = decltype(tag)::value;
        if (D == 64) Dv == 64 ? rows_by_mod<2, 2, LONG>(p, s) : rows_by_mod<2, 4, LONG>(p, s);
        else Dv == 64 ? rows_by_mod<4, 2, LONG>(p, s) : rows_by_mod<4, 4, LONG>(p, s);
    };
    if (scoremod_long(max_seqlen_k, p.dist_bias != nullptr)) launch(std::true_type{});
    else launch(std::false_type{});
    int rc = check_launch("nv_attn_scoremod_paged (rows)");
    if (rc != NV_OK || f.nsplit == 1) return rc;
    const dim3 grid((unsigned)(((int64_t)max_seqlen_q * p.H + 3) / 4), (unsigned)num_seqs);
    hipLaunchKernelGGL(scoremod_rows_merge_kernel, grid, dim3(256), 0, s, p, Dv);
    return check_launch("nv_attn_scoremod_paged (rows, merge)");
}

}  // namespace nv
