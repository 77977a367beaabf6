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
// What bounds it: waiting.  A key tile takes 2.1 us by itself and 3.2 beside the CU's other workgroup, where 64 soft-capped scores cost a SIMD about 70
// cycles (two exponentials and a reciprocal at quarter rate with what is around them) beside 32 of matrix products, and fewer vector
// instructions do not help: 3 us more with a polynomial in place of the cap's exponential and reciprocal.  The compiler cannot tell a transposed
// read from the LDS-DMA in flight and puts a wait for all vector memory in front of the first one of every tile, so for the next
// tile, whose loads start at the head of the same step; and the products of the first key block each wait for the two reads just before them.
// 4 prompts of 1777 .. 2048 tokens, 16 / 8 heads of 128, soft cap and sink, the call with its preparation of 21 us: 117 us (127 with an XCD's pairs
// one after the other, see there; 129 with the denominator as a product of rounded weights with ones); with the launch on 16 x 16
// tiles, values transposed through registers, which other sizes still take, 496 us (44 of them preparation).
#include <algorithm>
#include <type_traits>

#include "attn_scoremod_rows.h"

namespace nv {

constexpr int kSrTile = 64;
constexpr float kSrLog2e = 1.4426950408889634f;
constexpr float kSrInit = -1.0e30f;

typedef __attribute__((ext_vector_type(8))) short sr_s16x8;
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

template <int D32, int V32, int MOD>
__global__ __launch_bounds__(256, 2) void scoremod_rows_kernel(const ScoremodRowsParams p) {
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
    // 16 / 4 heads of 64, 16 chunks of 300 rows on 600 .. 4000 keys 121 us, together 145, 6 prompts of 300 .. 1300 50 and 57, 6 of 466 .. 862 50 and 37.
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
    const int i16 = lane & 15, g16 = (lane >> 4) & 1;
    const int qpos = rw0 + r + shift;                 // last key this lane's row sees
    const int wave_last = min(rw0 + 31, n_q - 1) + shift;
    int entry = 0;                                    // block-table entry of the tile staged next, fetched a tile ahead
    if (t_begin < nt) stage(std::integral_constant<int, 0>{}, t_begin, bt[t_begin / tpb]);
    if (t_begin + 1 < nt) entry = bt[(t_begin + 1) / tpb];

    auto tile_step = [&](auto buf_tag, int t) {
        constexpr int B = decltype(buf_tag)::value;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this tile has landed, and everybody is done with the other buffer
        __syncthreads();
        const int use = entry;
        if (t + 2 < nt) entry = bt[(t + 2) / tpb];
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
                if (MOD == kSrCap || (MOD == kSrGeneral && p.softcap > 0.f))       // cap tanh(s / cap) = cap - 2 cap / (exp(2 s / cap) + 1)
                    x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * p.cap_in) + 1.0f);
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
                sr_s16x8 va;
                va[0] = v1[0]; va[1] = v1[1]; va[2] = v1[2]; va[3] = v1[3];
                va[4] = v2[0]; va[5] = v2[1]; va[6] = v2[2]; va[7] = v2[3];
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va), pb, oacc[d], 0, 0, 0);
            }
        }
    };
    for (int t = t_begin; t < nt; t += 2) {
        tile_step(std::integral_constant<int, 0>{}, t);
        if (t + 1 < nt) tile_step(std::integral_constant<int, 1>{}, t + 1);
    }

    float l = sr_sum_xor32(l_run);
    __syncthreads();                                  // every wave is done with the tiles
    if (!wave_live) return;
    unsigned char* stg = lds + wave * (32 * STG);
    const int rows_here = min(32, n_q - rw0);
    // lane (r, hh): row rw0 + r, columns 32 d + 8 (i >> 2) + 4 hh + (i & 3)
    if (p.nsplit > 1) {                               // the state of this key range; an empty one leaves l = 0
        constexpr int PS = 32 * V32 + 2;
        float* dst = p.part + (((int64_t)(q_begin + rw0 + r) * p.H + hq) * p.nsplit + split) * PS;
        if (r < rows_here) {
            if (hh == 0) {
                dst[32 * V32] = m_run;
                dst[32 * V32 + 1] = l;
            }
            if (t_begin < nt) {
#pragma unroll
                for (int d = 0; d < V32; ++d)
#pragma unroll
                    for (int i = 0; i < 16; i += 2)
                        *(float2*)(dst + 32 * d + 8 * (i >> 2) + 4 * hh + (i & 3)) = make_float2(oacc[d][i], oacc[d][i + 1]);
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
            *(uint2*)(stg + r * STG + (32 * d + 2 * i + 4 * hh) * 2) =
                make_uint2(pack_bf16(oacc[d][i] * inv, oacc[d][i + 1] * inv), pack_bf16(oacc[d][i + 2] * inv, oacc[d][i + 3] * inv));
    constexpr int LPR = 4 * V32, RPI = 64 / LPR;      // lanes a row (16 bytes each), rows an instruction
    unsigned char* out = (unsigned char*)(p.out + (int64_t)(q_begin + rw0) * p.out_stride + (int64_t)hq * (32 * V32));
#pragma unroll
    for (int it = 0; it < (32 + RPI - 1) / RPI; ++it) {
        const int rr = RPI * it + lane / LPR, c = lane % LPR;
        if (lane < RPI * LPR && rr < rows_here) *(uint4*)(out + rr * p.out_stride * 2 + c * 16) = *(const uint4*)(stg + rr * STG + c * 16);
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

template <int D32, int V32>
static void rows_by_mod(const ScoremodRowsParams& p, hipStream_t s) {
    const dim3 grid((unsigned)(p.grid_base * p.nsplit));
    if (p.dist_bias != nullptr) hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrGeneral>), grid, dim3(256), 0, s, p);
    else if (p.softcap > 0.f) hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrCap>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((scoremod_rows_kernel<D32, V32, kSrPlain>), grid, dim3(256), 0, s, p);
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
    if (D == 64) Dv == 64 ? rows_by_mod<2, 2>(p, s) : rows_by_mod<2, 4>(p, s);
    else Dv == 64 ? rows_by_mod<4, 2>(p, s) : rows_by_mod<4, 4>(p, s);
    int rc = check_launch("nv_attn_scoremod_paged (rows)");
    if (rc != NV_OK || f.nsplit == 1) return rc;
    const dim3 grid((unsigned)(((int64_t)max_seqlen_q * p.H + 3) / 4), (unsigned)num_seqs);
    hipLaunchKernelGGL(scoremod_rows_merge_kernel, grid, dim3(256), 0, s, p, Dv);
    return check_launch("nv_attn_scoremod_paged (rows, merge)");
}

}  // namespace nv
