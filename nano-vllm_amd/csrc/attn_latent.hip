// Paged attention in latent space on the matrix cores: every query head of a sequence attends to ONE cached row per token
// whose first Dv columns are also the token's value (bf16, causal, fp32 softmax, an optional learned sink per head that
// joins the denominator only).
//
// With one key row for all heads the queries of a sequence are simply the rows (token, head) of a matrix
// [len_q * H, D], in the order the projection leaves them.  Both kernels work on wave tiles of 32 such rows:
//     S^T (keys x rows) = C Q^T       v_mfma_f32_32x32x16_bf16: A = cached rows from LDS, B = Q^T held in registers
//     O^T (Dv x rows)  += C^T P^T     A = the SAME rows of LDS read transposed (ds_read_b64_tr_b16), B = P^T straight from the
//                                     S^T accumulators
// so a cached row is fetched once, by LDS-DMA, and serves as key and value.  A lane holds half the scores of one row: the
// running maximum is per lane pair and raised only when a score exceeds it by 2^8, so the accumulators are seldom rescaled.
//
//   rows kernel    sequences with several tokens in the step: a workgroup of four waves takes 128 rows; key tiles of 64
//                  (32 for wide rows) are staged once for the four waves by loads that the compiler does not know (it would wait for all of
//                  them in front of a tile's first transposed read).  Where a wave has a SIMD to itself (rows beyond 160 columns, but for 192 with
//                  values of 128) it multiplies the next tile's scores beside the weights of this one, with operands four and eight products ahead, the
//                  accumulators held in their half of the registers, so that no tile moves them: 26 % fewer cycles, matrix cores busy in 55 % of
//                  them instead of 40, at 1.70 GHz instead of 1.84 (power).  16 heads, 256 columns, 1024 rows of each of 2 sequences of 3000 and 6001 keys: the call 160 -> 139 us; a prompt
//                  of 2000 tokens 71 -> 62, 37 rows on 3000 keys 34 -> 29.  One wave a SIMD for rows of 160 columns too: 54 us instead of 58 for a
//                  prompt of 2000, but 66 for 59 where 700 rows come on top of up to 2300 keys.
//                  Elsewhere two to four waves take turns, a tile's work one after the other, operands of the first product two ahead.  With the next
//                  scores beside, rows of 32, 64 and 96 columns lost a wave a SIMD or two: 4 prompts of 1900 .. 2048, rows of 64, 44.3 us before, 47.9
//                  so, 43.4 as it is; rows of 96 57.8, 60.6 and 54.2.  The second product is in order with operands four ahead for those, and left to
//                  the compiler for wider ones, whose waves are often alone at a launch's end: 3 prompts of 700 .. 1900, rows of 160, 48.3 before, 48.7
//                  in order, 47.1 as it is; the 4 prompts 85.2, 79.7 and 79.8; rows of 64, 3 prompts, 30.3, 29.3 and 30.4.
//   single kernel  sequences with one token: a workgroup takes up to 32 heads; its four waves take the key tiles of 32 in
//                  turn, each staging its own (no barrier in the loop), and join their states through LDS.  Rows up to 192 columns in order with operands
//                  ahead, by loads that the compiler does not know; wider ones, one wave a SIMD, in the compiler's order by loads that it knows (the
//                  addresses of 32 and more pieces a tile do not stay in scalar registers).  In order / in the compiler's, us: 256 sequences of
//                  513 .. 768 keys, rows of 160 25.3 / 26.1, 256 36.1 / 34.1;  32 of 500 .. 4000, 128 heads, rows of 576, 144 / 134.
//
// When a launch would leave most of the chip idle the keys are cut into ranges; the ranges' unnormalised states go through
// a workspace and a second launch.
//
// LDS image of a tile: 8-row x 32-column subtiles of 512 bytes, the 16-byte chunk within a subtile row XOR-ed by bits 2..3
// of the row; conflict-free for the row reads and for the transposed reads.
#include <algorithm>
#include <type_traits>

#include "launch_order.h"
#include "nv_common.h"
#include "../../include/nanovllm_hip_mixers.h"

namespace nv {

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

constexpr float kLatRunInit = -1.0e30f;        // finite initial running maximum (keeps exp2 NaN-free)
constexpr float kLatRaise = 8.0f;              // log2 units: weights stay below 2^8 between raises
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kLatRows = 32;                   // rows of a wave
constexpr int64_t kLatHeader = 64;             // bytes of the workspace in front of the states
constexpr int kLatStageRow = 144;              // bytes per row of the output staging area (128 + 16: spreads the banks)

struct LatentParams {
    const __bf16* q;             // [T, H, D]
    const __bf16* cache;         // [num_blocks, block_size, D]
    __bf16* out;                 // [T, H, Dv]
    float* part;                 // [T * H, nsplit, Dv + 2] when nsplit > 1
    const int *cu_q, *cu_k, *block_tables;
    const float* sink;
    int B, H, max_blocks, block_size, tiles_per_block;
    int64_t num_blocks;
    float scale_log2;
    int Dv, dv_groups;           // value columns, and how many workgroups share them (wide rows: the accumulators of all
                                 // columns beside the queries would not fit the registers)
    int row_tiles;               // rows kernel: 128-row tiles of the longest sequence
    int head_groups;             // single kernel: groups of 32 heads
    int nsplit, tiles_per_split; // rows kernel: the most ranges a row can have, and the fewest tiles of one
    int slots;                   // rows kernel: workgroups that the chip holds at a time; 0: neither the order nor even ranges matter
    int* share;                  // [1]: tiles of a range of the rows kernel, where slots > 0
};

__device__ __forceinline__ float lat_max_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float lat_sum_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// byte offset of 16-byte chunk `ch` of row `row` in the image of a tile whose rows are 32 * D32 columns wide
template <int D32>
__device__ __forceinline__ int lat_off(int row, int ch) {
    return 512 * D32 * (row >> 3) + 512 * (ch >> 2) + 64 * (row & 7) + 16 * ((ch & 3) ^ ((row >> 2) & 3));
}

// One 1-KiB piece of a tile: lane l fills bytes 16 l .. of it.  Which (row, chunk) of the tile that is.
template <int D32>
__device__ __forceinline__ void lat_piece(int piece, int lane, int& row, int& ch) {
    const int sub = 2 * piece + (lane >> 5);
    row = 8 * (sub / D32) + ((lane & 31) >> 2);
    ch = 4 * (sub % D32) + ((lane & 3) ^ ((row >> 2) & 3));
}

// The state of one wave: 32 rows of queries against the keys it is shown.
template <int D32, int DV32, int KB, bool HOLD>
struct LatentWave {
    bf16x8 qf[2 * D32];
    f32x16 oacc[DV32];
    float m_run, l_run;
    uint32_t key_at[2], value_at[2];           // where the lane's operands of a tile at LDS address 0 begin

    __device__ __forceinline__ void init(const __bf16* qrow, int lane, int dv0) {
        const int r = lane & 31, h = lane >> 5, i16 = lane & 15, g16 = (lane >> 4) & 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            key_at[i] = lat_off<D32>(r, 2 * i + h);
            value_at[i] = lat_off<D32>(8 * i + 4 * h + (i16 >> 2), 2 * g16 + ((i16 & 3) >> 1)) + 8 * (i16 & 1) + 512 * dv0;
        }
#pragma unroll
        for (int s = 0; s < 2 * D32; ++s) qf[s] = *(const bf16x8*)(qrow + 16 * s + 8 * h);
#pragma unroll
        for (int d = 0; d < DV32; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) oacc[d][i] = 0.f;
        m_run = kLatRunInit;
        l_run = 0.f;
    }

    // Rows kernel with several waves a SIMD, rows of 128 columns and more: the weights and the second product in the compiler's order (see the header).
    static constexpr bool FREE = !HOLD && KB == 2 && D32 >= 4;
    static constexpr int KSTEPS = 2 * D32, VSTEPS = 2 * KB * DV32;                      // products a key block and tile
    static constexpr int AHEAD = HOLD ? 4 : 2, KA = KSTEPS < AHEAD ? KSTEPS : AHEAD, VA = VSTEPS < 2 * AHEAD ? VSTEPS : 2 * AHEAD;
    typedef bf16x8 Keys[KA][KB];
    typedef bf16x8 Values[VA];
    // The lane's way through a tile; operands lie at constant distances from it.
    struct Tile {
        const lds_byte *key[2], *value[2];
    };
    __device__ __forceinline__ Tile tile(uint32_t at) const {
        return {{lds_pointer(key_at[0] + at), lds_pointer(key_at[1] + at)}, {lds_pointer(value_at[0] + at), lds_pointer(value_at[1] + at)}};
    }
    // Operand c of the first product: 32 keys of each block, columns 16 c ...
    __device__ __forceinline__ void keys(const Tile& t, int c, Keys& a) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            a[c % KA][kb] = *(const __attribute__((address_space(3))) bf16x8*)(t.key[c & 1] + 2048 * D32 * kb + 512 * (c >> 1));
    }
    __device__ __forceinline__ void first_keys(const Tile& t, Keys& a) {
#pragma unroll
        for (int c = 0; c < KA; ++c) keys(t, c, a);
    }
    // Scores of a tile's 32 KB keys (register i of block kb is key 32 kb + (i & 3) + 8 (i >> 2) + 4 h of the tile).  The first operands are in
    // `a`, the others come as many products ahead; beside() is what the wave does beside the products of a step.
    template <class F>
    __device__ __forceinline__ void scores(const Tile& t, f32x16 (&s)[KB], Keys& a, F beside) {
        constexpr f32x16 zero = {};
#pragma unroll
        for (int c = 0; c < KSTEPS; ++c) {
            __builtin_amdgcn_sched_barrier(0);                       // (left alone, a product waits for the read just before it)
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c % KA][kb], qf[c], c ? s[kb] : zero, 0, 0, 0);
            if (c + KA < KSTEPS) keys(t, c + KA, a);
            beside(c);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // Weights of the scores, as operands of the second product; their sum goes to `sum`.  Score i in three steps that lie apart beside products.
    typedef float Scores[16 * KB];             // (numbers, not vectors: they would be carried in the accumulators' half of the registers)
    __device__ __forceinline__ void relate(Scores& s, int i, float scale_log2) { s[i] = __builtin_fmaf(s[i], scale_log2, -m_run); }
    __device__ __forceinline__ void power(Scores& s, int i) { s[i] = __builtin_amdgcn_exp2f(s[i]); }
    __device__ __forceinline__ void take(Scores& s, int i, bf16x8 (&p)[2 * KB], float (&sum)[2]) {
        sum[i & 1] += s[i];
        if ((i & 7) == 7) {
#pragma unroll
            for (int j = 0; j < 8; ++j) p[i >> 3][j] = (__bf16)s[i - 7 + j];
            if constexpr (!FREE) asm volatile("" : "+v"(p[i >> 3]));  // (here and not where it is needed)
        }
    }
    // Operand n of the second product: 16 keys (n / DV32) x 32 columns (n % DV32, from 32 dv0 on), transposed on its way.  Keys of element
    // j: 16 (n / DV32) + 8 (j >> 2) + 4 h + (j & 3).
    __device__ __forceinline__ bf16x8 value(const Tile& t, int n) {
        const int off = 1024 * D32 * (n / DV32) + 512 * (n % DV32);
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t.value[0] + off));
        const s16x4 v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t.value[1] + off));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(v1, v2, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    // Adds the tile's values with these weights; the first VA operands are in `a`, the others come as many products ahead.  beside() as in scores().
    template <class F>
    __device__ __forceinline__ void values(const Tile& t, const bf16x8 (&p)[2 * KB], Values& a, F beside) {
#pragma unroll
        for (int n = 0; n < VSTEPS; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            oacc[n % DV32] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[n % VA], p[n / DV32], oacc[n % DV32], 0, 0, 0);
            if (n + VA < VSTEPS) a[n % VA] = value(t, n + VA);
            beside(n);
        }
        __builtin_amdgcn_sched_barrier(0);
        hold();
    }
    __device__ __forceinline__ void values(const Tile& t, const bf16x8 (&p)[2 * KB]) {
        if constexpr (FREE) {
#pragma unroll
            for (int n = 0; n < VSTEPS; ++n) oacc[n % DV32] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(value(t, n), p[n / DV32], oacc[n % DV32], 0, 0, 0);
            return;
        }
        Values a;
#pragma unroll
        for (int n = 0; n < VA; ++n) a[n] = value(t, n);
        values(t, p, a, [](int) {});
    }
    // The lane's row sees keys <= qpos of a tile that starts at key kt.
    __device__ __forceinline__ void mask(Scores& s, int lane, int kt, int qpos) {
        asm volatile("");                                            // (a branch around it, not 32 selections in every tile)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kt + kb * 32 + (i & 3) + 8 * (i >> 2) + 4 * (lane >> 5);
                s[16 * kb + i] = key <= qpos ? s[16 * kb + i] : -INFINITY;
            }
    }
    // Raises the running maximum where a row's largest score (`tmax`, in log2 units) asks for it.
    __device__ __forceinline__ bool high(float tmax) { return !__all(tmax <= m_run + kLatRaise); }       // rare after the first tiles
    __device__ __forceinline__ void raise(float tmax) {
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < DV32; ++d) {                             // (a block at a time: all of them would drive others out of their registers)
            if constexpr (HOLD) asm volatile("" : "+a"(oacc[d]));
#pragma unroll
            for (int i = 0; i < 16; ++i) oacc[d][i] *= alpha;
            if constexpr (HOLD) asm volatile("" : "+a"(oacc[d]));
            else asm volatile("" : "+v"(oacc[d]));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The queries have come (the compiler would wait for them, and with them for the tiles on their way, in front of every product).
    __device__ __forceinline__ void settle() {
#pragma unroll
        for (int s = 0; s < 2 * D32; ++s) {
            if constexpr (HOLD) asm volatile("" : "+a"(qf[s]));
            else asm volatile("" : "+v"(qf[s]));
        }
    }
    // The accumulators stay in the accumulators' half of the registers where the raise joins the way past it.
    __device__ __forceinline__ void hold() {
#pragma unroll
        for (int d = 0; d < DV32; ++d) {
            if constexpr (HOLD) asm volatile("" : "+a"(oacc[d]));
            else asm volatile("" : "+v"(oacc[d]));
        }
    }
    __device__ __forceinline__ float largest(const Scores& s) {
        float top = s[0];
#pragma unroll
        for (int i = 0; i < 16 * KB; ++i) top = fmaxf(top, s[i]);
        return top;
    }
    // A tile by itself, the first of its keys key kt (masked: some row of the wave does not see all of the tile).
    __device__ __forceinline__ void step(uint32_t at, int lane, int kt, int qpos, bool masked, float scale_log2) {
        Scores s;
        first(at, s, lane, kt, qpos, masked, scale_log2);
        last(at, s, scale_log2);
    }
    // The same in the compiler's order, from a tile at `lds` that came by loads which the compiler knows.
    __device__ __forceinline__ void plain_step(const unsigned char* lds, int lane, int kt, int qpos, bool masked, float scale_log2, int dv0) {
        const int r = lane & 31, h = lane >> 5, i16 = lane & 15, g16 = (lane >> 4) & 1;
        f32x16 s[KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
            for (int c = 0; c < KSTEPS; ++c)
                s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(lds + lat_off<D32>(kb * 32 + r, 2 * c + h)), qf[c], s[kb], 0, 0, 0);
        }
        if (masked) {
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) s[kb][i] = kt + kb * 32 + (i & 3) + 8 * (i >> 2) + 4 * h <= qpos ? s[kb][i] : -INFINITY;
        }
        float tmax = s[0][0];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[kb][i]);
        tmax = lat_max_xor32(tmax) * scale_log2;                 // (scale > 0)
        if (high(tmax)) {
            const float m_new = fmaxf(m_run, tmax), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < DV32; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[d][i] *= alpha;
        }
        float psum = 0.f;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[kb][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][i], scale_log2, -m_run));
                psum += s[kb][i];
            }
        l_run += psum;
#pragma unroll
        for (int k = 0; k < 2 * KB; ++k) {
            bf16x8 pb;
#pragma unroll
            for (int j = 0; j < 8; ++j) pb[j] = (__bf16)s[k >> 1][8 * (k & 1) + j];
            const int row = 16 * k + 4 * h + (i16 >> 2);
#pragma unroll
            for (int d = 0; d < DV32; ++d) {
                const unsigned char* at = lds + 512 * dv0 + 8 * (i16 & 1);
                const int ch = d * 4 + 2 * g16 + ((i16 & 3) >> 1);
                const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + lat_off<D32>(row, ch)));
                const s16x4 v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + lat_off<D32>(row + 8, ch)));
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, __builtin_shufflevector(v1, v2, 0, 1, 2, 3, 4, 5, 6, 7)), pb, oacc[d], 0, 0, 0);
            }
        }
    }
    __device__ __forceinline__ void first(uint32_t at, Scores& s, int lane, int kt, int qpos, bool masked, float scale_log2) {
        const Tile t = tile(at);
        Keys a;
        f32x16 n[KB];
        first_keys(t, a);
        scores(t, n, a, [](int) {});
#pragma unroll
        for (int i = 0; i < 16 * KB; ++i) s[i] = n[i >> 4][i & 15];
        if (masked) mask(s, lane, kt, qpos);
        const float tmax = lat_max_xor32(largest(s)) * scale_log2;   // (scale > 0)
        if (high(tmax)) raise(tmax);
        keep(s);
    }
    // The scores stay in the other half from one tile to the next.
    __device__ __forceinline__ void keep(Scores& s) {
#pragma unroll
        for (int i = 0; i < 16 * KB; ++i)
            if constexpr (!FREE) asm volatile("" : "+v"(s[i]));
    }
    // The weights and values of the tile at `now`, whose scores are s, and beside them the scores of the one at `next` (its first key kt), which
    // take their place: the weights beside the products of the scores, the largest of those beside the products of the values.  The first
    // operands of `next` are in `a`, those of the tile behind it are when it returns; half_way() is called between the two, begin() and
    // load(i), where there are loads, beside the products of the values.
    template <int LOADS, class S, class B, class F>
    __device__ __forceinline__ void turn(uint32_t now_at, uint32_t next_at, uint32_t behind_at, Scores& s, Keys& a, int lane, int kt, int qpos,
                                         bool masked, float scale_log2, S half_way, B begin, F load) {
        const Tile now = tile(now_at), next = tile(next_at), behind = tile(behind_at);
        f32x16 n[KB];
        bf16x8 p[2 * KB];
        Values v;
        float sum[2] = {0.f, 0.f};
        constexpr int ALL = 16 * KB, W = KSTEPS > 4 ? KSTEPS - 2 : KSTEPS, PER = (ALL + W - 1) / W;
        auto weigh = [&](int c) {
#pragma unroll
            for (int i = 0; i < ALL; ++i) {
                if (i / PER == c) relate(s, i, scale_log2);
                if (i / PER == c - 1) power(s, i);
                if (i / PER == c - 2) take(s, i, p, sum);
            }
        };
        scores(next, n, a, [&](int c) {
            weigh(c);
#pragma unroll
            for (int i = 0; i < VA; ++i)                             // (its first operands, where no more keys come)
                if (c == (KSTEPS > KA ? KSTEPS - KA + i * KA / VA : KSTEPS - 1)) v[i] = value(now, i);
        });
#pragma unroll
        for (int c = KSTEPS; c <= (ALL - 1) / PER + 2; ++c) weigh(c);
        l_run += sum[0] + sum[1];
        asm volatile("" : "+v"(l_run));                              // (here, not behind the products of the values)
        half_way();
        // The scores are in the accumulators' half of the registers; they move a block at a time, well behind the last product of theirs.
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) asm volatile("" : "+a"(n[kb]));
        constexpr bool LONG = VSTEPS >= 8 * KB;                      // (products enough to do it beside)
        constexpr int MOVE = LONG ? VSTEPS / 8 : 0, MAXES = LONG ? VSTEPS / 2 / KB : 1, EACH = 16 / MAXES + (16 % MAXES != 0);
        constexpr int END = MOVE + (LONG ? MAXES : 0) * KB;
        float top[2] = {-INFINITY, -INFINITY};
        values(now, p, v, [&](int c) {
            if constexpr (LOADS > 0) {
                if (c == 0) begin();
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                    if (c == (VSTEPS > 4 ? 1 : 0) + i * VSTEPS / (2 * LOADS)) load(i);    // (in the first half)
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const int at = c - MOVE - kb * MAXES;
                if (LONG ? at == 0 : c == 0) asm volatile("" : "+v"(n[kb]));
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (LONG ? i / EACH == at : c == 0) top[i & 1] = fmaxf(top[i & 1], n[kb][i]);
            }
            if (LONG && c == END) top[0] = lat_max_xor32(fmaxf(top[0], top[1])) * scale_log2;
            if (c == VSTEPS - 1) first_keys(behind, a);
        });
        if constexpr (!LONG || END >= VSTEPS) top[0] = lat_max_xor32(fmaxf(top[0], top[1])) * scale_log2;
#pragma unroll
        for (int i = 0; i < ALL; ++i) s[i] = n[i >> 4][i & 15];
        if (masked) {
            mask(s, lane, kt, qpos);
            top[0] = lat_max_xor32(largest(s)) * scale_log2;
        }
        if (high(top[0])) raise(top[0]);
        keep(s);
    }
    __device__ __forceinline__ void last(uint32_t at, Scores& s, float scale_log2) {
        bf16x8 p[2 * KB];
        float sum[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 16 * KB; ++i) {
            relate(s, i, scale_log2);
            power(s, i);
            take(s, i, p, sum);
        }
        l_run += sum[0] + sum[1];
        values(tile(at), p);
    }
};

// first byte of the tile that starts at key `kt` (tiles do not straddle blocks; table entries are clamped into the cache)
__device__ __forceinline__ const unsigned char* lat_tile_base(const LatentParams& p, int entry, int off, int row_bytes) {
    const int64_t phys = min(max(entry, 0), (int)p.num_blocks - 1);         // (fewer than 2^31)
    return (const unsigned char*)p.cache + (phys * p.block_size + off) * (int64_t)row_bytes;
}

// 1 / denominator of a finished row, with the sink in it, and the factor of the accumulators
__device__ __forceinline__ float lat_finish(float m, float l, const float* sink, int head) {
    float f = 1.f;
    if (sink != nullptr) {
        const float s2 = sink[head] * kLog2e, m2 = fmaxf(m, s2);
        f = __builtin_amdgcn_exp2f(m - m2);
        l = l * f + __builtin_amdgcn_exp2f(s2 - m2);
    }
    return f / l;
}

// ------------------------------------------------------------------------------------------------ several tokens
// Key tiles of a range: what the step has for every slot, not less than the launch has room for.  All row tiles get a whole range
// first, longest first, and what is left of the long ones goes to the slots whose row tile was short: 16 heads, 256 columns, 1024 rows
// of each of 2 sequences of 3000 and 6001 keys take 63 tiles the longest way, where ranges of half the longest sequence take 94:
// 152 -> 137 us a call; 500 rows of each of 4 sequences of 1000 .. 3000 keys 87 -> 82; with the order of the workgroups alone 16 prompts of 200 .. 512 tokens
// 56 -> 43 (device times, 256 columns; rows of one range write no state).
template <int KT>
__device__ __forceinline__ int lat_share(const LatentParams& p, int lane) {
    int64_t total = 0;
    int least = 0x7fffffff, longest = 0;                     // keys in front of a sequence's rows, keys of a sequence
    for (int b = lane; b < p.B; b += 64) {
        const int n_q = p.cu_q[b + 1] - p.cu_q[b], n_k = p.cu_k[b + 1] - p.cu_k[b];
        if (n_q <= 1) continue;
        const int64_t tiles = ((int64_t)n_q * p.H + 4 * kLatRows - 1) / (4 * kLatRows);
        total += tiles * (n_k - n_q / 2) / KT + tiles;
        least = min(least, n_k - n_q);
        longest = max(longest, n_k);
    }
    for (int o = 32; o > 0; o >>= 1) {
        total += __shfl_xor(total, o);
        least = min(least, __shfl_xor(least, o));
        longest = max(longest, __shfl_xor(longest, o));
    }
    return latent_alike(least, longest) ? p.tiles_per_split : latent_share(total, p.slots, p.tiles_per_split);
}

// EVEN: the launch is more than the chip holds at a time, so the order and the ranges of its workgroups matter.
template <int D32, int DV32, int KB, int OCC, bool EVEN>
__global__ __launch_bounds__(256, OCC) void attn_latent_rows_kernel(const LatentParams p) {
    constexpr int D = 32 * D32, KT = 32 * KB, kTile = KT * D * 2, kPieces = D32 * KB / 2;
    constexpr bool TURN = OCC == 1;                          // the next tile's scores beside this one's weights
    static_assert(D32 * KB % 2 == 0, "a wave stages whole pieces");
    // A tile each; two waves' output staging areas at the end.  Only the wait for the loads and the barrier, half way through a turn or at the head
    // of a step, keep a tile's reads apart from the loads into its buffer.
    constexpr int BUF = kTile > 2 * kLatRows * kLatStageRow ? kTile : 2 * kLatRows * kLatStageRow;
    __shared__ __attribute__((aligned(16))) unsigned char buf[TURN ? 4 : 2][BUF];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = blockIdx.y, dv0 = blockIdx.z * DV32, Dv = p.Dv;
    // The latest (heaviest) tiles first, the sequences in turn.  A workgroup's index gives its XCD (of eight) and there its shader engine
    // (of four, eight CUs each), and it waits for that one, others idle or not.  So a launch of more than one round turns every 32
    // workgroups by another amount, or two sequences would keep to half of the engines each (without key ranges only where they would); with
    // key ranges, which come in rounds of their own, it takes the sequences one after the other.
    const int first = blockIdx.x & ~31, x = EVEN && first + 32 <= (int)gridDim.x ? first + ((blockIdx.x + 13 * (first >> 5)) & 31) : (int)blockIdx.x;
    const bool one_by_one = EVEN && p.nsplit > 1;
    const int b = one_by_one ? x / p.row_tiles : x % p.B, qt = p.row_tiles - 1 - (one_by_one ? x % p.row_tiles : x / p.B);
    const int q_begin = p.cu_q[b], n_q = p.cu_q[b + 1] - q_begin, n_k = p.cu_k[b + 1] - p.cu_k[b];
    const int rows = n_q * p.H, row0 = qt * 4 * kLatRows;
    const int share = EVEN && p.nsplit > 1 ? __builtin_amdgcn_readfirstlane(lat_share<KT>(p, lane)) : p.tiles_per_split;
    if (EVEN && p.nsplit > 1 && blockIdx.x == 0 && split == 0 && blockIdx.z == 0 && tid == 0) *p.share = share;        // (for the merge)
    if (n_q <= 1 || row0 >= rows) return;                    // (single tokens belong to the other kernel)
    const int start = n_k - n_q;
    const int rw0 = row0 + wave * kLatRows;                  // the wave's first row
    const bool wave_live = rw0 < rows;
    const int my_row = min(rw0 + r, rows - 1);
    const int qpos = start + my_row / p.H;
    const int tiles = latent_tiles(start + (min(row0 + 4 * kLatRows, rows) - 1) / p.H, KT, p.nsplit, p.tiles_per_split);
    const int t_begin = split * share, t_end = min(tiles, t_begin + share);
    const int ranges = EVEN ? latent_ranges(tiles, share) : p.nsplit;
    if (split >= ranges) return;
    const int wave_first_pos = start + min(rw0, rows - 1) / p.H, wave_last_pos = start + min(rw0 + kLatRows - 1, rows - 1) / p.H;

    LatentWave<D32, DV32, KB, TURN> w;
    w.init(p.q + ((int64_t)q_begin * p.H + my_row) * D, lane, dv0);

    const int* table = p.block_tables + (int64_t)b * p.max_blocks;
    uint32_t dma_off[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        int row, ch;
        lat_piece<D32>(wave * kPieces + i, lane, row, ch);
        dma_off[i] = (uint32_t)(row * (D * 2) + ch * 16);
    }
    // The tile that is staged next: its number, its place in its block, and the block's entry of the table, fetched a tile ahead (the first
    // ones together: the wait for an entry is one for the tiles in front of it too).  Without branches, so that it goes beside products.
    const int first_block = t_begin / p.tiles_per_block, last_block = max(t_end - 1, 0) / p.tiles_per_block;
    constexpr int EARLY = TURN ? 3 : 2;
    int st = t_begin, st_in = t_begin - first_block * p.tiles_per_block, st_block = first_block, entry[EARLY];
#pragma unroll
    for (int i = 0, in = st_in, at = first_block; i < EARLY; ++i) {
        entry[i] = table[min(at, last_block)];
        const int wrap = ++in == p.tiles_per_block;
        in = wrap ? 0 : in;
        at += wrap;
    }
#pragma unroll
    for (int i = 0; i < EARLY; ++i) entry[i] = __builtin_amdgcn_readfirstlane(entry[i]);
    const unsigned char* st_base = nullptr;
    const uint32_t buf_at = lds_address(buf);
    uint32_t st_to = 0;
    auto stage_from = [&](int to) {
        st_base = lat_tile_base(p, __builtin_amdgcn_readfirstlane(entry[0]), st_in * KT, D * 2);
        st_to = buf_at + to * BUF + wave * kPieces * 1024;
        ++st;
        const int wrap = ++st_in == p.tiles_per_block;
        st_in = wrap ? 0 : st_in;
        st_block += wrap;
    };
    auto next_entry = [&] { entry[0] = table[min(st_block, last_block)]; };       // (in front of the tile's loads: there when the wait for them is over)
    auto stage_piece = [&](int i) { lds_load16(st_base, dma_off[i], st_to + i * 1024); };
    auto stage = [&](int to, auto next) {
        const int last = n_k - 1 - st * KT;                  // rows behind the sequence's end re-read its last row (no tile comes behind that one)
        if (last < KT - 1) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                int row, ch;
                lat_piece<D32>(wave * kPieces + i, lane, row, ch);
                dma_off[i] -= (uint32_t)(max(row - last, 0) * (D * 2));
            }
        }
        stage_from(to);
        next();
#pragma unroll
        for (int i = 0; i < kPieces; ++i) stage_piece(i);
    };
    auto shift = [&] {
#pragma unroll
        for (int i = 1; i < EARLY; ++i) entry[i - 1] = entry[i];
    };
    const int w_end = wave_live ? min(t_end, wave_last_pos / KT + 1) : t_begin;      // behind the wave's last tile
    const int full = wave_first_pos + 1 - KT;                // a tile that starts there at the latest is seen by all rows of the wave
    int t = t_begin, now = 0;
    if constexpr (TURN) {
        // Tile t's values and tile t + 1's scores in a step.  Half way through it tile t + 2 has landed for all and tile t - 1 is done with, so
        // the loads of tile t + 3 go out.
        auto sync = [&] {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        if (t < t_end) stage(0, shift);
        if (t + 1 < t_end) stage(1, shift);
        if (t + 2 < t_end) {
            stage(2, next_entry);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kPieces) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        w.settle();
        __syncthreads();
        typename LatentWave<D32, DV32, KB, TURN>::Scores sc;
        typename LatentWave<D32, DV32, KB, TURN>::Keys keys;
        if (t < w_end) {
            w.first(buf_at, sc, lane, t * KT, qpos, t * KT > full, p.scale_log2);
            w.first_keys(w.tile(buf_at + BUF), keys);
        }
        auto turn = [&](auto more) {
            w.template turn<decltype(more)::value ? kPieces : 0>(
                buf_at + now * BUF, buf_at + ((now + 1) & 3) * BUF, buf_at + ((now + 2) & 3) * BUF, sc, keys, lane, (t + 1) * KT, qpos, (t + 1) * KT > full,
                p.scale_log2,
                [&] {
                    sync();
                    if constexpr (!decltype(more)::value)
                        if (t + 3 < t_end) stage((now + 3) & 3, next_entry);
                },
                [&] {
                    stage_from((now + 3) & 3);
                    next_entry();
                },
                stage_piece);
        };
        const int whole = min(t_end, n_k / KT);              // (a tile that the sequence ends in is staged by itself)
        for (; t + 1 < w_end && t + 3 < whole; ++t, now = (now + 1) & 3) turn(std::true_type{});
        for (; t + 1 < w_end; ++t, now = (now + 1) & 3) turn(std::false_type{});
        if (t < w_end) w.last(buf_at + now * BUF, sc, p.scale_log2);
        for (; t < t_end; ++t, now = (now + 1) & 3) {        // (loads for the waves that have more tiles)
            sync();
            if (t + 3 < t_end) stage((now + 3) & 3, next_entry);
        }
    } else {
        if (t < t_end) stage(0, shift);
        w.settle();
        auto head = [&] {                                    // tile t has landed for all, the other buffer is free
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (t + 1 < t_end) stage(now ^ 1, next_entry);
        };
        for (; t < w_end; ++t, now ^= 1) {
            head();
            w.step(buf_at + now * BUF, lane, t * KT, qpos, t * KT > full, p.scale_log2);
        }
        for (; t < t_end; ++t, now ^= 1) head();
    }
    const float l_tot = lat_sum_xor32(w.l_run);
    __syncthreads();                                         // every wave is done reading tiles
    if (!wave_live) return;
    // Lane (r, h) holds columns 32 d + 8 (i >> 2) + 4 h + (i & 3) of row r: through the wave's staging area to 128-byte row
    // segments.
    unsigned char* stg = buf[wave >> 1] + (wave & 1) * (kLatRows * kLatStageRow);
    const int rows_here = rows - rw0;
    const int64_t grow = (int64_t)q_begin * p.H + rw0;
    if (ranges > 1) {
        float* dst = p.part + (grow * p.nsplit + split) * (Dv + 2);
        const int64_t ld = (int64_t)p.nsplit * (Dv + 2);
        if (dv0 == 0 && h == 0 && r < rows_here) {
            dst[r * ld + Dv] = w.m_run;
            dst[r * ld + Dv + 1] = l_tot;
        }
        if (!EVEN && t_begin >= t_end) return;               // no keys in this range: l = 0 says so
#pragma unroll
        for (int d = 0; d < DV32; ++d) {
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(float4*)(stg + r * kLatStageRow + (8 * g + 4 * h) * 4) =
                    make_float4(w.oacc[d][4 * g], w.oacc[d][4 * g + 1], w.oacc[d][4 * g + 2], w.oacc[d][4 * g + 3]);
#pragma unroll
            for (int it = 0; it < 8; ++it) {                 // (states are 8-byte aligned)
                const int c = it * 64 + lane, rr = c >> 4;
                const float2 v = *(const float2*)(stg + rr * kLatStageRow + (c & 15) * 8);
                if (rr < rows_here) *(float2*)(dst + rr * ld + (dv0 + d) * 32 + (c & 15) * 2) = v;
            }
        }
        return;
    }
    const float inv = lat_finish(w.m_run, l_tot, p.sink, my_row % p.H);
    __bf16* dst = p.out + grow * Dv + dv0 * 32;
#pragma unroll
    for (int d0 = 0; d0 < DV32; d0 += 2) {
        constexpr int kMax = 2;
        const int nd = d0 + kMax <= DV32 ? kMax : 1;
#pragma unroll
        for (int dd = 0; dd < kMax; ++dd) {
            if (d0 + dd >= DV32) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x16& o = w.oacc[d0 + dd < DV32 ? d0 + dd : 0];
                *(uint2*)(stg + r * kLatStageRow + (dd * 32 + 8 * g + 4 * h) * 2) =
                    make_uint2(pack_bf16(o[4 * g] * inv, o[4 * g + 1] * inv), pack_bf16(o[4 * g + 2] * inv, o[4 * g + 3] * inv));
            }
        }
        const int per = 4 * nd;                              // 16-byte pieces per row
        for (int c = lane; c < kLatRows * per; c += 64) {
            const int rr = c / per, pc = c % per;
            const uint4 v = *(const uint4*)(stg + rr * kLatStageRow + pc * 16);
            if (rr < rows_here) *(uint4*)(dst + (int64_t)rr * Dv + d0 * 32 + pc * 8) = v;
        }
    }
}

// ------------------------------------------------------------------------------------------------ one token
template <int D32, int DV32, int NBUF, int OCC>
__global__ __launch_bounds__(256, OCC) void attn_latent_single_kernel(const LatentParams p) {
    constexpr int D = 32 * D32, Dw = 32 * DV32, KT = 32, kTile = KT * D * 2, kPieces = 2 * D32;
    constexpr bool PLAIN = OCC == 1;                         // (see the header)
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // [4 waves][NBUF tiles], then [4][32] (m, l)
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x, hg = blockIdx.z / p.dv_groups, split = blockIdx.y, Dv = p.Dv;
    const int dv0 = (blockIdx.z % p.dv_groups) * DV32;
    const int t0 = p.cu_q[b];
    if (p.cu_q[b + 1] - t0 != 1) return;                     // longer portions belong to the other kernel
    const int n_k = p.cu_k[b + 1] - p.cu_k[b];
    const int head0 = hg * kLatRows, heads = min(kLatRows, p.H - head0);
    const int t_begin = split * p.tiles_per_split, t_end = min((n_k + KT - 1) / KT, t_begin + p.tiles_per_split);

    const int* table = p.block_tables + (int64_t)b * p.max_blocks;
    unsigned char* mine = lds + wave * (NBUF * kTile);
    int row0, ch0;                                           // piece i is piece 0 shifted by 2 i subtiles
    lat_piece<D32>(0, lane, row0, ch0);
    auto stage = [&](int buf, int t) {
        const int entry = __builtin_amdgcn_readfirstlane(table[t / p.tiles_per_block]);
        const unsigned char* base = lat_tile_base(p, entry, (t % p.tiles_per_block) * KT, D * 2);
        const int last = n_k - 1 - t * KT;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            int row, ch;
            lat_piece<D32>(i, lane, row, ch);
            const uint32_t off = (uint32_t)(min(row, last) * (D * 2) + ch * 16);
            unsigned char* to = mine + buf * kTile + i * 1024;
            if constexpr (PLAIN)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off), (__attribute__((address_space(3))) void*)to, 16, 0, 0);
            else
                lds_load16(base, off, lds_address(to));
        }
    };
    LatentWave<D32, DV32, 1, false> w;
    int t = t_begin + wave, buf = 0;
    if (t < t_end) stage(0, t);
    w.init(p.q + ((int64_t)t0 * p.H + head0 + min(r, heads - 1)) * D, lane, dv0);
    for (; t < t_end; t += 4) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this wave's own tile has landed
        if (NBUF == 2 && t + 4 < t_end) stage(buf ^ 1, t + 4);
        if constexpr (PLAIN) w.plain_step(mine + buf * kTile, lane, t * KT, n_k - 1, t * KT + KT > n_k, p.scale_log2, dv0);
        else w.step(lds_address(mine + buf * kTile), lane, t * KT, n_k - 1, t * KT + KT > n_k, p.scale_log2);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // its reads are done before the buffer is filled again
        if (NBUF == 1 && t + 4 < t_end) stage(0, t + 4);
        if (NBUF == 2) buf ^= 1;
    }
    // ---- join the four waves: maxima and denominators, then the accumulators, 16 rows at a time through the tile areas ----
    const float l_tot = lat_sum_xor32(w.l_run);
    float* ml = (float*)(lds + 4 * NBUF * kTile);
    if (h == 0) {
        ml[(wave * kLatRows + r) * 2] = w.m_run;
        ml[(wave * kLatRows + r) * 2 + 1] = l_tot;
    }
    __syncthreads();
    float m_all = kLatRunInit;
#pragma unroll
    for (int i = 0; i < 4; ++i) m_all = fmaxf(m_all, ml[(i * kLatRows + r) * 2]);
    const float f = __builtin_amdgcn_exp2f(w.m_run - m_all);
    float* accs = (float*)lds;                               // [4 waves][16 rows][Dw]: at most the tile areas (Dw <= D)
    constexpr int kArea = NBUF * kTile / 4;                  // floats from one wave's area to the next
    static_assert(16 * Dw * 4 <= NBUF * kTile, "the join area fits a wave's tiles");
    for (int half = 0; half < 2 && half * 16 < heads; ++half) {
        __syncthreads();
        if ((r >> 4) == half) {
#pragma unroll
            for (int d = 0; d < DV32; ++d)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *(float4*)(accs + wave * kArea + (r & 15) * Dw + d * 32 + 8 * g + 4 * h) =
                        make_float4(w.oacc[d][4 * g] * f, w.oacc[d][4 * g + 1] * f, w.oacc[d][4 * g + 2] * f, w.oacc[d][4 * g + 3] * f);
        }
        __syncthreads();
        const int n_rows = min(16, heads - half * 16);
        for (int i = tid; i < n_rows * (Dw / 4); i += 256) {
            const int row = i / (Dw / 4), c = (i % (Dw / 4)) * 4, hr = half * 16 + row;
            float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const float4 a = *(const float4*)(accs + x * kArea + row * Dw + c);
                s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
            }
            float m = kLatRunInit, l = 0.f;
#pragma unroll
            for (int x = 0; x < 4; ++x) m = fmaxf(m, ml[(x * kLatRows + hr) * 2]);
#pragma unroll
            for (int x = 0; x < 4; ++x) l += ml[(x * kLatRows + hr) * 2 + 1] * __builtin_amdgcn_exp2f(ml[(x * kLatRows + hr) * 2] - m);
            const int64_t grow = (int64_t)t0 * p.H + head0 + hr;
            if (p.nsplit > 1) {
                float* dst = p.part + (grow * p.nsplit + split) * (Dv + 2);
                *(float2*)(dst + dv0 * 32 + c) = make_float2(s.x, s.y);
                *(float2*)(dst + dv0 * 32 + c + 2) = make_float2(s.z, s.w);
                if (dv0 == 0 && c == 0) {
                    dst[Dv] = m;
                    dst[Dv + 1] = l;
                }
            } else {
                const float inv = lat_finish(m, l, p.sink, head0 + hr);
                *(uint2*)(p.out + grow * Dv + dv0 * 32 + c) = make_uint2(pack_bf16(s.x * inv, s.y * inv), pack_bf16(s.z * inv, s.w * inv));
            }
        }
    }
}

// Joins the key ranges of a row (token, head): one wave per row.  only: 1 = rows of single-token sequences, 2 = the others.
__global__ __launch_bounds__(256) void attn_latent_merge_kernel(const LatentParams p, int Dv, int64_t total_rows, int only, int tile_keys) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= total_rows) return;
    const int lane = threadIdx.x & 63;
    const int t = (int)(row / p.H), even = only == 2 && p.slots > 0, share = even ? *p.share : 0;
    int lo = 0, hi = p.B;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (p.cu_q[mid] <= t) lo = mid; else hi = mid;
    }
    const int q_begin = p.cu_q[lo], n_q = p.cu_q[lo + 1] - q_begin;
    if ((n_q == 1) != (only == 1)) return;
    int ranges = p.nsplit;
    if (even) {                                              // (a row of one range has its output already)
        const int n_k = p.cu_k[lo + 1] - p.cu_k[lo], end = (int)((row - (int64_t)q_begin * p.H) / (4 * kLatRows) + 1) * (4 * kLatRows);
        ranges = latent_ranges(latent_tiles(n_k - n_q + (min(end, n_q * p.H) - 1) / p.H, tile_keys, p.nsplit, p.tiles_per_split), share);
        if (ranges == 1) return;
    }
    const float* base = p.part + row * p.nsplit * (Dv + 2);
    // lane s holds range s (at most 32 of them): its share of the denominator and the factor of its accumulators
    float m = kLatRunInit, l = 0.f;
    if (lane < ranges) {
        const float2 ml = *(const float2*)(base + lane * (Dv + 2) + Dv);
        l = ml.y;
        if (l > 0.f) m = ml.x;
    }
    float m_all = m;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) m_all = fmaxf(m_all, __shfl_xor(m_all, o));
    m_all = __shfl(m_all, 0);                                // (lanes 32.. hold nothing)
    const float f = l > 0.f ? __builtin_amdgcn_exp2f(m - m_all) : 0.f;      // 0: the range had no keys, its state is not read
    const float inv = lat_finish(m_all, wave_sum(l * f), p.sink, (int)(row % p.H));
    for (int c = 2 * lane; c < Dv; c += 128) {               // (Dv is even)
        float ox = 0.f, oy = 0.f;
#pragma unroll 8
        for (int s = 0; s < ranges; ++s) {
            const float fs = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), s));   // (some lanes may sit this out)
            const float2 v = *(const float2*)(base + s * (Dv + 2) + c);
            ox += fs > 0.f ? fs * v.x : 0.f;
            oy += fs > 0.f ? fs * v.y : 0.f;
        }
        *(uint32_t*)(p.out + row * Dv + c) = pack_bf16(ox * inv, oy * inv);
    }
}

// ------------------------------------------------------------------------------------------------ launch plan
static bool latent_built(int D, int Dv) {
    if (D % 32 || Dv % 32) return false;
    const int d = D / 32, v = Dv / 32;
    if (d == v) return (d >= 1 && d <= 8) || d == 10 || d == 12 || d == 16;
    return (d == 5 && v == 4) || (d == 6 && v == 4) || (d == 8 && v == 6) || (d == 10 && v == 8) || (d == 18 && v == 16);
}
static int latent_tile_keys(int D) { return D <= 256 ? 64 : 32; }

struct LatentPlan {
    int nsplit, tiles_per_split;
};
// Key ranges: enough workgroups for the chip (a few per CU), not fewer than `min_tiles` tiles each.
static LatentPlan latent_plan(int64_t wgs, int max_k, int tile, int64_t want, int min_tiles) {
    const int tiles = std::max(1, (max_k + tile - 1) / tile);
    int64_t n = wgs > 0 ? (want + wgs - 1) / wgs : 1;
    n = std::max<int64_t>(1, std::min<int64_t>({n, (int64_t)tiles / min_tiles, (int64_t)32}));
    const int per = (int)((tiles + n - 1) / n);
    return {(tiles + per - 1) / per, per};
}
static LatentPlan latent_rows_plan(int B, int H, int max_q, int max_k, int D) {
    return latent_plan((int64_t)B * (((int64_t)max_q * H + 127) / 128), max_k, latent_tile_keys(D), 384, 8);
}
static LatentPlan latent_single_plan(int B, int H, int max_k) {
    return latent_plan((int64_t)B * ((H + 31) / 32), max_k, 32, 512, 8);
}

template <int D32, int DV32>
static int launch_latent_rows(LatentParams& p, int64_t total_q, int max_q, int max_k, hipStream_t s) {
    constexpr int KB = D32 <= 8 ? 2 : 1, OCC = D32 <= 5 || (D32 == 6 && DV32 == 4) ? 2 : 1, D = 32 * D32;
    const LatentPlan plan = latent_rows_plan(p.B, p.H, max_q, max_k, D);
    p.nsplit = plan.nsplit;
    p.tiles_per_split = plan.tiles_per_split;
    p.row_tiles = (int)(((int64_t)max_q * p.H + 127) / 128);
    p.tiles_per_block = p.block_size / (32 * KB);
    p.dv_groups = p.Dv / (32 * DV32);
    const int slots = std::max(1, 256 * OCC / p.dv_groups);
    p.slots = (int64_t)p.B * p.row_tiles * p.nsplit > slots && (p.nsplit > 1 || latent_turns(p.B, total_q, max_q, max_k)) ? slots : 0;
    const dim3 grid((unsigned)(p.B * p.row_tiles), (unsigned)p.nsplit, (unsigned)p.dv_groups);
    if (p.slots > 0) hipLaunchKernelGGL((attn_latent_rows_kernel<D32, DV32, KB, OCC, true>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((attn_latent_rows_kernel<D32, DV32, KB, OCC, false>), grid, dim3(256), 0, s, p);
    return check_launch("nv_attn_latent_paged (rows kernel)");
}
template <int D32, int DV32>
static int launch_latent_single(LatentParams p, int max_k, hipStream_t s) {
    constexpr int OCC = D32 <= 6 ? 2 : 1, NBUF = D32 <= 5 ? 2 : 1, D = 32 * D32;
    constexpr size_t single_lds = (size_t)4 * NBUF * 32 * D * 2 + 4 * kLatRows * 8;
    static_assert(single_lds <= 160 * 1024, "LDS of a compute unit");
    const void* fn = (const void*)attn_latent_single_kernel<D32, DV32, NBUF, OCC>;
    static bool raised = single_lds <= 64 * 1024;              // beyond the default limit of dynamic LDS: raise it once
    if (!raised) {
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)single_lds) != hipSuccess) return NV_ERR_LAUNCH;
        raised = true;
    }
    const LatentPlan plan = latent_single_plan(p.B, p.H, max_k);
    p.nsplit = plan.nsplit;
    p.tiles_per_split = plan.tiles_per_split;
    p.head_groups = (p.H + 31) / 32;
    p.dv_groups = p.Dv / (32 * DV32);
    p.tiles_per_block = p.block_size / 32;
    hipLaunchKernelGGL((attn_latent_single_kernel<D32, DV32, NBUF, OCC>), dim3((unsigned)p.B, (unsigned)p.nsplit, (unsigned)(p.head_groups * p.dv_groups)),
                       dim3(256), single_lds, s, p);
    return check_launch("nv_attn_latent_paged (single kernel)");
}

}  // namespace nv

extern "C" int nv_attn_latent_ok(int D, int Dv, int block_size) {
    return nv::latent_built(D, Dv) && block_size > 0 && block_size % 64 == 0 ? 1 : 0;
}

extern "C" int64_t nv_attn_latent_workspace_bytes(int num_seqs, int64_t T, int H, int D, int Dv, int max_seqlen_q, int max_seqlen_k) {
    using namespace nv;
    if (num_seqs <= 0 || T <= 0 || H <= 0 || Dv <= 0 || max_seqlen_k <= 0) return 0;
    int n = latent_single_plan(num_seqs, H, max_seqlen_k).nsplit;
    if (max_seqlen_q > 1) n = std::max(n, latent_rows_plan(num_seqs, H, max_seqlen_q, max_seqlen_k, D).nsplit);
    return n > 1 ? kLatHeader + T * H * n * (int64_t)(Dv + 2) * (int64_t)sizeof(float) : 0;
}

extern "C" int nv_attn_latent_paged(const void* q, const void* cache, void* out, const int32_t* cu_seqlens_q,
                                    const int32_t* cu_seqlens_k, const int32_t* block_tables, int num_seqs,
                                    int max_blocks_per_seq, int64_t T, int H, int D, int Dv, int64_t num_blocks, int block_size,
                                    float scale, const float* sink, int max_seqlen_q, int max_seqlen_k, int single_rows,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
    using namespace nv;
    NV_REQUIRE(num_seqs >= 0 && T >= 0 && H > 0 && num_blocks > 0 && max_blocks_per_seq > 0, NV_ERR_INVALID_ARG,
               "nv_attn_latent_paged: bad sizes");
    NV_REQUIRE(nv_attn_latent_ok(D, Dv, block_size), NV_ERR_UNSUPPORTED,
               "nv_attn_latent_paged: no kernel for rows of %d, values of %d, blocks of %d", D, Dv, block_size);
    NV_REQUIRE(scale > 0.f, NV_ERR_UNSUPPORTED, "nv_attn_latent_paged: the scale must be positive");
    if (T == 0 || num_seqs == 0) return NV_OK;
    NV_REQUIRE(q && cache && out && cu_seqlens_q && cu_seqlens_k && block_tables, NV_ERR_INVALID_ARG,
               "nv_attn_latent_paged: null pointer");
    NV_REQUIRE(max_seqlen_q > 0 && max_seqlen_k > 0, NV_ERR_INVALID_ARG, "nv_attn_latent_paged: the longest lengths must be given");
    NV_REQUIRE(((uintptr_t)q | (uintptr_t)cache | (uintptr_t)out) % 16 == 0, NV_ERR_INVALID_ARG,
               "nv_attn_latent_paged: pointers must be 16-byte aligned");
    NV_REQUIRE(T * H < (1LL << 31) && num_seqs < 65536 * 16 && (int64_t)num_seqs * (((int64_t)max_seqlen_q * H + 127) / 128) < (1LL << 31) &&
                   num_blocks < (1LL << 31),
               NV_ERR_UNSUPPORTED, "nv_attn_latent_paged: launch too large");
    const int64_t need = nv_attn_latent_workspace_bytes(num_seqs, T, H, D, Dv, max_seqlen_q, max_seqlen_k);
    NV_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && (uintptr_t)workspace % 16 == 0), NV_ERR_WORKSPACE,
               "nv_attn_latent_paged: workspace of %lld bytes, need %lld", (long long)workspace_bytes, (long long)need);
    const bool several = max_seqlen_q > 1, singles = single_rows != 0 || !several;
    LatentParams p{};
    p.q = (const __bf16*)q;
    p.cache = (const __bf16*)cache;
    p.out = (__bf16*)out;
    p.share = (int*)workspace;
    p.part = workspace ? (float*)((char*)workspace + kLatHeader) : nullptr;
    p.cu_q = cu_seqlens_q;
    p.cu_k = cu_seqlens_k;
    p.block_tables = block_tables;
    p.sink = sink;
    p.B = num_seqs;
    p.H = H;
    p.max_blocks = max_blocks_per_seq;
    p.block_size = block_size;
    p.num_blocks = num_blocks;
    p.scale_log2 = scale * kLog2e;
    p.Dv = Dv;
    hipStream_t s = (hipStream_t)stream;
    const auto merge = [&](const LatentPlan& plan, int only) {
        if (plan.nsplit <= 1) return (int)NV_OK;
        p.nsplit = plan.nsplit;
        hipLaunchKernelGGL(attn_latent_merge_kernel, dim3((unsigned)((T * H + 3) / 4)), dim3(256), 0, s, p, Dv, T * H, only, latent_tile_keys(D));
        return check_launch("nv_attn_latent_paged (merge)");
    };
    int rc = NV_ERR_UNSUPPORTED;
    // row columns / 32, value columns / 32, value columns / 32 per workgroup
#define NV_LAT_ALL(X)                                                                                                      \
    X(1, 1, 1) X(2, 2, 2) X(3, 3, 3) X(4, 4, 4) X(5, 5, 5) X(6, 6, 6) X(7, 7, 7) X(8, 8, 8) X(10, 10, 5) X(12, 12, 6) X(16, 16, 8) \
        X(5, 4, 4) X(6, 4, 4) X(8, 6, 6) X(10, 8, 8) X(18, 16, 8)
    if (several) {
        switch (D / 32 * 100 + Dv / 32) {
#define NV_LAT_CASE(A, V, W) case A * 100 + V: rc = launch_latent_rows<A, W>(p, T, max_seqlen_q, max_seqlen_k, s); break;
            NV_LAT_ALL(NV_LAT_CASE)
#undef NV_LAT_CASE
        }
        if (rc == NV_OK) rc = merge(latent_rows_plan(num_seqs, H, max_seqlen_q, max_seqlen_k, D), 2);
        NV_REQUIRE(rc == NV_OK, rc, "nv_attn_latent_paged: the rows kernel could not be launched");
    }
    if (singles) {
        switch (D / 32 * 100 + Dv / 32) {
#define NV_LAT_CASE(A, V, W) case A * 100 + V: rc = launch_latent_single<A, W>(p, max_seqlen_k, s); break;
            NV_LAT_ALL(NV_LAT_CASE)
#undef NV_LAT_CASE
        }
        if (rc == NV_OK) rc = merge(latent_single_plan(num_seqs, H, max_seqlen_k), 1);
        NV_REQUIRE(rc == NV_OK, rc, "nv_attn_latent_paged: the single kernel could not be launched");
    }
    return NV_OK;
}
