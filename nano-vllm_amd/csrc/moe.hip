// Routed experts (mixture of experts with small clamped-GLU experts), without a host round trip:
//
// nv_moe_route          per token, from fp32 router logits [T, E]: the `top` largest (lowest index first among equals),
//                       their weights = softmax over the chosen logits only.  ids [T, top] int32, weights [T, top] fp32.
// nv_moe_route_softmax  the same shape of answer from softmax scores over ALL experts: the choice is made on score +
//                       correction, the weights are the plain scores times a constant.  Ids beyond the experts that have
//                       tensors (experts that hand their input through) are left out by nv_moe_align.
// nv_moe_align          sorts the T * top (token, choice) pairs by expert: sorted_pairs[position] = pair index, and a
//                       table of row tiles (expert, first position, rows) of at most `tile_rows` rows that never
//                       straddle two experts, plus their count, all on the device.
// nv_moe_gate_up        y[position, :] = act(G_e h, U_e h) for every sorted position (expert e, token of the pair):
//                       g = min(G_e h, limit), u = clamp(U_e h, -limit, limit), act = g * sigmoid(alpha g) * (u + 1).
// nv_moe_down           out[pair, :] = weight[pair] * (D_e y[position, :]), fp32, at the pair's own row: the caller sums
//                       the `top` rows of a token in a fixed order (no atomics, bitwise reproducible).
//
// Both products are grouped matrix products on the matrix cores, a row tile (16 to 128 rows of ONE expert) and some columns a workgroup of
// four waves, in one of three kernels:
//   moe_big_kernel      tiles of 128 rows, bf16: 256 weight rows, both operands by LDS-DMA, v_mfma_f32_32x32x16_bf16
//   moe_rows_kernel     tiles of 16, 32 and 64 rows, bf16, few tiles that read the same weights: 64 weight rows straight from memory into
//                       the operands' registers, the waves share the contraction
//   moe_grouped_kernel  everything else (float32, sizes and addresses that are not in 16-byte pieces, many small tiles of the same
//                       weights): 64 or 128 weight rows, 64-deep (fp32: 32-deep) slices of both operands through LDS, the next slices
//                       on their way into registers, v_mfma_f32_16x16x32_bf16 or v_mfma_f32_16x16x4_f32 (true fp32)
// Weights are [E, rows_out, rows_in] with the contraction index contiguous, as stored.  The launch is sized for the most tiles any
// routing can produce; workgroups beyond the table's count return at once.
#include <algorithm>
#include <type_traits>

#include "launch_order.h"
#include "mfma_tile.h"
#include "../../include/nanovllm_hip_mixers.h"

namespace nv {

constexpr int kMoeMaxTop = 16;
constexpr int kMoeBN = 64;

// One wave per token: a lane keeps the logits e = lane, lane + 64, ... in registers (PER of them; more experts than
// that are re-read from memory), and every choice is a wave-wide arg-max (larger value, then lower index) after which the winner's
// lane strikes its element out.  Lane j keeps choice j: arrays indexed by the choice would lie in private memory (8192 tokens, top 4 of
// 32 experts: 13 -> 7 us for the launch).
constexpr int kMoeRoutePerLane = 8;            // experts <= 512 stay in registers
constexpr int kMoeNone = 0x7fffffff;
__device__ __forceinline__ void moe_better(float& v, int& e, float ov, int oe) {
    const bool take = (oe != kMoeNone) & ((e == kMoeNone) | (ov > v) | ((ov == v) & (oe < e)));      // (no branches)
    v = take ? ov : v;
    e = take ? oe : e;
}
template <int CTRL>
__device__ __forceinline__ void moe_better_dpp(float& v, int& e) {
    const float ov = dpp_f32<CTRL>(v);
    moe_better(v, e, ov, __builtin_amdgcn_update_dpp(0, e, CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float moe_first(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
// The choices of one token, a wave's work: lane j < top gets choice j and its weight.
template <int PER>
__device__ __forceinline__ void moe_route_token(const float* __restrict__ z, int E, int top, int lane, int& id, float& weight) {
    float reg[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        reg[i] = e < E ? z[e] : -INFINITY;
    }
    unsigned taken = 0;                                // bit i: this lane's element i is chosen
    float val = -INFINITY;
    id = 0;
    for (int j = 0; j < top; ++j) {
        float bv = -INFINITY;
        int be = kMoeNone;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane + 64 * i;
            if (e < E && !((taken >> i) & 1u) && (be == kMoeNone || reg[i] > bv)) { bv = reg[i]; be = e; }
        }
        for (int e = lane + 64 * PER; e < E; e += 64) {                  // the part that is not in registers
            bool gone = false;
            for (int i = 0; i < j; ++i) gone |= __builtin_amdgcn_readlane(id, i) == e;
            const float v = z[e];
            if (!gone && (be == kMoeNone || v > bv)) { bv = v; be = e; }
        }
        moe_better_dpp<0xB1>(bv, be);                  // lanes 1 and 2 apart, mirrored halves of 8, of 16, then 16 and 32 apart
        moe_better_dpp<0x4E>(bv, be);
        moe_better_dpp<0x141>(bv, be);
        moe_better_dpp<0x140>(bv, be);
        moe_better(bv, be, __shfl_xor(bv, 16), __shfl_xor(be, 16));
        moe_better(bv, be, __shfl_xor(bv, 32), __shfl_xor(be, 32));
        be = __builtin_amdgcn_readfirstlane(be);
        bv = moe_first(bv);
        if ((be & 63) == lane && be < 64 * PER) taken |= 1u << (be >> 6);
        if (lane == j) { id = be; val = bv; }
    }
    const float ex = expf(val - moe_first(val));
    float sum = 0.f;
    for (int j = 0; j < top; ++j) sum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ex), j));
    weight = ex / sum;
}

// The same for at most 64 experts, four tokens of a wave side by side: 16 lanes a token, four logits each, so that a choice takes no
// exchange beyond a row of 16 lanes.
__device__ __forceinline__ void moe_load_logits(const float* __restrict__ z, int E, int l16, float (&reg)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) reg[i] = l16 + 16 * i < E ? z[l16 + 16 * i] : -INFINITY;
}
__device__ __forceinline__ void moe_route_four(const float (&reg)[4], int E, int top, int l16, int& id, float& weight) {
    unsigned open = 0;                                 // bit i: element l16 + 16 i is there and not chosen yet
#pragma unroll
    for (int i = 0; i < 4; ++i) open |= l16 + 16 * i < E ? 1u << i : 0u;
    float val = -INFINITY;
    id = 0;
    for (int j = 0; j < top; ++j) {
        float bv = -INFINITY;
        int be = kMoeNone;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (((open >> i) & 1u) && (be == kMoeNone || reg[i] > bv)) { bv = reg[i]; be = l16 + 16 * i; }
        moe_better_dpp<0xB1>(bv, be);
        moe_better_dpp<0x4E>(bv, be);
        moe_better_dpp<0x141>(bv, be);
        moe_better_dpp<0x140>(bv, be);
        be = __builtin_amdgcn_update_dpp(0, be, 0x150, 0xF, 0xF, true);        // (of the row's first lane)
        bv = dpp_f32<0x150>(bv);
        if ((be & 15) == l16) open &= ~(1u << (be >> 4));
        if (l16 == j) { id = be; val = bv; }
    }
    const float ex = expf(val - dpp_f32<0x150>(val));
    float sum = 0.f;
#define NV_MOE_ADD(J) if (J < top) sum += dpp_f32<0x150 + J>(ex)
    NV_MOE_ADD(0); NV_MOE_ADD(1); NV_MOE_ADD(2); NV_MOE_ADD(3); NV_MOE_ADD(4); NV_MOE_ADD(5); NV_MOE_ADD(6); NV_MOE_ADD(7);
    NV_MOE_ADD(8); NV_MOE_ADD(9); NV_MOE_ADD(10); NV_MOE_ADD(11); NV_MOE_ADD(12); NV_MOE_ADD(13); NV_MOE_ADD(14); NV_MOE_ADD(15);
#undef NV_MOE_ADD
    weight = ex / sum;
}

template <int PER>
__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ logits, int* __restrict__ ids,
                                                        float* __restrict__ wgt, int64_t T, int E, int top) {
    constexpr int G = PER == 1 ? 4 : 1;                // tokens of a wave
    const int lane = threadIdx.x & 63, at = lane & (64 / G - 1);
    const int64_t t0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * G, t = t0 + lane / (64 / G);
    if (t0 >= T) return;                               // (whole waves leave together)
    int id;
    float weight;
    if constexpr (PER == 1) {
        float reg[4];
        moe_load_logits(logits + min(t, T - 1) * E, E, at, reg);
        moe_route_four(reg, E, top, at, id, weight);
    } else {
        moe_route_token<PER>(logits + t * E, E, top, lane, id, weight);
    }
    if (at < top && t < T) {
        ids[t * top + at] = id;
        wgt[t * top + at] = weight;
    }
}

// Sigmoid scores with a selection bias and a choice limited to the best consecutive blocks of experts.  One wave per
// token: the biased scores go to LDS, a lane adds up the top two of its block, every group counts how many
// groups beat it (larger merit, then lower index) and is open when fewer than `keep` do; the choice is the wave-wide
// arg-max of nv_moe_route over the experts of open groups, and the weights are the plain sigmoids of the chosen.
constexpr int kMoeGroupedMaxE = 512;
__global__ __launch_bounds__(64) void moe_route_grouped_kernel(const float* __restrict__ logits, const float* __restrict__ corr,
                                                               int* __restrict__ ids, float* __restrict__ wgt, int E, int top,
                                                               int n_groups, int keep) {
    __shared__ float choice[kMoeGroupedMaxE];
    __shared__ float merit[kMoeGroupedMaxE];
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const float* z = logits + t * E;
    const int gs = E / n_groups;
    for (int e = lane; e < E; e += 64) {
        const float s = 1.0f / (1.0f + expf(-z[e]));
        choice[e] = corr != nullptr ? s + corr[e] : s;
    }
    __syncthreads();
    if (n_groups > 1) {
        for (int g = lane; g < n_groups; g += 64) {
            float a = -INFINITY, b = -INFINITY;                // the largest and the second largest of the group
            for (int i = 0; i < gs; ++i) {
                const float c = choice[g * gs + i];
                if (c > a) { b = a; a = c; } else if (c > b) b = c;
            }
            merit[g] = gs > 1 ? a + b : a;
        }
        __syncthreads();
        for (int g = lane; g < n_groups; g += 64) {
            const float mine = merit[g];
            int ahead = 0;
            for (int o = 0; o < n_groups; ++o) ahead += (merit[o] > mine || (merit[o] == mine && o < g)) ? 1 : 0;
            if (ahead >= keep)
                for (int i = 0; i < gs; ++i) choice[g * gs + i] = -INFINITY;
        }
        __syncthreads();
    }
    unsigned taken = 0;
    for (int j = 0; j < top; ++j) {
        float bv = -INFINITY;
        int be = 0x7fffffff;
        for (int i = 0; i < kMoeGroupedMaxE / 64; ++i) {
            const int e = lane + 64 * i;
            if (e < E && !((taken >> i) & 1u) && (be == 0x7fffffff || choice[e] > bv)) { bv = choice[e]; be = e; }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off);
            const int oe = __shfl_xor(be, off);
            const bool mine_valid = be != 0x7fffffff, other_valid = oe != 0x7fffffff;
            if (other_valid && (!mine_valid || ov > bv || (ov == bv && oe < be))) { bv = ov; be = oe; }
        }
        if ((be & 63) == lane) taken |= 1u << (be >> 6);
        if (lane == 0) {
            ids[t * top + j] = be;
            wgt[t * top + j] = 1.0f / (1.0f + expf(-z[be]));
        }
    }
}

// Softmax scores over all experts, a choice on score + correction, weights = scale * score of the chosen.  One wave per
// token: scores and choice values live in LDS, each choice is a wave-wide arg-max (larger value, then lower index) after
// which the winner's lane strikes it out.
constexpr int kMoeSoftmaxMaxE = 1024;
__global__ __launch_bounds__(64) void moe_route_softmax_kernel(const float* __restrict__ logits, const float* __restrict__ corr,
                                                               int* __restrict__ ids, float* __restrict__ wgt, int E, int top,
                                                               float scale) {
    __shared__ float score[kMoeSoftmaxMaxE];
    __shared__ float choice[kMoeSoftmaxMaxE];
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const float* z = logits + t * E;
    float zmax = -INFINITY;
    for (int e = lane; e < E; e += 64) zmax = fmaxf(zmax, z[e]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) zmax = fmaxf(zmax, __shfl_xor(zmax, off));
    float sum = 0.f;
    for (int e = lane; e < E; e += 64) {
        const float p = expf(z[e] - zmax);
        score[e] = p;
        sum += p;
    }
    const float inv = 1.0f / wave_sum(sum);
    for (int e = lane; e < E; e += 64) {               // (a lane reads back what it wrote itself)
        const float s = score[e] * inv;
        score[e] = s;
        choice[e] = corr != nullptr ? s + corr[e] : s;
    }
    __syncthreads();
    unsigned taken = 0;                                // bit i: expert lane + 64 i is chosen
    for (int j = 0; j < top; ++j) {
        float bv = -INFINITY;
        int be = E;                                    // E: nothing found
        for (int i = 0, e = lane; e < E; ++i, e += 64)
            if (!((taken >> i) & 1u) && (be == E || choice[e] > bv)) { bv = choice[e]; be = e; }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off);
            const int oe = __shfl_xor(be, off);
            if (oe < E && (be == E || ov > bv || (ov == bv && oe < be))) { bv = ov; be = oe; }
        }
        if ((be & 63) == lane) taken |= 1u << (be >> 6);
        if (lane == 0) {
            ids[t * top + j] = be;
            wgt[t * top + j] = scale * score[be < E ? be : 0];
        }
    }
}

// One workgroup.  meta: [0] = number of tiles, then (expert, first position, rows) per tile.  A pair whose id is not in
// 0 .. E - 1 (a choice that needs no product) gets no position.  Every wave counts and places its own range of the pairs through
// counters of its own (COPIES of them; one for few pairs and when they would not fit LDS): 64 lanes on one table beside 15 other waves spent the time
// on each other's additions (32768 pairs, 32 experts: 43 -> 21 us).
template <int COPIES>
__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids, int* __restrict__ sorted_pairs,
                                                         int* __restrict__ meta, int64_t P, int E, int tile_rows) {
    extern __shared__ int sm[];                    // [COPIES][E] counts, then cursors; [E + 1] first position, [E + 1] first tile
    int* first = sm + COPIES * E;
    int* first_tile = first + E + 1;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int* mine = sm + (COPIES > 1 ? wave : 0) * E;
    for (int i = tid; i < COPIES * E; i += 1024) sm[i] = 0;
    __syncthreads();
    const int64_t per = ((P + 15) / 16 + 63) / 64 * 64, p0 = wave * per, p1 = p0 + per < P ? p0 + per : P;
    for (int64_t p = p0 + lane; p < p1; p += 256) {          // four loads on their way
        int e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = p + 64 * u < p1 ? ids[p + 64 * u] : -1;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (e[u] >= 0 && e[u] < E) atomicAdd(&mine[e[u]], 1);
    }
    __syncthreads();
    for (int e = tid; e < E; e += 1024) {          // counts to the copies' offsets within the expert, the total to first[e + 1]
        int off = 0;
        for (int c = 0; c < COPIES; ++c) {
            const int n = sm[c * E + e];
            sm[c * E + e] = off;
            off += n;
        }
        first[e + 1] = off;
        first_tile[e + 1] = (off + tile_rows - 1) / tile_rows;
    }
    __syncthreads();
    if (tid == 0) {
        first[0] = first_tile[0] = 0;
        for (int e = 0; e < E; ++e) {
            first[e + 1] += first[e];
            first_tile[e + 1] += first_tile[e];
        }
        meta[0] = first_tile[E];
    }
    __syncthreads();
    for (int e = tid; e < E; e += 1024) {
        for (int c = 0; c < COPIES; ++c) sm[c * E + e] += first[e];
        for (int n = first_tile[e], m = first[e]; n < first_tile[e + 1]; ++n, m += tile_rows) {
            meta[1 + 3 * n] = e;
            meta[2 + 3 * n] = m;
            meta[3 + 3 * n] = min(tile_rows, first[e + 1] - m);
        }
    }
    __syncthreads();
    for (int64_t p = p0 + lane; p < p1; p += 256) {
        int e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = p + 64 * u < p1 ? ids[p + 64 * u] : -1;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (e[u] >= 0 && e[u] < E) sorted_pairs[atomicAdd(&mine[e[u]], 1)] = (int)(p + 64 * u);
    }
}

// Routing and sort together.  Few tokens: one launch of one workgroup, the pairs' ids and places stay in registers.  More: the
// first launch routes a few tokens a workgroup and leaves every workgroup's counts per expert, the second one adds them up
// and places the pairs; the single workgroup of moe_align_kernel spends its time on 32768 additions to LDS.  Beyond 64 experts a token takes a
// wave for a microsecond a choice, so that a wave has one as long as the counts of the workgroups stay few.
// Two launches of their own against these, us:
//   top 4 of 32 experts, 32 tokens 11.1 -> 4.7, 128: 11.5 -> 7.7, 256: 11.8 -> 7.4, 8192: 36.2 -> 12.8
//   top 8 of 65: 8 tokens 17.6 -> 9.2, 128: 18.6 -> 12.1 (82 in one workgroup), 1024: 23.6 -> 17.4 (35 with four tokens a wave), 8192: 66.5 -> 60.9
//   top 8 of 512: 8 tokens 45 -> 11.4, 128: 47 -> 16.9, 1024: 52 -> 32.5, 8192: 104 -> 84;  top 2 of 65, 4096 and 8192: 17.6 -> 18.4, 24.8 -> 25.5
constexpr int kMoeSortMaxE = 512, kMoeSortGroups = 256;
constexpr __host__ __device__ int moe_sort_few(int E) { return E <= 64 ? 128 : 16; }
constexpr __host__ __device__ int moe_sort_least(int E) { return E <= 64 ? 16 : 4; }         // a token a wave, four side by side up to 64 experts

// first / first_tile [E + 1] from the counts by one wave (in LDS)
__device__ __forceinline__ void moe_scan(const int* counts, int* first, int* first_tile, int E, int tile_rows, int lane) {
    int base = 0, base_tile = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int n = e0 + lane < E ? counts[e0 + lane] : 0, m = (n + tile_rows - 1) / tile_rows;
        int sum = n, tiles = m;
#pragma unroll
        for (int off = 1; off < 64; off *= 2) {
            const int a = __shfl_up(sum, off), b = __shfl_up(tiles, off);
            if (lane >= off) { sum += a; tiles += b; }
        }
        if (e0 + lane < E) {
            first[e0 + lane] = base + sum - n;
            first_tile[e0 + lane] = base_tile + tiles - m;
        }
        base += __builtin_amdgcn_readlane(sum, 63);
        base_tile += __builtin_amdgcn_readlane(tiles, 63);
    }
    if (lane == 0) {
        first[E] = base;
        first_tile[E] = base_tile;
    }
}
__device__ __forceinline__ void moe_put_tiles(const int* first, const int* first_tile, int* __restrict__ meta, int E, int tile_rows, int tid, int threads) {
    if (tid == 0) meta[0] = first_tile[E];
    for (int e = tid; e < E; e += threads) {
        for (int n = first_tile[e], m = first[e]; n < first_tile[e + 1]; ++n, m += tile_rows) {
            meta[1 + 3 * n] = e;
            meta[2 + 3 * n] = m;
            meta[3 + 3 * n] = min(tile_rows, first[e + 1] - m);
        }
    }
}

template <int PER>
__global__ __launch_bounds__(1024) void moe_route_sort_few_kernel(const float* __restrict__ logits, int* __restrict__ ids, float* __restrict__ wgt,
                                                                  int* __restrict__ sorted_pairs, int* __restrict__ meta, int T, int E, int top,
                                                                  int tile_rows) {
    __shared__ int counts[64 * PER], first[64 * PER + 1], first_tile[64 * PER + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int e = tid; e < E; e += 1024) counts[e] = 0;
    __syncthreads();
    constexpr int G = PER == 1 ? 4 : 1, N = moe_sort_few(64 * PER) / (16 * G);       // tokens of a wave side by side; times
    const int at = lane & (64 / G - 1), mine = wave * G + lane / (64 / G);
    int id[N], place[N];
    float reg[PER == 1 ? N : 1][4];
    if constexpr (PER == 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) moe_load_logits(logits + min(mine + 16 * G * i, T - 1) * (int64_t)E, E, at, reg[i]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int t = mine + 16 * G * i;
        if ((wave + 16 * i) * G < T) {
            float weight;
            if constexpr (PER == 1) moe_route_four(reg[i], E, top, at, id[i], weight);
            else moe_route_token<PER>(logits + (int64_t)t * E, E, top, lane, id[i], weight);
            if (at < top && t < T) {
                ids[t * top + at] = id[i];
                wgt[t * top + at] = weight;
                place[i] = atomicAdd(&counts[id[i]], 1);
            }
        }
    }
    __syncthreads();
    if (wave == 0) moe_scan(counts, first, first_tile, E, tile_rows, lane);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int t = mine + 16 * G * i;
        if (t < T && at < top) sorted_pairs[first[id[i]] + place[i]] = t * top + at;
    }
    moe_put_tiles(first, first_tile, meta, E, tile_rows, tid, 1024);
}

template <int PER>
__global__ __launch_bounds__(256) void moe_route_count_kernel(const float* __restrict__ logits, int* __restrict__ ids, float* __restrict__ wgt,
                                                              int* __restrict__ counts, int64_t T, int E, int top, int tokens) {
    __shared__ int mine[64 * PER];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int e = tid; e < E; e += 256) mine[e] = 0;
    __syncthreads();
    constexpr int G = PER == 1 ? 4 : 1;                // tokens of a wave side by side
    const int at = lane & (64 / G - 1);
    const int64_t t0 = (int64_t)blockIdx.x * tokens, t1 = min(t0 + tokens, T);
    for (int64_t tw = t0 + wave * G; tw < t1; tw += 4 * G) {
        const int64_t t = tw + lane / (64 / G);
        int id;
        float weight;
        if constexpr (PER == 1) {
            float reg[4];
            moe_load_logits(logits + min(t, T - 1) * E, E, at, reg);
            moe_route_four(reg, E, top, at, id, weight);
        } else {
            moe_route_token<PER>(logits + t * E, E, top, lane, id, weight);
        }
        if (at < top && t < t1) {
            ids[t * top + at] = id;
            wgt[t * top + at] = weight;
            atomicAdd(&mine[id], 1);
        }
    }
    __syncthreads();
    for (int e = tid; e < E; e += 256) counts[(int64_t)blockIdx.x * E + e] = mine[e];
}

// grid: as many workgroups as counted.  columns: the power of two that holds E, at most 256; the other threads share the workgroups.
__global__ __launch_bounds__(256) void moe_place_kernel(const int* __restrict__ ids, const int* __restrict__ counts, int* __restrict__ sorted_pairs,
                                                        int* __restrict__ meta, int64_t pairs, int E, int tile_rows, int per_group, int columns) {
    __shared__ int all[kMoeSortMaxE], before[kMoeSortMaxE], first[kMoeSortMaxE + 1], first_tile[kMoeSortMaxE + 1];
    const int tid = threadIdx.x, groups = gridDim.x, me = blockIdx.x;
    for (int e = tid; e < E; e += 256) all[e] = before[e] = 0;
    __syncthreads();
    const int shares = 256 / columns, per = (groups + shares - 1) / shares;
    const int g0 = tid / columns * per, g1 = min(g0 + per, groups);
    for (int e = tid % columns; e < E; e += columns) {
        int sum = 0, ahead = 0;
#pragma unroll 8
        for (int g = g0; g < g1; ++g) {
            const int n = counts[(int64_t)g * E + e];
            sum += n;
            ahead += g < me ? n : 0;
        }
        atomicAdd(&all[e], sum);
        atomicAdd(&before[e], ahead);
    }
    __syncthreads();
    if (tid < 64) moe_scan(all, first, first_tile, E, tile_rows, tid);
    __syncthreads();
    if (me == 0) moe_put_tiles(first, first_tile, meta, E, tile_rows, tid, 256);
    const int64_t p0 = (int64_t)me * per_group, p1 = min(p0 + per_group, pairs);
    for (int64_t p = p0 + tid; p < p1; p += 256) {
        const int e = ids[p];
        sorted_pairs[first[e] + atomicAdd(&before[e], 1)] = (int)p;
    }
}

// The gated unit of all three kernels below.  (On the hardware's exponential and reciprocal the tiles of 128 rows would save 17 of
// the 497 us of the call measured there, at one or two units in the last place more and with nothing left of a denormal reciprocal.)
__device__ __forceinline__ float moe_glu(float g, float u, float limit, float alpha, float shift) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-alpha * g)) * (u + shift);
}

// Many rows per expert, bf16: a workgroup of four waves takes 128 rows of one expert and 256 weight rows (gate and up: 128 columns of
// both), a wave 64 x 128 of it on v_mfma_f32_32x32x16_bf16 (weights as the first operand, so that a lane holds four neighbouring
// columns of a row).  Slices 64 deep, whole cache lines of every row, go straight into LDS (LDS-DMA, chunks swizzled by row so that the
// 16-byte operand reads are free of bank conflicts).  A wave reads all operands of its slice into registers; the next slice then goes into the same
// 48 KiB while it multiplies, and the other workgroup of the CU has its turn at LDS.  Rows past the tile repeat its first one, weight rows past N the last
// ones; neither is written.
// Launches that leave a CU one workgroup, and rows or weights 4 GiB apart, take slices 32 deep by address, three buffers and two slices in flight.
// What bounds it: the way of the slices from L2 (11 TB/s through the CUs' vector caches).  Slices 32 deep take half a cache line of every row
// and the same line again for the next slice: 340 and 240 us for both products of the call below.  Without any loads behind the first slice it
// is 217 and 136 us, with all of them in the vector caches 226 and 145, in L2 263 and 160 (these, and the next lines', with the cheaper gated unit).
// Buffer loads, because the compiler waits for all LDS reads behind a global load into LDS (and has no 64-bit addresses to add up): 336 -> 281
// us; the products at a higher priority than the other workgroup's reads: 299 -> 281.  256 x 256 by one workgroup a CU, two buffers: four
// waves of 128 x 128 319 and 211 us, eight of 64 x 128 349 and 220; a load of the lines two slices ahead into L2: no gain.
// 8192 tokens, top 4 of 32 experts, width 2048, ff 1024: gate and up 340 -> 297 us, down 240 -> 187; the call 604 -> 497, with the outputs past the caches 485.
constexpr int kMoeBigRows = 128;

// D: depth of a slice, 64 or 32.  A piece of 1 KiB is 512 / D rows of 2 D bytes, lane l fills bytes 16 l .. of it.
template <int D>
__device__ __forceinline__ int big_off(int row, int ch) {
    return row * 2 * D + ((ch ^ (D == 64 ? (row >> 1) & 7 : (row >> 2) & 3)) * 16);
}
// STREAM: outputs pass by the caches (moe_streams_out).
template <int MODE, int D, bool STREAM = false>
__global__ __launch_bounds__(256, 2) void moe_big_kernel(
    const __bf16* __restrict__ a, int64_t a_stride, const __bf16* __restrict__ w, const int* __restrict__ sorted_pairs,
    const int* __restrict__ meta, const float* __restrict__ pair_w, __bf16* __restrict__ y, float* __restrict__ out, int top, int N,
    int K, float limit, float alpha, float up_shift) {
    constexpr bool GATE_UP = MODE == 1, GATHER = MODE != 0;
    constexpr int COLS = GATE_UP ? 128 : 256, XB = kMoeBigRows * 2 * D, BUF = XB + 256 * 2 * D;       // bytes: rows' slice, both slices
    __shared__ __attribute__((aligned(16))) unsigned char buf[BUF], buf1[D == 64 ? 16 : BUF], buf2[D == 64 ? 16 : BUF];
    __shared__ int src_row[kMoeBigRows];
    __shared__ float weight[MODE == 0 ? kMoeBigRows : 1];
    // Workgroups go to the eight XCDs in turn; an XCD takes a run of the tiles that there are, all column blocks of a tile next to each
    // other: its L2 then holds a tile's rows for all of them and an expert's weights for its tiles (tiles next to each other instead:
    // no difference at the call above).
    const int n_cols = (N + COLS - 1) / COLS, items = meta[0] * n_cols, per_xcd = (items + 7) / 8, at = blockIdx.x / 8;
    const int item = (blockIdx.x & 7) * per_xcd + at;
    if (at >= per_xcd || item >= items) return;
    const int tile = item / n_cols, n0 = (item % n_cols) * COLS;
    const int e = meta[1 + 3 * tile], row0 = meta[2 + 3 * tile], rows = meta[3 + 3 * tile];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5, wr = wave >> 1, wc = wave & 1;
    for (int i = tid; i < kMoeBigRows; i += 256) {
        src_row[i] = sorted_pairs[row0 + min(i, rows - 1)];
        if constexpr (MODE == 0) weight[i] = pair_w[src_row[i]];
    }
    __syncthreads();
    const __bf16* we = w + (int64_t)e * ((GATE_UP ? 2 : 1) * (int64_t)N) * K;
    // a wave stages XP pieces of the rows and WP of the weight rows
    constexpr int PR = 512 / D, XP = kMoeBigRows / PR / 4, WP = 256 / PR / 4;
    const int p_row = lane / (D / 8), p_ch = lane % (D / 8);
    // 64 deep: 32-bit offsets from the first row and from the expert's first weight row (the launch sees to it that they fit)
    const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(GATHER ? a : a + (int64_t)row0 * a_stride), 0, -1, 0x00020000);
    const auto wr_ = __builtin_amdgcn_make_buffer_rsrc((void*)we, 0, -1, 0x00020000);
    uint32_t x_lane[4], w_lane[2], w_piece[8];
    const char *xp[2], *wp[4];                        // 32 deep: addresses
    if constexpr (D == 64) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int r = (wave * XP + i) * PR + p_row;
            x_lane[i] = ((uint32_t)(GATHER ? src_row[r] / top : min(r, rows - 1)) * (uint32_t)a_stride + (p_ch ^ ((r >> 1) & 7)) * 8) * 2u;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) w_lane[i] = (uint32_t)(p_row * K + (p_ch ^ (i * 4 + (p_row >> 1))) * 8) * 2u;
        // (N is a multiple of 8: a piece's weight rows are all there or none of them is)
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int lr = (wave * WP + i) * PR;      // first weight row of the piece: gate rows, then up rows
            w_piece[i] = (uint32_t)(GATE_UP ? (lr >> 7) * N + min(n0 + (lr & 127), N - 8) : min(n0 + lr, N - 8)) * (uint32_t)K * 2u;
        }
    } else {
        const int ch = p_ch ^ ((p_row >> 2) & 3);
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int r = (wave * XP + i) * PR + p_row;
            const int64_t at = GATHER ? (int64_t)(src_row[r] / top) : row0 + min(r, rows - 1);
            xp[i] = (const char*)(a + at * a_stride + ch * 8);
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int lr = (wave * WP + i) * PR + p_row;
            const int64_t n = GATE_UP ? (lr >> 7) * (int64_t)N + min(n0 + (lr & 127), N - 1) : min(n0 + lr, N - 1);
            wp[i] = (const char*)(we + n * K + ch * 8);
        }
    }
    auto stage = [&](unsigned char* dst, int t) {     // (32 deep: the slices one after the other)
        if constexpr (D == 64) {
#pragma unroll
            for (int i = 0; i < WP; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(wr_, (__attribute__((address_space(3))) void*)(dst + XB + (wave * WP + i) * 1024), 16,
                                                         w_lane[i & 1], w_piece[i] + t * 128, 0, 0);
#pragma unroll
            for (int i = 0; i < XP; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(dst + (wave * XP + i) * 1024), 16, x_lane[i],
                                                         t * 128, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)xp[i],
                                                 (__attribute__((address_space(3))) void*)(dst + (wave * XP + i) * 1024), 16, 0, 0);
                xp[i] += 64;
            }
#pragma unroll
            for (int i = 0; i < WP; ++i) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)wp[i],
                                                 (__attribute__((address_space(3))) void*)(dst + XB + (wave * WP + i) * 1024), 16, 0, 0);
                wp[i] += 64;
            }
        }
    };
    f32x16 acc[4][2];                                 // [weight block: gate 0, 1, up 0, 1 | 0 .. 3][row block]
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[j][x][i] = 0.f;
    bf16x8 xf[D / 16][2], wf[D / 16][4];              // operands of the 16-deep steps of a slice
    auto read = [&](const unsigned char* src, int s) {
#pragma unroll
        for (int x = 0; x < 2; ++x) xf[s][x] = *(const bf16x8*)(src + big_off<D>(wr * 64 + x * 32 + l32, 2 * s + hh));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int lr = GATE_UP ? (j >> 1) * 128 + wc * 64 + (j & 1) * 32 : wc * 128 + j * 32;
            wf[s][j] = *(const bf16x8*)(src + XB + big_off<D>(lr + l32, 2 * s + hh));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int x = 0; x < 2; ++x) acc[j][x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[s][j], xf[s][x], acc[j][x], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int slices = K / D;
    if constexpr (D == 64) {
        stage(buf, 0);
        for (int t = 0; t < slices; ++t) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x70);         // vmcnt(0) lgkmcnt(0): this wave's part of the slice has landed
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int s = 0; s < 4; ++s) read(buf, s);
            if (t + 1 < slices) {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the wave has read the slice
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                stage(buf, t + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int s = 0; s < 4; ++s) multiply(s);
            __builtin_amdgcn_s_setprio(0);
        }
    } else {
        // One slice: this wave's part of it has landed (all but the newest six loads have) and the wave is done reading the one before;
        // past the barrier so it is for all waves, and the slice after the next one goes where the one before was.  An LDS object per buffer and
        // no condition inside the loop: the compiler waits for the loads just issued in front of every read otherwise (36 -> 48 us).
        auto step = [&](bool more, bool stages, const unsigned char* now, unsigned char* after_next) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);        // (nor may the products sink below the wait)
            if (more) __builtin_amdgcn_s_waitcnt(0x76);       // vmcnt(6) lgkmcnt(0): the six of the next slice stay in flight
            else __builtin_amdgcn_s_waitcnt(0x70);    // vmcnt(0) lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (stages) stage(after_next, 0);
            __builtin_amdgcn_sched_barrier(0);        // (the compiler would start the loads behind the products)
#pragma unroll
            for (int s = 0; s < 2; ++s) read(now, s);
#pragma unroll
            for (int s = 0; s < 2; ++s) multiply(s);
        };
        stage(buf, 0);                                // (at least 2 slices: K is a multiple of 64)
        stage(buf1, 0);
        int t = 0;
        for (; t + 4 < slices; t += 3) {
            step(true, true, buf, buf2);
            step(true, true, buf1, buf);
            step(true, true, buf2, buf1);
        }
        const int left = slices - t;                  // 2 .. 4
        step(true, left > 2, buf, buf2);
        step(left > 2, left > 3, buf1, buf);
        if (left > 2) step(left > 3, false, buf2, buf1);
        if (left > 3) step(false, false, buf, buf2);
    }
    __syncthreads();                                  // the slices are done with: each wave turns its blocks through LDS of its own
    // lane (l32, hh) holds of row 64 wr + 32 x + l32 the weight rows 8 (i >> 2) + 4 hh + (i & 3) of each block
    if constexpr (MODE != 0) {
        constexpr int CW = GATE_UP ? 64 : 128, LD = CW * 2 + 16;       // columns of the wave; bytes of a staged row
        unsigned char* st = D == 64 ? buf + wave * 32 * LD : (wave < 2 ? buf : buf1) + (wave & 1) * 32 * LD;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
            for (int j = 0; j < (GATE_UP ? 2 : 4); ++j)
#pragma unroll
                for (int i = 0; i < 16; i += 4) {
                    float v[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        if constexpr (GATE_UP) {
                            v[t] = moe_glu(acc[j][x][i + t], acc[j + 2][x][i + t], limit, alpha, up_shift);
                        } else {
                            const float u = fmaxf(acc[j][x][i + t], 0.f);
                            v[t] = u * u;
                        }
                    }
                    *(uint2*)(st + l32 * LD + (j * 32 + 2 * i + 4 * hh) * 2) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            constexpr int LPR = CW / 8;               // lanes a row, 16 bytes each
#pragma unroll
            for (int it = 0; it < 32 * LPR / 64; ++it) {
                const int rr = it * (64 / LPR) + lane / LPR, c = (lane % LPR) * 8, r = wr * 64 + x * 32 + rr, n = n0 + wc * CW + c;
                const uint4 v = *(const uint4*)(st + rr * LD + c * 2);
                if (r < rows && n < N) *(uint4*)(y + (int64_t)(row0 + r) * N + n) = v;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    } else {
        constexpr int LD = 64 * 4 + 16;
        unsigned char* st = D == 64 ? buf + wave * 32 * LD : (wave < 2 ? buf : buf1) + (wave & 1) * 32 * LD;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {    // 64 columns at a time
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        const f32x16& c = acc[2 * half + j][x];
                        *(float4*)(st + l32 * LD + (j * 32 + 2 * i + 4 * hh) * 4) = make_float4(c[i], c[i + 1], c[i + 2], c[i + 3]);
                    }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    const int rr = it * 4 + (lane >> 4), c = (lane & 15) * 4, r = wr * 64 + x * 32 + rr, n = n0 + wc * 128 + half * 64 + c;
                    float4 v = *(const float4*)(st + rr * LD + c * 4);
                    if (r < rows && n < N) {
                        const int pair = src_row[r];
                        const float f = weight[r];
                        const f32x4 o = {v.x * f, v.y * f, v.z * f, v.w * f};
                        f32x4* to = (f32x4*)(out + (int64_t)pair * N + n);
                        if constexpr (STREAM) __builtin_nontemporal_store(o, to);
                        else *to = o;
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
    }
}

// Few rows per expert, bf16: bound by the expert's weights, which stream from memory straight into the operands of the matrix cores, past LDS.
// A workgroup takes a tile of at most 16 MT rows and 64 weight rows (gate and up: 32 columns of both); its four waves take a quarter of the
// contraction each and add their sums up in LDS, so that every wave has 16 KiB of weights on their way and a CU that holds two to
// four workgroups 128 to 256 (the kernel below has 16 a workgroup).  Top 4 of 32 experts, width 2048, ff 1024, 32 tokens: gate and up 66 -> 48.5 us
// (5.5 TB/s), down 28 -> 26.5 (5.1); the call with 1 token 47 -> 23.  Steps 32 deep for 64 rows, three workgroups a CU: 64 -> 75 us at 256 tokens.  Rows past the tile repeat its first one, weight rows past N the
// last one; neither is written.
template <int MODE, int MT>
__global__ __launch_bounds__(256, MT == 1 ? 4 : MT == 2 ? 3 : 2) void moe_rows_kernel(
    const __bf16* __restrict__ a, int64_t a_stride, const __bf16* __restrict__ w, const int* __restrict__ sorted_pairs,
    const int* __restrict__ meta, const float* __restrict__ pair_w, __bf16* __restrict__ y, float* __restrict__ out, int top, int N,
    int K, float limit, float alpha, float up_shift) {
    constexpr bool GATE_UP = MODE == 1, GATHER = MODE != 0;
    constexpr int NB = 4, COLS = GATE_UP ? 32 : 64;
    __shared__ f32x4 part[MT > 1 ? 2 : 1][4][NB][64];
    // An XCD takes a run of the items, the tiles of an expert next to each other: they read its weights once from memory.
    const int tiles = meta[0], n_cols = (N + COLS - 1) / COLS, items = tiles * n_cols, per_xcd = (items + 7) / 8, at = blockIdx.x / 8;
    const int item = (blockIdx.x & 7) * per_xcd + at;
    if (at >= per_xcd || item >= items) return;
    const int tile = item % tiles, n0 = (item / tiles) * COLS;
    const int e = meta[1 + 3 * tile], row0 = meta[2 + 3 * tile], rows = meta[3 + 3 * tile];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
    const int steps = K / 64, per = (steps + 3) / 4, s0 = min(wave * per, steps), s1 = min(s0 + per, steps);
    const __bf16* we = w + (int64_t)e * ((GATE_UP ? 2 : 1) * (int64_t)N) * K + s0 * 64 + 8 * g;
    const __bf16 *wp[NB], *xp[MT];
    int src[MT];                                      // on its way in front of the weights, which do not need it
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        src[m] = row0 + (m * 16 + l16 < rows ? m * 16 + l16 : 0);
        if constexpr (GATHER) src[m] = sorted_pairs[src[m]];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int64_t n = GATE_UP ? (j >> 1) * (int64_t)N + min(n0 + (j & 1) * 16 + l16, N - 1) : min(n0 + j * 16 + l16, N - 1);
        wp[j] = we + n * K;
    }
    f32x4 acc[MT][NB];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int D = 2;                              // a step: 64 deep, whole cache lines of every row
    struct Step {
        bf16x8 w[NB][D], x[MT][D];
    };
    auto load_w = [&](Step& f) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
#pragma unroll
            for (int i = 0; i < D; ++i) f.w[j][i] = *(const bf16x8*)(wp[j] + i * 32);
            wp[j] += 32 * D;
        }
    };
    auto load_x = [&](Step& f) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int i = 0; i < D; ++i) f.x[m][i] = *(const bf16x8*)(xp[m] + i * 32);
            xp[m] += 32 * D;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load = [&](Step& f) {
        load_w(f);
        load_x(f);
    };
    auto multiply = [&](const Step& f) {
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j][i], f.x[m][i], acc[m][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    Step f0, f1;
    int n = (s1 - s0) * (2 / D);
    if (n > 0) load_w(f0);
    if (n > 1) load_w(f1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; ++m) xp[m] = a + (int64_t)(GATHER ? src[m] / top : src[m]) * a_stride + s0 * 64 + 8 * g;
    if (n > 0) load_x(f0);
    if (n > 1) load_x(f1);
#pragma unroll 1
    for (; n > 3; n -= 2) {
        multiply(f0);
        load(f0);
        multiply(f1);
        load(f1);
    }
    if (n > 0) multiply(f0);
    if (n > 2) load(f0);
    if (n > 1) multiply(f1);
    if (n > 2) multiply(f0);
    // lane (l16, g) holds of row 16 m + l16 the weight rows 4 g + i of each block
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (m > 0 && m * 16 >= rows) break;           // (for the whole workgroup)
        auto& p = part[MT > 1 ? m & 1 : 0];
#pragma unroll
        for (int j = 0; j < NB; ++j) p[wave][j][lane] = acc[m][j];
        __syncthreads();                              // (the buffer's last reads lie in front of the barrier before)
        auto sum = [&](int j) { return (p[0][j][lane] + p[1][j][lane]) + (p[2][j][lane] + p[3][j][lane]); };
        const int r = m * 16 + l16, c = n0 + (GATE_UP ? wave & 1 : wave) * 16 + 4 * g;
        const bool live = r < rows && c < N && (!GATE_UP || wave < 2);
        if (!live) {
        } else if constexpr (GATE_UP) {
            const f32x4 gs = sum(wave), us = sum(wave + 2);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = moe_glu(gs[i], us[i], limit, alpha, up_shift);
            *(uint2*)(y + (int64_t)(row0 + r) * N + c) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        } else if constexpr (MODE == 2) {
            const f32x4 us = sum(wave);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float u = fmaxf(us[i], 0.f);
                v[i] = u * u;
            }
            *(uint2*)(y + (int64_t)(row0 + r) * N + c) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        } else {
            const int pair = sorted_pairs[row0 + r];
            *(f32x4*)(out + (int64_t)pair * N + c) = sum(wave) * pair_w[pair];
        }
    }
}

// MODE 1 (gate and up): A rows are gathered token rows, B holds the expert's gate rows and up rows, the epilogue is the
//         gated activation.
// MODE 2 (up alone):   A rows are gathered token rows, B the expert's up rows, the epilogue is max(x, 0)^2.
// MODE 0 (down):       A rows are the sorted activation rows, B the expert's down rows, the epilogue weights and scatters.
// The slices of the next step are fetched into registers while the current ones are multiplied out of LDS.
template <typename T, int MT, int NT, int MODE>
__global__ __launch_bounds__(256) void moe_grouped_kernel(
    const T* __restrict__ a, int64_t a_stride, const T* __restrict__ w, const int* __restrict__ sorted_pairs,
    const int* __restrict__ meta, const float* __restrict__ pair_w, T* __restrict__ y, float* __restrict__ out, int top,
    int N, int K, float limit, float alpha, float up_shift, int vec_ok, int max_tiles) {
    using M = TileMma<T>;
    constexpr bool GATE_UP = MODE == 1, GATHER = MODE != 0;
    constexpr int BK = M::kBK, BM = 16 * MT, BN = 64 * NT, NB = GATE_UP ? 2 : 1, LD = BK + M::kPad, KV = BK / M::kVec;
    constexpr int A_IT = (BM * KV + 255) / 256, B_IT = (NB * BN * KV + 255) / 256;
    __shared__ __attribute__((aligned(16))) T As[BM * LD];
    __shared__ __attribute__((aligned(16))) T Bs[NB * BN * LD];
    __shared__ int src_row[BM];                    // gathered rows: token of the row; else the pair of the row; -1 past the tile
    // Workgroups go to the chip's 8 XCDs (each with its own L2) round robin by their index: index i runs item
    // (i % 8) * (items / 8) + i / 8, so one XCD works through neighbouring row tiles -- the tiles of one expert, which
    // share their weight slices in that L2.  Items: row tile fastest, then the column block.
    const int items = gridDim.x, per_xcd = items / 8;
    int item = blockIdx.x;
    if (item < per_xcd * 8) item = (item % 8) * per_xcd + item / 8;
    const int tile = item % max_tiles, n0 = (item / max_tiles) * BN;
    if (tile >= meta[0]) return;
    const int e = meta[1 + 3 * tile], row0 = meta[2 + 3 * tile], rows = meta[3 + 3 * tile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lq = lane & 15, lg = lane >> 4;
    for (int i = tid; i < BM; i += 256) {
        const int pair = i < rows ? sorted_pairs[row0 + i] : -1;
        src_row[i] = pair < 0 ? -1 : (GATHER ? pair / top : pair);
    }
    __syncthreads();
    const T* we = w + (int64_t)e * (NB * (int64_t)N) * K;     // [NB * N, K] of this expert
    // what this thread stages: row pointers are fixed over the K loop
    const T* a_row[A_IT];
    const T* b_row[B_IT];
#pragma unroll
    for (int i = 0; i < A_IT; ++i) {
        const int it = tid + 256 * i, r = it / KV;
        a_row[i] = nullptr;
        if (it < BM * KV && r < rows) a_row[i] = GATHER ? a + (int64_t)src_row[r] * a_stride : a + (int64_t)(row0 + r) * a_stride;
    }
#pragma unroll
    for (int i = 0; i < B_IT; ++i) {
        const int it = tid + 256 * i, r = it / KV, n = n0 + (r % BN);
        b_row[i] = (it < NB * BN * KV && n < N) ? we + ((int64_t)(r / BN) * N + n) * K : nullptr;
    }
    uint4 a_reg[A_IT], b_reg[B_IT];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < A_IT; ++i) a_reg[i] = tile_fetch<T>(a_row[i], k0 + ((tid + 256 * i) % KV) * M::kVec, K, vec_ok != 0);
#pragma unroll
        for (int i = 0; i < B_IT; ++i) b_reg[i] = tile_fetch<T>(b_row[i], k0 + ((tid + 256 * i) % KV) * M::kVec, K, vec_ok != 0);
    };
    f32x4 acc[NB * NT][MT];
#pragma unroll
    for (int b = 0; b < NB * NT; ++b)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[b][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
        __syncthreads();                               // the previous slices have been consumed
#pragma unroll
        for (int i = 0; i < A_IT; ++i) {
            const int it = tid + 256 * i;
            if (it < BM * KV) *(uint4*)(As + (it / KV) * LD + (it % KV) * M::kVec) = a_reg[i];
        }
#pragma unroll
        for (int i = 0; i < B_IT; ++i) {
            const int it = tid + 256 * i;
            if (it < NB * BN * KV) *(uint4*)(Bs + (it / KV) * LD + (it % KV) * M::kVec) = b_reg[i];
        }
        __syncthreads();
        if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += M::kStep) {
#pragma unroll
            for (int b = 0; b < NB * NT; ++b) {      // b = (gate | up) * NT + column sub-tile of this wave
                const T* brow = Bs + ((b / NT) * BN + (wave * NT + b % NT) * 16 + lq) * LD + kk;
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[b][m] = M::run(As + (m * 16 + lq) * LD + kk, brow, lg, acc[b][m]);
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + (wave * NT + nt) * 16 + lq;
        if (n >= N) continue;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = m * 16 + 4 * lg + i;
                if (r >= rows) continue;
                if constexpr (GATE_UP) {
                    y[(int64_t)(row0 + r) * N + n] = (T)moe_glu(acc[nt][m][i], acc[NT + nt][m][i], limit, alpha, up_shift);
                } else if constexpr (MODE == 2) {
                    const float u = fmaxf(acc[nt][m][i], 0.f);
                    y[(int64_t)(row0 + r) * N + n] = (T)(u * u);
                } else {
                    const int pair = src_row[r];
                    out[(int64_t)pair * N + n] = acc[nt][m][i] * pair_w[pair];
                }
            }
        }
    }
}

// Tiles of 32 and 128 rows are for whole 64-deep slices and 16-byte pieces of the rows and weights that they are suggested for.
static bool moe_pieces_ok(int dtype, const void* a, int64_t a_stride, const void* w, int N, int K) {
    return dtype == NV_DTYPE_BF16 && K % 64 == 0 && N % 8 == 0 && a_stride % 8 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
}

// Offsets from the first row and from the expert's first weight row are 32 bits in bytes, 64 deep; an input or an expert's matrix of 4 GiB takes
// slices 32 deep by address.
static bool moe_offsets_ok(int64_t a_rows, int64_t a_stride, int64_t w_rows, int K) {
    return a_rows * a_stride < (1LL << 31) - K && w_rows * K < (1LL << 31) - K;
}

template <typename T, int MODE>
static void launch_grouped(const void* a, int64_t a_stride, const void* w, const int* sorted_pairs, const int* meta,
                           const float* pair_w, void* y, float* out, int top, int N, int K, float limit, float alpha,
                           float up_shift, int64_t pairs, int E, int tile_rows, int64_t a_rows, hipStream_t s) {
    const int max_tiles = (int)nv_moe_max_tiles(pairs, E, tile_rows);
    // activations and outputs that do not start on 16 bytes take the general launch, in tiles of any size
    const bool pieces = sizeof(T) == 2 && (MODE == 0 ? (uintptr_t)out : (uintptr_t)y) % 16 == 0 && moe_pieces_ok(NV_DTYPE_BF16, a, a_stride, w, N, K);
    if constexpr (sizeof(T) == 2) {
        if (pieces && tile_rows == kMoeBigRows) {
            constexpr int cols = MODE == 1 ? 128 : 256;
            const int n_cols = (N + cols - 1) / cols;
            const dim3 grid((unsigned)(((int64_t)max_tiles * n_cols + 7) / 8 * 8));
#define NV_MOE_BIG(D, STREAM)                                                                                                            \
    hipLaunchKernelGGL((moe_big_kernel<MODE, D, STREAM>), grid, dim3(256), 0, s, (const T*)a, a_stride, (const T*)w, sorted_pairs, meta, pair_w, \
                       (T*)y, out, top, N, K, limit, alpha, up_shift)
            if (moe_few_blocks(pairs, E, n_cols) || !moe_offsets_ok(MODE == 0 ? kMoeBigRows : a_rows, a_stride, (MODE == 1 ? 2 : 1) * (int64_t)N, K))
                NV_MOE_BIG(32, false);
            else if (MODE == 0 && moe_streams_out(pairs, N, E, K))
                NV_MOE_BIG(64, MODE == 0);
            else
                NV_MOE_BIG(64, false);
#undef NV_MOE_BIG
            return;
        }
    }
    if constexpr (sizeof(T) == 2) {
        if (pieces && moe_streams(tile_rows, pairs, E, MODE == 0 ? K : N)) {
            const int64_t items = (int64_t)max_tiles * ((N + (MODE == 1 ? 31 : 63)) / (MODE == 1 ? 32 : 64));
#define NV_MOE_ROWS(MT)                                                                                                              \
    hipLaunchKernelGGL((moe_rows_kernel<MODE, MT>), dim3((unsigned)((items + 7) / 8 * 8)), dim3(256), 0, s, (const T*)a, a_stride, (const T*)w, \
                       sorted_pairs, meta, pair_w, (T*)y, out, top, N, K, limit, alpha, up_shift)
            if (tile_rows == 64) NV_MOE_ROWS(4);
            else if (tile_rows == 32) NV_MOE_ROWS(2);
            else NV_MOE_ROWS(1);
#undef NV_MOE_ROWS
            return;
        }
    }
    const int vec = TileMma<T>::kVec;
    const int vec_ok = K % vec == 0 && a_stride % vec == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
    // many rows per expert: 64 x 128 tiles (a wave owns 32 columns; 128 rows of this kernel measured slower: one workgroup per CU);
    // few: 16 x 64 tiles, more workgroups per weight byte
#define NV_MOE_LAUNCH(MT, NT)                                                                                          \
    hipLaunchKernelGGL((moe_grouped_kernel<T, MT, NT, MODE>), dim3((unsigned)(max_tiles * ((N + 64 * NT - 1) / (64 * NT)))), \
                       dim3(256), 0, s, (const T*)a, a_stride, (const T*)w, sorted_pairs, meta, pair_w, (T*)y, out, top, N, K,  \
                       limit, alpha, up_shift, vec_ok, max_tiles)
    if constexpr (sizeof(T) == 2) {
        if (tile_rows == kMoeBigRows || tile_rows == 32) {
            if (tile_rows == 32) NV_MOE_LAUNCH(2, 1);
            else NV_MOE_LAUNCH(8, 1);
            return;
        }
    }
    if (tile_rows == 64 && sizeof(T) == 2) NV_MOE_LAUNCH(4, 2);
    else if (tile_rows == 64) NV_MOE_LAUNCH(4, 1);
    else NV_MOE_LAUNCH(1, 1);
#undef NV_MOE_LAUNCH
}

}  // namespace nv

extern "C" int nv_moe_route(const float* logits, int32_t* ids, float* weights, int64_t T, int E, int top, void* stream) {
    using namespace nv;
    NV_REQUIRE(T >= 0 && E > 0 && top >= 1 && top <= E && top <= kMoeMaxTop, NV_ERR_INVALID_ARG,
               "nv_moe_route: top=%d must lie in 1 .. min(E=%d, %d)", top, E, kMoeMaxTop);
    if (T == 0) return NV_OK;
    NV_REQUIRE(logits && ids && weights, NV_ERR_INVALID_ARG, "nv_moe_route: null pointer");
    NV_REQUIRE((T + 3) / 4 < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_route: launch too large");
    if (E <= 64) hipLaunchKernelGGL(moe_route_kernel<1>, dim3((unsigned)((T + 15) / 16)), dim3(256), 0, (hipStream_t)stream, logits, ids, weights, T, E, top);
    else
        hipLaunchKernelGGL(moe_route_kernel<kMoeRoutePerLane>, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, (hipStream_t)stream, logits, ids,
                           weights, T, E, top);
    return check_launch("nv_moe_route");
}

extern "C" int nv_moe_tile_rows(int64_t pairs, int E) { return pairs >= 32 * (int64_t)E ? 64 : 16; }

// By pairs per expert: tiles of 16 rows below 8, of 32 below 21, of 64 (all of these stream the weights past LDS, which costs little more with
// more rows a tile and saves the second reading of an expert that has more), then of 128 staged through LDS, which wants enough of its
// 128 x 256 blocks to fill the chip.  Whole calls, us, tiles of 16 / 32 / 64 / 128 rows:
//   top 4 of 32 experts, width 2048, ff 1024:  6 pairs an expert 83 / 86 / 89 / 108, 16: 107 / 96 / 101 / 113, 24: 134 / 107 / 105 / 115,
//   32: 149 / 121 / 112 / 116, 40: 174 / 142 / 118 / 117, 64: 252 / 178 / 156 / 123
//   top 2 of 32, 1024, 1024:  16: 53 / 48 / 51 / 54, 32: 78 / 63 / 57 / 56, 48: 105 / 79 / 65 / 59
//   top 2 of 16, 1024, 512:  6: 18 / 18 / 20 / 38, 24: 27 / 29 / 25 / 40, 64: 47 / 39 / 39 / 42, 96: 61 / 52 / 40 / 42, 128: 73 / 58 / 59 / 45
//   top 4 of 16, 2048, 512:  12: 36 / 30 / 30 / 53, 48: 66 / 51 / 39 / 57, 96: 104 / 83 / 64 / 59
// It is the first expert with more rows than a tile that decides, so routings differ, and more experts have one earlier.  Both products, us:
//   tiles of 32 / 64: 16 of 2048, 1024:  20: 41 / 44, 23 with one of 33 rows: 56 / 45
//   tiles of 64 in four routings and of 128:  16 of 2048, 1024:  48: 53, 53, 52, 54 and 57, 52: 67, 54, 54, 70 and 57, 56: 69, 72, 73, 72 and 57
//     32 of 1024, 512:  44: 34, 33, 34, 34 and 37, 48: 43, 34, 34, 41 and 37;  32 of 2048, 512:  48: 69, 57, 59, 68 and 56
// Short rows of many blocks, from 21 to 31 pairs: 16-row tiles through LDS, 32 of 1024, 1024:  24: 40 us, tiles of 64 47 (weights from memory 50 and 51).
extern "C" int nv_moe_tile_rows_for(int64_t pairs, int E, int width, int ff, const void* h, int64_t h_stride, const void* up,
                                    const void* down, int dtype) {
    using namespace nv;
    if (!moe_pieces_ok(dtype, h, h_stride, up, ff, width) || !moe_pieces_ok(dtype, nullptr, ff, down, width, ff)) return nv_moe_tile_rows(pairs, E);
    const int64_t blocks = (int64_t)E * ((ff + 127) / 128);           // of the first product, a tile an expert
    if (pairs >= (blocks >= 256 ? 40 : blocks < 128 ? 84 : E < 32 ? 52 : 48) * (int64_t)E) return kMoeBigRows;
    if (pairs >= 21 * (int64_t)E) return blocks >= 256 && width <= 1024 && pairs < 32 * (int64_t)E ? 16 : 64;
    return pairs >= 8 * (int64_t)E ? 32 : 16;
}

extern "C" int64_t nv_moe_max_tiles(int64_t pairs, int E, int tile_rows) {
    return pairs / tile_rows + std::min<int64_t>(pairs, E);
}

static bool moe_tile_ok(int rows) { return rows == 16 || rows == 32 || rows == 64 || rows == 128; }

extern "C" int nv_moe_align(const int32_t* ids, int32_t* sorted_pairs, int32_t* meta, int64_t pairs, int E,
                            int tile_rows, void* stream) {
    using namespace nv;
    NV_REQUIRE(pairs >= 0 && E > 0 && E <= 4096 && moe_tile_ok(tile_rows), NV_ERR_INVALID_ARG,
               "nv_moe_align: bad sizes");
    NV_REQUIRE(ids && sorted_pairs && meta, NV_ERR_INVALID_ARG, "nv_moe_align: null pointer");
    NV_REQUIRE(pairs < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_align: too many pairs");
    const size_t tables = sizeof(int) * 2 * ((size_t)E + 1);
    // few pairs: one table, since joining the copies then costs more than the additions (128 pairs: 0.6 us of the whole call)
    if (E <= 512 && pairs >= 4096)
        hipLaunchKernelGGL(moe_align_kernel<16>, dim3(1), dim3(1024), sizeof(int) * 16 * (size_t)E + tables, (hipStream_t)stream, ids,
                           sorted_pairs, meta, pairs, E, tile_rows);
    else
        hipLaunchKernelGGL(moe_align_kernel<1>, dim3(1), dim3(1024), sizeof(int) * (size_t)E + tables, (hipStream_t)stream, ids,
                           sorted_pairs, meta, pairs, E, tile_rows);
    return check_launch("nv_moe_align");
}

// Tokens of a workgroup of the first launch.  Beyond 64 experts a wave's next token costs a microsecond a choice, and a workgroup more
// costs every workgroup of the second launch E counts, about a microsecond for 5200.
static int moe_sort_tokens(int64_t T, int E, int top) {
    const int whole = nv::moe_sort_least(E);
    int64_t n = (T + nv::kMoeSortGroups - 1) / nv::kMoeSortGroups;
    n = (n + whole - 1) / whole * whole;
    while (E > 64 && n * n * top * 1300 < T * E) n += whole;
    return (int)n;
}
extern "C" int64_t nv_moe_route_sort_words(int64_t T, int E) {
    if (T <= nv::moe_sort_few(E) || E > nv::kMoeSortMaxE) return 0;
    const int tokens = moe_sort_tokens(T, E, nv::kMoeMaxTop);         // (the most workgroups of any number of choices)
    return (T + tokens - 1) / tokens * E;
}
extern "C" int nv_moe_route_sort(const float* logits, int32_t* ids, float* weights, int32_t* sorted_pairs, int32_t* meta, int32_t* counts,
                                 int64_t T, int E, int top, int tile_rows, void* stream) {
    using namespace nv;
    NV_REQUIRE(T >= 0 && E > 0 && top >= 1 && top <= E && top <= kMoeMaxTop && moe_tile_ok(tile_rows), NV_ERR_INVALID_ARG,
               "nv_moe_route_sort: top=%d must lie in 1 .. min(E=%d, %d), tiles have 16, 32, 64 or 128 rows", top, E, kMoeMaxTop);
    if (T == 0 || E > kMoeSortMaxE) {
        const int rc = nv_moe_route(logits, ids, weights, T, E, top, stream);
        return rc != NV_OK ? rc : nv_moe_align(ids, sorted_pairs, meta, T * top, E, tile_rows, stream);
    }
    NV_REQUIRE(logits && ids && weights && sorted_pairs && meta && (counts || T <= moe_sort_few(E)), NV_ERR_INVALID_ARG, "nv_moe_route_sort: null pointer");
    NV_REQUIRE(T * top < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_route_sort: too many pairs");
    hipStream_t s = (hipStream_t)stream;
    if (T <= moe_sort_few(E)) {
        if (E <= 64)
            hipLaunchKernelGGL(moe_route_sort_few_kernel<1>, dim3(1), dim3(1024), 0, s, logits, ids, weights, sorted_pairs, meta, (int)T, E, top, tile_rows);
        else
            hipLaunchKernelGGL(moe_route_sort_few_kernel<kMoeRoutePerLane>, dim3(1), dim3(1024), 0, s, logits, ids, weights, sorted_pairs, meta,
                               (int)T, E, top, tile_rows);
        return check_launch("nv_moe_route_sort");
    }
    const int tokens = moe_sort_tokens(T, E, top);
    const unsigned groups = (unsigned)((T + tokens - 1) / tokens);
    int columns = 16;
    while (columns < E && columns < 256) columns *= 2;
    if (E <= 64) hipLaunchKernelGGL(moe_route_count_kernel<1>, dim3(groups), dim3(256), 0, s, logits, ids, weights, counts, T, E, top, tokens);
    else
        hipLaunchKernelGGL(moe_route_count_kernel<kMoeRoutePerLane>, dim3(groups), dim3(256), 0, s, logits, ids, weights, counts, T, E, top, tokens);
    hipLaunchKernelGGL(moe_place_kernel, dim3(groups), dim3(256), 0, s, ids, counts, sorted_pairs, meta, T * top, E, tile_rows, tokens * top, columns);
    return check_launch("nv_moe_route_sort");
}

extern "C" int nv_moe_gate_up(const void* h, int64_t h_stride, const void* gate_up, const int32_t* sorted_pairs,
                              const int32_t* meta, void* y, int dtype, int64_t pairs, int E, int top, int width, int ff,
                              float limit, float alpha, int tile_rows, void* stream) {
    return nv_moe_gate_up_act(h, h_stride, gate_up, sorted_pairs, meta, y, dtype, pairs, E, top, width, ff, limit, alpha,
                              1.0f, tile_rows, stream);
}

extern "C" int nv_moe_gate_up_act(const void* h, int64_t h_stride, const void* gate_up, const int32_t* sorted_pairs,
                                  const int32_t* meta, void* y, int dtype, int64_t pairs, int E, int top, int width,
                                  int ff, float limit, float alpha, float up_shift, int tile_rows, void* stream) {
    using namespace nv;
    NV_REQUIRE(pairs >= 0 && E > 0 && top > 0 && width > 0 && ff > 0 && moe_tile_ok(tile_rows),
               NV_ERR_INVALID_ARG, "nv_moe_gate_up: bad sizes");
    if (pairs == 0) return NV_OK;
    NV_REQUIRE(h && gate_up && sorted_pairs && meta && y, NV_ERR_INVALID_ARG, "nv_moe_gate_up: null pointer");
    NV_REQUIRE(dtype == NV_DTYPE_BF16 || dtype == NV_DTYPE_F32, NV_ERR_INVALID_ARG, "nv_moe_gate_up: bad dtype");
    NV_REQUIRE((tile_rows != 128 && tile_rows != 32) || moe_pieces_ok(dtype, h, h_stride, gate_up, ff, width), NV_ERR_UNSUPPORTED,
               "nv_moe_gate_up: tiles of 32 or 128 rows take bf16 rows in whole pieces");
    const int64_t tiles = nv_moe_max_tiles(pairs, E, tile_rows);
    NV_REQUIRE(tiles * ((ff + kMoeBN - 1) / kMoeBN) < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_gate_up: launch too large");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == NV_DTYPE_BF16)
        launch_grouped<__bf16, 1>(h, h_stride, gate_up, sorted_pairs, meta, nullptr, y, nullptr, top, ff, width, limit,
                                     alpha, up_shift, pairs, E, tile_rows, pairs / top, s);
    else
        launch_grouped<float, 1>(h, h_stride, gate_up, sorted_pairs, meta, nullptr, y, nullptr, top, ff, width, limit,
                                    alpha, up_shift, pairs, E, tile_rows, pairs / top, s);
    return check_launch("nv_moe_gate_up");
}

extern "C" int nv_moe_down(const void* y, const void* down, const int32_t* sorted_pairs, const int32_t* meta,
                           const float* pair_weights, float* out, int dtype, int64_t pairs, int E, int width, int ff,
                           int tile_rows, void* stream) {
    using namespace nv;
    NV_REQUIRE(pairs >= 0 && E > 0 && width > 0 && ff > 0 && moe_tile_ok(tile_rows), NV_ERR_INVALID_ARG,
               "nv_moe_down: bad sizes");
    if (pairs == 0) return NV_OK;
    NV_REQUIRE(y && down && sorted_pairs && meta && pair_weights && out, NV_ERR_INVALID_ARG, "nv_moe_down: null pointer");
    NV_REQUIRE(dtype == NV_DTYPE_BF16 || dtype == NV_DTYPE_F32, NV_ERR_INVALID_ARG, "nv_moe_down: bad dtype");
    NV_REQUIRE((tile_rows != 128 && tile_rows != 32) || moe_pieces_ok(dtype, nullptr, ff, down, width, ff), NV_ERR_UNSUPPORTED,
               "nv_moe_down: tiles of 32 or 128 rows take bf16 rows in whole pieces");
    const int64_t tiles = nv_moe_max_tiles(pairs, E, tile_rows);
    NV_REQUIRE(tiles * ((width + kMoeBN - 1) / kMoeBN) < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_down: launch too large");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == NV_DTYPE_BF16)
        launch_grouped<__bf16, 0>(y, ff, down, sorted_pairs, meta, pair_weights, nullptr, out, 1, width, ff, 0.f, 0.f, 0.f,
                                      pairs, E, tile_rows, pairs, s);
    else
        launch_grouped<float, 0>(y, ff, down, sorted_pairs, meta, pair_weights, nullptr, out, 1, width, ff, 0.f, 0.f, 0.f,
                                     pairs, E, tile_rows, pairs, s);
    return check_launch("nv_moe_down");
}

extern "C" int nv_moe_route_grouped(const float* logits, const float* correction, int32_t* ids, float* weights, int64_t T,
                                    int E, int top, int n_groups, int keep_groups, void* stream) {
    using namespace nv;
    NV_REQUIRE(T >= 0 && E > 0 && E <= kMoeGroupedMaxE && top >= 1, NV_ERR_INVALID_ARG,
               "nv_moe_route_grouped: E=%d must lie in 1 .. %d", E, kMoeGroupedMaxE);
    NV_REQUIRE(n_groups >= 1 && E % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups, NV_ERR_INVALID_ARG,
               "nv_moe_route_grouped: %d groups must divide E=%d and hold the %d kept", n_groups, E, keep_groups);
    NV_REQUIRE(top <= keep_groups * (E / n_groups), NV_ERR_INVALID_ARG,
               "nv_moe_route_grouped: top=%d exceeds the %d experts of the kept groups", top, keep_groups * (E / n_groups));
    if (T == 0) return NV_OK;
    NV_REQUIRE(logits && ids && weights, NV_ERR_INVALID_ARG, "nv_moe_route_grouped: null pointer");
    NV_REQUIRE(T < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_route_grouped: launch too large");
    hipLaunchKernelGGL(moe_route_grouped_kernel, dim3((unsigned)T), dim3(64), 0, (hipStream_t)stream, logits, correction, ids,
                       weights, E, top, n_groups, keep_groups);
    return check_launch("nv_moe_route_grouped");
}

extern "C" int nv_moe_up_relu2(const void* h, int64_t h_stride, const void* up, const int32_t* sorted_pairs,
                               const int32_t* meta, void* y, int dtype, int64_t pairs, int E, int top, int width, int ff,
                               int tile_rows, void* stream) {
    using namespace nv;
    NV_REQUIRE(pairs >= 0 && E > 0 && top > 0 && width > 0 && ff > 0 && moe_tile_ok(tile_rows),
               NV_ERR_INVALID_ARG, "nv_moe_up_relu2: bad sizes");
    if (pairs == 0) return NV_OK;
    NV_REQUIRE(h && up && sorted_pairs && meta && y, NV_ERR_INVALID_ARG, "nv_moe_up_relu2: null pointer");
    NV_REQUIRE(dtype == NV_DTYPE_BF16 || dtype == NV_DTYPE_F32, NV_ERR_INVALID_ARG, "nv_moe_up_relu2: bad dtype");
    NV_REQUIRE((tile_rows != 128 && tile_rows != 32) || moe_pieces_ok(dtype, h, h_stride, up, ff, width), NV_ERR_UNSUPPORTED,
               "nv_moe_up_relu2: tiles of 32 or 128 rows take bf16 rows in whole pieces");
    const int64_t tiles = nv_moe_max_tiles(pairs, E, tile_rows);
    NV_REQUIRE(tiles * ((ff + kMoeBN - 1) / kMoeBN) < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_up_relu2: launch too large");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == NV_DTYPE_BF16)
        launch_grouped<__bf16, 2>(h, h_stride, up, sorted_pairs, meta, nullptr, y, nullptr, top, ff, width, 0.f, 0.f, 0.f,
                                  pairs, E, tile_rows, pairs / top, s);
    else
        launch_grouped<float, 2>(h, h_stride, up, sorted_pairs, meta, nullptr, y, nullptr, top, ff, width, 0.f, 0.f, 0.f,
                                 pairs, E, tile_rows, pairs / top, s);
    return check_launch("nv_moe_up_relu2");
}

extern "C" int nv_moe_route_softmax(const float* logits, const float* correction, int32_t* ids, float* weights, int64_t T,
                                    int E, int top, float scale, void* stream) {
    using namespace nv;
    NV_REQUIRE(T >= 0 && E > 0 && E <= kMoeSoftmaxMaxE, NV_ERR_INVALID_ARG, "nv_moe_route_softmax: E=%d must lie in 1 .. %d",
               E, kMoeSoftmaxMaxE);
    NV_REQUIRE(top >= 1 && top <= E, NV_ERR_INVALID_ARG, "nv_moe_route_softmax: top=%d must lie in 1 .. E=%d", top, E);
    if (T == 0) return NV_OK;
    NV_REQUIRE(logits && ids && weights, NV_ERR_INVALID_ARG, "nv_moe_route_softmax: null pointer");
    NV_REQUIRE(T < (1LL << 31), NV_ERR_UNSUPPORTED, "nv_moe_route_softmax: launch too large");
    hipLaunchKernelGGL(moe_route_softmax_kernel, dim3((unsigned)T), dim3(64), 0, (hipStream_t)stream, logits, correction, ids,
                       weights, E, top, scale);
    return check_launch("nv_moe_route_softmax");
}
