// Recurrences whose memory S [D, Dv] (key channel x value channel, fp32) decays with one factor per key channel and is
// rewritten along its own read-out.  Three forms; x0 .. x3 are the raw projections, everything after them is fp32:
//
//   gated    (x0 = q, x1 = k, x2 = a_raw)   k, q unit vectors (q times D^-1/2);  w = exp(-exp(c0_h) softplus(x2 + c1))
//            S <- diag(w) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//   general  (x0 = r, x1 = k, x2 = w_raw, x3 = a_raw)   u = k / |k|;  w = exp(-p0 sigmoid(x2 + c0));  a = sigmoid(x3 + c1)
//            S <- diag(w) S - (a u)(u^T S) + k v^T  (both terms read the old state);  o = S^T r
//   write    (x0 = q, x1 = f_raw)   w = c1 + (1 - c1) sigmoid(x1 + c0);  k = 1 - w;  S <- diag(w) S + k v^T;  o = S^T silu(q)
//
// A token-by-token loop is bound by its serial chain (one pass over the state a token and the LDS reads of the token's vectors
// by every lane), so portions run in CHUNKS, of 16 tokens here.  With G_t the product of the decays from the chunk's start through
// token t, and S the state in front of the chunk, each form is
//
//   C = K S, Q S         what the tokens' k and q (r) find in S: K_t = k_t G_t (general: k_t G_(t-1)), Q_t = q_t G_t, 16 rows each
//   U = T (V - K S)      gated; general: U = T (K S + PK V); write has none: the tokens' influence on each other, solved
//   O = Q S + PQ U       (general: + PV V; write: PV V alone)
//   S <- diag(G_16) S + K^^T V (general, write) + X^^T U (gated, general),   K^_t = k_t G_16 / G_t
//
// T is the inverse of a unit lower triangular 16 x 16 matrix by forward substitution, with the tokens' factors on either side; PQ, PV
// and PK are lower triangles; all come from the pair products P_ts = sum_d l_t,d r_s,d G_t / G_s, s <= t.  Gated keys and queries are
// scaled to unit length on their way into K, Q and X^, so that V - K S needs no factors.  All large products are
// v_mfma_f32_16x16x4_f32: operands and sums stay fp32.
//
// A zero of a triangle keeps a token's row out of a product only while the row is finite.  Where a chunk holds a value that is not, its
// sequence and head take these products token by token, so that no earlier token and, from q, no state sees it.
//
// G_t / G_s does not factor through one reference without overflow when a channel decays fast.  Both sides are taken relative to
// the middle of the chunk, eight factors on either side, where no channel of the chunk has eight that multiply to less than 2^-80 (a
// right side then keeps its 24 bits down to 2^-46 of the raw key).  Other chunks take the pairs in sets by where s and t part: in
// halves, quarters, eighths or neighbours of the chunk, each relative to the boundary between the two, where every factor is a decay
// and nothing is divided, and s = t; two sets, pairs across the halves and within a half relative to the half's middle, where no four
// factors multiply to less than 2^-80.  A chunk and head decide by themselves.  Gated, 16 prompts of 300 .. 500 tokens, 16 heads
// 128 x 128, a channel of every head at exp(-8) a token: 222 us with one set for all, 228 with two, 258 with five.
//
// Two launches: the first makes every chunk's operands (two waves per chunk and head, all chunks at once), the second walks the
// chunks of a (sequence, head, 16 value columns) with the state in MFMA accumulators (128 channels: 32 registers) and reads the
// operands from memory in the order of its lanes.  Operands prepared beside the products (one launch, everything through LDS) took the
// same issue slots: 653 us instead of 286 on gated, 4 prompts of 1501 .. 2048 tokens, 16 heads 128 x 128, in chunks of 8.
// Accumulators of one product are the operand of the next in place: a lane holds rows 4 g + e (g: its group of 16 lanes), so
// MFMA e of a tile contracts the four rows {4 g + e}, and the other operand is read in that order (16 bytes a lane); U, 16 rows, fills
// all four groups.  The chunk takes 104 (gated) / 144 (general) / 68 (write) MFMAs of 32 cycles per 16 columns of 128 channels.
//
// Why 16 tokens: the products per token are those of chunks of 8 (chunk_recurrence_short.hip, which short portions and full grids still
// take: `cr_chunk_tokens`), but a chunk's chain of exchange, triangle and update is paid half as often, and Q S, which no other product
// waits for, is multiplied while the parts of K S are exchanged.  Whole calls, chunks of 8 against 16, 16 heads 128 x 128, bf16 rows:
// gated, 4 prompts of 1501 .. 2048 tokens 285 -> 248 us; general, 3 prompts of 700 .. 2000: 286 -> 266; write, 8 portions of 509 over
// carried states: 114 -> 96, one prompt of 2048: 197 -> 119.  Token by token: gated 3123, general 3645, write 431; gated, 256 single
// tokens, the states of three layers in turn: 393 -> 113, and 99 past the caches (5.4 TB/s of states).
// In a profile of the 248-us call (286 us there) the first launch is 82 us, the second 177, 128 chunks in a row at 1.38 us: 0.83 us of MFMAs
// (15.3 ns each, back to back), the rest LDS latency and the chain; the read-outs' norm is 26.  Tried and slower: all large products as six bf16 products of three parts each, split by the
// movers (198 us for the second launch: the LDS traffic of the parts; 144 without them), the same for the updates alone (176), four
// waves a state on eight product waves (180).
//
// Against 64 bits (float32 rows, 64 and 128 channels, 8 to 1000 tokens a sequence, fresh and carried states), relative to the
// token-by-token launch: states gated 0.88 to 0.96 times its error, general 1.03 to 1.13, write 0.99 to 1.00; read-outs 0.91 to 1.06,
// 0.98 to 1.08 and 1.01 to 1.09 (a read-out near zero aside, which its norm blows up in either).  Three things keep them there.
// Decays are multiplied in 64 bits and each product is rounded once, where 15 roundings in a row are 15 factors of one channel's error.
// Sums over all key channels have their roundings one after the other, so C is four sums and a pair product eight (four: read-outs 2 to
// 5 % further off).  The removals of the general form are summed by themselves: on top of the state each of 16 terms is rounded at
// the state's size (states 1.35 to 1.67 times the token-by-token launch's error).  Of bf16 read-outs, which are 1.7e-3 off by their own
// rounding, none of it shows.
//
// The read-outs go to a scratch of fp32 rows, because a row's norm spans the workgroups of its value columns; a last launch
// norms, weights and gates them.  Single tokens run in a launch of their own that streams every state once.
#include <algorithm>

#include "chunk_recurrence_parts.h"
#include "launch_order.h"
#include "../../include/nanovllm_hip_mixers.h"

namespace nv {

constexpr int kCrChunk = 16;
// Where a chunk's operands lie in the workspace: one record per (head, chunk), in the order in which the lanes of the second
// launch read them, a head's chunks one after the other, beside them the chunks' rows of V ([head][record][16][Dv], zeros past the
// sequence's end); read-outs are [head][row][Dv] too.  The second launch has few loads in flight, so streams that stay within a page
// for several chunks matter to it (heads side by side, every chunk on pages of its own: 302 us instead of 264, chunks of 8).
template <int FORM, int D>
struct CrRecord {
    static constexpr int kRows = FORM == kCrWrite ? 16 : 32;      // of [K; Q]: write has no K
    static constexpr int kUpd = FORM == kCrGeneral ? 2 : 1;       // update operands: K^ and / or X^
    static constexpr int kMat = FORM == kCrWrite ? 1 : FORM == kCrGated ? 2 : 4;      // gated: T, PQ; general: T, PQ, PV, PK; write: PV
    static constexpr int kq = 0;                                  // [K, Q][tile][g][row][4 channels]
    static constexpr int upd = kq + kRows * D;                    // [operand][tile][g][channel][4 tokens]
    static constexpr int decay = upd + kUpd * 16 * D;             // [channel]
    static constexpr int m = decay + D;                           // [matrix][16][16]
    static constexpr int words = m + kMat * 256;
};
// ------------------------------------------------------------------------------------------------ first launch
// Two waves per (chunk, head), eight tokens each; a lane owns two neighbouring channels of its eight tokens, so running products need
// no exchange but of the halves' totals.  LDS turns the pair products' operands, K and Q into the order of the matrix cores; one wave
// multiplies the rows K and solves for T, the other one multiplies the rows Q.  One wave with all 16 tokens spills registers (general:
// 95 us where this takes 70, 3 prompts of 700 .. 2000 tokens; gated 88 and 83).
template <int D>
struct CrPrepLds {
    static constexpr int kRow = D + 4;                            // rows of D channels start on different banks
    float k[16 * kRow], q[16 * kRow], right[16 * kRow];           // left sides, then [K; Q]; right sides, then the halves' decays
    float kn[16], qn[16], beta[16];
    uint32_t odd[2], far[2];
};

template <typename T, int FORM, int D, bool VEC>
__global__ __launch_bounds__(128, FORM == kCrGeneral ? 2 : 3) void recurrence_chunks_kernel(const ChunkRecurrenceArgs a, const int first_seq) {
    constexpr int NM = D / 16, NX = FORM == kCrGated ? 3 : FORM == kCrGeneral ? 4 : 2, L = kCrChunk, N = L / 2;
    constexpr bool HAS_K = FORM != kCrWrite;
    typedef CrPrepLds<D> Lds;
    typedef CrRecord<FORM, D> Rec;
    typedef CrRaw<T> In;
    constexpr int ROW = Lds::kRow;
    __shared__ __attribute__((aligned(16))) Lds lds;
    const int lane = threadIdx.x & 63, half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4, h = blockIdx.y;
    const int64_t rec = blockIdx.x;
    const int row0 = a.cu_q[first_seq];
    int lo = first_seq, hi = a.num_seqs;              // the last sequence whose records start at or in front of this one
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cr_first_record<kCrChunk>(a.cu_q[mid] - row0, mid - first_seq) <= rec) lo = mid; else hi = mid;
    }
    const int b = lo, q0 = a.cu_q[b], len = a.cu_q[b + 1] - q0;
    const int64_t c64 = rec - cr_first_record<kCrChunk>(q0 - row0, b - first_seq);
    if (len < 2 || c64 * L >= len) return;            // (for the whole workgroup)
    const int t0 = q0 + (int)c64 * L, n16 = min(L, q0 + len - t0), n = min(N, max(n16 - half * N, 0)), th = half * N;
    float* out = a.chunks + (h * a.records + rec) * Rec::words;

    const bool in_row = D == 128 || 2 * lane < D;
    const int d = in_row ? 2 * lane : 0;
    CrPair<T, VEC> raw[NX][N];
    {
        const void* xs[4] = {a.x0, a.x1, a.x2, a.x3};
        const int64_t ss[4] = {a.s0, a.s1, a.s2, a.s3};
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int hj = (FORM == kCrGated && j < 2) ? h / a.group : h;
            const T* p = (const T*)xs[j] + (int64_t)t0 * ss[j] + (int64_t)hj * D;
#pragma unroll
            for (int t = 0; t < N; ++t) {             // (past the end: the chunk's first row, dropped below)
                const T* row = p + (t < n ? th + t : 0) * ss[j];
                raw[j][t].load(row + d);
            }
        }
    }
    float odd[4] = {};                                // NaN with a value that is not finite
    {
        const T* v = (const T*)a.v + (int64_t)t0 * a.sv + (int64_t)h * a.Dv;
        T* to = (T*)a.columns + ((h * a.records + rec) * L + th) * a.Dv;
        for (int c = 2 * lane; c < a.Dv; c += 128) {
            CrPair<T, VEC> r[N];
#pragma unroll
            for (int t = 0; t < N; ++t) r[t].load(v + (t < n ? th + t : 0) * a.sv + c);
#pragma unroll
            for (int t = 0; t < N; ++t) {
                r[t].keep(t < n);
                r[t].store(to + t * a.Dv + c);
                odd[t & 3] = fmaf(r[t].value(0), 0.f, odd[t & 3]);
                odd[t & 3] = fmaf(r[t].value(1), 0.f, odd[t & 3]);
            }
        }
    }
    float beta = 0.f;                                 // raw, of token lane % 8
    if constexpr (FORM == kCrGated)
        beta = CrRaw<T>::value(In::load((const T*)a.b_raw + (int64_t)(t0 + min(th + (lane & 7), n16 - 1)) * a.b_stride + h));
    float c0[2], c1[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        c0[i] = FORM == kCrGated ? expf(a.c0[h]) : a.c0[h * D + d + i];
        c1[i] = a.c1[h * D + d + i];
    }
    // Per token and channel: decay, and what else is not the raw projection itself (write: q; general: a k).
    float w[N][2], made[FORM == kCrGated ? 1 : N][2];
#pragma unroll
    for (int t = 0; t < N; ++t) {
#pragma unroll
        for (int j = 0; j < NX; ++j)
            if (HAS_K && j < 2) raw[j][t].keep(t < n && in_row);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float in[4];
#pragma unroll
            for (int j = 0; j < NX; ++j) in[j] = raw[j][t].value(i);
            const CrElem el = cr_elem<FORM>(in, c0[i], c1[i], a.p0);
            const bool live = t < n && in_row;
            w[t][i] = live ? el.w : 1.f;
            if constexpr (FORM == kCrWrite) made[t][i] = live ? el.q : 0.f;
            if constexpr (FORM == kCrGeneral) made[t][i] = live ? el.a : 0.f;
            odd[t & 3] = fmaf(w[t][i], 0.f, odd[t & 3]);
            if constexpr (FORM != kCrGated) odd[t & 3] = fmaf(made[t][i], 0.f, odd[t & 3]);
            if constexpr (FORM == kCrGeneral) odd[t & 3] = fmaf(raw[0][t].value(i), 0.f, odd[t & 3]);
        }
    }
    auto kf = [&](int t, int i) { return FORM == kCrWrite ? 1.f - w[t][i] : raw[1][t].value(i); };
    auto qf = [&](int t, int i) { return FORM == kCrWrite ? made[FORM == kCrGated ? 0 : t][i] : raw[0][t].value(i); };
    auto af = [&](int t, int i) { return made[FORM == kCrGated ? 0 : t][i]; };
    // 1 / |k| and 1 / |q| of token lane % 8 (where the form takes them)
    float kn = 1.f, qn = 1.f;
    if constexpr (HAS_K) {
        auto squares = [&](auto of) {                 // 8 tokens' sums over 64 lanes: halved three times over the lanes, then summed
            float s[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) s[t] = of(t);
            const bool o1 = lane & 1, o2 = lane & 2, o4 = lane & 4;
            float u[4], x[2];
#pragma unroll
            for (int t = 0; t < 4; ++t) u[t] = (o1 ? s[2 * t + 1] : s[2 * t]) + dpp_f32<0xB1>(o1 ? s[2 * t] : s[2 * t + 1]);
#pragma unroll
            for (int t = 0; t < 2; ++t) x[t] = (o2 ? u[2 * t + 1] : u[2 * t]) + dpp_f32<0x4E>(o2 ? u[2 * t] : u[2 * t + 1]);
            float r = (o4 ? x[1] : x[0]) + __shfl_xor(o4 ? x[0] : x[1], 4);
            r += __shfl_xor(r, 8);
            r += __shfl_xor(r, 16);
            return r + __shfl_xor(r, 32);
        };
        const bool in = (lane & 7) < n;
        const float ss = squares([&](int t) { return kf(t, 0) * kf(t, 0) + kf(t, 1) * kf(t, 1); });     // (all lanes take part)
        odd[0] += ss * 0.f;
        kn = in ? 1.0f / sqrtf(ss + a.p1) : 0.f;
        if constexpr (FORM == kCrGated) {
            const float qq = squares([&](int t) { return qf(t, 0) * qf(t, 0) + qf(t, 1) * qf(t, 1); });
            odd[1] += qq * 0.f + beta * 0.f;
            qn = 1.0f / sqrtf((qq + a.p1) * (float)D);
            beta = in ? cr_sigmoid(beta) : 0.f;
        }
        if (lane < 8) {
            lds.kn[th + lane] = kn;
            lds.qn[th + lane] = qn;
            lds.beta[th + lane] = beta;
        }
    }
    // decays from the half's first token through t, and behind t to the half's end
    float pre[2][N], suf[2][N];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        pre[i][0] = w[0][i];
        suf[i][N - 1] = 1.f;
#pragma unroll
        for (int t = 1; t < N; ++t) {
            pre[i][t] = pre[i][t - 1] * w[t][i];
            suf[i][N - 1 - t] = suf[i][N - t] * w[N - t][i];
        }
    }
    {
        // (false with a decay that is not a number)
        const bool near = __all(pre[0][N - 1] >= kCrNear && pre[1][N - 1] >= kCrNear);
        const bool near4 = __all(pre[0][N / 2 - 1] >= kCrNear && pre[1][N / 2 - 1] >= kCrNear &&
                                 suf[0][N / 2 - 1] >= kCrNear && suf[1][N / 2 - 1] >= kCrNear);
        const bool any_odd = __any((odd[0] + odd[1]) + (odd[2] + odd[3]) != 0.f);
        if (lane == 0) {
            lds.far[half] = near ? 0 : near4 ? 1 : 2;
            lds.odd[half] = any_odd;
        }
    }
    auto put = [&](float* rows, auto of) {            // this wave's 8 rows of this lane's two channels
        if (in_row) {
#pragma unroll
            for (int t = 0; t < N; ++t) *(float2*)(rows + (th + t) * ROW + d) = make_float2(of(t, 0), of(t, 1));
        }
    };
    __syncthreads();
    if (half == 0 && lane == 0) a.odd[h * a.records + rec] = lds.odd[0] | lds.odd[1];
    const uint32_t far = __builtin_amdgcn_readfirstlane(max(lds.far[0], lds.far[1]));     // 0, 1, 2: one set of pairs, two, five
    // ---- pair products: entry (row 4 g + e, column l16), rows k (first wave) or q (second), columns k or a k
    f32x4 pk = {0.f, 0.f, 0.f, 0.f}, pa = pk;
    {
        auto product = [&] {                          // of the operands in LDS
            f32x4 p[8] = {};
            const float* lf = (half ? lds.q : lds.k) + l16 * ROW + 4 * g;
            const float* rt = lds.right + l16 * ROW + 4 * g;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const f32x4 x = *(const f32x4*)(lf + 16 * m), y = *(const f32x4*)(rt + 16 * m);
#pragma unroll
                for (int e = 0; e < 4; ++e) p[4 * (m & 1) + e] = cr_mfma(x[e], y[e], p[4 * (m & 1) + e]);
            }
            return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        };
        // Relative to the middle: left sides G_t / G_8, right sides G_8 / G_t.  Otherwise part 8, 4, 2, 1 (0: s = t) one after the
        // other: left sides from the start of the part through the token, right sides behind the token to the end of its part; two
        // sets: part 4 relative to the half's middle.
#pragma unroll 1
        for (int part = 8; part >= 0; part = far == 0 || part == 0 || (far == 1 && part == 4) ? -1 : part / 2) {
            float lv[2][N], rv[2][N], first[2] = {1.f, 1.f};      // (first: left side of the first token's key, general)
            if (part == 8) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int t = 0; t < N; ++t) {
                        lv[i][t] = far == 0 && half == 0 ? __builtin_amdgcn_rcpf(suf[i][t]) : pre[i][t];
                        rv[i][t] = far == 0 && half == 1 ? __builtin_amdgcn_rcpf(pre[i][t]) : suf[i][t];
                    }
                    if (far == 0 && half == 0) first[i] = __builtin_amdgcn_rcpf(pre[i][N - 1]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float f = 1.f;
#pragma unroll
                    for (int t = 0; t < N; ++t) {
                        if ((t & (part - 1)) == 0) f = 1.f;
                        f *= part ? w[t][i] : 1.f;
                        lv[i][t] = f;
                    }
#pragma unroll
                    for (int t = N - 1; t >= 0; --t) {
                        if (((t + 1) & (part - 1)) == 0) f = 1.f;
                        rv[i][t] = part ? f : 1.f;
                        f *= w[t][i];
                    }
                    if (far == 1) {
                        first[i] = __builtin_amdgcn_rcpf(lv[i][N / 2 - 1]);
#pragma unroll
                        for (int t = 0; t < N / 2; ++t) lv[i][t] = __builtin_amdgcn_rcpf(rv[i][t]);
#pragma unroll
                        for (int t = N / 2; t < N; ++t) rv[i][t] = __builtin_amdgcn_rcpf(lv[i][t]);
                    }
                }
            }
            if constexpr (HAS_K)
                put(lds.k, [&](int t, int i) {        // (general: through the token before)
                    if constexpr (FORM != kCrGeneral) return kf(t, i) * lv[i][t];
                    return kf(t, i) * (t == 0 ? first[i] : (t & (part - 1)) == 0 ? 1.f : lv[i][t ? t - 1 : 0]);
                });
            put(lds.q, [&](int t, int i) { return qf(t, i) * lv[i][t]; });
            put(lds.right, [&](int t, int i) { return kf(t, i) * rv[i][t]; });
            // pairs whose tokens part at this part
            const bool middle = far == 0 || (far == 1 && part == 4);
            const uint32_t from = middle ? 0 : part, many = middle ? 2 * part : part ? part : 1;
            auto take = [&](f32x4& to, f32x4 of) {
#pragma unroll
                for (int e = 0; e < 4; ++e) to[e] = (uint32_t)((4 * g + e) ^ l16) - from < many ? of[e] : to[e];
            };
            __syncthreads();
            if (HAS_K || half) take(pk, product());
            __syncthreads();
            if constexpr (FORM == kCrGeneral) {
                put(lds.right, [&](int t, int i) { return af(t, i) * rv[i][t]; });
                __syncthreads();
                take(pa, product());
                __syncthreads();
            }
        }
    }
    // ---- [K; Q] (through LDS), K^, X^ and the chunk's decay; k and q are unit vectors from here on (gated).  Decays from the chunk's
    // start through a token (G) and behind it to the chunk's end (F).
    auto ku = [&](int t, int i) { return FORM == kCrGated ? kf(t, i) * cr_lane(kn, t) : kf(t, i); };
    auto qu = [&](int t, int i) { return FORM == kCrGated ? qf(t, i) * cr_lane(qn, t) : qf(t, i); };
    float G[2][N], F[2][N];
    double end[2] = {1.0, 1.0}, other[2];             // decays of this half, then of the chunk; of the other half
    {
        auto forward = [&](double (&f)[2]) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int t = 0; t < N; ++t) G[i][t] = (float)(f[i] *= (double)w[t][i]);
            }
        };
        auto backward = [&](double (&f)[2]) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int t = N - 1; t >= 0; --t) {
                    F[i][t] = (float)f[i];
                    f[i] *= (double)w[t][i];
                }
            }
        };
        double2* const totals = (double2*)lds.right;
        if (half) backward(end); else forward(end);
        if (in_row) totals[half * (D / 2) + d / 2] = make_double2(end[0], end[1]);
        __syncthreads();
        const double2 o = totals[(half ^ 1) * (D / 2) + d / 2];
        other[0] = end[0] = o.x;
        other[1] = end[1] = o.y;
        if (half) forward(end); else backward(end);
    }
    if constexpr (FORM == kCrGated) put(lds.k, [&](int t, int i) { return ku(t, i) * G[i][t]; });
    if constexpr (FORM == kCrGeneral) put(lds.k, [&](int t, int i) { return ku(t, i) * (t ? G[i][t ? t - 1 : 0] : half ? (float)other[i] : 1.f); });
    put(lds.q, [&](int t, int i) { return qu(t, i) * G[i][t]; });
    auto put_update = [&](int which, auto of) {       // lane (g, channel) of a tile: tokens 4 g .. 4 g + 3
        if (in_row) {
#pragma unroll
            for (int gg = 0; gg < 2; ++gg) {
                float* to = out + Rec::upd + which * 16 * D + (((d >> 4) * 4 + half * 2 + gg) * 16 + (d & 15)) * 4;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    f32x4 r;
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[e] = of(4 * gg + e, i) * F[i][4 * gg + e];
                    *(f32x4*)(to + 4 * i) = r;
                }
            }
        }
    };
    if constexpr (FORM == kCrGated) put_update(0, ku); else put_update(0, kf);
    if constexpr (FORM == kCrGeneral) put_update(1, af);
    if (half == 0 && in_row) *(float2*)(out + Rec::decay + d) = make_float2((float)end[0], (float)end[1]);
    __syncthreads();
    if (HAS_K || half) {
        const float* rows = (half ? lds.q : lds.k) + l16 * ROW + 4 * g;
        const int tile = HAS_K && half ? NM : 0;
#pragma unroll
        for (int m = 0; m < NM; ++m) *(f32x4*)(out + Rec::kq + ((tile + m) * 64 + lane) * 4) = *(const f32x4*)(rows + 16 * m);
    }
    // ---- T, and what the tokens' writes bring the read-outs
    float* mat = out + Rec::m;
    auto put_matrix = [&](int which, f32x4 p, int strict) {                   // s <= t (strict: s < t), zeros elsewhere
#pragma unroll
        for (int e = 0; e < 4; ++e) mat[which * 256 + (4 * g + e) * 16 + l16] = l16 + strict <= 4 * g + e ? p[e] : 0.f;
    };
    if constexpr (FORM == kCrWrite) {
        if (half) put_matrix(0, pk, 0);
        return;
    }
    // gated: u = T (v - K^T S), T = (I + A)^-1 diag(beta), A_ts = beta_t kn_t kn_s P_ts (s < t);  o_t = Q^T S + qn_t kn_s P_ts u_s
    // general: x = (I + A)^-1 diag(kn) (K^T S + PK v), A_ts = kn_t kn_s P_ts(k, a k), PK_ts = P_ts(k, k) (s < t); the writes along a k
    //          take u_s = -kn_s x_s, which T makes at once;  o_t = Q^T S + P_ts(r, k) v_s + P_ts(r, a k) u_s
    const float kc = lds.kn[l16];
    f32x4 rows, p = FORM == kCrGated ? pk : pa;
#pragma unroll
    for (int e = 0; e < 4; ++e) rows[e] = half ? (FORM == kCrGated ? lds.qn[4 * g + e] : 0.f) : lds.kn[4 * g + e];
    if (half) {
        if constexpr (FORM == kCrGated) p *= rows * kc;
        put_matrix(1, p, 0);
        if constexpr (FORM == kCrGeneral) put_matrix(2, pk, 0);
        return;
    }
    if constexpr (FORM == kCrGeneral) put_matrix(3, pk, 1);
    const float bc = FORM == kCrGated ? lds.beta[l16] : kc;
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] *= (FORM == kCrGated ? rows[e] * lds.beta[4 * g + e] : rows[e]) * kc;
    float y[L];                                       // column l16 of T
    f32x4 mine = {0.f, 0.f, 0.f, 0.f};                // its rows 4 g + e (an index by g into y would put y into memory)
#pragma unroll
    for (int t = 0; t < L; ++t) {
        float s0 = t == l16 ? bc : 0.f, s1 = 0.f;
#pragma unroll
        for (int i = 0; i < t; ++i) {
            const float f = cr_lane(p[t & 3], (t >> 2) * 16 + i);
            if (i & 1) s1 -= f * y[i]; else s0 -= f * y[i];
        }
        y[t] = s0 + s1;
        mine[t & 3] = g == (t >> 2) ? y[t] : mine[t & 3];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) mat[(4 * g + e) * 16 + l16] = mine[e] * (FORM == kCrGeneral ? -rows[e] : 1.f);
}

// ------------------------------------------------------------------------------------------------ second launch
// RS waves per (sequence, head, 16 value columns), each with D / RS key channels of the state in MFMA accumulators; RS = 2: the
// waves' parts of K S are exchanged through LDS while Q S is multiplied, and each takes half of what is added to Q S, which the movers
// add up.  A workgroup has four of these waves, one on each SIMD of a CU, and four that do nothing but move: records and columns of V four
// chunks ahead into registers and two ahead into LDS (three slots), read-outs from LDS to memory.  One barrier a chunk.  With the loads
// and stores in the products' waves every chunk also paid for their issue (chunks of 8: 264 us instead of 219).
template <typename T, int FORM, int D, int RS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void recurrence_states_kernel(
    const ChunkRecurrenceArgs a, const int first_seq) {
    constexpr int NM = D / 16 / RS;                   // tiles of a wave
    constexpr int L = kCrChunk;
    typedef CrRecord<FORM, D> Rec;
    constexpr int ROUNDS = (Rec::words + 1023) / 1024;
    constexpr int COLS = 64 / RS, PER = 4 / RS;       // value columns of the workgroup; elements of a row of V a thread moves
    __shared__ __attribute__((aligned(16))) float slots[3][Rec::words];
    __shared__ __attribute__((aligned(16))) float vs[3][L][COLS], os[2][RS][L][COLS];
    __shared__ f32x4 part[RS == 1 ? 1 : 2][4][64];
    // Workgroups go to the eight XCDs in turn: an XCD takes neighbouring heads.
    const int pair = gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
    const int b = first_seq + pair / a.H, h = pair % a.H;
    const int q0 = a.cu_q[b], len = a.cu_q[b + 1] - q0;
    if (len < 2) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int chunks = (len + L - 1) / L, Dv = a.Dv;

    if (wave >= 4) {
        // ---------------------------------------------------------------- the movers
        const int tid = threadIdx.x - 256;
        const int64_t first = (int64_t)h * a.records + cr_first_record<kCrChunk>(q0 - a.cu_q[first_seq], b - first_seq);
        const float* rec = a.chunks + first * Rec::words;
        const int tok = tid >> 4, col = (tid & 15) * PER, col_all = blockIdx.y * COLS + col;
        // (columns past the end: the last ones, used by waves that write nothing)
        const T* v = (const T*)a.columns + first * L * Dv + tok * Dv + min(col_all, Dv - PER);
        float* o = a.raw + ((int64_t)h * a.T + q0 + tok) * Dv + col_all;
        struct Staged {
            f32x4 r[ROUNDS];
            CrColumns<T, PER> v;
        };
        auto fetch = [&](int c, Staged& st) {
            c = min(c, chunks - 1);
            const float* rc = rec + (int64_t)c * Rec::words;
            st.v.load(v + (int64_t)c * L * Dv);
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i)
                if ((i + 1) * 1024 <= Rec::words || i * 1024 + tid * 4 < Rec::words) st.r[i] = *(const f32x4*)(rc + (uint32_t)(i * 1024 + tid * 4));
        };
        auto stage = [&](int at, const Staged& st) {
#pragma unroll
            for (int e = 0; e < PER; ++e) vs[at][tok][col + e] = st.v.value(e);
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i)
                if ((i + 1) * 1024 <= Rec::words || i * 1024 + tid * 4 < Rec::words) *(f32x4*)(slots[at] + i * 1024 + tid * 4) = st.r[i];
        };
        auto store = [&](int c) {
            if (c * L + tok < len && col_all < Dv) {
                float* to = o + (int64_t)c * L * Dv;
                if constexpr (RS == 1) *(f32x4*)to = *(const f32x4*)&os[c & 1][0][tok][col];
                else {
                    const float2 x = *(const float2*)&os[c & 1][0][tok][col], y = *(const float2*)&os[c & 1][RS - 1][tok][col];
                    *(float2*)to = make_float2(x.x + y.x, x.y + y.y);
                }
            }
        };
        Staged s0, s1;
        fetch(0, s0);
        fetch(1, s1);
        stage(0, s0);
        stage(1, s1);
        fetch(2, s0);
        fetch(3, s1);
        cr_group_barrier();
        int at = 2, c = 0;
        auto move = [&](int c, Staged& st) {          // behind the barrier of chunk c: st holds chunk c + 2 and takes c + 4
            cr_group_barrier();
            stage(at, st);
            at = at == 2 ? 0 : at + 1;
            fetch(c + 4, st);
            if (c > 0) store(c - 1);
        };
        for (; c + 1 < chunks; c += 2) {              // (no way out of the middle: the waits at the loop's head stay exact)
            move(c, s0);
            move(c + 1, s1);
        }
        if (c < chunks) move(c, s0);
        cr_group_barrier();
        store(chunks - 1);
        return;
    }

    // -------------------------------------------------------------------- the state
    const int rp = wave % RS, l16 = lane & 15, g = lane >> 4, d0 = rp * (D / RS);
    int tile = blockIdx.y * (4 / RS) + wave / RS;
    const bool live = tile * 16 < Dv, fresh = a.cu_k[b + 1] - a.cu_k[b] == len;
    if (!live) tile = 0;                              // (waves without columns repeat the first ones' and write nothing)
    const int in_group = (wave / RS) * 16 + l16;
    float* slot = a.state + ((int64_t)a.slots[b] * a.H + h) * (int64_t)D * Dv + (int64_t)(d0 + 4 * g) * Dv + tile * 16 + l16;
    f32x4 S[NM];                                      // rows 4 g + e of the wave's tiles
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[m][e] = fresh ? 0.f : slot[(int64_t)(16 * m + e) * Dv];
    }
    uint32_t odd = 0;                                 // some chunk of the sequence and head holds a value that is not finite
    {
        const uint32_t* flags = a.odd + (int64_t)h * a.records + cr_first_record<kCrChunk>(q0 - a.cu_q[first_seq], b - first_seq);
        for (int c = lane; c < chunks; c += 64) odd |= flags[c];
        odd = __any(odd != 0);
    }
    const int at_x = Rec::kq + lane * 4 + d0 * 16, at_upd = Rec::upd + lane * 4 + d0 * 16;
    const int at_dec = Rec::decay + d0 + ((l16 + 4 * g) & 15), at_m = Rec::m + l16 * 16 + 4 * g;
    constexpr bool HAS_K = FORM != kCrWrite, HAS_V = FORM != kCrGated;
    constexpr int MV = FORM == kCrGeneral ? 512 : 0;  // the matrix that takes V to the read-outs
    constexpr f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 x[NM];                                      // the first rows that a chunk multiplies: read behind the barrier in front of it
    auto read_x = [&](int at) {
#pragma unroll
        for (int m = 0; m < NM; ++m) x[m] = *(const f32x4*)(slots[at] + 256 * m + at_x);
    };
    // Rows of a lower triangular matrix times 16 rows of values, the wave's share of the 16; ODD: a zero above the diagonal keeps a later
    // token out only while that token's value is finite, so token by token, each from rows that end with it.
    constexpr int E0 = 4 / RS;
    typedef CrRow<E0> Share;
    const int at_share = at_m + rp * E0;
    auto share = [&](f32x4 x) {
        Share r;
#pragma unroll
        for (int e = 0; e < E0; ++e) r[e] = rp ? x[(E0 + e) & 3] : x[e];
        return r;
    };
    auto triangle = [&](auto odd_tag, auto mt, auto x, f32x4 onto) {
        constexpr bool ODD = decltype(odd_tag)::value;
        constexpr int E = sizeof(x) / sizeof(float);  // 4: all of the 16 rows
        auto sum = [&](int t, f32x4 c0) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int row = 4 * g + (E == 4 ? e : rp * E0 + e);
                c0 = cr_mfma(mt[e], ODD ? (row <= t ? x[e] : 0.f) : x[e], c0);        // (a sum that goes on costs a product no wait)
            }
            return c0;
        };
        if constexpr (!ODD) return sum(0, onto);
        f32x4 rows = zero;
#pragma unroll 1
        for (int t = 0; t < L; ++t) {
            const f32x4 r = sum(t, onto);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * g + e == t) rows[e] = r[e];
        }
        return rows;
    };
    // General: a chunk's removals, summed by themselves and added where the next products hide it (which costs 5 us of 227, one prompt of
    // 2048 tokens).
    f32x4 moved[FORM == kCrGeneral ? NM : 1] = {};
    cr_group_barrier();
    if (!HAS_K || odd == 0) read_x(0);
    int at = 0;
    // Chunk c from slot `at`.  LATE: operands when they are needed, since the triangles' loops take registers of their own (read
    // ahead there too, the kernels of a whole state a wave spilled and all their calls paid for it, 2 to 4 %).
    auto chunk = [&](auto odd_tag, int c) {
        constexpr bool LATE = HAS_K && decltype(odd_tag)::value;
        const float* rc = slots[at];
        float dec[NM];                                // lane e of group g: the decay of row 4 g + e of the tile
        f32x4 xq[NM], up[NM], ux[NM], vv, mt;
        Share mq, mv, mk;
        if constexpr (LATE) read_x(at);
        auto read_xq = [&] {
#pragma unroll
            for (int m = 0; m < NM; ++m) xq[m] = HAS_K ? *(const f32x4*)(rc + 16 * D + 256 * m + at_x) : x[m];
        };
        if constexpr (!LATE) read_xq();
#pragma unroll
        for (int e = 0; e < 4; ++e) vv[e] = vs[at][4 * g + e][in_group];
        if constexpr (FORM == kCrGeneral) mk = *(const Share*)(rc + 768 + at_share);
        if constexpr (HAS_V) mv = *(const Share*)(rc + MV + at_share);
        if constexpr (HAS_K) {
            mt = *(const f32x4*)(rc + at_m);
            mq = *(const Share*)(rc + 256 + at_share);
        }
        __builtin_amdgcn_sched_barrier(0);            // the reads are on their way before the products
        auto read_update = [&] {
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                dec[m] = rc[16 * m + at_dec];
                if constexpr (HAS_V) up[m] = *(const f32x4*)(rc + 256 * m + at_upd);
                if constexpr (HAS_K) ux[m] = *(const f32x4*)(rc + (Rec::kUpd - 1) * 16 * D + 256 * m + at_upd);
            }
        };
        // (four sums: a quarter of the roundings one after the other)
        f32x4 ck = zero, other = zero, o0 = zero, o1 = zero, o2 = zero, o3 = zero;
        auto q_tile = [&](int m) {
            o0 = cr_mfma(xq[m][0], S[m][0], o0);
            o1 = cr_mfma(xq[m][1], S[m][1], o1);
            o2 = cr_mfma(xq[m][2], S[m][2], o2);
            o3 = cr_mfma(xq[m][3], S[m][3], o3);
        };
        constexpr int QF = NM > 2 ? (NM + 1) / 2 : 1; // tiles of Q S in front of the barrier: while the parts of K S are written
        if constexpr (HAS_K) {
            f32x4 k1 = zero, k2 = zero, k3 = zero;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                if constexpr (FORM == kCrGeneral) S[m] += moved[m];
                ck = cr_mfma(x[m][0], S[m][0], ck);
                k1 = cr_mfma(x[m][1], S[m][1], k1);
                k2 = cr_mfma(x[m][2], S[m][2], k2);
                k3 = cr_mfma(x[m][3], S[m][3], k3);
            }
            f32x4 pk = zero;
            if constexpr (FORM == kCrGeneral) pk = triangle(odd_tag, mk, share(vv), zero);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LATE) read_xq(); else read_update();
            q_tile(0);
            __builtin_amdgcn_sched_barrier(0);
            ck = (ck + k1) + (k2 + k3);
            if constexpr (FORM == kCrGeneral) ck += pk;
            if constexpr (RS > 1) part[c & 1][wave][lane] = ck;
        } else {
            read_update();
            q_tile(0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 1; m < (LATE ? NM : QF); ++m) q_tile(m);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LATE) read_update();
        cr_group_barrier();                           // chunk c + 1 is in its slot; chunk c - 1's slot is free
        if constexpr (HAS_K && RS > 1) other = part[c & 1][wave ^ 1][lane];
        at = at == 2 ? 0 : at + 1;
        if constexpr (!LATE) read_x(at);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = LATE ? NM : QF; m < NM; ++m) q_tile(m);
        f32x4 o = zero;
        if constexpr (HAS_V) o = triangle(odd_tag, mv, share(vv), zero);
        __builtin_amdgcn_sched_barrier(0);
        o += (o0 + o1) + (o2 + o3);
        // the state moves on: rows 4 g + e of tile m decay, then take the chunk's writes
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            S[m][0] *= dpp_f32<0x150>(dec[m]);        // row_newbcast e: lane e of the group
            S[m][1] *= dpp_f32<0x151>(dec[m]);
            S[m][2] *= dpp_f32<0x152>(dec[m]);
            S[m][3] *= dpp_f32<0x153>(dec[m]);
        }
        if constexpr (HAS_V) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int m = 0; m < NM; ++m) S[m] = cr_mfma(up[m][e], vv[e], S[m]);
        }
        if constexpr (FORM == kCrGeneral) __builtin_amdgcn_sched_barrier(0);      // (they run while the other wave's part comes)
        if constexpr (HAS_K) {
            ck += other;
            const f32x4 u = triangle(odd_tag, mt, FORM == kCrGated ? vv - ck : ck, zero);
            if constexpr (FORM == kCrGated) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int m = 0; m < NM; ++m) S[m] = cr_mfma(ux[m][e], u[e], S[m]);
            } else {
#pragma unroll
                for (int m = 0; m < NM; ++m) moved[m] = cr_mfma(ux[m][0], u[0], zero);
#pragma unroll
                for (int e = 1; e < 4; ++e)
#pragma unroll
                    for (int m = 0; m < NM; ++m) moved[m] = cr_mfma(ux[m][e], u[e], moved[m]);
            }
            o += triangle(odd_tag, mq, share(u), zero);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) os[c & 1][rp][4 * g + e][in_group] = o[e];
    };
    if (odd == 0) {
        for (int c = 0; c < chunks; ++c) chunk(std::false_type{}, c);
    } else {
        for (int c = 0; c < chunks; ++c) chunk(std::true_type{}, c);
    }
    cr_group_barrier();
    if (!live) return;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        if constexpr (FORM == kCrGeneral) S[m] += moved[m];
#pragma unroll
        for (int e = 0; e < 4; ++e) slot[(int64_t)(16 * m + e) * Dv] = S[m][e];
    }
}

// ------------------------------------------------------------------------------------------------ read-outs
// out = o / sqrt(mean(o^2) + eps) * norm_w * sigmoid(gate) per token and head; 16 lanes a row, pieces of four columns.  A workgroup
// takes a token; SEARCH: tokens that are their sequence's only row are another launch's.
template <typename T, bool VEC, bool SEARCH>
__global__ __launch_bounds__(256) void recurrence_finish_kernel(const ChunkRecurrenceArgs a, const int first_seq) {
    const int t = a.cu_q[first_seq] + blockIdx.x, l16 = threadIdx.x & 15;
    if (t >= a.cu_q[a.num_seqs]) return;
    if constexpr (SEARCH) {
        int lo = 0, hi = a.num_seqs;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (a.cu_q[mid] <= t) lo = mid; else hi = mid;
        }
        if (a.cu_q[lo + 1] - a.cu_q[lo] < 2) return;
    }
    const int Dv = a.Dv;
    constexpr int V = VEC ? 4 : 1;
    constexpr int P = 16 / V;                         // pieces of a lane: up to 256 columns
    for (int h = threadIdx.x >> 4; h < a.H; h += 16) {
        const float* o = a.raw + ((int64_t)h * a.T + t) * Dv;
        const float* w = a.norm_w + (int64_t)h * a.norm_head_stride;
        const T* gate = (const T*)a.gate_raw + (int64_t)t * a.gate_stride + (int64_t)h * Dv;
        Cols<V> x[P], gt[P];
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int c = V * (l16 + 16 * j);
            if (c < Dv) {
                x[j] = row_load<V>(o + c);
                if (a.gate_raw != nullptr) gt[j] = row_load<V>(gate + c);
            }
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            if (V * (l16 + 16 * j) < Dv) {
#pragma unroll
                for (int e = 0; e < V; ++e) ss += x[j].v[e] * x[j].v[e];
            }
        }
        const float rstd = 1.0f / sqrtf(row16_sum(ss) / (float)Dv + a.eps);
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int c = V * (l16 + 16 * j);
            if (c < Dv) {
                const Cols<V> wt = row_load<V>(w + c);
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    x[j].v[e] *= rstd * wt.v[e];
                    if (a.gate_raw != nullptr) x[j].v[e] *= cr_sigmoid(gt[j].v[e]);
                }
                row_store<V>((T*)a.out + (int64_t)t * a.out_stride + (int64_t)h * Dv + c, x[j]);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ single tokens
// One token of a sequence: bound by its state, which is read and written once.  A workgroup per (sequence, head) holds the state in
// registers, four neighbouring columns of ROWS rows a thread (all loads in flight at once); what the token finds in the old state
// and what it reads out come from one pass: with p = S^T k (decayed as the form wants it) the read-out of the new state
// is that of the decayed old one plus the write's part, which is a number per token (k . q and the like) times the columns written.
// STREAM: the states pass by the caches (see recurrence_streams).
template <typename T, int FORM, int ROWS, bool STREAM>
__global__ __launch_bounds__(256) void single_recurrence_kernel(const ChunkRecurrenceArgs a, const int pieces) {
    constexpr int NX = FORM == kCrGated ? 3 : FORM == kCrGeneral ? 4 : 2;
    __shared__ float ws[256], ks[256], qs[256], as[256], red[4][4];
    __shared__ __attribute__((aligned(16))) float part[2][256 * 4];
    const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int t = a.cu_q[b], D = a.D, Dv = a.Dv;
    if (a.cu_q[b + 1] - t != 1) return;
    const bool fresh = a.cu_k[b + 1] - a.cu_k[b] == 1;
    const int c = (tid % pieces) * 4, group = tid / pieces, groups = 256 / pieces;      // (pieces is a power of two)
    const bool live = c < Dv;
    // the token's rows first: they are waited for first
    float x[4] = {};
    const int dd = tid < D ? tid : 0;
    {
        const void* xs[4] = {a.x0, a.x1, a.x2, a.x3};
        const int64_t ss[4] = {a.s0, a.s1, a.s2, a.s3};
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int hj = (FORM == kCrGated && j < 2) ? h / a.group : h;
            x[j] = (float)((const T*)xs[j])[(int64_t)t * ss[j] + (int64_t)hj * D + dd];
        }
    }
    const float c0 = FORM == kCrGated ? expf(a.c0[h]) : a.c0[(int64_t)h * D + dd], c1 = a.c1[(int64_t)h * D + dd];
    float v[4], gate[4], nw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = live ? (float)((const T*)a.v)[(int64_t)t * a.sv + (int64_t)h * Dv + c + e] : 0.f;
        gate[e] = (live && a.gate_raw != nullptr) ? (float)((const T*)a.gate_raw)[(int64_t)t * a.gate_stride + (int64_t)h * Dv + c + e] : 0.f;
        nw[e] = live ? a.norm_w[(int64_t)h * a.norm_head_stride + c + e] : 0.f;
    }
    float beta = 0.f;
    if constexpr (FORM == kCrGated) beta = (float)((const T*)a.b_raw)[(int64_t)t * a.b_stride + h];
    float* st = a.state + ((int64_t)a.slots[b] * a.H + h) * (int64_t)D * Dv + c;
    f32x4 S[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = group + i * groups;
        S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (live && d < D && !fresh) {
            const f32x4* from = (const f32x4*)(st + (int64_t)d * Dv);
            S[i] = STREAM ? __builtin_nontemporal_load(from) : *from;
        }
    }
    {
        CrElem el = cr_elem<FORM>(x, c0, c1, a.p0);
        if (tid >= D) el = CrElem{1.f, 0.f, 0.f, 0.f};
        const float s0 = wave_sum(el.k * el.k);
        const float s1 = wave_sum(FORM == kCrGated ? el.q * el.q : el.a * el.q), s2 = wave_sum(el.k * el.q);
        if ((tid & 63) == 0) {
            red[0][tid >> 6] = s0;
            red[1][tid >> 6] = s1;
            red[2][tid >> 6] = s2;
        }
        ws[tid] = el.w;
        ks[tid] = el.k;
        qs[tid] = el.q;
        as[tid] = el.a;
    }
    __syncthreads();
    const float kk = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]), s1 = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    const float kq = (red[2][0] + red[2][1]) + (red[2][2] + red[2][3]);
    const float kn = FORM == kCrWrite ? 1.f : 1.0f / sqrtf(kk + a.p1);
    const float qn = FORM == kCrGated ? 1.0f / sqrtf((s1 + a.p1) * (float)D) : 1.f;
    f32x4 pk = {0.f, 0.f, 0.f, 0.f}, pq = pk;         // S^T k (general: of the old state), (w S)^T q over this thread's rows
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int d = group + i * groups;
        if (d < D) {
            if constexpr (FORM == kCrGeneral) pk += S[i] * ks[d];
            S[i] *= ws[d];
            if constexpr (FORM == kCrGated) pk += S[i] * ks[d];
            pq += S[i] * qs[d];
        }
    }
    if constexpr (FORM != kCrWrite) *(f32x4*)(part[0] + tid * 4) = pk;
    *(f32x4*)(part[1] + tid * 4) = pq;
    __syncthreads();
    f32x4 sk = {0.f, 0.f, 0.f, 0.f}, sq = sk;
    for (int j = 0; j < groups; ++j) {
        if constexpr (FORM != kCrWrite) sk += *(const f32x4*)(part[0] + (j * pieces + tid % pieces) * 4);
        sq += *(const f32x4*)(part[1] + (j * pieces + tid % pieces) * 4);
    }
    const f32x4 vv = {v[0], v[1], v[2], v[3]};
    f32x4 o, add, sub = {0.f, 0.f, 0.f, 0.f};         // new state: decayed old + k add - a sub
    if constexpr (FORM == kCrGated) {
        add = (vv - sk * kn) * (cr_sigmoid(beta) * kn);
        o = (sq + add * kq) * qn;
    } else if constexpr (FORM == kCrGeneral) {
        add = vv;
        sub = sk * (kn * kn);
        o = sq + vv * kq - sub * s1;
    } else {
        add = vv;
        o = sq + vv * kq;
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int d = group + i * groups;
            if (d < D) {
                S[i] += add * ks[d];
                if constexpr (FORM == kCrGeneral) S[i] -= sub * as[d];
                f32x4* to = (f32x4*)(st + (int64_t)d * Dv);
                if constexpr (STREAM) __builtin_nontemporal_store(S[i], to);
                else *to = S[i];
            }
        }
    }
    float ss = live ? (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]) : 0.f;
    for (int m = 1; m < pieces; m *= 2) ss += __shfl_xor(ss, m);        // (pieces <= 64: a row's columns lie in one wave)
    if (live && group == 0) {
        const float rstd = 1.0f / sqrtf(ss / (float)Dv + a.eps);
        T* out = (T*)a.out + (int64_t)t * a.out_stride + (int64_t)h * Dv + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float r = o[e] * rstd * nw[e];
            if (a.gate_raw != nullptr) r *= cr_sigmoid(gate[e]);
            out[e] = (T)r;
        }
    }
}

// ------------------------------------------------------------------------------------------------ launches
// Sizes both launches take: the single tokens' one holds a state in at most 32 pieces of four columns a thread.
static bool recurrence_built(int D, int Dv) {
    return (D == 32 || D == 64 || D == 96 || D == 128) && Dv % 16 == 0 && Dv <= 256 && D * Dv <= 128 * 128;
}

// Two waves for a state's 16 columns while that leaves every workgroup (one a CU, two tiles of columns) a CU of its own.  Whole
// calls, one against two waves, sequences of 768 rows, 16 heads: gated 128 x 128, 128 tiles 114 -> 78 us, 512: 147 -> 113,
// 640: 158 -> 175, 1024: 190 -> 208; gated 64 x 64, 512: 122 -> 106, 640: 135 -> 155; general, 512: 188 -> 141, 640: 201 -> 223;
// write 128 x 128, 512: 100 -> 73, 640: 110 -> 118.
static bool cr_two_waves(int64_t seqs, int H, int Dv) { return seqs * H * ((Dv / 16 + 1) / 2) <= 256; }

// Tokens of a chunk, from the mean portion of the sequences behind the leading single tokens.  A chunk of 16 halves the serial chain but
// takes more products and registers a token, and a portion's last chunk is as dear half empty.  So it pays in long portions, later where the
// grid fills the chip by itself (one wave a state), later the more products the form has, and sooner where every workgroup of the
// first launch has a CU to itself.  Whole calls, 16 heads, chunks of 16 against 8, lines from 16 .. 2048 rows in 1 .. 128
// sequences:  write, 128 x 128: 8 of 64 rows 0.96, 32 of 64 0.92, 8 of 17 1.18, 64 x 64: 16 of 128 0.99, 32 of 72 1.10, 1 of 33 0.95;
// gated, 128 x 128: 4 of 192 0.94, 8 of 256 1.00, 16 of 256 0.96, 256 of 2 1.43, 64 x 64: 16 of 256 1.03, of 512 0.99, 32 x 32: 16 of 512
// 1.05, 1 of 128 0.95; general, 128 x 128: 2 of 512 0.94, 4 of 256 1.05, 16 of 512 1.03, 256 of 2 1.58, 1 of 192 0.96.
static int cr_chunk_tokens(int form, int64_t rows, int64_t seqs, int H, int D, int Dv) {
    const bool alone = (cr_first_record<kCrChunk>(rows, (int)seqs) + 1) * H <= 256, two = cr_two_waves(seqs, H, Dv);
    if (form == kCrGeneral && !two) return 8;
    const int64_t from = form == kCrWrite ? (alone ? 25 : D >= 128 ? 64 : 128)
                                          : form == kCrGated ? (alone ? 96 : two ? 192 : 128 * 256 / D) : (alone ? 128 : 512);
    return rows >= from * seqs ? kCrChunk : 8;
}

// The workspace of T rows in seqs sequences: records, their rows of V, read-outs, flags; the parts in front of the flags are whole
// 16-byte pieces.
struct CrWorkspace {
    int tokens;                                       // of a chunk
    int64_t records, chunks, columns, raw, odd;       // how many (per head); bytes of the parts
    CrWorkspace(int form, int chunk, int64_t T, int H, int D, int Dv, int seqs, int dtype) {
        tokens = chunk;
        const int words = tokens != kCrChunk ? short_recurrence_words(form, D)
                                             : (form == kCrWrite ? 16 : 32) * D + (form == kCrGeneral ? 2 : 1) * 16 * D + D +
                                                   (form == kCrWrite ? 256 : form == kCrGated ? 512 : 1024);
        records = tokens != kCrChunk ? short_recurrence_records(T, seqs) : cr_first_record<kCrChunk>(T, seqs) + 1;
        chunks = records * H * words * 4;
        columns = records * H * tokens * Dv * (dtype == NV_DTYPE_BF16 ? 2 : 4);
        raw = T * H * Dv * 4;
        odd = records * H * 4;
    }
    int64_t bytes() const { return chunks + columns + raw + odd; }
};

template <typename T, int FORM, int D>
static void chunks_of_size(const ChunkRecurrenceArgs& a, int first_seq, bool vec, int waves, hipStream_t s) {
    const dim3 prep((unsigned)a.records, (unsigned)a.H), block(512);
    const unsigned pairs = (unsigned)((a.num_seqs - first_seq) * a.H), tiles = (unsigned)(a.Dv / 16);
    if (vec) hipLaunchKernelGGL((recurrence_chunks_kernel<T, FORM, D, true>), prep, dim3(128), 0, s, a, first_seq);
    else hipLaunchKernelGGL((recurrence_chunks_kernel<T, FORM, D, false>), prep, dim3(128), 0, s, a, first_seq);
    if constexpr (FORM != kCrGeneral) {               // (general: steps of two waves only)
        if (waves == 1) {
            hipLaunchKernelGGL((recurrence_states_kernel<T, FORM, D, 1>), dim3(pairs, (tiles + 3) / 4), block, 0, s, a, first_seq);
            return;
        }
    }
    hipLaunchKernelGGL((recurrence_states_kernel<T, FORM, D, 2>), dim3(pairs, (tiles + 1) / 2), block, 0, s, a, first_seq);
}

template <typename T, int FORM>
static int chunks_of(const ChunkRecurrenceArgs& a, int first_seq, int tokens, bool singles_behind, int dtype, hipStream_t s) {
    const uintptr_t piece = 2 * sizeof(T) - 1;        // two channels by one load
    const bool pairs = a.sv % 2 == 0 && a.s0 % 2 == 0 && a.s1 % 2 == 0 && a.s2 % 2 == 0 && a.s3 % 2 == 0 &&
                       (((uintptr_t)a.v | (uintptr_t)a.x0 | (uintptr_t)a.x1 | (uintptr_t)a.x2 | (uintptr_t)a.x3) & piece) == 0;
    const int waves = cr_two_waves(a.num_seqs - first_seq, a.H, a.Dv) ? 2 : 1;
    if (tokens != kCrChunk) {
        launch_short_recurrence(FORM, a, first_seq, pairs, waves, dtype, s);
    } else {
        switch (a.D) {
            case 32: chunks_of_size<T, FORM, 32>(a, first_seq, pairs, waves, s); break;
            case 64: chunks_of_size<T, FORM, 64>(a, first_seq, pairs, waves, s); break;
            case 96: chunks_of_size<T, FORM, 96>(a, first_seq, pairs, waves, s); break;
            default: chunks_of_size<T, FORM, 128>(a, first_seq, pairs, waves, s); break;
        }
    }
    const dim3 rows((unsigned)a.T);
    const bool vec = a.gate_stride % 4 == 0 && a.out_stride % 4 == 0 &&
                     ((uintptr_t)a.gate_raw | (uintptr_t)a.out | (uintptr_t)a.norm_w | (uintptr_t)a.raw) % 16 == 0;
    if (vec && singles_behind) hipLaunchKernelGGL((recurrence_finish_kernel<T, true, true>), rows, dim3(256), 0, s, a, first_seq);
    else if (vec) hipLaunchKernelGGL((recurrence_finish_kernel<T, true, false>), rows, dim3(256), 0, s, a, first_seq);
    else hipLaunchKernelGGL((recurrence_finish_kernel<T, false, true>), rows, dim3(256), 0, s, a, first_seq);
    return check_launch("chunked recurrence");
}

template <typename T, int FORM, bool STREAM>
static void singles_rows(const ChunkRecurrenceArgs& a, int pieces, int rows, hipStream_t s) {
    const dim3 grid((unsigned)a.num_seqs, (unsigned)a.H), block(256);
    if (rows <= 4) hipLaunchKernelGGL((single_recurrence_kernel<T, FORM, 4, STREAM>), grid, block, 0, s, a, pieces);
    else if (rows <= 8) hipLaunchKernelGGL((single_recurrence_kernel<T, FORM, 8, STREAM>), grid, block, 0, s, a, pieces);
    else if (rows <= 16) hipLaunchKernelGGL((single_recurrence_kernel<T, FORM, 16, STREAM>), grid, block, 0, s, a, pieces);
    else hipLaunchKernelGGL((single_recurrence_kernel<T, FORM, 32, STREAM>), grid, block, 0, s, a, pieces);
}
// singles: sequences known to be of one token
template <typename T, int FORM>
static int singles_of(const ChunkRecurrenceArgs& a, int singles, hipStream_t s) {
    int pieces = 1;
    while (pieces * 4 < a.Dv) pieces *= 2;            // at most 64
    const int rows = (a.D + 256 / pieces - 1) / (256 / pieces);
    if (recurrence_streams(singles, a.H, a.D, a.Dv)) singles_rows<T, FORM, true>(a, pieces, rows, s);
    else singles_rows<T, FORM, false>(a, pieces, rows, s);
    return check_launch("single-token recurrence");
}

#define NV_CR_DISPATCH(FN, ...)                                                                                       \
    if (dtype == NV_DTYPE_BF16)                                                                                       \
        return form == kCrGated ? FN<__bf16, kCrGated>(__VA_ARGS__)                                                   \
                                : form == kCrGeneral ? FN<__bf16, kCrGeneral>(__VA_ARGS__) : FN<__bf16, kCrWrite>(__VA_ARGS__); \
    return form == kCrGated ? FN<float, kCrGated>(__VA_ARGS__)                                                        \
                            : form == kCrGeneral ? FN<float, kCrGeneral>(__VA_ARGS__) : FN<float, kCrWrite>(__VA_ARGS__)

static int launch_chunk_recurrence(int form, const ChunkRecurrenceArgs& a, int first_seq, int tokens, bool singles_behind, int dtype,
                                   hipStream_t s) {
    NV_CR_DISPATCH(chunks_of, a, first_seq, tokens, singles_behind, dtype, s);
}
static int launch_single_recurrence(int form, const ChunkRecurrenceArgs& a, int singles, int dtype, hipStream_t s) {
    NV_CR_DISPATCH(singles_of, a, singles, s);
}
#undef NV_CR_DISPATCH

bool run_recurrence_portions(int form, ChunkRecurrenceArgs a, int lead, int portions, int dtype, void* workspace,
                             int64_t workspace_bytes, hipStream_t s, int* rc) {
    *rc = NV_OK;
    // (T = 0: not known, as from the entry points without portions; there may be longer portions then)
    const bool rest = lead < a.num_seqs && (a.T <= 0 || a.T > lead) && (portions & (NV_PORTION_FEW | NV_PORTION_LONG));
    const bool singles_behind = lead < a.num_seqs && (portions & NV_PORTION_SINGLE);
    // (rows, and sequences times heads, number workgroups in 32 bits; strides are 64 bits throughout)
    if (!recurrence_built(a.D, a.Dv) || (uintptr_t)a.state % 16 != 0 || a.T >= (1LL << 31) || (int64_t)a.num_seqs * a.H >= (1LL << 31) ||
        (rest && (workspace == nullptr || a.T <= 0)))
        return false;
    const CrWorkspace ws(form, cr_chunk_tokens(form, a.T - lead, a.num_seqs - lead, a.H, a.D, a.Dv), a.T, a.H, a.D, a.Dv, a.num_seqs - lead, dtype);
    const int64_t need = ws.bytes();
    if (rest && workspace_bytes < need) {
        set_error("recurrence: workspace of %lld bytes, need %lld", (long long)workspace_bytes, (long long)need);
        *rc = NV_ERR_WORKSPACE;
        return true;
    }
    if (lead > 0 || singles_behind) {
        ChunkRecurrenceArgs one = a;
        if (!singles_behind) one.num_seqs = lead;
        *rc = launch_single_recurrence(form, one, recurrence_singles(a.num_seqs, lead, rest), dtype, s);
        if (*rc != NV_OK) return true;
    }
    a.chunks = (float*)workspace;
    a.columns = (char*)workspace + ws.chunks;
    a.raw = (float*)((char*)a.columns + ws.columns);
    a.odd = (uint32_t*)((char*)a.raw + ws.raw);
    a.records = ws.records;
    if (rest) *rc = launch_chunk_recurrence(form, a, lead, ws.tokens, singles_behind, dtype, s);
    return true;
}

}  // namespace nv

extern "C" int64_t nv_recurrence_workspace_bytes(int form, int64_t T, int H, int D, int Dv, int num_seqs, int leading_singles,
                                                 int dtype) {
    if (form < 0 || form > 2 || T <= 0 || H <= 0 || D <= 0 || Dv <= 0 || leading_singles < 0 || num_seqs <= leading_singles ||
        !nv::recurrence_built(D, Dv))
        return 0;
    // (never less than chunks of 8 would need: more rows in as many sequences need no less, whichever they are taken in)
    const int seqs = num_seqs - leading_singles;
    int64_t need = nv::CrWorkspace(form, 8, T, H, D, Dv, seqs, dtype).bytes();
    if (nv::cr_chunk_tokens(form, T - leading_singles, seqs, H, D, Dv) == nv::kCrChunk)
        need = std::max(need, nv::CrWorkspace(form, nv::kCrChunk, T, H, D, Dv, seqs, dtype).bytes());
    return need;
}
