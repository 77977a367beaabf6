// The recurrences of chunk_recurrence.hip in chunks of 8 tokens, for short portions and full grids (the rule is `cr_chunk_tokens`): a
// chunk of 16 that holds a few tokens costs what a full one does, and its operands are twice the memory.
//
// With the names of that file, 16 rows take both K and Q here, and what the tokens do to each other is solved into one matrix:
//
//   C = [K; Q] S        16 rows, K_t = k_t G_t (general: u_t G_(t-1)), Q_t = q_t G_t
//   [U; O] = M C + M2 V 16 x 16 and 16 x 8 matrices of the chunk alone (write has no U and no M: O = C + M2 V)
//   S <- diag(G_8) S + K^^T V (general, write) + X^^T U (gated, general),   K^_t = k_t G_8 / G_t
//
// M and M2 come from the pair products and the inverse of a unit lower triangular 8 x 8 matrix by forward substitution.  The pair
// products' two sides are taken relative to the middle of the chunk, four factors on either side, where no channel of the chunk has four
// that multiply to less than 2^-80, else in four sets by where s and t part.  A wave decides by its chunk alone.
//
// Two launches: a wave per chunk and head makes the operands; the second walks the chunks of a (sequence, head, 16 value columns).
// U comes out in the lower half of the lanes; v_permlane32_swap spreads its 8 rows over all four groups, so that an update of
// a 16-channel tile takes two MFMAs.  A chunk takes 54 (gated) / 70 (general) / 50 (write) MFMAs of 32 cycles per 16 columns of 128
// channels, 0.81 us with its chain of exchange, M and update.
//
// Against 64 bits: states 0.98 to 1.03 (gated), 1.30 to 1.51 (general), 1.00 (write) times the token-by-token launch's error, all below
// 3.4e-7; read-outs 0.98 to 1.10, 1.0 to 1.25, 1.02 to 1.12 times.
#include "chunk_recurrence_parts.h"
#include "../../include/nanovllm_hip_mixers.h"

namespace nv {

constexpr int kCrShort = 8;

// The lower half's `lo` in the lower half of the lanes, the lower half's `hi` in the upper one.
__device__ __forceinline__ float cr_spread(float lo, float hi) {
    return __builtin_bit_cast(float, __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, lo), __builtin_bit_cast(int, hi), false, false)[0]);
}
// LDS writes of this wave are done.
__device__ __forceinline__ void cr_wave_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// One record per (head, chunk), in the order in which the second launch's lanes read it.
template <int FORM, int D>
struct CrShortRecord {
    static constexpr int kRows = FORM == kCrWrite ? 8 : 16;       // of [K; Q]: write has no K
    static constexpr int kUpd = FORM == kCrGeneral ? 2 : 1;       // update operands: K^ and / or X^
    static constexpr int kq = 0;                                  // [tile][g][row][4 channels]
    static constexpr int upd = kq + kRows * D;                    // [operand][tile][g][channel][2 tokens]
    static constexpr int decay = upd + kUpd * 8 * D;              // [channel]
    static constexpr int m = decay + D;                           // [16][16]
    static constexpr int m2 = m + (FORM == kCrWrite ? 0 : 256);   // [16][8] (write: [8][8])
    static constexpr int words = m2 + 8 * kRows;
};

// ------------------------------------------------------------------------------------------------ first launch
// A wave per (chunk, head); a lane owns two neighbouring channels and all 8 tokens, so running products need no exchange.  LDS
// (the wave's own) only turns the pair products' operands and [K; Q] into the order of the matrix cores.
template <typename T, int FORM, int D>
struct CrShortLds {
    static constexpr int kRow = D + 4;                            // rows of D channels start on different banks
    static constexpr int kRight = FORM == kCrGeneral ? 16 : 8;
    float left[16 * kRow], right[kRight * kRow];                  // pair products' operands; then left holds [K; Q]
};

template <typename T, int FORM, int D, bool VEC>
__global__ __launch_bounds__(256) void short_recurrence_chunks_kernel(const ChunkRecurrenceArgs a, const int first_seq) {
    constexpr int NM = D / 16, NX = FORM == kCrGated ? 3 : FORM == kCrGeneral ? 4 : 2;
    typedef CrShortLds<T, FORM, D> Lds;
    typedef CrShortRecord<FORM, D> Rec;
    typedef CrRaw<T> In;
    constexpr int ROW = Lds::kRow;
    __shared__ __attribute__((aligned(16))) Lds all[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4, h = blockIdx.y * 4 + wave;
    const int64_t rec = blockIdx.x;
    const int row0 = a.cu_q[first_seq];
    int lo = first_seq, hi = a.num_seqs;              // the last sequence whose records start at or in front of this one
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cr_first_record<kCrShort>(a.cu_q[mid] - row0, mid - first_seq) <= rec) lo = mid; else hi = mid;
    }
    const int b = lo, q0 = a.cu_q[b], len = a.cu_q[b + 1] - q0;
    const int64_t c64 = rec - cr_first_record<kCrShort>(q0 - row0, b - first_seq);
    if (len < 2 || c64 * kCrShort >= len || h >= a.H) return;
    const int t0 = q0 + (int)c64 * kCrShort, n = min(kCrShort, q0 + len - t0);
    float* out = a.chunks + (h * a.records + rec) * Rec::words;
    Lds& lds = all[wave];

    const bool in_row = 2 * lane < D;
    const int d = in_row ? 2 * lane : 0;
    CrPair<T, VEC> raw[NX][8];
    {
        const void* xs[4] = {a.x0, a.x1, a.x2, a.x3};
        const int64_t ss[4] = {a.s0, a.s1, a.s2, a.s3};
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int hj = (FORM == kCrGated && j < 2) ? h / a.group : h;
            const T* p = (const T*)xs[j] + (int64_t)t0 * ss[j] + (int64_t)hj * D;
#pragma unroll
            for (int t = 0; t < 8; ++t) {             // (past the end: the chunk's first row, dropped below)
                const T* row = p + (t < n ? t : 0) * ss[j];
                raw[j][t].load(row + d);
            }
        }
    }
    float odd[8] = {};                                // NaN with a value that is not finite
    {
        const T* v = (const T*)a.v + (int64_t)t0 * a.sv + (int64_t)h * a.Dv;
        T* to = (T*)a.columns + (h * a.records + rec) * 8 * a.Dv;
        for (int c = 2 * lane; c < a.Dv; c += 128) {
            CrPair<T, VEC> r[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) r[t].load(v + (t < n ? t : 0) * a.sv + c);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                r[t].keep(t < n);
                r[t].store(to + t * a.Dv + c);
                odd[t] += r[t].value(0) * 0.f;
                odd[t] += r[t].value(1) * 0.f;
            }
        }
    }
    float beta = 0.f;                                 // raw, of token lane % 8
    if constexpr (FORM == kCrGated) beta = CrRaw<T>::value(In::load((const T*)a.b_raw + (int64_t)(t0 + min(lane & 7, n - 1)) * a.b_stride + h));
    float c0[2], c1[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        c0[i] = FORM == kCrGated ? expf(a.c0[h]) : a.c0[h * D + d + i];
        c1[i] = a.c1[h * D + d + i];
    }
    CrElem el[8][2];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float in[4];
#pragma unroll
            for (int j = 0; j < NX; ++j) {
                in[j] = raw[j][t].value(i);
                odd[t] += in[j] * 0.f;
            }
            el[t][i] = cr_elem<FORM>(in, c0[i], c1[i], a.p0);
            if (t >= n || !in_row) el[t][i] = CrElem{1.f, 0.f, 0.f, 0.f};
        }
    }
    const float sum_odd = ((odd[0] + odd[1]) + (odd[2] + odd[3])) + ((odd[4] + odd[5]) + (odd[6] + odd[7])) + beta * 0.f;
    const bool any_odd = __any(sum_odd != 0.f);
    if (lane == 0) a.odd[h * a.records + rec] = any_odd;
    float kk = 0.f, qq = 0.f;                         // sums of squares of token lane % 8
    if constexpr (FORM != kCrWrite) {
        auto squares = [&](auto of) {                 // 8 tokens' sums over 64 lanes: halved three times over the lanes, then summed
            float s[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) s[t] = of(t);
            const bool o1 = lane & 1, o2 = lane & 2, o4 = lane & 4;
            float u[4], w[2];
#pragma unroll
            for (int t = 0; t < 4; ++t) u[t] = (o1 ? s[2 * t + 1] : s[2 * t]) + dpp_f32<0xB1>(o1 ? s[2 * t] : s[2 * t + 1]);
#pragma unroll
            for (int t = 0; t < 2; ++t) w[t] = (o2 ? u[2 * t + 1] : u[2 * t]) + dpp_f32<0x4E>(o2 ? u[2 * t] : u[2 * t + 1]);
            float r = (o4 ? w[1] : w[0]) + __shfl_xor(o4 ? w[0] : w[1], 4);
            r += __shfl_xor(r, 8);
            r += __shfl_xor(r, 16);
            return r + __shfl_xor(r, 32);
        };
        kk = squares([&](int t) { return el[t][0].k * el[t][0].k + el[t][1].k * el[t][1].k; });
        if constexpr (FORM == kCrGated) qq = squares([&](int t) { return el[t][0].q * el[t][0].q + el[t][1].q * el[t][1].q; });
    }
    // ---- pair products: entry (row 4 g + e, column l16): rows k | q, columns k | a k
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
    auto products = [&] {                             // of the operands in LDS
        cr_wave_sync();
        f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0, p2 = p0, p3 = p0;
        const int lrow = FORM == kCrWrite ? (8 + (l16 & 7)) : l16;
        const float* lf = lds.left + lrow * ROW + 4 * g;
        const float* rt = lds.right + (Lds::kRight == 16 ? l16 : (l16 & 7)) * ROW + 4 * g;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const f32x4 x = *(const f32x4*)(lf + 16 * m), y = *(const f32x4*)(rt + 16 * m);
            p0 = cr_mfma(x[0], y[0], p0);
            p1 = cr_mfma(x[1], y[1], p1);
            p2 = cr_mfma(x[2], y[2], p2);
            p3 = cr_mfma(x[3], y[3], p3);
        }
        return (p0 + p1) + (p2 + p3);
    };
    // relative to the middle: left sides G_t / G_4, right sides G_4 / G_t
    float side[2][8];
    bool near = true;                                 // (false with a decay that is not a number)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        side[i][3] = 1.f;                             // of tokens 0 .. 3: products behind the token; 4 .. 7: through the token
#pragma unroll
        for (int t = 2; t >= 0; --t) side[i][t] = side[i][t + 1] * el[t + 1][i].w;
        side[i][4] = el[4][i].w;
#pragma unroll
        for (int t = 5; t < 8; ++t) side[i][t] = side[i][t - 1] * el[t][i].w;
        near = near && side[i][0] * el[0][i].w >= kCrNear && side[i][7] >= kCrNear;
    }
    if (__all(near)) {
        if (in_row) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                float lv[2], rv[2], hb[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float inv = __builtin_amdgcn_rcpf(side[i][t]);
                    lv[i] = t < 4 ? inv : side[i][t];
                    rv[i] = t < 4 ? side[i][t] : inv;
                    if constexpr (FORM == kCrGeneral) // the old state: through the token before
                        hb[i] = t == 0 ? __builtin_amdgcn_rcpf(side[i][0] * el[0][i].w)
                                       : t < 4 ? __builtin_amdgcn_rcpf(side[i][t - 1]) : t == 4 ? 1.f : side[i][t - 1];
                    else hb[i] = lv[i];
                }
                if constexpr (FORM != kCrWrite) *(float2*)(lds.left + t * ROW + d) = make_float2(el[t][0].k * hb[0], el[t][1].k * hb[1]);
                *(float2*)(lds.left + (8 + t) * ROW + d) = make_float2(el[t][0].q * lv[0], el[t][1].q * lv[1]);
                *(float2*)(lds.right + t * ROW + d) = make_float2(el[t][0].k * rv[0], el[t][1].k * rv[1]);
                if constexpr (FORM == kCrGeneral)
                    *(float2*)(lds.right + (8 + t) * ROW + d) = make_float2(el[t][0].a * rv[0], el[t][1].a * rv[1]);
            }
        }
        p = products();
    } else {
#pragma unroll 1
        for (int part = 4; part >= 0; part = part == 1 ? 0 : part == 0 ? -1 : part / 2) {       // 4, 2, 1; 0: s = t
            if (in_row) {
                float lv[2] = {1.f, 1.f}, rv[2] = {1.f, 1.f};
#pragma unroll
                for (int t = 0; t < 8; ++t) {         // from the start of its part through the token
                    if ((t & (part - 1)) == 0) lv[0] = lv[1] = 1.f;
                    const float before[2] = {lv[0], lv[1]};
#pragma unroll
                    for (int i = 0; i < 2; ++i) lv[i] *= part ? el[t][i].w : 1.f;
                    const float* kv = FORM == kCrGeneral ? before : lv;
                    if constexpr (FORM != kCrWrite) *(float2*)(lds.left + t * ROW + d) = make_float2(el[t][0].k * kv[0], el[t][1].k * kv[1]);
                    *(float2*)(lds.left + (8 + t) * ROW + d) = make_float2(el[t][0].q * lv[0], el[t][1].q * lv[1]);
                }
#pragma unroll
                for (int t = 7; t >= 0; --t) {        // behind the token to the end of its part
                    if (((t + 1) & (part - 1)) == 0) rv[0] = rv[1] = 1.f;
                    *(float2*)(lds.right + t * ROW + d) = make_float2(el[t][0].k * rv[0], el[t][1].k * rv[1]);
                    if constexpr (FORM == kCrGeneral)
                        *(float2*)(lds.right + (8 + t) * ROW + d) = make_float2(el[t][0].a * rv[0], el[t][1].a * rv[1]);
#pragma unroll
                    for (int i = 0; i < 2; ++i) rv[i] *= part ? el[t][i].w : 1.f;
                }
            }
            const f32x4 of = products();
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int apart = ((4 * g + e) & 7) ^ (l16 & 7);
                if (part ? apart >= part && apart < 2 * part : apart == 0) p[e] = of[e];
            }
            cr_wave_sync();
        }
    }
    // ---- [K; Q], K^, X^ and the chunk's decay
    float G[2][8], F[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        G[i][0] = el[0][i].w;
        F[i][7] = 1.f;
#pragma unroll
        for (int t = 1; t < 8; ++t) {
            G[i][t] = G[i][t - 1] * el[t][i].w;
            F[i][7 - t] = F[i][8 - t] * el[8 - t][i].w;
        }
    }
    cr_wave_sync();
    if (in_row) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            if constexpr (FORM == kCrGated)
                *(float2*)(lds.left + t * ROW + d) = make_float2(el[t][0].k * G[0][t], el[t][1].k * G[1][t]);
            if constexpr (FORM == kCrGeneral)
                *(float2*)(lds.left + t * ROW + d) = make_float2(t ? el[t][0].k * G[0][t ? t - 1 : 0] : el[t][0].k,
                                                                 t ? el[t][1].k * G[1][t ? t - 1 : 0] : el[t][1].k);
            *(float2*)(lds.left + (8 + t) * ROW + d) = make_float2(el[t][0].q * G[0][t], el[t][1].q * G[1][t]);
        }
        *(float2*)(out + Rec::decay + d) = make_float2(G[0][7], G[1][7]);
        // token pairs in the order of the lane groups that supply them: of V 0 1 | 2 3 | 4 5 | 6 7, of U 0 1 | 4 5 | 2 3 | 6 7
        auto store = [&](int which, auto of, bool u) {
#pragma unroll
            for (int pos = 0; pos < 4; ++pos) {
                const int t = u ? (pos == 1 ? 4 : pos == 2 ? 2 : 2 * pos) : 2 * pos;
                float* to = out + Rec::upd + which * 8 * D + (((d >> 4) * 4 + pos) * 16 + (d & 15)) * 2;
                *(f32x4*)to = f32x4{of(t, 0) * F[0][t], of(t + 1, 0) * F[0][t + 1], of(t, 1) * F[1][t], of(t + 1, 1) * F[1][t + 1]};
            }
        };
        if constexpr (FORM == kCrGated) store(0, [&](int t, int i) { return el[t][i].k; }, true);
        else store(0, [&](int t, int i) { return el[t][i].k; }, false);
        if constexpr (FORM == kCrGeneral) store(1, [&](int t, int i) { return el[t][i].a; }, true);
    }
    cr_wave_sync();
    if constexpr (FORM == kCrWrite) {
        // lanes: (tile, g, row) of 8 rows, 16 bytes each
#pragma unroll
        for (int i = 0; i < NM / 2; ++i) {
            const int at = i * 64 + lane;             // tile at / 32, g (at / 8) % 4, row at % 8
            *(f32x4*)(out + Rec::kq + at * 4) = *(const f32x4*)(lds.left + (8 + (at & 7)) * ROW + 16 * (at >> 5) + 4 * ((at >> 3) & 3));
        }
    } else {
#pragma unroll
        for (int m = 0; m < NM; ++m) *(f32x4*)(out + Rec::kq + (m * 64 + lane) * 4) = *(const f32x4*)(lds.left + l16 * ROW + 16 * m + 4 * g);
    }
    // ---- M and M2
    float* m = out + Rec::m;
    float* m2 = out + Rec::m2;
    if constexpr (FORM == kCrWrite) {
        if (g < 2 && l16 < 8) {
#pragma unroll
            for (int e = 0; e < 4; ++e) m2[(4 * g + e) * 8 + l16] = l16 <= 4 * g + e ? p[e] : 0.f;
        }
        return;
    }
    const int j = lane & 7;
    const bool in = j < n;
    const float kn = in ? 1.0f / sqrtf(kk + a.p1) : 0.f;                               // of token lane % 8
    const float qn = FORM == kCrGated ? 1.0f / sqrtf((qq + a.p1) * (float)D) : 1.0f;
    // Lanes 0 - 7: columns of M for the rows K; lanes 8 - 15: columns of M2; lanes 16 - 23: columns of M for the rows Q.
    const int kind = lane >> 3;
    float y[8], o[8];
    if constexpr (FORM == kCrGated) {
        // u = T beta (v - kn K^T S), T = (I + A)^-1, A_ts = beta_t kn_t kn_s P_ts (s < t);  y_t = kn_t u_t is what X^ = k G_8 / G_t
        // takes, o_t = qn_t (Q^T S + sum_(s <= t) P'_ts y_s)
        beta = in ? cr_sigmoid(beta) : 0.f;
        const float rhs = kind == 0 ? -beta * kn * kn : kind == 1 ? beta * kn : 0.f;
        const float scale = beta * kn * kn;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < t; ++i) s += cr_lane(p[t & 3], (t >> 2) * 16 + i) * y[i];
            y[t] = (t == j ? rhs : 0.f) - cr_lane(scale, t) * s;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float s = (kind == 2 && t == j) ? 1.f : 0.f;
#pragma unroll
            for (int i = 0; i <= t; ++i) s += cr_lane(p[t & 3], (2 + (t >> 2)) * 16 + i) * y[i];
            o[t] = s * cr_lane(qn, t);
        }
    } else {
        // x_t = u_t^T S_(t-1) = kn_t (K^T S + sum_(s < t) P_ts(k, k) v_s - P_ts(k, a k) kn_s x_s);  y_t = kn_t x_t, taken with
        // a minus sign by X^ = a k G_8 / G_t;  o_t = Q^T S + sum_(s <= t) P_ts(r, k) v_s - P_ts(r, a k) y_s
        const float kn2 = kn * kn;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float nt = __shfl(p[t & 3], (t >> 2) * 16 + j);
            float s = kind == 0 ? (t == j ? 1.f : 0.f) : kind == 1 ? (t > j ? nt : 0.f) : 0.f;
#pragma unroll
            for (int i = 0; i < t; ++i) s -= cr_lane(p[t & 3], (t >> 2) * 16 + 8 + i) * y[i];
            y[t] = cr_lane(kn2, t) * s;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float bt = __shfl(p[t & 3], (2 + (t >> 2)) * 16 + j);
            float s = kind == 2 ? (t == j ? 1.f : 0.f) : kind == 1 ? (t >= j ? bt : 0.f) : 0.f;
#pragma unroll
            for (int i = 0; i <= t; ++i) s -= cr_lane(p[t & 3], (2 + (t >> 2)) * 16 + 8 + i) * y[i];
            o[t] = s;
        }
    }
    if (kind < 3) {
        float* to = kind == 1 ? m2 + j : m + (kind == 2 ? 8 : 0) + j;
        const int ld = kind == 1 ? 8 : 16;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            to[t * ld] = FORM == kCrGeneral ? -y[t] : y[t];
            to[(8 + t) * ld] = o[t];
        }
    }
}

// ------------------------------------------------------------------------------------------------ second launch
// RS waves per (sequence, head, 16 value columns), each with D / RS key channels of the state in MFMA accumulators; RS = 2: the
// waves' parts of [K; Q] S are exchanged through LDS.  A workgroup has four of these waves, one on each SIMD of a CU, and four that
// do nothing but move: records and columns of V four chunks ahead into registers and two ahead into LDS (three slots), read-outs from LDS to
// memory.  One barrier a chunk.  The products alone are bound by their chain (product, exchange, M, update); with the loads and
// stores in the same waves every chunk also paid for their issue (gated, 4 x 1501 .. 2048 tokens, 16 heads: 264 us instead of 219).
template <typename T, int FORM, int D, int RS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void short_recurrence_states_kernel(
    const ChunkRecurrenceArgs a, const int first_seq) {
    constexpr int NM = D / 16 / RS;                   // tiles of a wave
    typedef CrShortRecord<FORM, D> Rec;
    constexpr int ROUNDS = (Rec::words + 1023) / 1024;
    constexpr int COLS = 64 / RS, PER = 2 / RS;       // value columns of the workgroup; elements of a row of V a thread moves
    __shared__ __attribute__((aligned(16))) float slots[3][Rec::words];
    __shared__ __attribute__((aligned(8))) float vs[3][kCrShort][COLS], os[2][kCrShort][COLS];
    __shared__ f32x4 part[RS == 1 ? 1 : 2][4][64];
    // Workgroups go to the eight XCDs in turn: an XCD takes neighbouring heads.
    const int pair = gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
    const int b = first_seq + pair / a.H, h = pair % a.H;
    const int q0 = a.cu_q[b], len = a.cu_q[b + 1] - q0;
    if (len < 2) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int chunks = (len + kCrShort - 1) / kCrShort, Dv = a.Dv;

    if (wave >= 4) {
        // ---------------------------------------------------------------- the movers
        const int tid = threadIdx.x - 256;
        const int64_t first = (int64_t)h * a.records + cr_first_record<kCrShort>(q0 - a.cu_q[first_seq], b - first_seq);
        const float* rec = a.chunks + first * Rec::words;
        const int tok = tid >> 5, col = (tid & 31) * PER, col_all = blockIdx.y * COLS + col;
        // (columns past the end: the last ones, used by waves that write nothing)
        const T* v = (const T*)a.columns + first * 8 * Dv + tok * Dv + min(col_all, Dv - PER);
        float* o = a.raw + ((int64_t)h * a.T + q0 + tok) * Dv + col_all;
        struct Staged {
            f32x4 r[ROUNDS];
            CrColumns<T, PER> v;
        };
        auto fetch = [&](int c, Staged& st) {
            c = min(c, chunks - 1);
            const float* rc = rec + (int64_t)c * Rec::words;
            st.v.load(v + (int64_t)c * 8 * Dv);
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
            if (c * kCrShort + tok < len && col_all < Dv) {
#pragma unroll
                for (int e = 0; e < PER; ++e) o[(int64_t)c * kCrShort * Dv + e] = os[c & 1][tok][col + e];
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
        const uint32_t* flags = a.odd + (int64_t)h * a.records + cr_first_record<kCrShort>(q0 - a.cu_q[first_seq], b - first_seq);
        for (int c = lane; c < chunks; c += 64) odd |= flags[c];
        odd = __any(odd != 0);
    }
    const int at_kq = Rec::kq + (FORM == kCrWrite ? (g * 8 + (l16 & 7)) * 4 + d0 * 8 : lane * 4 + d0 * 16);
    constexpr int kq_tile = 16 * Rec::kRows;
    const int at_upd = Rec::upd + lane * 2 + d0 * 8, at_dec = Rec::decay + d0 + ((l16 + 4 * g) & 15), at_m = Rec::m + l16 * 16 + 4 * g;
    const int at_m2 = Rec::m2 + (FORM == kCrWrite ? l16 & 7 : l16) * 8 + 2 * g;
    f32x4 x[NM];
    auto read_x = [&](int at) {
#pragma unroll
        for (int m = 0; m < NM; ++m) x[m] = *(const f32x4*)(slots[at] + kq_tile * m + at_kq);
    };
    cr_group_barrier();
    read_x(0);
    int at = 0;
    auto chunk = [&](auto odd_tag, int c) {           // chunk c from slot `at`
        constexpr bool ODD = decltype(odd_tag)::value;
        const float* rc = slots[at];
        f32x4 y;
        float dec[NM];                                // lane e of group g: the decay of row 4 g + e of the tile
        float2 uk[NM], ux[NM];
        float vv[2];
        const float2 y2 = *(const float2*)(rc + at_m2);
#pragma unroll
        for (int e = 0; e < 2; ++e) vv[e] = vs[at][2 * g + e][in_group];
        if constexpr (FORM != kCrWrite) y = *(const f32x4*)(rc + at_m);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            dec[m] = rc[16 * m + at_dec];
            if constexpr (FORM != kCrGated) uk[m] = *(const float2*)(rc + 128 * m + at_upd);
            if constexpr (FORM != kCrWrite) ux[m] = *(const float2*)(rc + (Rec::kUpd - 1) * 8 * D + 128 * m + at_upd);
        }
        f32x4 c0 = {0.f, 0.f, 0.f, 0.f}, d = c0, c1 = c0, c2 = c0, c3 = c0;   // (four sums: a quarter of the roundings one after the other)
        __builtin_amdgcn_sched_barrier(0);            // the reads are on their way before the products
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            c0 = cr_mfma(x[m][0], S[m][0], c0);
            c1 = cr_mfma(x[m][1], S[m][1], c1);
            c2 = cr_mfma(x[m][2], S[m][2], c2);
            c3 = cr_mfma(x[m][3], S[m][3], c3);
        }
        d = cr_mfma(y2.x, vv[0], d);
        d = cr_mfma(y2.y, vv[1], d);
        __builtin_amdgcn_sched_barrier(0);            // (d's products run while the last of C comes out: 298 -> 286 us, gated)
        c0 = (c0 + c1) + (c2 + c3);
        if constexpr (RS > 1) part[c & 1][wave][lane] = c0;
        cr_group_barrier();                           // chunk c + 1 is in its slot; chunk c - 1's slot is free
        f32x4 other;
        if constexpr (RS > 1) other = part[c & 1][wave ^ 1][lane];
        at = at == 2 ? 0 : at + 1;
        read_x(at);
        // the state moves on: rows 4 g + e of tile m decay, then take the chunk's writes
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            S[m][0] *= dpp_f32<0x150>(dec[m]);        // row_newbcast e: lane e of the group
            S[m][1] *= dpp_f32<0x151>(dec[m]);
            S[m][2] *= dpp_f32<0x152>(dec[m]);
            S[m][3] *= dpp_f32<0x153>(dec[m]);
        }
        if constexpr (FORM != kCrGated) {
#pragma unroll
            for (int m = 0; m < NM; ++m) S[m] = cr_mfma(uk[m].x, vv[0], S[m]);
#pragma unroll
            for (int m = 0; m < NM; ++m) S[m] = cr_mfma(uk[m].y, vv[1], S[m]);
        }
        if constexpr (RS > 1) c0 += other;
        if constexpr (!ODD) {
            if constexpr (FORM != kCrWrite) {
#pragma unroll
                for (int e = 0; e < 4; ++e) d = cr_mfma(y[e], c0[e], d);
            }
        } else {
            // A zero above the diagonal keeps a later token out only while that token's value is finite: token by token, each
            // from operands that end with it; a row of Q counts for its own read-out alone.
            f32x4 rows = d;
#pragma unroll 1
            for (int t = 0; t < kCrShort; ++t) {
                f32x4 u = {0.f, 0.f, 0.f, 0.f};
                u = cr_mfma(y2.x, 2 * g <= t ? vv[0] : 0.f, u);
                u = cr_mfma(y2.y, 2 * g + 1 <= t ? vv[1] : 0.f, u);
                f32x4 o = u;
                if constexpr (FORM != kCrWrite) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int at = (4 * g + e) & 7;
                        u = cr_mfma(y[e], g < 2 && at <= t ? c0[e] : 0.f, u);
                        o = cr_mfma(y[e], (g < 2 ? at <= t : at == t) ? c0[e] : 0.f, o);
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (((4 * g + e) & 7) == t) rows[e] = g < 2 ? u[e] : o[e];
            }
            d = rows;
        }
        if constexpr (FORM == kCrWrite) {
            d += c0;
        } else {
            // tokens 0, 1 | 4, 5 of U sit in groups 0 | 1, tokens 2, 3 | 6, 7 move to groups 2 | 3
            const float u0 = cr_spread(d[0], d[2]), u1 = cr_spread(d[1], d[3]);
#pragma unroll
            for (int m = 0; m < NM; ++m) S[m] = cr_mfma(ux[m].x, u0, S[m]);
#pragma unroll
            for (int m = 0; m < NM; ++m) S[m] = cr_mfma(ux[m].y, u1, S[m]);
        }
        // write: rows 0 - 7 of the products are the read-outs (8 - 15 repeat them), else rows 8 - 15
        if (rp == 0 && (FORM == kCrWrite ? g < 2 : g >= 2)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) os[c & 1][4 * (g & 1) + e][in_group] = d[e];
        }
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
#pragma unroll
        for (int e = 0; e < 4; ++e) slot[(int64_t)(16 * m + e) * Dv] = S[m][e];
    }
}

// ------------------------------------------------------------------------------------------------ launches
int64_t short_recurrence_records(int64_t rows, int seqs) { return cr_first_record<kCrShort>(rows, seqs) + 1; }
int short_recurrence_words(int form, int D) {
    const int rows = form == kCrWrite ? 8 : 16;
    return rows * D + (form == kCrGeneral ? 2 : 1) * 8 * D + D + (form == kCrWrite ? 0 : 256) + 8 * rows;
}

template <typename T, int FORM, int D>
static void short_chunks_of_size(const ChunkRecurrenceArgs& a, int first_seq, bool vec, int waves, hipStream_t s) {
    const dim3 prep((unsigned)a.records, (unsigned)((a.H + 3) / 4)), block(512);
    const unsigned pairs = (unsigned)((a.num_seqs - first_seq) * a.H), tiles = (unsigned)(a.Dv / 16);
    if (vec) hipLaunchKernelGGL((short_recurrence_chunks_kernel<T, FORM, D, true>), prep, dim3(256), 0, s, a, first_seq);
    else hipLaunchKernelGGL((short_recurrence_chunks_kernel<T, FORM, D, false>), prep, dim3(256), 0, s, a, first_seq);
    if (waves == 2) hipLaunchKernelGGL((short_recurrence_states_kernel<T, FORM, D, 2>), dim3(pairs, (tiles + 1) / 2), block, 0, s, a, first_seq);
    else hipLaunchKernelGGL((short_recurrence_states_kernel<T, FORM, D, 1>), dim3(pairs, (tiles + 3) / 4), block, 0, s, a, first_seq);
}

template <typename T, int FORM>
static void short_chunks_of(const ChunkRecurrenceArgs& a, int first_seq, bool vec, int waves, hipStream_t s) {
    switch (a.D) {
        case 32: short_chunks_of_size<T, FORM, 32>(a, first_seq, vec, waves, s); break;
        case 64: short_chunks_of_size<T, FORM, 64>(a, first_seq, vec, waves, s); break;
        case 96: short_chunks_of_size<T, FORM, 96>(a, first_seq, vec, waves, s); break;
        default: short_chunks_of_size<T, FORM, 128>(a, first_seq, vec, waves, s); break;
    }
}

void launch_short_recurrence(int form, const ChunkRecurrenceArgs& a, int first_seq, bool vec, int waves, int dtype, hipStream_t s) {
    if (dtype == NV_DTYPE_BF16) {
        if (form == kCrGated) short_chunks_of<__bf16, kCrGated>(a, first_seq, vec, waves, s);
        else if (form == kCrGeneral) short_chunks_of<__bf16, kCrGeneral>(a, first_seq, vec, waves, s);
        else short_chunks_of<__bf16, kCrWrite>(a, first_seq, vec, waves, s);
    } else {
        if (form == kCrGated) short_chunks_of<float, kCrGated>(a, first_seq, vec, waves, s);
        else if (form == kCrGeneral) short_chunks_of<float, kCrGeneral>(a, first_seq, vec, waves, s);
        else short_chunks_of<float, kCrWrite>(a, first_seq, vec, waves, s);
    }
}

}  // namespace nv
