// What the launches of the recurrences share: decays and vectors of a token from its raw projections, loads of rows, products.
#pragma once
#include <type_traits>

#include "chunk_recurrence.h"
#include "row_pieces.h"

namespace nv {

constexpr float kCrNear = 8.27180613e-25f;            // 2^-80

__device__ __forceinline__ float cr_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
// log(1 + exp(x)) = max(x, 0) + log(1 + u), u = exp(-|x|) <= 1; log(1 + u) = 2 atanh(s), s = u / (2 + u) <= 1/3, by its series
// (the first term left out is below 2^-26 of the sum).  s carries the roundings of 2 + u and of the reciprocal.  Within 4 % of
// log1pf's error, and 7 instead of 19 us of a 285 us call (gated, 4 prompts of 1501 .. 2048 tokens); the hardware's logarithm and exponential took none of
// these, with 1.35 times the error in a decay.
__device__ __forceinline__ float cr_softplus(float x) {
    const float u = expf(-fabsf(x)), n = 2.0f + u, lost = u - (n - 2.0f), r = __builtin_amdgcn_rcpf(n);
    float s = u * r;
    s = fmaf(fmaf(-s, lost, fmaf(-s, n, u)), r, s);
    const float z = s * s;
    float p = 1.0f / 15.0f;
    p = fmaf(p, z, 1.0f / 13.0f);
    p = fmaf(p, z, 1.0f / 11.0f);
    p = fmaf(p, z, 1.0f / 9.0f);
    p = fmaf(p, z, 1.0f / 7.0f);
    p = fmaf(p, z, 1.0f / 5.0f);
    p = fmaf(p, z, 1.0f / 3.0f);
    return fmaxf(x, 0.f) + fmaf(2.0f * s * z, p, 2.0f * s);
}

// Decay and vectors of one token and channel from its raw projections (x: in the order of x0 .. x3).
struct CrElem {
    float w, k, q, a;                                 // decay; k (raw scale); q / r; removal rate times k (general)
};
template <int FORM>
__device__ __forceinline__ CrElem cr_elem(const float* x, float c0, float c1, float p0) {
    CrElem e;
    if constexpr (FORM == kCrGated) {
        e.w = expf(-c0 * cr_softplus(x[2] + c1));     // c0: exp(A_log)
        e.k = x[1];
        e.q = x[0];
        e.a = 0.f;
    } else if constexpr (FORM == kCrGeneral) {
        e.w = expf(-p0 * cr_sigmoid(x[2] + c0));
        e.k = x[1];
        e.q = x[0];
        e.a = cr_sigmoid(x[3] + c1) * x[1];
    } else {
        e.w = c1 + (1.0f - c1) * cr_sigmoid(x[1] + c0);
        e.k = 1.0f - e.w;
        e.q = x[0] * cr_sigmoid(x[0]);
        e.a = 0.f;
    }
    return e;
}

// An element on its way from memory in a register of its own: packed halves would make every load wait for the one before.
template <typename T> struct CrRaw;
template <> struct CrRaw<__bf16> {
    typedef uint32_t type;
    static __device__ __forceinline__ uint32_t load(const __bf16* p) { return *(const uint16_t*)p; }
    static __device__ __forceinline__ float value(uint32_t r) { return __builtin_bit_cast(float, r << 16); }
};
// Two neighbouring elements by one load (VEC) or two.
template <typename T, bool VEC> struct CrPair;
template <> struct CrPair<__bf16, true> {
    uint32_t r;
    __device__ __forceinline__ void load(const __bf16* p) { r = *(const uint32_t*)p; }
    __device__ __forceinline__ float value(int i) const { return i ? bf16_hi(r) : bf16_lo(r); }
    __device__ __forceinline__ void keep(bool in) { r = in ? r : 0u; }
    __device__ __forceinline__ void store(__bf16* p) const { *(uint32_t*)p = r; }
};
template <> struct CrPair<float, true> {
    float2 r;
    __device__ __forceinline__ void load(const float* p) { r = *(const float2*)p; }
    __device__ __forceinline__ float value(int i) const { return i ? r.y : r.x; }
    __device__ __forceinline__ void keep(bool in) { r = in ? r : make_float2(0.f, 0.f); }
    __device__ __forceinline__ void store(float* p) const { *(float2*)p = r; }
};
template <typename T> struct CrPair<T, false> {
    typename CrRaw<T>::type r[2];
    __device__ __forceinline__ void load(const T* p) {
        r[0] = CrRaw<T>::load(p);
        r[1] = CrRaw<T>::load(p + 1);
    }
    __device__ __forceinline__ float value(int i) const { return CrRaw<T>::value(r[i]); }
    __device__ __forceinline__ void keep(bool in) {
        r[0] = in ? r[0] : 0;
        r[1] = in ? r[1] : 0;
    }
    __device__ __forceinline__ void store(T* p) const {
        p[0] = (T)value(0);
        p[1] = (T)value(1);
    }
};
template <> struct CrRaw<float> {
    typedef float type;
    static __device__ __forceinline__ float load(const float* p) { return *p; }
    static __device__ __forceinline__ float value(float r) { return r; }
};

__device__ __forceinline__ f32x4 cr_mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float cr_lane(float x, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
// LDS writes of the workgroup's waves are done; loads from memory stay in flight.
__device__ __forceinline__ void cr_group_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int N> using CrRow = __attribute__((ext_vector_type(N))) float;
// PER neighbouring elements of a row of V by one load.
template <typename T, int PER> struct CrColumns : CrPair<T, true> {};
template <typename T> struct CrColumns<T, 1> {
    typename CrRaw<T>::type r;
    __device__ __forceinline__ void load(const T* p) { r = CrRaw<T>::load(p); }
    __device__ __forceinline__ float value(int) const { return CrRaw<T>::value(r); }
};
template <> struct CrColumns<__bf16, 4> {
    uint2 r;
    __device__ __forceinline__ void load(const __bf16* p) { r = *(const uint2*)p; }
    __device__ __forceinline__ float value(int i) const { return i & 1 ? bf16_hi(i < 2 ? r.x : r.y) : bf16_lo(i < 2 ? r.x : r.y); }
};
template <> struct CrColumns<float, 4> {
    f32x4 r;
    __device__ __forceinline__ void load(const float* p) { r = *(const f32x4*)p; }
    __device__ __forceinline__ float value(int i) const { return r[i]; }
};

// Records of a sequence start at (first row + (CHUNK - 1) x its number) / CHUNK: enough for the chunks in front, whatever the lengths,
// without a scan over them (rows and numbers counted from the first sequence of the launch).
template <int CHUNK>
__device__ __host__ __forceinline__ int64_t cr_first_record(int64_t first_row, int seq) {
    return (first_row + (int64_t)(CHUNK - 1) * seq) / CHUNK;
}

}  // namespace nv
