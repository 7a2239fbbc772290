// Per-event operand preparation and the write update of the routed GDN2
// recurrence, shared by the forward kernel and the backward replay so both
// execute the identical FP32 operation sequence (the backward replays the
// forward trajectory exactly from its snapshots).
//
// Reference: _pack (role_bank_dispatch.py:47-73: eb = b*p and ew = w*p rounded
// to the source dtype once), decay_transform (routed_update.py:5-13: eg = g*p
// in FP32) and _write (role_bank_kernel.py:35-43):
//   hd = diag(exp(eg)) M;  a = eb * k;  u = ew * v - a^T hd;  M' = hd + k u^T
#pragma once

#include "bdm_common.h"

namespace bdm {

// Row-side operands of one write event (one token, one head).
template <int S>
struct WriteRows {
    float key[S];    // k
    float decay[S];  // exp(eg)
    float eb[S];     // bf(b*p)
    float a[S];      // eb * k
};

// eg = g*p (routed decay) or g; eb = bf(b*p) in the controller dtype T.
template <typename T, int S>
__device__ __forceinline__ void prepare_write_rows(const float (&k)[S], const float (&g)[S], const float (&b)[S],
                                                   float pw, bool routed_decay, WriteRows<S> &w) {
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const float eg = routed_decay ? g[r] * pw : g[r];
        w.key[r] = k[r];
        w.decay[r] = __expf(eg);
        w.eb[r] = round_to<T>(b[r] * pw);
        w.a[r] = w.eb[r] * k[r];
    }
}

// Apply one write to the CPL columns a lane owns.  ew = bf(w*p) per column.
template <int S, int CPL>
__device__ __forceinline__ void apply_write(float (&h)[S][CPL], const WriteRows<S> &w, const float (&ew)[CPL],
                                            const float (&value)[CPL]) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        float erase = 0.f;
#pragma unroll
        for (int r = 0; r < S; ++r) {
            h[r][c] *= w.decay[r];
            erase = fmaf(w.a[r], h[r][c], erase);
        }
        const float u = fmaf(ew[c], value[c], -erase);
#pragma unroll
        for (int r = 0; r < S; ++r) h[r][c] = fmaf(w.key[r], u, h[r][c]);
    }
}

// Sums over lane pairs l, l + 32: lanes 0..31 return a(l) + a(l + 32), lanes
// 32..63 return b(l - 32) + b(l) (v_permlane32_swap exchanges a's upper half
// with b's lower half).
__device__ __forceinline__ float half_pair_sum(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sums over 16-lane row pairs (0, 1) and (2, 3): rows 0 and 2 return a
// summed with the next row, rows 1 and 3 return b summed with the previous
// row (v_permlane16_swap exchanges a's odd rows with b's even rows).
__device__ __forceinline__ float row_pair_sum(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sum over the row groups of a column, in every lane.
template <int RG>
__device__ __forceinline__ float sum_row_groups(float x) {
    if constexpr (RG >= 2) x = half_pair_sum(x, x);
    if constexpr (RG >= 4) x = row_pair_sum(x, x);
    return x;
}

// Two adjacent columns of T as loaded (BF16 pairs stay packed).
template <typename T>
struct Pair;
template <>
struct Pair<bf16_t> {
    using raw = uint32_t;
    static __device__ __forceinline__ raw load(const bf16_t *p) { return *reinterpret_cast<const uint32_t *>(p); }
    static __device__ __forceinline__ float lo(raw r) { return __uint_as_float(r << 16); }
    static __device__ __forceinline__ float hi(raw r) { return __uint_as_float(r & 0xffff0000u); }
    // bf(x*p) of both halves, packed
    static __device__ __forceinline__ raw scaled(raw r, float pw) { return pack_bf16x2(lo(r) * pw, hi(r) * pw); }
    static __device__ __forceinline__ raw zero() { return 0u; }
};
template <>
struct Pair<float> {
    using raw = float2;
    static __device__ __forceinline__ raw load(const float *p) { return *reinterpret_cast<const float2 *>(p); }
    static __device__ __forceinline__ float lo(raw r) { return r.x; }
    static __device__ __forceinline__ float hi(raw r) { return r.y; }
    static __device__ __forceinline__ raw scaled(raw r, float pw) { return make_float2(r.x * pw, r.y * pw); }
    static __device__ __forceinline__ raw zero() { return make_float2(0.f, 0.f); }
};

// Columns of T as loaded: a pair (CPL = 2, one load) or one.
template <typename T, int CPL>
struct LaneCols {
    T x;
    __device__ __forceinline__ void load(const T *at) { x = *at; }
    __device__ __forceinline__ float get(int) const { return to_f32(x); }
};
template <typename T>
struct LaneCols<T, 2> {
    typename Pair<T>::raw x;
    __device__ __forceinline__ void load(const T *at) { x = Pair<T>::load(at); }
    __device__ __forceinline__ float get(int c) const { return c ? Pair<T>::hi(x) : Pair<T>::lo(x); }
};

// A lane's columns into a row of E: one store for a pair (even columns).
template <int CPL>
__device__ __forceinline__ void store_cols(bf16_t *at, const float (&x)[CPL]) {
    if constexpr (CPL == 2) *reinterpret_cast<uint32_t *>(at) = pack_bf16x2(x[0], x[1]);
    else at[0] = from_f32<bf16_t>(x[0]);
}
template <int CPL>
__device__ __forceinline__ void store_cols(float *at, const float (&x)[CPL]) {
    if constexpr (CPL == 2) *reinterpret_cast<float2 *>(at) = make_float2(x[0], x[1]);
    else at[0] = x[0];
}

}  // namespace bdm
