// Rows of the layer's elementwise kernels: a lane's run of channels as loaded,
// element conversions and parameters of a runtime dtype.
#pragma once

#include <type_traits>

#include "kda_common.h"

namespace kda {

// channels per lane of q, k and v: 16 bytes (fewer where a row is a fraction of
// a wave's run)
template <typename XT> constexpr int kLaneCh = 16 / static_cast<int>(sizeof(XT));
// Runs of 64 n channels, a wave's, in rows of D.
__host__ __device__ constexpr int64_t segments(int64_t D, int n) { return (D + 64 * n - 1) / (64 * n); }
// Whether a row of D channels takes more than half a wave at n channels a lane.
constexpr bool fills(int64_t D, int n) { return D > 32 * n; }
constexpr int kGateSeg = 256;  // channels per wave of the gate, 4 a lane

template <typename XT> __device__ __forceinline__ float to_f(XT x);
template <> __device__ __forceinline__ float to_f<float>(float x) { return x; }
template <> __device__ __forceinline__ float to_f<_Float16>(_Float16 x) { return static_cast<float>(x); }
template <> __device__ __forceinline__ float to_f<bf16_t>(bf16_t x) { return bf16_bits_to_f32(x.bits); }

template <typename XT> __device__ __forceinline__ XT from_f(float x);
template <> __device__ __forceinline__ float from_f<float>(float x) { return x; }
template <> __device__ __forceinline__ _Float16 from_f<_Float16>(float x) {
    // x as the 32-bit value it is: v_fma_mixlo_f16, which the compiler takes in
    // some kernels and not in others, would round a product before it to 16 bits at once
    asm("" : "+v"(x));
    return static_cast<_Float16>(x);
}
template <> __device__ __forceinline__ bf16_t from_f<bf16_t>(float x) { return bf16_t{f32_to_bf16_bits(x)}; }

// Round to XT and back: the value an XT tensor would hold.
template <typename XT>
__device__ __forceinline__ float round_to(float x) {
    return to_f(from_f<XT>(x));
}

// N consecutive elements held as loaded.  Rows are aligned to their
// element only (the layer's rows of H (2 K + V) + H + 256 elements are not a
// multiple of 16 bytes for every H); the compiler emits what that allows.
template <typename XT, int N>
struct Raw {
    static constexpr int W = sizeof(XT) * N / 4;     // words
    uint32_t w[W];
};
template <int N, typename XT>
__device__ __forceinline__ Raw<XT, N> ldn(const XT* p) {
    Raw<XT, N> r;
    __builtin_memcpy(r.w, p, sizeof(r.w));
    return r;
}
template <typename XT, int N>
__device__ __forceinline__ void unpack(const Raw<XT, N>& r, float (&x)[N]) {
#pragma unroll
    for (int c = 0; c < N; ++c) {
        if constexpr (sizeof(XT) == 4) {
            x[c] = __uint_as_float(r.w[c]);
        } else {
            const uint16_t u = static_cast<uint16_t>(r.w[c / 2] >> (16 * (c % 2)));
            x[c] = Elem<XT>::code == KDA_DTYPE_F16 ? static_cast<float>(__builtin_bit_cast(_Float16, u))
                                                   : bf16_bits_to_f32(u);
        }
    }
}
template <typename XT, int N>
__device__ __forceinline__ void stn(XT* p, const float (&x)[N]) {
    XT v[N];
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] = from_f<XT>(x[c]);
    __builtin_memcpy(p, v, sizeof(v));
}

// N consecutive parameters of a runtime dtype from element i on: as loaded, and
// as fp32.  Apart, so that the wait for them comes where they are used: a
// conversion beside the load would wait for it before the loads after it.
template <int N>
struct RawParams {
    uint32_t w[N];
};
template <int N>
__device__ __forceinline__ RawParams<N> ld_params(const void* p, int64_t i, int dtype) {
    RawParams<N> r;
    if (dtype == KDA_DTYPE_F32) __builtin_memcpy(r.w, static_cast<const float*>(p) + i, N * 4);
    else __builtin_memcpy(r.w, static_cast<const uint16_t*>(p) + i, N * 2);
    return r;
}
template <int N>
__device__ __forceinline__ void decode(const RawParams<N>& r, int dtype, float (&x)[N]) {
    const auto half = [&](int c) { return static_cast<uint16_t>(r.w[c / 2] >> (16 * (c % 2))); };
    if (dtype == KDA_DTYPE_F32) {
#pragma unroll
        for (int c = 0; c < N; ++c) x[c] = __uint_as_float(r.w[c]);
    } else if (dtype == KDA_DTYPE_F16) {
#pragma unroll
        for (int c = 0; c < N; ++c) x[c] = static_cast<float>(__builtin_bit_cast(_Float16, half(c)));
    } else {
#pragma unroll
        for (int c = 0; c < N; ++c) x[c] = bf16_bits_to_f32(half(c));
    }
}

// x of lane I of each four lanes, to all four.
template <int I>
__device__ __forceinline__ float quad_bcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x55 * I, 0xF, 0xF, true));
}

// sum_c x[c] y[c] over a head of DH channels of XT, N a lane (the lanes of a
// head in their order; all-reduce).  The order of the additions is that of
// kLaneCh channels a lane, whatever N: those in their order, the rest as
// lanes_sum adds lanes.  So a row gives the same bits in every kernel's layout.
template <typename XT, int DH, int N>
__device__ __forceinline__ float head_dot(const float (&x)[N], const float (&y)[N]) {
    constexpr int R = kLaneCh<XT>, G = DH / R, L = R / N;        // channels of a run, runs, lanes of a run
    static_assert(L == 1 || (R == 8 && (L == 2 || L == 4)), "a run in one, two or four lanes");
    const auto chain = [&](float s) {
#pragma unroll
        for (int c = 0; c < N; ++c) s = fmaf(x[c], y[c], s);
        return s;
    };
    float s = chain(0.f);
    if constexpr (L == 1) return lanes_sum<G>(s);
    if constexpr (L == 2) {                              // the second lane of two goes on from the first
        s = chain(__int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xA0, 0xF, 0xF, true)));  // [0,0,2,2]
        s = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xF5, 0xF, 0xF, true));         // [1,1,3,3]
    }
    if constexpr (L == 4) {
        s = chain(quad_bcast<0>(s));
        s = chain(quad_bcast<1>(s));
        s = chain(quad_bcast<2>(s));
        s = quad_bcast<3>(s);
    }
    const auto xor16 = [](float v) {
        const unsigned u = __float_as_uint(v);
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    const auto xor32 = [](float v) {
        const unsigned u = __float_as_uint(v);
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    const auto dpp = [](auto ctrl, float v) {
        return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    using Ror8 = std::integral_constant<int, 0x128>;
    using Ror4 = std::integral_constant<int, 0x124>;
    using Ror2 = std::integral_constant<int, 0x122>;
    using Quad2 = std::integral_constant<int, 0x4E>;     // quad [2,3,0,1]
    using Half = std::integral_constant<int, 0x141>;     // row_half_mirror: the other four lanes of eight
    if constexpr (G == 8) {                              // runs 1, 2, 4 apart in turn
        if constexpr (L == 2) s = dpp(Quad2{}, s);
        s = dpp(Half{}, s);
        s = dpp(Ror8{}, s);
        if constexpr (L == 4) s = xor16(s);
    } else {                                             // runs 8, 4, 2, 1 apart in turn, then 16
        if constexpr (L == 4) s = xor32(s);
        s = xor16(s);
        s = dpp(Ror8{}, s);
        s = dpp(Ror4{}, s);
        if constexpr (L == 2) s = dpp(Ror2{}, s);
        if constexpr (G == 32) s = xor32(s);
    }
    static_assert(L == 1 || G == 8 || G == 16 || (G == 32 && L == 2), "heads of 64, 128 and 256 channels, within a wave");
    return s;
}

}  // namespace kda
