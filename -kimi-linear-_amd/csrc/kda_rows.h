// Rows of the layer's elementwise kernels: a lane's run of channels as loaded,
// element conversions and parameters of a runtime dtype.
#pragma once

#include "kda_common.h"

namespace kda {

// channels per lane of q, k and v: 16 bytes
template <typename XT> constexpr int kLaneCh = 16 / static_cast<int>(sizeof(XT));
// Runs of 64 n channels, a wave's, in rows of D.
__host__ __device__ constexpr int64_t segments(int64_t D, int n) { return (D + 64 * n - 1) / (64 * n); }
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

// sum_c x[c] y[c] over a head of DH channels, N a lane (all-reduce).
template <typename XT, int DH, int N>
__device__ __forceinline__ float head_dot(const float (&x)[N], const float (&y)[N]) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < N; ++c) s = fmaf(x[c], y[c], s);
    return lanes_sum<DH / N>(s);
}

}  // namespace kda
