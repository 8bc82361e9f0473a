// y = x W^T for the few rows of a decode step or a short prompt, on gfx950.
//
// With up to 64 rows a projection is a read of its weight: every byte of W is
// used once, and the matrix cores have nothing to wait for but it.  One
// workgroup takes 16 or 32 rows of W; its waves split the contraction, each issues
// all loads of up to eight 32-deep steps before its first MFMA, and the waves'
// sums meet in LDS in a fixed order.  At N = 2048, K = 2048 that is 128
// workgroups of 8 waves with 64 KiB of W in flight each: the whole weight is
// requested at once.  Where a decode step has two small projections side by
// side (the gates' up-projections, K = 128) one launch does both, and the
// residual stream's add can take place on the result, rounded to the
// activation type first as a separate add would find it.
//
// A wave's MFMA takes 16 rows of W as its A operand and 16 rows of x as B, so
// a lane ends up with four neighbouring outputs of one row: one 8-byte store.
#include <hip/hip_runtime.h>

#include "kda_common.h"
#include "kda_hip.h"
#include "kda_launch.h"

namespace kda {
namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

template <typename T> struct Mat;
template <> struct Mat<_Float16> {
    static __device__ __forceinline__ f4 mma(uint4 a, uint4 b, f4 c) {
        return mfma16x16x32(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c);
    }
};
template <> struct Mat<bf16_t> {
    static __device__ __forceinline__ f4 mma(uint4 a, uint4 b, f4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0,
                                                       0);
    }
};

constexpr int kDepth = 8;        // steps whose loads are in flight together

// N steps of 32 from the lane's addresses on.
template <typename T, int MT, int NT, int N>
__device__ __forceinline__ void steps(const T* const (&w)[NT], const T* const (&x)[MT], int64_t off,
                                      f4 (&acc)[NT][MT]) {
    uint4 wr[N][NT], xr[N][MT];
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
        for (int t = 0; t < NT; ++t) wr[i][t] = *reinterpret_cast<const uint4*>(w[t] + off + 32 * i);
#pragma unroll
        for (int m = 0; m < MT; ++m) xr[i][m] = *reinterpret_cast<const uint4*>(x[m] + off + 32 * i);
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[t][m] = Mat<T>::mma(wr[i][t], xr[i][m], acc[t][m]);
}

// Grid (max N / (16 NT), matrices), 64 SPLIT threads; K a multiple of 32 SPLIT.
// MT 16-row tiles of x cover its M rows, NT those of W a workgroup's; a lane
// past the last row of either reads that row and stores nothing.
template <typename T, int MT, int NT, int SPLIT>
__global__ __launch_bounds__(64 * SPLIT) void linear_kernel(kda_linear_args a) {
    const int mat = blockIdx.y;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (16 * NT), N = a.N[mat];
    if (n0 >= N) return;
    const int lane = threadIdx.x & 63, wave = SPLIT == 1 ? 0 : threadIdx.x >> 6;
    const int ln = lane & 15, lg = lane >> 4;
    const int64_t per = a.K / 32 / SPLIT, k0 = wave * per * 32 + lg * 8;
    const T* w[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        w[t] = static_cast<const T*>(a.w[mat]) + min(n0 + 16 * t + ln, N - 1) * a.K + k0;
    const T* x[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
        x[m] = static_cast<const T*>(a.x[mat]) + min(static_cast<int64_t>(16 * m + ln), a.M - 1) * a.x_stride[mat] + k0;
    f4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = f4{0.f, 0.f, 0.f, 0.f};
    int64_t s = 0;
    for (; s + kDepth <= per; s += kDepth) steps<T, MT, NT, kDepth>(w, x, 32 * s, acc);
    if (s + 4 <= per) {
        steps<T, MT, NT, 4>(w, x, 32 * s, acc);
        s += 4;
    }
    for (; s < per; ++s) steps<T, MT, NT, 1>(w, x, 32 * s, acc);

    constexpr int kTiles = NT * MT;
    __shared__ f4 part[SPLIT == 1 ? 1 : SPLIT * kTiles * 64];
    if constexpr (SPLIT > 1) {
#pragma unroll
        for (int i = 0; i < kTiles; ++i) part[(wave * kTiles + i) * 64 + lane] = acc[i / MT][i % MT];
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
        if (SPLIT > 1 && i % SPLIT != wave) continue;
        f4 r = acc[i / MT][i % MT];
        if constexpr (SPLIT > 1) {
            r = part[i * 64 + lane];
#pragma unroll
            for (int v = 1; v < SPLIT; ++v) {
                const f4 p = part[(v * kTiles + i) * 64 + lane];
#pragma unroll
                for (int j = 0; j < 4; ++j) r[j] += p[j];
            }
        }
        const int64_t row = 16 * (i % MT) + ln, n = n0 + 16 * (i / MT) + 4 * lg;
        if (row >= a.M || n >= N) continue;
        T out[4];
        if (a.residual) {
            const uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const T*>(a.residual) +
                                                              row * a.residual_stride + n);
            T res[4];
            __builtin_memcpy(res, &raw, 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] = Elem<T>::ld(&res[j]) + round_elem<T>(r[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) Elem<T>::st(&out[j], r[j]);
        uint2 raw;
        __builtin_memcpy(&raw, out, 8);
        *reinterpret_cast<uint2*>(static_cast<T*>(a.y[mat]) + row * N + n) = raw;
    }
}

template <typename T, int MT, int NT>
int launch(const kda_linear_args& a, hipStream_t stream) {
    const int mats = a.x[1] ? 2 : 1;
    const int64_t n = mats == 2 && a.N[1] > a.N[0] ? a.N[1] : a.N[0];
    const dim3 grid(static_cast<unsigned>((n + 16 * NT - 1) / (16 * NT)), static_cast<unsigned>(mats));
    // as many waves as leave each at least four steps (8 at K >= 1024, 4 at
    // 512, one at 128), where the steps divide evenly
    const int64_t st = a.K / 32;
    if (st >= 32 && st % 8 == 0) linear_kernel<T, MT, NT, 8><<<grid, 512, 0, stream>>>(a);
    else if (st >= 16 && st % 4 == 0) linear_kernel<T, MT, NT, 4><<<grid, 256, 0, stream>>>(a);
    else linear_kernel<T, MT, NT, 1><<<grid, 64, 0, stream>>>(a);
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

template <typename T, int NT>
int launch_rows(const kda_linear_args& a, hipStream_t stream) {
    if (a.M <= 16) return launch<T, 1, NT>(a, stream);
    if (a.M <= 32) return launch<T, 2, NT>(a, stream);
    return launch<T, 4, NT>(a, stream);
}

// 32 rows of W a workgroup halve the reads of x, but only a wide projection
// still has workgroups for the chip's 256 CUs: at N = 6416, K = 2048, 1 and 16
// rows 8.0 and 9.9 us -> 6.9 and 8.1; at N = 4096, 256 workgroups of 16 rows
// against 128 of 32: 5.8 and 6.3 against 6.6 and 8.0.
template <typename T>
int launch_type(const kda_linear_args& a, hipStream_t stream) {
    return a.N[0] >= 6144 ? launch_rows<T, 2>(a, stream) : launch_rows<T, 1>(a, stream);
}

}  // namespace

// The shapes this kernel is the better one for.  Each workgroup reads all rows
// of x, which with up to 16 costs less than the 16 or 32 rows of W beside
// them; with more it still wins where the library's product is bound by its
// launch.  us a product in a graph of 40, library / here, fp16 (N, K, rows):
//   6416, 2048:  1: 8.8 / 6.9   16: 8.8 / 8.1   32: 8.8 / 9.8   64: 9.5 / 13.6
//   2048, 2048:  1: 7.8 / 4.6   16: 8.0 / 6.0   32: 8.2 / 7.8   64: 8.6 / 11.4
//   3344, 1024:  1: 4.5 / 3.4   16: 4.8 / 4.2   32: 7.8 / 5.1   64: 7.0 / 7.0
//   1808,  512:  1: 3.6 / 2.4   16: 3.6 / 2.8   32: 4.8 / 3.4   64: 5.5 / 4.4
//   2048,  128:  1: 3.2 / 1.9   16: 3.5 / 2.1   32: 3.5 / 2.2   64: 3.7 / 2.7
// (two of the last in one launch: 2.0 and 2.8 us at 1 and 64 rows).  At one
// row the 6416 x 2048 weight goes by at 3.8 TB/s, 5.3 without the launch.
bool linear_supported(const kda_linear_args& a) {
    if (a.M > 64 || a.K % 32 != 0) return false;
    return a.M <= 16 || a.K <= (a.M <= 32 ? 1024 : 512);
}

int linear_launch(const kda_linear_args& a, hipStream_t stream) {
    return a.dtype == KDA_DTYPE_F16 ? launch_type<_Float16>(a, stream) : launch_type<bf16_t>(a, stream);
}

}  // namespace kda
