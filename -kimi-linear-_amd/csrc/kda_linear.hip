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

// Four neighbouring elements in one store.
template <typename T>
__device__ __forceinline__ void store4(T* p, f4 v) {
    struct alignas(4 * sizeof(T)) { T e[4]; } out;
#pragma unroll
    for (int j = 0; j < 4; ++j) Elem<T>::st(&out.e[j], v[j]);
    __builtin_memcpy(__builtin_assume_aligned(p, 4 * sizeof(T)), &out, sizeof(out));
}

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
        if (a.residual) {
            const uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const T*>(a.residual) +
                                                              row * a.residual_stride + n);
            T res[4];
            __builtin_memcpy(res, &raw, 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] = Elem<T>::ld(&res[j]) + round_elem<T>(r[j]);
        }
        store4(static_cast<T*>(a.y[mat]) + row * N + n, r);
    }
}

// As many waves as leave each at least four steps (8 at K >= 1024, 4 at 512,
// one at 128), where the steps divide evenly.
int waves(int64_t K) {
    const int64_t st = K / 32;
    return st >= 32 && st % 8 == 0 ? 8 : (st >= 16 && st % 4 == 0 ? 4 : 1);
}

template <typename T, int MT, int NT>
int launch(const kda_linear_args& a, hipStream_t stream) {
    const int mats = a.x[1] ? 2 : 1;
    const int64_t n = mats == 2 && a.N[1] > a.N[0] ? a.N[1] : a.N[0];
    const dim3 grid(static_cast<unsigned>((n + 16 * NT - 1) / (16 * NT)), static_cast<unsigned>(mats));
    switch (waves(a.K)) {
        case 8: linear_kernel<T, MT, NT, 8><<<grid, 512, 0, stream>>>(a); break;
        case 4: linear_kernel<T, MT, NT, 4><<<grid, 256, 0, stream>>>(a); break;
        default: linear_kernel<T, MT, NT, 1><<<grid, 64, 0, stream>>>(a);
    }
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

template <typename T, int NT>
int launch_rows(const kda_linear_args& a, hipStream_t stream) {
    if (a.M <= 16) return launch<T, 1, NT>(a, stream);
    if (a.M <= 32) return launch<T, 2, NT>(a, stream);
    return launch<T, 4, NT>(a, stream);
}

// 32 rows of W a workgroup halve the reads of x, where 16 are more workgroups
// than the chip's 256 CUs.  us, 16 / 32 rows a workgroup, fp16, 1 and 16 rows of
// x: K = 2048, N = 4096 5.9 / 6.7 and 6.6 / 8.1, N = 4112 7.2 / 6.8 and 9.4 / 8.1,
// N = 6416 8.1 / 7.0 and 10.1 / 8.3; K = 512, N = 4112 3.0 / 3.1 and 3.7 / 3.6.
// With one wave a workgroup it is always 16 (K = 2080, N = 6416 9.8 / 14.1).
template <typename T>
int launch_type(const kda_linear_args& a, hipStream_t stream) {
    return a.N[0] > 4096 && waves(a.K) > 1 ? launch_rows<T, 2>(a, stream) : launch_rows<T, 1>(a, stream);
}

// ---- dW = dy^T x over many rows --------------------------------------------
// The weight gradient of the gates' up-projections: few outputs (N K =
// 2048 x 128) that each sum over every token, which the library's product
// leaves to 64 workgroups.  A wave takes 64 rows and 128 columns of dW and a
// share of the tokens, 32 a step; four waves meet in LDS and the workgroups'
// sums, enough of them to fill the chip, in a second kernel, both in a fixed
// order.  Both operands have the contraction along their rows: a lane loads 4
// neighbouring channels of 8 tokens and turns them into four fragments of 8
// tokens in registers, so the tile's rows are n0 + 4 i + j for fragment j, and
// four column fragments end in 16 contiguous bytes of dW.
// The loads bound it: one step of each wave is in flight behind the current
// one, with 128 accumulators a wave leaving room for one wave a SIMD.  us in
// a graph of 40, bf16, library / here: 8192 tokens, N = 2048 63.5 / 20.2
// (1.7 TB/s of dy), 32768 tokens 150 / 59.6, N = 512 at 8192 tokens 63.8 /
// 15.8; 1024 tokens, N = 2048 11.3 / 10.5, 256 tokens 6.5 / 6.6.
constexpr int kWgN = 64, kWgK = 128;

struct Rows8 {
    uint2 r[8];
};
// 8 tokens' 4 channels -> fragment J: channel J of the 8 tokens
template <int J>
__device__ __forceinline__ uint4 frag(const Rows8& v) {
    constexpr uint32_t sel = J % 2 == 0 ? 0x05040100u : 0x07060302u;
    const auto word = [&](int i) { return J / 2 == 0 ? v.r[i].x : v.r[i].y; };
    return uint4{__builtin_amdgcn_perm(word(1), word(0), sel), __builtin_amdgcn_perm(word(3), word(2), sel),
                 __builtin_amdgcn_perm(word(5), word(4), sel), __builtin_amdgcn_perm(word(7), word(6), sel)};
}

template <typename T>
__device__ __forceinline__ void load_rows(Rows8& v, const T* p, int64_t stride, int64_t row, int64_t M) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v.r[i] = *reinterpret_cast<const uint2*>(p + min(row + i, M - 1) * stride);
    if (row + 8 > M) {                                  // tokens past the last count as zero
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (row + i >= M) v.r[i] = uint2{0, 0};
    }
}

// Grid (N / 64 * K / 128, splits); out: fp32 [splits, N, K].
template <typename T>
__global__ __launch_bounds__(256) void wgrad_kernel(kda_linear_wgrad_args a, float* out, int64_t per) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ln = lane & 15, lg = lane >> 4;
    const int64_t nt = a.N / kWgN;
    const int64_t n0 = blockIdx.x % nt * kWgN, k0 = blockIdx.x / nt * kWgK;
    const T* dy = static_cast<const T*>(a.dy) + n0 + 4 * ln;
    const T* x = static_cast<const T*>(a.x) + k0 + 4 * ln;
    const int64_t end = min((static_cast<int64_t>(blockIdx.y) + 1) * per, (a.M + 31) / 32);
    int64_t s = static_cast<int64_t>(blockIdx.y) * per + wave;

    f4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    Rows8 na, nb[2];
    const auto fetch = [&](int64_t step) {
        const int64_t row = 32 * step + 8 * lg;
        load_rows(na, dy, a.dy_stride, row, a.M);
        load_rows(nb[0], x, a.x_stride, row, a.M);
        load_rows(nb[1], x + 64, a.x_stride, row, a.M);
    };
    if (s < end) fetch(s);
    for (; s < end; s += 4) {
        const uint4 fa[4] = {frag<0>(na), frag<1>(na), frag<2>(na), frag<3>(na)};
        const uint4 fb[8] = {frag<0>(nb[0]), frag<1>(nb[0]), frag<2>(nb[0]), frag<3>(nb[0]),
                             frag<0>(nb[1]), frag<1>(nb[1]), frag<2>(nb[1]), frag<3>(nb[1])};
        if (s + 4 < end) fetch(s + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = Mat<T>::mma(fa[i], fb[j], acc[i][j]);
    }

    // waves 2 and 3 hand their sums to 0 and 1; those exchange halves
    __shared__ f4 red[2][32][64];
    if (wave >= 2) {
#pragma unroll
        for (int i = 0; i < 32; ++i) red[wave - 2][i][lane] = acc[i / 8][i % 8];
    }
    __syncthreads();
    if (wave < 2) {
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i / 8][i % 8] += red[wave][i][lane];
    }
    __syncthreads();
    if (wave < 2) {
#pragma unroll
        for (int i = 0; i < 32; ++i)
            if (i / 16 != wave) red[wave][i][lane] = acc[i / 8][i % 8];
    }
    __syncthreads();
    if (wave >= 2) return;
    out += static_cast<int64_t>(blockIdx.y) * a.N * a.K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i / 2 != wave) continue;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] += red[1 - wave][8 * i + j][lane];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t n = n0 + 4 * (4 * lg + q) + i;
                store4(out + n * a.K + k0 + 64 * h + 4 * ln,
                       f4{acc[i][4 * h][q], acc[i][4 * h + 1][q], acc[i][4 * h + 2][q], acc[i][4 * h + 3][q]});
            }
    }
}

// dw[e] = the sum of the splits' shares, in order; four elements a thread.
template <typename T>
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const float* part, T* dw, int64_t n, int splits) {
    const int64_t e = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (e >= n) return;
    f4 s = *reinterpret_cast<const f4*>(part + e);
#pragma unroll 8
    for (int i = 1; i < splits; ++i) s += *reinterpret_cast<const f4*>(part + i * n + e);
    store4(dw + e, s);
}

// One workgroup a CU, each with at least two steps a wave; two or more, with at
// most 64 tiles and at least 16 steps.
int64_t wgrad_splits(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = (N / kWgN) * (K / kWgK), steps = (M + 31) / 32;
    return min(256 / tiles, steps / 8);
}

template <typename T>
int launch_wgrad(const kda_linear_wgrad_args& a, hipStream_t stream) {
    const int64_t splits = wgrad_splits(a.M, a.N, a.K), steps = (a.M + 31) / 32;
    const int64_t per = (steps + splits - 1) / splits;
    const dim3 grid(static_cast<unsigned>((a.N / kWgN) * (a.K / kWgK)), static_cast<unsigned>(splits));
    float* part = static_cast<float*>(a.workspace);
    wgrad_kernel<T><<<grid, 256, 0, stream>>>(a, part, per);
    if (hipGetLastError() != hipSuccess) return KDA_ERR_LAUNCH;
    const int64_t n = a.N * a.K;
    wgrad_sum_kernel<T><<<static_cast<unsigned>((n / 4 + 255) / 256), 256, 0, stream>>>(part, static_cast<T*>(a.dw), n,
                                                                                        static_cast<int>(splits));
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

}  // namespace

// Each workgroup reads all rows of x, which with up to 16 costs less than the 16
// or 32 rows of W beside them; with more it still wins where the library's
// product is bound by its launch.  us a product in a graph of 24, library / here,
// fp16 (N, K, rows):
//   6416, 2048:  1: 8.9 / 7.0   16: 8.9 / 8.3
//   2048, 2048:  1: 7.8 / 4.7   16: 8.1 / 6.0
//   4096, 1024:  1: 5.5 / 3.7   16: 5.8 / 4.4   32: 8.1 / 5.4
//   2048,  512:  1: 3.7 / 2.6   16: 3.8 / 3.0   32: 4.9 / 3.5   64: 5.5 / 4.5
//   2048,  128:  1: 3.2 / 1.9   16: 3.6 / 2.1   32: 3.5 / 2.3   64: 3.7 / 2.6
// (two of the last in one launch: 2.0 and 2.8 us at 1 and 64 rows).  At one
// row the 6416 x 2048 weight goes by at 3.8 TB/s, 5.3 without the launch.  The
// layer takes the library's product for the widths and depths where it is the
// faster one (layer.py, _few_rows).
bool linear_supported(const kda_linear_args& a) {
    if (a.M > 64 || a.K % 32 != 0) return false;
    return a.M <= 16 || a.K <= (a.M <= 32 ? 1024 : 512);
}

int linear_launch(const kda_linear_args& a, hipStream_t stream) {
    return a.dtype == KDA_DTYPE_F16 ? launch_type<_Float16>(a, stream) : launch_type<bf16_t>(a, stream);
}

// From 512 tokens on (measured above); up to 64 tiles, beyond which the
// library's product has workgroups enough by itself.
bool linear_wgrad_supported(int64_t M, int64_t N, int64_t K) {
    return M >= 512 && N > 0 && K > 0 && N % kWgN == 0 && K % kWgK == 0 && N <= 4096 && K <= 4096 &&
           (N / kWgN) * (K / kWgK) <= 64 && M <= int64_t{1} << 40;
}
int64_t linear_wgrad_workspace_bytes(int64_t M, int64_t N, int64_t K) { return wgrad_splits(M, N, K) * N * K * 4; }

int linear_wgrad_launch(const kda_linear_wgrad_args& a, hipStream_t stream) {
    return a.dtype == KDA_DTYPE_F16 ? launch_wgrad<_Float16>(a, stream) : launch_wgrad<bf16_t>(a, stream);
}

}  // namespace kda
