// Pre- and post-processing of the KDA layer around the core, for gfx950.
//
// kda_prep_fwd replaces the elementwise part of _projections
// (kimi_linear/kda.py:399-461): per q/k/v channel the causal short
// convolution (kda.py:282-310), SiLU, and for q and k the per-head L2
// normalisation (kda.py:313-325); the forget gate g = -exp(A_log) *
// softplus(gk + dt_bias) and beta = sigmoid(.) (kda.py:452-460).  The
// reference runs these as ~20 separate elementwise kernels with fp16
// round trips between them; here every projection element is read once (plus
// the conv_size - 1 rows of context a token tile needs) and every core input
// is written once, all arithmetic in fp32 and each output rounded once.  A
// call without g and beta outputs skips the gates: the layer hands gk and the
// beta logits to the gated core entry points, whose loaders form them.
//
// kda_output_fwd replaces HeadwiseRMSNorm and the sigmoid output gate of
// _output (kda.py:258-279, 464-470): one read of the core output and of the
// gate projection, one write of the o_proj input.
//
// Both are streaming kernels with the lanes across channels, eight adjacent
// ones a lane (16 bytes of a 16-bit row), so a wave takes 512 channels of a
// row: the heads' sums of squares are DPP sums over K / 8 lanes, and the
// per-row work (addresses, the sum's exchange, the row's rsqrt) is shared by
// eight channels.  A row of at most 256 channels takes four a lane (the output
// kernel two up to 128), which keeps lanes that would be idle at work, and so
// does a decode step of the pre-processing, whose time is its chain's; the
// norms' sums keep their order (head_dot), so the bits are the same.  Every load of a unit is issued unconditionally before its
// first use (rows past the data re-read a valid row and are masked), so a
// wave keeps all of its rows in flight at once instead of waiting on each.
// The parameters' loads come before the rows': used first in a row's store,
// which is conditional, a later load of theirs was waited for in every row,
// and with it the store of the row before (B=4 T=3048 H=16 V=128 bf16, output:
// 26.4 -> 24.0 us; B=48 T=184 20.2 -> 18.9).
#include <type_traits>

#include "kda_common.h"
#include "kda_rows.h"

namespace kda {

namespace {

constexpr int kTile = 16;      // tokens per prep unit at most; an in-place conv cache needs T <= this
constexpr int kMaxConv = 4;    // largest conv_size
// ---- prep: 64 N channels of q, k or v over a token tile ---------------------
// DH: the head size whose L2 norm is taken (q and k), 0 for none (v).  CS:
// conv_size, so that the taps of a lane's channels are a few wide loads: with a
// runtime size each was a load and a wait of its own (us, bf16 unless said: a
// decode step at B=33 H=16 K=V=128 conv_size 2 6.0 -> 3.0, two channels a lane
// took 3.7; B=4 T=125 H=16 fp16 conv_size 3 with the gates 12.1 -> 7.6, 9.6).
template <typename XT, int DH, int TILE, int CS, int N>
__device__ __forceinline__ void conv_unit(const kda_prep_args& a, int i, int64_t b, int64_t t0, int64_t seg, int lane) {
    constexpr int cs = CS, cm = cs - 1, kRows = TILE + cm;
    const int64_t D = a.H * (DH ? DH : a.V);
    const bool valid = seg * (64 * N) + N * lane < D;
    const int64_t ch0 = valid ? seg * (64 * N) + N * lane : 0;
    const int64_t T = a.T;
    const int n = static_cast<int>((T - t0) < TILE ? (T - t0) : TILE);
    const XT* x = static_cast<const XT*>(a.x[i]) + b * a.x_stride[i][0];
    const XT* hist = static_cast<const XT*>(a.hist_in[i]);
    const XT* hrow = hist != nullptr ? hist + b * cm * D : x;

    // the parameters first: what waits for a row has them then
    const RawParams<N * cs> rw = ld_params<N * cs>(a.conv_w[i], ch0 * cs, a.w_dtype);
    RawParams<N> rb{};
    if (a.conv_b[i] != nullptr) rb = ld_params<N>(a.conv_b[i], ch0, a.w_dtype);

    // window row r holds token t0 - cm + r: a token of this call, a cached
    // input (t < 0) or zero.  Every row is loaded unconditionally (rows with
    // no data read token 0 and are masked) so that all loads are in flight
    // together.
    Raw<XT, N> win[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int64_t tok = t0 - cm + r;
        const bool in_x = tok >= 0 && tok < T;
        const bool in_h = tok < 0 && hist != nullptr;
        const XT* src = in_x ? x + tok * a.x_stride[i][1] : (in_h ? hrow + (cm + tok) * D : x);
        win[r] = ldn<N>(src + ch0);
        if (!(in_x || in_h)) {
#pragma unroll
            for (int c = 0; c < Raw<XT, N>::W; ++c) win[r].w[c] = 0u;
        }
    }
    float w[cs][N], wc[N * cs], bias[N];
    decode(rw, a.w_dtype, wc);
    decode(rb, a.w_dtype, bias);
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < cs; ++j) w[j][c] = wc[cs * c + j];

    XT* out = static_cast<XT*>(i == 0 ? a.q : (i == 1 ? a.k : a.v)) + (b * T + t0) * D + ch0;
    const float inv_eps = 1.f / a.l2_eps;
    // tap j of tile token t reads window row t + j (token t0 + t - cm + j)
    float xs[cs][N];
#pragma unroll
    for (int j = 0; j < cm; ++j) unpack(win[j], xs[j]);
#pragma unroll
    for (int t = 0; t < TILE; ++t) {
        unpack(win[t + cm], xs[(t + cm) % cs]);
        float s[N];
#pragma unroll
        for (int c = 0; c < N; ++c) {
            float u = bias[c];
#pragma unroll
            for (int j = 0; j < cs; ++j) u = fmaf(w[j][c], xs[(t + j) % cs][c], u);
            s[c] = u * sigmoid_f(u);
        }
        if constexpr (DH != 0) {
            // l2 norm over the head: x * min(rsqrt(sum x^2), 1/eps)
            const float rn = fminf(rsqrtf(head_dot<XT, DH>(s, s)), inv_eps);
#pragma unroll
            for (int c = 0; c < N; ++c) s[c] *= rn;
        }
        if (t < n && valid) stn(out + t * D, s);
    }

    // the next call's conv cache: inputs T - cm .. T - 1 = window rows n + r
    if (a.hist_out[i] != nullptr && t0 + n == T && valid) {
        XT* ho = static_cast<XT*>(a.hist_out[i]) + b * cm * D + ch0;
#pragma unroll
        for (int r = 0; r < cm; ++r) {
            Raw<XT, N> hv = win[r];
#pragma unroll
            for (int rr = 0; rr < kRows; ++rr)
                if (rr == n + r) hv = win[rr];
            __builtin_memcpy(ho + r * D, hv.w, sizeof(hv.w));
        }
    }
}

// ---- prep: the forget gate of 256 channels over a token tile, and the betas
// of their heads.  Four channels a lane: g is stored in 32 bits, 16 bytes a
// lane (eight channels in two stores of 32-byte lanes took 107 us where this
// takes 78 at B=4 T=2048 H=16 K=128 bf16, the projections included).
template <typename XT, int DH, int TILE>
__device__ __forceinline__ void gate_unit(const kda_prep_args& a, int64_t b, int64_t t0, int64_t seg, int lane) {
    constexpr int kHeads = kGateSeg / DH;        // heads per unit
    const int64_t D = a.H * DH;
    const bool valid = seg * kGateSeg + 4 * lane < D;
    const int64_t ch0 = valid ? seg * kGateSeg + 4 * lane : 0;
    const int64_t T = a.T;
    const int n = static_cast<int>((T - t0) < TILE ? (T - t0) : TILE);
    const XT* gk = static_cast<const XT*>(a.gk) + b * a.gk_stride[0] + ch0;

    const RawParams<4> ra = ld_params<4>(a.a_log, ch0, a.p_dtype), rd = ld_params<4>(a.dt_bias, ch0, a.p_dtype);
    // every load first (rows past the end re-read the last token)
    Raw<XT, 4> z[TILE];
#pragma unroll
    for (int t = 0; t < TILE; ++t) z[t] = ldn<4>(gk + (t0 + (t < n ? t : n - 1)) * a.gk_stride[1]);
    // entry e of the unit's TILE x kHeads betas: token e / kHeads, head e % kHeads
    constexpr int kB = (TILE * kHeads + 63) / 64;
    RawElem rl[kB];
    int64_t bt[kB], bh[kB];
    bool bv[kB];
#pragma unroll
    for (int e = 0; e < kB; ++e) {
        const int k = lane + 64 * e;
        bt[e] = t0 + k / kHeads;
        bh[e] = seg * kHeads + k % kHeads;
        bv[e] = k < n * kHeads && bh[e] < a.H;
        rl[e] = load_raw_elem(a.beta_logit,
                              b * a.beta_stride[0] + (bv[e] ? bt[e] * a.beta_stride[1] + bh[e] : t0 * a.beta_stride[1]),
                              a.x_dtype);
    }
    float neg_a[4], dtb[4];
    decode(ra, a.p_dtype, neg_a);
    decode(rd, a.p_dtype, dtb);
#pragma unroll
    for (int c = 0; c < 4; ++c) neg_a[c] = -__expf(neg_a[c]);
    float* g = static_cast<float*>(a.g) + (b * T + t0) * D + ch0;
#pragma unroll
    for (int t = 0; t < TILE; ++t) {
        float x[4], o[4];
        unpack(z[t], x);
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = neg_a[c] * softplus(x[c] + dtb[c]);
        if (t < n && valid) stn(g + t * D, o);
    }
#pragma unroll
    for (int e = 0; e < kB; ++e)
        if (bv[e]) static_cast<float*>(a.beta)[(b * T + bt[e]) * a.H + bh[e]] = sigmoid_f(decode_elem(rl[e], a.x_dtype));
}

// Bound by memory from a few thousand tokens on (4.4-4.6 of the 5.2 TB/s of a
// copy, reading three rows in sixteen twice).  us, two channels a lane and a
// wave a head -> this, fp16 unless said: B=16 T=2048 H=16 d=128 bf16 210 -> 184;
// B=4 T=2048 53.5 -> 44; B=1 T=1000 12.0 -> 8.8; a decode step at B=1 4.1 ->
// 3.5, at B=64 5.6 -> 4.0.
//
// One wave per (batch, tile, 64 N channels of q, k, v and, unless the call
// leaves the gates to the core, of the gate).  The host keeps the number of
// units below 2^31, so the unit index is split with 32-bit arithmetic.
template <typename XT, int K, int TILE, int N>
__global__ __launch_bounds__(256) void prep_kernel(const kda_prep_args a, uint32_t ntiles, uint32_t units) {
    const int lane = threadIdx.x & 63;
    const uint32_t unit = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= units) return;
    const uint32_t H = static_cast<uint32_t>(a.H);
    const uint32_t segk = segments(H * K, N), segv = segments(H * static_cast<uint32_t>(a.V), N);
    const uint32_t per = 2 * segk + segv + (a.g != nullptr ? (H * K + kGateSeg - 1) / kGateSeg : 0);
    uint32_t s = unit % per;
    const uint32_t bt = unit / per;
    const int64_t t0 = static_cast<int64_t>(bt % ntiles) * TILE, b = bt / ntiles;
    const auto conv = [&](auto dh, int i, int64_t seg) {
        constexpr int DH = decltype(dh)::value;
        switch (a.conv_size) {
            case 4: conv_unit<XT, DH, TILE, 4, N>(a, i, b, t0, seg, lane); break;
            case 3: conv_unit<XT, DH, TILE, 3, N>(a, i, b, t0, seg, lane); break;
            case 2: conv_unit<XT, DH, TILE, 2, N>(a, i, b, t0, seg, lane); break;
            default: conv_unit<XT, DH, TILE, 1, N>(a, i, b, t0, seg, lane);
        }
    };
    if (s < 2 * segk) {
        conv(std::integral_constant<int, K>{}, s >= segk, s - (s >= segk) * segk);
    } else if (s < 2 * segk + segv) {
        conv(std::integral_constant<int, 0>{}, 2, s - 2 * segk);
    } else {
        gate_unit<XT, K, TILE>(a, b, t0, s - 2 * segk - segv, lane);
    }
}

// ---- output: one wave per (batch, tile of tokens, 64 N channels) ------------
// At copy rate from a few thousand tokens on; us at H=16 V=128 fp16, a wave a
// head -> this: B=4 T=2048 19.9 -> 19.6 (bf16 21.0 -> 19.2), B=1 T=1000 4.8 ->
// 3.9, a decode step at B=64 2.9 -> 2.5.  Units of 2 tokens where units of 8
// leave SIMDs without two waves.
constexpr int kOutRows = 8;      // tokens per unit (1 for a decode step)

template <typename XT, int V, int TILE, int N>
__global__ __launch_bounds__(256) void output_kernel(const kda_output_args a, uint32_t ntiles, uint32_t units) {
    const int lane = threadIdx.x & 63;
    const uint32_t unit = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= units) return;
    const uint32_t D = static_cast<uint32_t>(a.H) * V;
    const uint32_t segs = segments(D, N);
    const uint32_t ch = (unit % segs) * (64 * N) + N * lane, bt = unit / segs;
    const bool valid = ch < D;
    const int64_t c0 = valid ? ch : 0, h = c0 / V;
    const int64_t t0 = static_cast<int64_t>(bt % ntiles) * TILE, b = bt / ntiles;
    const int n = static_cast<int>((a.T - t0) < TILE ? (a.T - t0) : TILE);

    // every load first, the weights' before the rows' (rows past the end re-read the last token)
    const RawParams<N> rw = ld_params<N>(a.weight, c0, a.w_dtype);
    const XT* op = static_cast<const XT*>(a.o) + b * a.o_stride[0] + h * a.o_stride[2] + c0 % V;
    const XT* gp = static_cast<const XT*>(a.gate) + b * a.gate_stride[0] + c0;
    Raw<XT, N> o[TILE], gt[TILE];
#pragma unroll
    for (int r = 0; r < TILE; ++r) {
        const int64_t t = t0 + (r < n ? r : n - 1);
        o[r] = ldn<N>(op + t * a.o_stride[1]);
        gt[r] = ldn<N>(gp + t * a.gate_stride[1]);
    }
    float w[N];
    decode(rw, a.w_dtype, w);

    XT* yp = static_cast<XT*>(a.y) + (b * a.T + t0) * D + c0;
#pragma unroll
    for (int r = 0; r < TILE; ++r) {
        float x[N], g[N];
        unpack(o[r], x);
        unpack(gt[r], g);
        const float rstd = rsqrtf(head_dot<XT, V>(x, x) / static_cast<float>(V) + a.eps);
        float y[N];
#pragma unroll
        for (int c = 0; c < N; ++c) y[c] = round_to<XT>((x[c] * rstd) * w[c]) * sigmoid_f(g[c]);
        if (r < n && valid) stn(yp + r * static_cast<int64_t>(D), y);
    }
}

// ---- host side --------------------------------------------------------------
bool dtype_ok(int32_t d) { return d == KDA_DTYPE_F32 || d == KDA_DTYPE_F16 || d == KDA_DTYPE_BF16; }
int64_t esize(int32_t d) { return d == KDA_DTYPE_F32 ? 4 : 2; }
bool head_ok(int64_t d) { return d == 64 || d == 128 || d == 256; }

// A vector access of `cpl` elements needs the pointer and every stride aligned to it.
bool vec_ok(const void* p, const int64_t* strides, int n, int64_t cpl, int32_t dtype) {
    if (reinterpret_cast<uintptr_t>(p) % static_cast<uintptr_t>(cpl * esize(dtype)) != 0) return false;
    for (int i = 0; i < n; ++i)
        if (strides[i] % cpl != 0) return false;
    return true;
}

bool overlap(const void* a, int64_t na, const void* b, int64_t nb) {
    const auto a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
    return a0 < b0 + static_cast<uintptr_t>(nb) && b0 < a0 + static_cast<uintptr_t>(na);
}

// Tokens per unit: 16; 4 where units of 16 would leave SIMDs without a wave
// (each also reads the conv_size - 1 rows before it; B=1 T=1000 H=16 K=128
// without the gates 8.8 us, 9.9 in units of 8; B=2 T=2048 25 us in units of
// 16, 30 in units of 4; with the gates, whose waves are shorter, B=4 T=2048 H=4
// 24 us in units of 4 and 28.5 in units of 16); 1 for a decode step.  A conv
// cache updated in place needs all its tokens in one unit, which then reads
// the old rows before it writes the new ones: 8 or 16.
template <typename XT, int K, int N>
void launch_prep_n(const kda_prep_args& a, hipStream_t stream) {
    const int64_t per = 2 * segments(a.H * K, N) + segments(a.H * a.V, N) +
                        (a.g != nullptr ? (a.H * K + kGateSeg - 1) / kGateSeg : 0);
    auto go = [&](auto tile) {
        constexpr int TILE = decltype(tile)::value;
        const int64_t ntiles = (a.T + TILE - 1) / TILE, units = a.B * ntiles * per;
        hipLaunchKernelGGL((prep_kernel<XT, K, TILE, N>), dim3(static_cast<unsigned>((units + 3) / 4)), dim3(256), 0,
                           stream, a, static_cast<uint32_t>(ntiles), static_cast<uint32_t>(units));
    };
    if constexpr (N == 4) {
        if (a.T == 1) return go(std::integral_constant<int, 1>{});
    }
    const int64_t kWaves = a.g != nullptr ? 4096 : 1280;
    bool in_place = false;
    for (int i = 0; i < 3; ++i) in_place = in_place || (a.hist_in[i] != nullptr && a.hist_in[i] == a.hist_out[i]);
    const bool few = a.B * ((a.T + kTile - 1) / kTile) * per < kWaves;
    if (few && (!in_place || a.T <= 4)) go(std::integral_constant<int, 4>{});
    else if (few && a.T <= 8) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, kTile>{});
}
template <typename XT, int K>
void launch_prep(const kda_prep_args& a, hipStream_t stream) {
    // us, eight channels a lane -> this: decode step, B=9 H=2 d=64 bf16 3.2 -> 2.8,
    // B=16 H=32 K=64 V=128 3.7 -> 2.7 (two channels a lane 2.8 and 3.9)
    if constexpr (kLaneCh<XT> == 8) {
        if (a.T > 1 && fills(a.H * K, 8) && fills(a.H * a.V, 8)) return launch_prep_n<XT, K, 8>(a, stream);
    }
    launch_prep_n<XT, K, 4>(a, stream);
}

template <typename XT>
int launch_prep_dims(const kda_prep_args& a, hipStream_t stream) {
    switch (a.K) {
        case 64: launch_prep<XT, 64>(a, stream); break;
        case 128: launch_prep<XT, 128>(a, stream); break;
        case 256: launch_prep<XT, 256>(a, stream); break;
        default: return KDA_ERR_UNSUPPORTED;
    }
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

template <typename XT, int V, int N>
void launch_output_n(const kda_output_args& a, hipStream_t stream) {
    const int64_t segs = segments(a.H * V, N);
    auto go = [&](auto tile) {
        constexpr int TILE = decltype(tile)::value;
        const int64_t ntiles = (a.T + TILE - 1) / TILE, units = a.B * ntiles * segs;
        hipLaunchKernelGGL((output_kernel<XT, V, TILE, N>), dim3(static_cast<unsigned>((units + 3) / 4)), dim3(256), 0,
                           stream, a, static_cast<uint32_t>(ntiles), static_cast<uint32_t>(units));
    };
    if (a.T == 1) go(std::integral_constant<int, 1>{});
    else if (a.B * ((a.T + kOutRows - 1) / kOutRows) * segs < 2048) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, kOutRows>{});
}
template <typename XT, int V>
void launch_output(const kda_output_args& a, hipStream_t stream) {
    const int64_t D = a.H * V;
    // us, eight channels a lane with the weights after the rows -> this (a wave a
    // head): H=1 V=64, B=5 T=2230 bf16 5.3 -> 3.5 (4.0), B=16 T=338 fp16 4.4 -> 2.7 (3.2)
    if constexpr (kLaneCh<XT> == 8) {
        if (a.T == 1 || fills(D, 8)) return launch_output_n<XT, V, 8>(a, stream);
        if constexpr (V <= 128) {
            if (D <= 128) return launch_output_n<XT, V, 2>(a, stream);
        }
    }
    launch_output_n<XT, V, 4>(a, stream);
}

template <typename XT>
int launch_output_dims(const kda_output_args& a, hipStream_t stream) {
    switch (a.V) {
        case 64: launch_output<XT, 64>(a, stream); break;
        case 128: launch_output<XT, 128>(a, stream); break;
        case 256: launch_output<XT, 256>(a, stream); break;
        default: return KDA_ERR_UNSUPPORTED;
    }
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

int validate_prep(const kda_prep_args* a) {
    if (a == nullptr) return KDA_ERR_NULL_POINTER;
    if (a->B < 0 || a->T < 0 || a->H < 0 || a->K <= 0 || a->V <= 0) return KDA_ERR_BAD_SHAPE;
    if (a->conv_size < 1 || a->conv_size > kMaxConv) return KDA_ERR_UNSUPPORTED;
    if (!head_ok(a->K) || !head_ok(a->V)) return KDA_ERR_UNSUPPORTED;
    if (!dtype_ok(a->x_dtype) || !dtype_ok(a->w_dtype) || !dtype_ok(a->p_dtype)) return KDA_ERR_BAD_DTYPE;
    if (!(a->l2_eps > 0.f)) return KDA_ERR_BAD_SHAPE;
    if (a->B == 0 || a->H == 0) return KDA_OK;
    // no tokens: nothing to compute, and a requested conv cache would need a copy
    if (a->T == 0) {
        for (int i = 0; i < 3; ++i)
            if (a->hist_out[i] != nullptr) return KDA_ERR_BAD_SHAPE;
        return KDA_OK;
    }
    const int64_t cm = a->conv_size - 1;
    for (int i = 0; i < 3; ++i) {
        if (a->x[i] == nullptr || a->conv_w[i] == nullptr) return KDA_ERR_NULL_POINTER;
        const int64_t cpl = (i == 2 ? a->V : a->K) / 64;
        if (!vec_ok(a->x[i], a->x_stride[i], 2, cpl, a->x_dtype)) return KDA_ERR_BAD_SHAPE;
        const int64_t D = a->H * (i == 2 ? a->V : a->K);
        if (a->hist_in[i] && !vec_ok(a->hist_in[i], nullptr, 0, cpl, a->x_dtype)) return KDA_ERR_BAD_SHAPE;
        if (a->hist_out[i]) {
            if (!vec_ok(a->hist_out[i], nullptr, 0, cpl, a->x_dtype)) return KDA_ERR_BAD_SHAPE;
            // in place only when one tile holds every token: the wave that
            // writes the cache is then the one that read it
            const int64_t nb = a->B * cm * D * esize(a->x_dtype);
            if (a->hist_in[i] && overlap(a->hist_in[i], nb, a->hist_out[i], nb) &&
                !(a->hist_in[i] == a->hist_out[i] && a->T <= kTile))
                return KDA_ERR_ALIAS;
        }
    }
    if (!a->q || !a->k || !a->v) return KDA_ERR_NULL_POINTER;
    // g and beta both absent: the gates are left to the core's gated entry points
    const bool gates = a->g != nullptr || a->beta != nullptr;
    if (gates && (!a->gk || !a->a_log || !a->dt_bias || !a->beta_logit || !a->g || !a->beta))
        return KDA_ERR_NULL_POINTER;
    const int64_t ck = a->K / 64, cv = a->V / 64;
    if (!vec_ok(a->q, nullptr, 0, ck, a->x_dtype) || !vec_ok(a->k, nullptr, 0, ck, a->x_dtype) ||
        !vec_ok(a->v, nullptr, 0, cv, a->x_dtype))
        return KDA_ERR_BAD_SHAPE;
    if (gates && (!vec_ok(a->gk, a->gk_stride, 2, ck, a->x_dtype) || !vec_ok(a->g, nullptr, 0, ck, KDA_DTYPE_F32)))
        return KDA_ERR_BAD_SHAPE;
    const int64_t ntiles = (a->T + kTile - 1) / kTile;
    if (a->B * ntiles * 4 * a->H > INT32_MAX) return KDA_ERR_BAD_SHAPE;
    return KDA_OK;
}

int validate_output(const kda_output_args* a) {
    if (a == nullptr) return KDA_ERR_NULL_POINTER;
    if (a->B < 0 || a->T < 0 || a->H < 0 || a->V <= 0) return KDA_ERR_BAD_SHAPE;
    if (!head_ok(a->V)) return KDA_ERR_UNSUPPORTED;
    if (!dtype_ok(a->x_dtype) || !dtype_ok(a->w_dtype)) return KDA_ERR_BAD_DTYPE;
    if (!(a->eps >= 0.f)) return KDA_ERR_BAD_SHAPE;
    if (a->B == 0 || a->T == 0 || a->H == 0) return KDA_OK;
    if (!a->o || !a->gate || !a->weight || !a->y) return KDA_ERR_NULL_POINTER;
    const int64_t cpl = a->V / 64;
    if (!vec_ok(a->o, a->o_stride, 3, cpl, a->x_dtype) || !vec_ok(a->gate, a->gate_stride, 2, cpl, a->x_dtype) ||
        !vec_ok(a->y, nullptr, 0, cpl, a->x_dtype))
        return KDA_ERR_BAD_SHAPE;
    if (a->B * ((a->T + kOutRows - 1) / kOutRows) * a->H > INT32_MAX) return KDA_ERR_BAD_SHAPE;
    return KDA_OK;
}

}  // namespace

}  // namespace kda

extern "C" {

int kda_prep_fwd(const kda_prep_args* args, void* stream) {
    const int st = kda::validate_prep(args);
    if (st != KDA_OK || args->B == 0 || args->H == 0 || args->T == 0) return st;
    const auto s = static_cast<hipStream_t>(stream);
    switch (args->x_dtype) {
        case KDA_DTYPE_F16: return kda::launch_prep_dims<_Float16>(*args, s);
        case KDA_DTYPE_BF16: return kda::launch_prep_dims<kda::bf16_t>(*args, s);
        default: return kda::launch_prep_dims<float>(*args, s);
    }
}

int kda_output_fwd(const kda_output_args* args, void* stream) {
    const int st = kda::validate_output(args);
    if (st != KDA_OK || args->B == 0 || args->T == 0 || args->H == 0) return st;
    const auto s = static_cast<hipStream_t>(stream);
    switch (args->x_dtype) {
        case KDA_DTYPE_F16: return kda::launch_output_dims<_Float16>(*args, s);
        case KDA_DTYPE_BF16: return kda::launch_output_dims<kda::bf16_t>(*args, s);
        default: return kda::launch_output_dims<float>(*args, s);
    }
}

}  // extern "C"
