// Gradients of the KDA layer's pre- and post-processing (kda_prep_fwd,
// kda_output_fwd), for gfx950.
//
// Training differentiates the whole layer (the reference by autograd through
// _projections and _output, kimi_linear/kda.py:399-470; it trains the layer in
// scripts/train_musicgpt_fp16.py:519-523).  The core has its own backward
// (kda_chunkwise_bwd); these kernels carry the gradients the rest of the way:
//
//   prep_bwd_kernel, one workgroup per (batch, 64-token tile, run of channels),
//     eight channels a lane as in the forward.  q, k, v: the forward is re-evaluated
//     from the saved projections (conv, SiLU, L2 norm), then
//       ds = rn dy - s rn^3 <s, dy>      (L2 norm; ds = dy / eps when clamped)
//       du = ds sigmoid(u) (1 + u (1 - sigmoid(u)))          (SiLU)
//       dx[t] = sum_j w[j] du[t + cm - j]                     (causal conv)
//     and the tile's shares of dw[j] = sum_t du[t] x[t - cm + j], db = sum du.
//     Gates: dgk = dg (-exp(A_log)) sigmoid(z),
//     dbeta_logit = dbeta beta (1 - beta), and the tile's shares of
//     dA_log = sum dg g and ddt_bias = sum dgk.
//   output_bwd_kernel, one wave per (batch, 32-token tile, head):
//       n = o r w, r = rsqrt(mean o^2 + eps), y = n sigmoid(z)
//       dn = dy sigmoid(z),  dz = dy n sigmoid(z) (1 - sigmoid(z))
//       do = r w dn - o r^3 <o, w dn> / V,  and the tile's share of dw = sum dn o r.
//   colsum_kernel: the parameter gradients as sums of the tiles' shares, in
//     tile order (fp32; identical from run to run).
//
// Both are HBM-streaming: every input element is read once per use (plus the
// conv halo), every gradient written once.
#include "kda_common.h"
#include "kda_rows.h"

namespace kda {

namespace {

constexpr int kMaxConvB = 4;      // largest conv_size (as the forward)
constexpr int kGroup = 4;         // tokens per step of a conv unit: the convolution's window, so a row's slot is its index
constexpr int kStep = 8;          // tokens per step of a gate unit
constexpr int kPrepTile = 64;     // tokens per prep unit, a workgroup's
constexpr int kSub = 4;           // its waves, a quarter of the tile each
constexpr int kOutStep = 8;       // tokens per step of an output unit
constexpr int kOutTile = 32;      // tokens per output unit

template <typename XT, int CPL>
struct alignas(sizeof(XT) * CPL) Vec {
    XT e[CPL];
};
template <typename XT, int CPL>
__device__ __forceinline__ void vld(const XT* p, float (&x)[CPL]) {
    const Vec<XT, CPL> v = *reinterpret_cast<const Vec<XT, CPL>*>(p);
#pragma unroll
    for (int c = 0; c < CPL; ++c) x[c] = to_f(v.e[c]);
}
template <typename XT, int CPL>
__device__ __forceinline__ void vst(XT* p, const float (&x)[CPL]) {
    Vec<XT, CPL> v;
#pragma unroll
    for (int c = 0; c < CPL; ++c) v.e[c] = from_f<XT>(x[c]);
    *reinterpret_cast<Vec<XT, CPL>*>(p) = v;
}

// Shares of the parameter gradients, one row per unit tile:
// conv i: [rows][D_i * conv_size] weights and [rows][D_i] biases; gates
// [rows][H K] for A_log and for dt_bias.
struct PrepParts {
    float* dw[3];
    float* db[3];
    float* da;
    float* ddt;
    int64_t rows;
};

int64_t prep_rows(int64_t B, int64_t T) { return B * ((T + kPrepTile - 1) / kPrepTile); }

PrepParts prep_parts(void* ws, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t cs) {
    PrepParts p;
    p.rows = prep_rows(B, T);
    float* f = static_cast<float*>(ws);
    const int64_t D[3] = {H * K, H * K, H * V};
    for (int i = 0; i < 3; ++i) {
        p.dw[i] = f;
        f += p.rows * D[i] * cs;
        p.db[i] = f;
        f += p.rows * D[i];
    }
    p.da = f;
    f += p.rows * H * K;
    p.ddt = f;
    return p;
}

int64_t prep_ws_floats(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t cs) {
    return prep_rows(B, T) * ((2 * H * K + H * V) * (cs + 1) + 2 * H * K);
}

// Sums over the waves of a tile, in their order; wave 0 has them.
template <int N>
__device__ __forceinline__ void sum_waves(float (&v)[N], float* red, int wave, int lane) {
    if (wave > 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) red[((wave - 1) * N + i) * 64 + lane] = v[i];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < kSub - 1; ++w)
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] += red[(w * N + i) * 64 + lane];
    }
}

// ---- q, k or v: 64 N channels over a token tile ------------------------------
// DH: the head size whose L2 norm is taken (q and k), 0 for none (v).  CS:
// conv_size, so that the taps are a few wide loads (one load and wait for each
// took 60.6 us at B=20 T=704 H=1 d=64 conv_size 2, before this split 37.0).  The tokens go by once: du[t] needs the x
// rows t - 3 .. t and completes dx[t - 3], so four x rows and four partial dx
// rows are held, in slots by the token's index modulo 4, and a wave's last
// three dx take du of three tokens past its own.  tw: tokens a wave, a quarter
// of the tile, or of a shorter sequence, in whole groups.  wl[L] is the tap of lag L:
// u[t] = sum_L wl[L] x[t - L], dx[t] = sum_L wl[L] du[t + L].
template <typename XT, int DH, int CS, int N>
__device__ __forceinline__ void conv_bwd_unit(const kda_prep_bwd_args& a, const PrepParts& pp, int i, int64_t b,
                                              int64_t tile, int64_t seg, int wave, int lane, int tw, float* red) {
    constexpr int G = kGroup;
    static_assert(G == kMaxConvB, "a row's slot is its index in the group");
    const int64_t D = a.H * (DH ? DH : a.V), T = a.T;
    const bool valid = seg * (64 * N) + N * lane < D;
    const int64_t ch0 = valid ? seg * (64 * N) + N * lane : 0;
    constexpr int cs = CS, cm = cs - 1;
    const int64_t dxs = a.dx_stride ? a.dx_stride : D;
    const XT* x = static_cast<const XT*>(a.x[i]) + b * a.x_stride[i][0] + ch0;
    const XT* dy = static_cast<const XT*>(a.dy[i]) + b * T * D + ch0;
    XT* dx = static_cast<XT*>(a.dx[i]) + b * T * dxs + ch0;
    const int64_t t0 = tile * kPrepTile + wave * tw;
    const int n = static_cast<int>(T - t0 < tw ? T - t0 : tw);      // <= 0: no token

    Raw<XT, N> nx[G], ny[G];
    const auto fetch = [&](int idx) {                   // rows past the end re-read the last token
#pragma unroll
        for (int r = 0; r < G; ++r) {
            const int64_t tok = t0 + idx + r < T ? t0 + idx + r : T - 1;
            nx[r] = ldn<N>(x + tok * a.x_stride[i][1]);
            ny[r] = ldn<N>(dy + tok * D);
        }
    };
    fetch(0);
    float xs[G][N], dxa[G][N], wl[cs][N], wc[N * cs], bias[N], dws[cs][N], dbs[N];
#pragma unroll
    for (int r = 1; r < G; ++r) {                       // tokens t0 - 3 .. t0 - 1
        const int64_t tok = t0 - G + r;
        const Raw<XT, N> h = ldn<N>(x + (tok < 0 ? 0 : (tok < T ? tok : T - 1)) * a.x_stride[i][1]);
        unpack(h, xs[r]);
        if (tok < 0) {
#pragma unroll
            for (int c = 0; c < N; ++c) xs[r][c] = 0.f;
        }
    }
#pragma unroll
    for (int c = 0; c < N; ++c) bias[c] = dbs[c] = 0.f;
    if (a.conv_b[i] != nullptr) decode(ld_params<N>(a.conv_b[i], ch0, a.w_dtype), a.w_dtype, bias);
    decode(ld_params<N * cs>(a.conv_w[i], ch0 * cs, a.w_dtype), a.w_dtype, wc);
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int L = 0; L < cs; ++L) {
            wl[L][c] = wc[cs * c + cm - L];
            dws[L][c] = 0.f;
        }
#pragma unroll
    for (int L = 0; L < G; ++L)
#pragma unroll
        for (int c = 0; c < N; ++c) dxa[L][c] = 0.f;
    const float inv_eps = 1.f / a.l2_eps;

    for (int idx0 = 0; n > 0 && idx0 < n + G - 1; idx0 += G) {
        Raw<XT, N> cx[G], cy[G];
#pragma unroll
        for (int r = 0; r < G; ++r) cx[r] = nx[r], cy[r] = ny[r];
        fetch(idx0 + G);
#pragma unroll
        for (int r = 0; r < G; ++r) {
            const int idx = idx0 + r;
            float d[N], u[N], sg[N], s[N];
            unpack(cx[r], xs[r]);
            unpack(cy[r], d);
#pragma unroll
            for (int c = 0; c < N; ++c) {
                u[c] = bias[c];
#pragma unroll
                for (int L = cm; L >= 0; --L) u[c] = fmaf(wl[L][c], xs[(r - L + G) % G][c], u[c]);
                sg[c] = sigmoid_f(u[c]);
                s[c] = u[c] * sg[c];
            }
            if constexpr (DH != 0) {
                // y = s min(rsqrt(sum s^2), 1/eps): a clamped row is s / eps
                const float rn = rsqrtf(head_dot<XT, DH>(s, s)), dot = head_dot<XT, DH>(s, d);
                const bool clamped = !(rn < inv_eps);
                const float k3 = rn * rn * rn * dot;
#pragma unroll
                for (int c = 0; c < N; ++c) d[c] = clamped ? d[c] * inv_eps : fmaf(rn, d[c], -s[c] * k3);
            }
            const bool in = t0 + idx < T;
#pragma unroll
            for (int c = 0; c < N; ++c) {
                d[c] *= sg[c] * fmaf(u[c], 1.f - sg[c], 1.f);
                d[c] = in ? d[c] : 0.f;
                dxa[r][c] = wl[0][c] * d[c];
#pragma unroll
                for (int L = 1; L < cs; ++L)
                    dxa[(r - L + G) % G][c] = fmaf(wl[L][c], d[c], dxa[(r - L + G) % G][c]);
            }
            if (idx < n) {                              // the tile's own tokens
#pragma unroll
                for (int c = 0; c < N; ++c) {
                    dbs[c] += d[c];
#pragma unroll
                    for (int L = 0; L < cs; ++L)
                        dws[L][c] = fmaf(d[c], xs[(r - L + G) % G][c], dws[L][c]);
                }
            }
            const int e = idx - (G - 1);
            if (e >= 0 && e < n && valid) stn(dx + (t0 + e) * dxs, dxa[(r + 1) % G]);
        }
    }
    float sums[(cs + 1) * N];
#pragma unroll
    for (int c = 0; c < N; ++c) {
#pragma unroll
        for (int L = 0; L < cs; ++L) sums[L * N + c] = dws[L][c];
        sums[cs * N + c] = dbs[c];
    }
    sum_waves(sums, red, wave, lane);
    if (!valid || wave > 0) return;
    const int64_t row = b * ((T + kPrepTile - 1) / kPrepTile) + tile;
#pragma unroll
    for (int c = 0; c < N; ++c) {
#pragma unroll
        for (int L = 0; L < cs; ++L) pp.dw[i][(row * D + ch0 + c) * cs + cm - L] = sums[L * N + c];
        if (a.db[i] != nullptr) pp.db[i][row * D + ch0 + c] = sums[cs * N + c];
    }
}

// ---- the gates of 256 channels over a token tile, and the betas of their heads
template <typename XT, int DH>
__device__ __forceinline__ void gate_bwd_unit(const kda_prep_bwd_args& a, const PrepParts& pp, int64_t b, int64_t tile,
                                              int64_t seg, int wave, int lane, int tw, float* red) {
    constexpr int N = 4, kHeads = kGateSeg / DH;
    const int64_t D = a.H * DH, T = a.T;
    const bool valid = seg * kGateSeg + N * lane < D;
    const int64_t ch0 = valid ? seg * kGateSeg + N * lane : 0;
    float neg_a[N], dtb[N], sa[N], sd[N];
    decode(ld_params<N>(a.a_log, ch0, a.p_dtype), a.p_dtype, neg_a);
    decode(ld_params<N>(a.dt_bias, ch0, a.p_dtype), a.p_dtype, dtb);
#pragma unroll
    for (int c = 0; c < N; ++c) {
        neg_a[c] = -__expf(neg_a[c]);
        sa[c] = sd[c] = 0.f;
    }
    const XT* gk = static_cast<const XT*>(a.gk) + b * a.gk_stride[0] + ch0;
    const float* dg = a.dg + b * T * D + ch0;
    XT* dgk = static_cast<XT*>(a.dgk) + b * T * D + ch0;
    const int64_t dls = a.dx_stride ? a.dx_stride : a.H;
    const int64_t t0 = tile * kPrepTile + wave * tw;
    const int64_t t1 = t0 + tw < T ? t0 + tw : T;
    // lane e < kStep kHeads of a step takes the beta of its token e / kHeads, head e % kHeads
    const int64_t bh = seg * kHeads + lane % kHeads;
    const bool beta_lane = lane < kStep * kHeads && bh < a.H;
    for (int64_t s0 = t0; s0 < t1; s0 += kStep) {
        Raw<XT, N> z[kStep];
        Raw<float, N> d[kStep];
#pragma unroll
        for (int t = 0; t < kStep; ++t) {
            const int64_t tok = s0 + t < t1 ? s0 + t : s0;
            z[t] = ldn<N>(gk + tok * a.gk_stride[1]);
            d[t] = ldn<N>(dg + tok * D);
        }
#pragma unroll
        for (int t = 0; t < kStep; ++t) {
            if (s0 + t >= t1) break;
            float zz[N], dd[N], o[N];
            unpack(z[t], zz);
            unpack(d[t], dd);
#pragma unroll
            for (int c = 0; c < N; ++c) {
                zz[c] += dtb[c];
                // softplus(z) = z above torch's threshold (20), and its
                // derivative 1 there; sigmoid(z) below
                const float sp = softplus(zz[c]);
                const float sl = zz[c] > 20.f ? 1.f : sigmoid_f(zz[c]);
                o[c] = dd[c] * neg_a[c] * sl;
                sd[c] += o[c];
                sa[c] = fmaf(dd[c], neg_a[c] * sp, sa[c]);
            }
            if (valid) stn(dgk + (s0 + t) * D, o);
        }
        const int64_t tok = s0 + lane / kHeads;
        if (beta_lane && tok < t1) {
            const float x = load_elem(a.beta_logit, b * a.beta_stride[0] + tok * a.beta_stride[1] + bh, a.x_dtype);
            const float bt = sigmoid_f(x);
            const float g = a.dbeta[(b * T + tok) * a.H + bh] * bt * (1.f - bt);
            store_elem(a.dbeta_logit, (b * T + tok) * dls + bh, a.x_dtype, g);
        }
    }
    float sums[2 * N];
#pragma unroll
    for (int c = 0; c < N; ++c) sums[c] = sa[c], sums[N + c] = sd[c];
    sum_waves(sums, red, wave, lane);
    if (!valid || wave > 0) return;
    const int64_t row = b * ((T + kPrepTile - 1) / kPrepTile) + tile;
#pragma unroll
    for (int c = 0; c < N; ++c) {
        pp.da[row * D + ch0 + c] = sums[c];
        pp.ddt[row * D + ch0 + c] = sums[N + c];
    }
}

// One workgroup per (batch, tile, 64 N channels of q, k, v or kGateSeg of the
// gates), the gates' shorter units last, into what the others leave free.
// Bound by the arithmetic on the channels (about 40 operations each, two of
// them transcendental) at two waves a SIMD.  A wave a head, two channels a
// lane, took 11 rows of du for 8 tokens and a 64-lane sum a row.  us of
// kda_prep_backward, then -> this, H=16 d=128 unless said, a wave a whole tile
// in brackets: B=4 T=2048 bf16 213 -> 135 (139), fp16 177 -> 138 (141), fp32
// 202 -> 184 (197); B=1 T=2048 bf16 65 -> 42 (55); B=1 T=500 52 -> 22 (49);
// B=1 T=1024 H=8 d=64 fp16 42 -> 20 (48).
template <typename XT, int K, int CS, int N>
__global__ __launch_bounds__(64 * kSub, 2) void prep_bwd_kernel(const kda_prep_bwd_args a, const PrepParts pp,
                                                         uint32_t ntiles, uint32_t convs, int tw) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __shared__ float red[(kSub - 1) * ((CS + 1) * N > 8 ? (CS + 1) * N : 8) * 64];    // (the gates: 8 sums a lane)
    if (blockIdx.x >= convs) {
        const uint32_t u = blockIdx.x - convs, segs = (static_cast<uint32_t>(a.H) * K + kGateSeg - 1) / kGateSeg;
        const uint32_t bt = u / segs;
        gate_bwd_unit<XT, K>(a, pp, bt / ntiles, bt % ntiles, u % segs, wave, lane, tw, red);
        return;
    }
    const uint32_t segk = static_cast<uint32_t>(segments(a.H * K, N)), segv = static_cast<uint32_t>(segments(a.H * a.V, N));
    const uint32_t per = 2 * segk + segv, s = blockIdx.x % per, bt = blockIdx.x / per;
    const int64_t tile = bt % ntiles, b = bt / ntiles;
    if (s < 2 * segk) {
        const int i = s >= segk;
        conv_bwd_unit<XT, K, CS, N>(a, pp, i, b, tile, s - i * segk, wave, lane, tw, red);
    } else {
        conv_bwd_unit<XT, 0, CS, N>(a, pp, 2, b, tile, s - 2 * segk, wave, lane, tw, red);
    }
}

// ---- output: one wave per (batch, 32-token tile, head) ---------------------
template <typename XT, int CPL>
__global__ __launch_bounds__(256) void output_bwd_kernel(const kda_output_bwd_args a, float* part, uint32_t ntiles,
                                                         uint32_t units) {
    const int lane = threadIdx.x & 63;
    const uint32_t unit = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= units) return;
    const uint32_t H = static_cast<uint32_t>(a.H);
    const int64_t h = unit % H;
    const uint32_t bt = unit / H;
    const int64_t tile = bt % ntiles, b = bt / ntiles;
    const int64_t V = 64 * CPL, T = a.T;
    const int64_t c0 = lane * CPL;
    const XT* op = static_cast<const XT*>(a.o) + b * a.o_stride[0] + h * a.o_stride[2] + c0;
    const XT* gp = static_cast<const XT*>(a.gate) + b * a.gate_stride[0] + h * V + c0;
    const XT* dyp = static_cast<const XT*>(a.dy) + b * T * a.H * V + h * V + c0;
    XT* dop = static_cast<XT*>(a.d_o) + b * T * a.H * V + h * V + c0;
    XT* dgp = static_cast<XT*>(a.dgate) + b * T * a.H * V + h * V + c0;
    float w[CPL], dws[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        w[c] = load_elem(a.weight, h * V + c0 + c, a.w_dtype);
        dws[c] = 0.f;
    }
    const float inv_v = 1.f / static_cast<float>(V);
    const int64_t t0 = tile * kOutTile;
    for (int step = 0; step < kOutTile / kOutStep; ++step) {
        const int64_t s0 = t0 + step * kOutStep;
        if (s0 >= T) break;
        float o[kOutStep][CPL], z[kOutStep][CPL], d[kOutStep][CPL];
#pragma unroll
        for (int r = 0; r < kOutStep; ++r) {
            const int64_t t = s0 + r < T ? s0 + r : s0;
            vld<XT, CPL>(op + t * a.o_stride[1], o[r]);
            vld<XT, CPL>(gp + t * a.gate_stride[1], z[r]);
            vld<XT, CPL>(dyp + t * a.H * V, d[r]);
        }
#pragma unroll
        for (int r = 0; r < kOutStep; ++r) {
            if (s0 + r >= T) break;
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < CPL; ++c) ss = fmaf(o[r][c], o[r][c], ss);
            const float rs = rsqrtf(wave_sum(ss) * inv_v + a.eps);
            float dn[CPL], dz[CPL], pr = 0.f;
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const float sg = sigmoid_f(z[r][c]);
                const float n = to_f(from_f<XT>((o[r][c] * rs) * w[c]));
                dn[c] = d[r][c] * sg;
                dz[c] = d[r][c] * n * sg * (1.f - sg);
                dws[c] = fmaf(dn[c], o[r][c] * rs, dws[c]);
                pr = fmaf(o[r][c], w[c] * dn[c], pr);
            }
            const float k3 = rs * rs * rs * wave_sum(pr) * inv_v;
            float g[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) g[c] = fmaf(rs * w[c], dn[c], -o[r][c] * k3);
            vst<XT, CPL>(dop + (s0 + r) * a.H * V, g);
            vst<XT, CPL>(dgp + (s0 + r) * a.H * V, dz);
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) part[(b * ntiles + tile) * a.H * V + h * V + c0 + c] = dws[c];
}

// ---- sums of the tiles' shares ---------------------------------------------
struct ColSum {
    const float* src;              // [rows][n]
    void* dst;                     // [n]
    int64_t n;
    int32_t dtype;                 // of dst
};
struct ColSums {
    ColSum s[8];
    int64_t rows;
};

__global__ __launch_bounds__(256) void colsum_kernel(const ColSums c) {
    const ColSum d = c.s[blockIdx.y];
    const int64_t k = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (d.src == nullptr || k >= d.n) return;
    // eight independent partial sums keep eight loads in flight; the order of
    // the additions is fixed
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int64_t r = 0;
    for (; r + 8 <= c.rows; r += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[u] += d.src[(r + u) * d.n + k];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (r + u < c.rows) acc[u] += d.src[(r + u) * d.n + k];
    store_elem(d.dst, k, d.dtype,
               ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7])));
}

int launch_colsum(const ColSums& c, int count, hipStream_t stream) {
    int64_t nmax = 0;
    for (int i = 0; i < count; ++i) nmax = c.s[i].n > nmax ? c.s[i].n : nmax;
    if (nmax == 0 || count == 0) return KDA_OK;
    hipLaunchKernelGGL(colsum_kernel, dim3(static_cast<unsigned>((nmax + 255) / 256), static_cast<unsigned>(count)),
                       dim3(256), 0, stream, c);
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

bool dtype_ok(int32_t d) { return d == KDA_DTYPE_F32 || d == KDA_DTYPE_F16 || d == KDA_DTYPE_BF16; }
int64_t esize(int32_t d) { return d == KDA_DTYPE_F32 ? 4 : 2; }
bool head_ok(int64_t d) { return d == 64 || d == 128; }
bool aligned(const void* p, int64_t bytes) { return reinterpret_cast<uintptr_t>(p) % static_cast<uintptr_t>(bytes) == 0; }

int validate_prep_bwd(const kda_prep_bwd_args* a) {
    if (a == nullptr) return KDA_ERR_NULL_POINTER;
    if (a->B < 0 || a->T < 0 || a->H < 0 || a->K <= 0 || a->V <= 0) return KDA_ERR_BAD_SHAPE;
    if (a->conv_size < 1 || a->conv_size > kMaxConvB) return KDA_ERR_UNSUPPORTED;
    if (!head_ok(a->K) || !head_ok(a->V)) return KDA_ERR_UNSUPPORTED;
    if (!dtype_ok(a->x_dtype) || !dtype_ok(a->w_dtype) || (a->gk && !dtype_ok(a->p_dtype))) return KDA_ERR_BAD_DTYPE;
    if (!(a->l2_eps > 0.f)) return KDA_ERR_BAD_SHAPE;
    if (a->B == 0 || a->H == 0 || a->T == 0) return KDA_OK;
    for (int i = 0; i < 3; ++i) {
        if (!a->x[i] || !a->conv_w[i] || !a->dy[i] || !a->dx[i] || !a->dw[i]) return KDA_ERR_NULL_POINTER;
        const int64_t cpl = (i == 2 ? a->V : a->K) / 64, vb = cpl * esize(a->x_dtype);
        if (!aligned(a->x[i], vb) || a->x_stride[i][0] % cpl || a->x_stride[i][1] % cpl || !aligned(a->dy[i], vb) ||
            !aligned(a->dx[i], vb))
            return KDA_ERR_BAD_SHAPE;
    }
    if (a->gk) {
        if (!a->a_log || !a->dt_bias || !a->beta_logit || !a->dg || !a->dbeta || !a->dgk || !a->dbeta_logit ||
            !a->da_log || !a->ddt_bias)
            return KDA_ERR_NULL_POINTER;
        const int64_t cpl = a->K / 64, vb = cpl * esize(a->x_dtype);
        if (!aligned(a->gk, vb) || a->gk_stride[0] % cpl || a->gk_stride[1] % cpl || !aligned(a->dgk, vb) ||
            !aligned(a->dg, cpl * 4))
            return KDA_ERR_BAD_SHAPE;
    }
    if (!a->workspace) return KDA_ERR_NULL_POINTER;
    if (!aligned(a->workspace, 16)) return KDA_ERR_BAD_SHAPE;
    if (prep_rows(a->B, a->T) * 4 * a->H > INT32_MAX) return KDA_ERR_BAD_SHAPE;
    const int64_t hk = a->H * a->K, hv = a->H * a->V;
    if (a->dx_stride != 0 && (a->dx_stride < (hk > hv ? hk : hv) || a->dx_stride % (a->K > a->V ? a->K / 64 : a->V / 64)))
        return KDA_ERR_BAD_SHAPE;
    return KDA_OK;
}

int validate_output_bwd(const kda_output_bwd_args* a) {
    if (a == nullptr) return KDA_ERR_NULL_POINTER;
    if (a->B < 0 || a->T < 0 || a->H < 0 || a->V <= 0) return KDA_ERR_BAD_SHAPE;
    if (!head_ok(a->V)) return KDA_ERR_UNSUPPORTED;
    if (!dtype_ok(a->x_dtype) || !dtype_ok(a->w_dtype)) return KDA_ERR_BAD_DTYPE;
    if (!(a->eps >= 0.f)) return KDA_ERR_BAD_SHAPE;
    if (a->B == 0 || a->T == 0 || a->H == 0) return KDA_OK;
    if (!a->o || !a->gate || !a->weight || !a->dy || !a->d_o || !a->dgate || !a->dweight || !a->workspace)
        return KDA_ERR_NULL_POINTER;
    const int64_t cpl = a->V / 64, vb = cpl * esize(a->x_dtype);
    if (!aligned(a->o, vb) || a->o_stride[0] % cpl || a->o_stride[1] % cpl || a->o_stride[2] % cpl ||
        !aligned(a->gate, vb) || a->gate_stride[0] % cpl || a->gate_stride[1] % cpl || !aligned(a->dy, vb) ||
        !aligned(a->d_o, vb) || !aligned(a->dgate, vb) || !aligned(a->workspace, 16))
        return KDA_ERR_BAD_SHAPE;
    if (a->B * ((a->T + kOutTile - 1) / kOutTile) * a->H > INT32_MAX) return KDA_ERR_BAD_SHAPE;
    return KDA_OK;
}

template <typename XT, int K, int CS, int N>
int launch_prep_bwd_n(const kda_prep_bwd_args& a, hipStream_t stream) {
    const PrepParts pp = prep_parts(a.workspace, a.B, a.T, a.H, a.K, a.V, a.conv_size);
    const int64_t ntiles = (a.T + kPrepTile - 1) / kPrepTile, hk = a.H * a.K, hv = a.H * a.V;
    const int64_t convs = pp.rows * (2 * segments(hk, N) + segments(hv, N));
    const int64_t gates = a.gk != nullptr ? pp.rows * ((hk + kGateSeg - 1) / kGateSeg) : 0;
    const dim3 grid(static_cast<unsigned>(convs + gates));
    const uint32_t nt = static_cast<uint32_t>(ntiles), nc = static_cast<uint32_t>(convs);
    // a sequence of one tile is shared out among its waves (us with 16 tokens a
    // wave -> this: B=52 T=18 H=8 d=128 bf16 32.8 -> 24.1, B=16 T=24 H=16 d=64 fp16
    // conv 2 16.6 -> 12.6; a wave a head took 27.0 and 14.2)
    const int tw = ntiles > 1 ? kPrepTile / kSub : static_cast<int>((a.T + kGroup * kSub - 1) / (kGroup * kSub)) * kGroup;
    hipLaunchKernelGGL((prep_bwd_kernel<XT, K, CS, N>), grid, dim3(64 * kSub), 0, stream, a, pp, nt, nc, tw);
    if (hipGetLastError() != hipSuccess) return KDA_ERR_LAUNCH;
    ColSums c{};
    c.rows = pp.rows;
    int n = 0;
    const int64_t D[3] = {a.H * a.K, a.H * a.K, a.H * a.V};
    const int32_t wt = a.typed_param_grads ? a.w_dtype : KDA_DTYPE_F32;
    const int32_t pt = a.typed_param_grads ? a.p_dtype : KDA_DTYPE_F32;
    for (int i = 0; i < 3; ++i) {
        c.s[n++] = ColSum{pp.dw[i], a.dw[i], D[i] * a.conv_size, wt};
        if (a.db[i] != nullptr) c.s[n++] = ColSum{pp.db[i], a.db[i], D[i], wt};
    }
    if (a.gk != nullptr) {
        c.s[n++] = ColSum{pp.da, a.da_log, a.H * a.K, pt};
        c.s[n++] = ColSum{pp.ddt, a.ddt_bias, a.H * a.K, pt};
    }
    return launch_colsum(c, n, stream);
}

template <typename XT, int K, int CS>
int launch_prep_bwd(const kda_prep_bwd_args& a, hipStream_t stream) {
    // us, eight channels a lane -> four: B=39 T=348 H=2 K=64 V=128 fp16 57.0 -> 43.4,
    // B=42 T=210 H=1 K=128 V=64 fp16 43.4 -> 34.2 (a wave a head 46.6 and 42.2)
    if constexpr (kLaneCh<XT> == 8) {
        if (fills(a.H * K, 8) && fills(a.H * a.V, 8)) return launch_prep_bwd_n<XT, K, CS, 8>(a, stream);
    }
    return launch_prep_bwd_n<XT, K, CS, 4>(a, stream);
}

template <typename XT, int K>
int launch_prep_bwd_conv(const kda_prep_bwd_args& a, hipStream_t stream) {
    switch (a.conv_size) {
        case 4: return launch_prep_bwd<XT, K, 4>(a, stream);
        case 3: return launch_prep_bwd<XT, K, 3>(a, stream);
        case 2: return launch_prep_bwd<XT, K, 2>(a, stream);
        default: return launch_prep_bwd<XT, K, 1>(a, stream);
    }
}

template <typename XT>
int launch_prep_bwd_dims(const kda_prep_bwd_args& a, hipStream_t stream) {
    return a.K == 64 ? launch_prep_bwd_conv<XT, 64>(a, stream) : launch_prep_bwd_conv<XT, 128>(a, stream);
}

template <typename XT>
int launch_output_bwd(const kda_output_bwd_args& a, hipStream_t stream) {
    const int64_t ntiles = (a.T + kOutTile - 1) / kOutTile;
    const int64_t units = a.B * ntiles * a.H;
    float* part = static_cast<float*>(a.workspace);
    const dim3 grid(static_cast<unsigned>((units + 3) / 4)), block(256);
    const uint32_t nt = static_cast<uint32_t>(ntiles), nu = static_cast<uint32_t>(units);
    if (a.V == 64)
        hipLaunchKernelGGL((output_bwd_kernel<XT, 1>), grid, block, 0, stream, a, part, nt, nu);
    else
        hipLaunchKernelGGL((output_bwd_kernel<XT, 2>), grid, block, 0, stream, a, part, nt, nu);
    if (hipGetLastError() != hipSuccess) return KDA_ERR_LAUNCH;
    ColSums c{};
    c.rows = a.B * ntiles;
    c.s[0] = ColSum{part, a.dweight, a.H * a.V, a.typed_param_grads ? a.w_dtype : KDA_DTYPE_F32};
    return launch_colsum(c, 1, stream);
}

}  // namespace

}  // namespace kda

extern "C" {

size_t kda_prep_bwd_workspace_size(int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t conv_size) {
    if (B <= 0 || T <= 0 || H <= 0 || K <= 0 || V <= 0 || conv_size < 1) return 0;
    return static_cast<size_t>(kda::prep_ws_floats(B, T, H, K, V, conv_size)) * sizeof(float);
}

int kda_prep_bwd(const kda_prep_bwd_args* args, void* stream) {
    const int st = kda::validate_prep_bwd(args);
    if (st != KDA_OK || args->B == 0 || args->H == 0 || args->T == 0) return st;
    const auto s = static_cast<hipStream_t>(stream);
    switch (args->x_dtype) {
        case KDA_DTYPE_F16: return kda::launch_prep_bwd_dims<_Float16>(*args, s);
        case KDA_DTYPE_BF16: return kda::launch_prep_bwd_dims<kda::bf16_t>(*args, s);
        default: return kda::launch_prep_bwd_dims<float>(*args, s);
    }
}

size_t kda_output_bwd_workspace_size(int64_t B, int64_t T, int64_t H, int64_t V) {
    if (B <= 0 || T <= 0 || H <= 0 || V <= 0) return 0;
    return static_cast<size_t>(B * ((T + kda::kOutTile - 1) / kda::kOutTile) * H * V) * sizeof(float);
}

int kda_output_bwd(const kda_output_bwd_args* args, void* stream) {
    const int st = kda::validate_output_bwd(args);
    if (st != KDA_OK || args->B == 0 || args->T == 0 || args->H == 0) return st;
    const auto s = static_cast<hipStream_t>(stream);
    switch (args->x_dtype) {
        case KDA_DTYPE_F16: return kda::launch_output_bwd<_Float16>(*args, s);
        case KDA_DTYPE_BF16: return kda::launch_output_bwd<kda::bf16_t>(*args, s);
        default: return kda::launch_output_bwd<float>(*args, s);
    }
}

}  // extern "C"
