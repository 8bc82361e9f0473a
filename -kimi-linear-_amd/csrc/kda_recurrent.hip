// Token-by-token KDA recurrence (decode step) for gfx950.
//
// Replaces the body of kda_recurrent (kimi_linear/kda.py:196-219).  Per token
// the reference makes ~8 elementwise passes over the [K, V] fp32 state; this
// kernel keeps the state of one (batch, head, V-tile) in registers for the
// whole call, so each state element is read from HBM once and written once.
//
// Per token, with a = exp(g), q~ = q * scale (single-pass form of Eq. 1):
//   S' = Diag(a) S,   u = S'^T k,   r = S'^T q~,   d = beta (v - u)
//   S  = S' + k d^T,  o = r + (q~ . k) d            (== S^T q~ after the update)
//
// Work split: one workgroup of NW waves per (b, h, V-tile of 4 CPL NW
// columns); wave w owns 4 CPL columns of the tile for all K rows, lane l the
// four columns 4 (l % CPL) .. +3 of K CPL / 64 rows: a row segment is one
// 16-byte access.  Both K-reductions (u, r) are sums over the lanes of one
// column group, inside the wave (permlane swaps and DPP row rotations, all
// on the VALU): no LDS round and no barrier.  q~, k and a of a token are
// staged once per workgroup in LDS.
//
// Order of the sums over K.  The rows form 16 groups: RV = min(4, K / 16)
// adjacent rows, RV v .. RV v + RV - 1, of every 16 RV belong to group v.  A
// group's rows are summed in order, then the groups as a tree: v with v + 8,
// then + 4, + 2, + 1.  Every kernel and lane layout here keeps that order
// (and q.k's: runs of 8 channels in order, then lanes_sum), so a token gives
// the same bits alone or in a span, whatever the number of sequences.
//
// Gated calls (kda_recurrent_gated_fwd) take the gate's up-projection gk and
// the beta logits instead of g and beta and form, while staging the token,
// a = exp(-exp(A_log) softplus(gk + dt_bias)) and beta = sigmoid(logit) in
// fp32 (kimi_linear/kda.py:452-460).
//
// A call of several tokens runs recurrent_seq_kernel (below): the work split
// above hides a token's loads only behind other waves, and puts 32 x 4 state
// values in a lane, so a chain of tokens took 2.5 us a token.
#include <type_traits>

#include "kda_common.h"
#include "kda_launch.h"

namespace kda {

namespace {

constexpr int rows_run(int K) { return K / 16 < 4 ? K / 16 : 4; }   // RV

// Sum over the 64 / CPL lanes that share l % CPL (all-reduce): lane bit 5
// first, then 4, 3, 2 (lane groups with their indices' higher bits first).
template <int CPL>
__device__ __forceinline__ float colgroup_sum(float x) {
    {
        const unsigned u = __float_as_uint(x);
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    {
        const unsigned u = __float_as_uint(x);
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if constexpr (CPL <= 8)
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xF, 0xF, true));   // row_ror:8
    if constexpr (CPL == 4)
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xF, 0xF, true));   // row_ror:4
    return x;
}

// q.k of a staged token, in every lane: runs of 8 channels, then lanes_sum.
template <int K>
__device__ __forceinline__ float staged_qk(const float* q, const float* k, int lane) {
    constexpr int TPR = K / 8;
    const int c = 8 * (lane % TPR);
    float x = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) x = fmaf(q[c + j], k[c + j], x);
    return lanes_sum<TPR>(x);
}

// VEC: the state is read (unless absent) and written as 16-byte-aligned fp32
// rows with buffer loads/stores; otherwise element by element in any dtype.
// A separate instantiation keeps the generic path's registers out of the
// fast one.
//
// Lane l of a wave holds 4 adjacent state columns (column group l % CPL) of
// the row groups v = l / CPL + NG m, NG = 64 / CPL.
template <int K, int NW, int CPL, bool VEC>
__global__ __launch_bounds__(64 * NW) void recurrent_kernel(const kda_fwd_args a, const kda_gate_args gate) {
    static_assert(CPL == 4 || CPL == 8 || CPL == 16, "column groups per wave");
    constexpr int RPL = K * CPL / 64;           // rows per lane
    constexpr int VT = 4 * CPL * NW;            // columns per workgroup
    constexpr int RV = rows_run(K);             // adjacent rows of a row group
    constexpr int NG = 64 / CPL;                // lane groups
    constexpr int NM = 16 / NG;                 // row groups per lane
    constexpr int NP = K / (16 * RV);           // runs per row group
    static_assert(RPL == RV * NM * NP, "a lane's rows");
    // the row of a lane's value (run p of row group m, j-th row) past its first
    auto row = [](int p, int m, int j) { return 16 * RV * p + RV * NG * m + j; };
    auto index = [](int p, int m, int j) { return (m * NP + p) * RV + j; };

    __shared__ float s_q[K], s_k[K], s_a[K];

    const int64_t H = a.H, T = a.T, V = a.V;
    const int nvt = static_cast<int>(V / VT);
    int bid = blockIdx.x;
    const int vt = bid % nvt;
    bid /= nvt;
    const int64_t h = bid % H;
    const int64_t b = bid / H;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int cg = lane % CPL, rg = lane / CPL;
    const int r0 = RV * rg;
    const int64_t col0 = static_cast<int64_t>(vt) * VT + 4 * CPL * wave + 4 * cg;
    const int64_t sbase = (b * H + h) * static_cast<int64_t>(K) * V;

    // fp32 state rows go through one buffer descriptor per head: the lane
    // offset is one register and the row offset a scalar
    const uint32_t row_bytes = static_cast<uint32_t>(V) * 4u;
    const uint32_t lane_off = static_cast<uint32_t>(r0) * row_bytes + static_cast<uint32_t>(col0) * 4u;
    // The state is read once per call, and each element's last read comes
    // right before its write: non-temporal loads (nt) keep the read lines from
    // being retained in the caches, which measured 30.7 -> 22.5 us per B=64
    // H=16 d=128 decode step when the state comes from HBM (in place), at a
    // small cost when it sits in the Infinity Cache (20.9 -> 22.2 us).
    constexpr int kLoadNonTemporal = 2;
    // The new state is stored streaming as well (nt with sc1): a decode step
    // over states larger than the Infinity Cache (five rotating 64 MiB sets at
    // B=64 H=16 d=128) measured 24.35 -> 23.30 us per step against plain
    // stores, in place 23.40 -> 23.21 us; one cache-resident set stepped into
    // a fresh tensor pays 23.1 -> 24.1 us.
    constexpr int kStoreStreaming = 2 | 16;
    float S[RPL][4];
    auto each_row = [&](auto&& f) {              // f(index in S, row past the lane's first)
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int j = 0; j < RV; ++j) f(index(p, m, j), row(p, m, j));
    };
    if (a.state_in == nullptr) {
#pragma unroll
        for (int j = 0; j < RPL; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) S[j][c] = 0.f;
    } else if (VEC) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(static_cast<const float*>(a.state_in) + sbase), static_cast<short>(0),
            static_cast<int>(K * row_bytes), 0x00020000);
        each_row([&](int i, int r) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(lane_off),
                                                                  static_cast<int>(r * row_bytes), kLoadNonTemporal);
            S[i][0] = __uint_as_float(x[0]); S[i][1] = __uint_as_float(x[1]);
            S[i][2] = __uint_as_float(x[2]); S[i][3] = __uint_as_float(x[3]);
        });
    } else {
        each_row([&](int i, int r) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                S[i][c] = load_elem(a.state_in, sbase + static_cast<int64_t>(r0 + r) * V + col0 + c,
                                    a.state_in_dtype);
        });
    }

    // channels this thread stages per token, and for a gated call their
    // exp(A_log) and dt_bias, fetched once (beside the state loads)
    constexpr int KPT = (K + 64 * NW - 1) / (64 * NW);
    float gcoef[KPT], gbias[KPT];
    if (gate.a_log) {
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
            const int i = tid + 64 * NW * j;
            gcoef[j] = i < K ? expf(gate.a_log[h * K + i]) : 0.f;
            gbias[j] = i < K ? gate.dt_bias[h * K + i] * kLog2e : 0.f;
        }
    }
    const float scale = a.scale;
    for (int64_t t = 0; t < T; ++t) {
        // ---- stage token t: q~, k, exp(g) for all K rows; v, beta per lane.
        // Every load is issued before any is decoded.
        const int64_t tq = b * a.q_stride[0] + t * a.q_stride[1] + h * a.q_stride[2];
        const int64_t tk = b * a.k_stride[0] + t * a.k_stride[1] + h * a.k_stride[2];
        const int64_t tg = b * a.g_stride[0] + t * a.g_stride[1] + h * a.g_stride[2];
        const int64_t tv = b * a.v_stride[0] + t * a.v_stride[1] + h * a.v_stride[2] + col0;
        RawElem rv[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) rv[c] = load_raw_elem(a.v, tv + c, a.qkv_dtype);
        const RawElem rb =
            load_raw_elem(a.beta, b * a.beta_stride[0] + t * a.beta_stride[1] + h * a.beta_stride[2], a.beta_dtype);
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
            const int i = tid + 64 * NW * j;
            if (i >= K) break;
            const RawElem rq = load_raw_elem(a.q, tq + i, a.qkv_dtype);
            const RawElem rk = load_raw_elem(a.k, tk + i, a.qkv_dtype);
            const RawElem rg = load_raw_elem(a.g, tg + i, a.g_dtype);
            s_q[i] = decode_elem(rq, a.qkv_dtype) * scale;
            s_k[i] = decode_elem(rk, a.qkv_dtype);
            const float gv = decode_elem(rg, a.g_dtype);
            s_a[i] = gate.a_log ? gate_decay(fmaf(gv, kLog2e, gbias[j]), gcoef[j]) : fast_exp(gv);
        }
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = decode_elem(rv[c], a.qkv_dtype);
        const float beta = gate.a_log ? sigmoid_f(decode_elem(rb, a.beta_dtype)) : decode_elem(rb, a.beta_dtype);
        __syncthreads();

        // ---- decay, then the K-reductions: each row group of the lane in
        // order, the lane's groups as a tree (v with v + 8, then + 4), then the
        // lanes
        const float qk = staged_qk<K>(s_q, s_k, lane);
        float pu[NM][4], pr[NM][4];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
#pragma unroll
            for (int c = 0; c < 4; ++c) pu[m][c] = pr[m][c] = 0.f;
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int j = 0; j < RV; ++j) {
                    const int i = index(p, m, j), r = r0 + row(p, m, j);
                    const float al = s_a[r], qq = s_q[r], kk = s_k[r];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        S[i][c] *= al;
                        pu[m][c] = fmaf(S[i][c], kk, pu[m][c]);
                        pr[m][c] = fmaf(S[i][c], qq, pr[m][c]);
                    }
                }
        }
#pragma unroll
        for (int w = NM / 2; w > 0; w /= 2)
#pragma unroll
            for (int m = 0; m < w; ++m)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    pu[m][c] += pu[m + w][c];
                    pr[m][c] += pr[m + w][c];
                }
        float d[4], rr[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            d[c] = beta * (v[c] - colgroup_sum<CPL>(pu[0][c]));
            rr[c] = colgroup_sum<CPL>(pr[0][c]);
        }
        each_row([&](int i, int r) {
            const float kk = s_k[r0 + r];
#pragma unroll
            for (int c = 0; c < 4; ++c) S[i][c] = fmaf(kk, d[c], S[i][c]);
        });
        if (rg == 0) {
            const int64_t io = ((b * T + t) * H + h) * V + col0;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float o = fmaf(qk, d[c], rr[c]);
                if (a.clamp_fp16_out && a.qkv_dtype == KDA_DTYPE_F16) o = clamp_fp16_safe(o);
                store_elem(a.o, io + c, a.qkv_dtype, o);
            }
        }
        if (t + 1 < T) __syncthreads();   // the next token's staging overwrites s_*
    }

    if (VEC) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(static_cast<float*>(a.state_out) + sbase,
                                                          static_cast<short>(0), static_cast<int>(K * row_bytes),
                                                          0x00020000);
        typedef unsigned int u4 __attribute__((ext_vector_type(4)));
        each_row([&](int i, int r) {
            __builtin_amdgcn_raw_buffer_store_b128(
                u4{__float_as_uint(S[i][0]), __float_as_uint(S[i][1]), __float_as_uint(S[i][2]),
                   __float_as_uint(S[i][3])},
                rs, static_cast<int>(lane_off), static_cast<int>(r * row_bytes), kStoreStreaming);
        });
    } else {
        each_row([&](int i, int r) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                store_elem(a.state_out, sbase + static_cast<int64_t>(r0 + r) * V + col0 + c, a.state_out_dtype,
                           S[i][c]);
        });
    }
}

// Several tokens: the same recurrence, split so that a token is short.
//
// One workgroup of four waves per (b, h, 16 C columns); a wave owns 4 C
// columns, lane l the C columns C (l / 16) .. of K / 16 rows (row group
// l % 16: pieces of up to four adjacent rows, one piece in every 16, so the
// 16 row groups read one contiguous line of a token's q, k or a from LDS).
// The K-reductions run inside a 16-lane DPP row, and a lane holds K C / 16
// state values (8 C at K = 128) instead of 128.
//
// Tokens are staged in groups of G: a thread converts 8 channels of one
// token's q, k and g, fetched a group ahead, and their part of q.k.  Groups
// alternate between two LDS buffers, one barrier a group.  The lane of row
// group i holds v of the group's token i and keeps that token's outputs: one
// store a group, issued after the next group's wait for its loads (the
// counter that wait reads also counts stores).
//
// ckpt: the chunk records' fp32 states (kda_chunkwise_fwd_ckpt of fp32
// activations), stored before every 32-token chunk.
//
// Bound by the chain of a token (the sums, their exchange, the update: about
// 60 VALU instructions a wave at C = 1), not by memory.  B=2 T=1024 H=16
// K=V=128 fp32: 2630 us in recurrent_kernel, 191 here (187 ns a token); a
// span of 37 tokens at B=4 95 -> 15.6 us.  The error against float64 is that
// of recurrent_kernel (state 4.7e-8; outputs 9.4e-8 where it has 1.2e-7).
//
// ROWS says how rows of q, k and g are fetched: 16-byte loads of 16-bit q, k
// and g (kRows16), 16-bit q, k and 32-bit g (kRowsMixed) or all 32-bit
// (kRows32), every row 16-byte aligned; or element by element in any types
// (kRowsAny).  In the first three the loop's loads are free of branches:
// a token past T reads row T - 1 again, whose values nothing uses.  (A branch
// around a load, or a type chosen between two loads, made the compiler wait
// for the loads right after issuing them: 239 us in place of 199.)
enum Rows { kRowsAny, kRows16, kRowsMixed, kRows32 };
template <int K, int C, Rows ROWS>
__global__ __launch_bounds__(256) void recurrent_seq_kernel(const kda_fwd_args a, const kda_gate_args gate,
                                                            float* ckpt) {
    constexpr int G = K <= 128 ? 16 : 8;         // tokens per group
    constexpr int R = K / 16;                    // rows per lane
    constexpr int RV = rows_run(K);              // rows per piece
    constexpr int NP = R / RV;                   // pieces
    constexpr int TPR = K / 8;                   // staging threads per token
    static_assert(G * TPR <= 256 && 32 % G == 0, "a group is staged in one pass; records start at group starts");
    typedef float fv __attribute__((ext_vector_type(RV)));
    typedef float f2 __attribute__((ext_vector_type(2)));

    // token i of group buffer b is row b G + i; one row more, since a token's
    // operands are read while the token before it runs, the group's last too
    __shared__ fv s_q[2 * G + 1][K / RV], s_k[2 * G + 1][K / RV], s_a[2 * G + 1][K / RV];
    __shared__ f2 s_b[2 * G + 1];                // beta and q.k of a token

    const int64_t H = a.H, T = a.T, V = a.V;
    const int nvt = static_cast<int>(V / (16 * C));
    int bid = blockIdx.x;
    const int vt = bid % nvt;
    bid /= nvt;
    const int64_t h = bid % H;
    const int64_t b = bid / H;

    const int tid = threadIdx.x;
    const int rg = tid & 15, cl = (tid >> 4) & 3, wave = tid >> 6;
    const int64_t col0 = static_cast<int64_t>(vt) * (16 * C) + 4 * C * wave + C * cl;
    const int64_t sbase = (b * H + h) * static_cast<int64_t>(K) * V + col0;
    auto row = [&](int e) { return (e / RV) * 16 * RV + RV * rg + e % RV; };

    // ---- staging: this thread's token of a group and its 8 channels
    const int st = tid / TPR, sc = 8 * (tid % TPR);
    const bool stager = st < G;
    const bool q32 = ROWS == kRowsAny ? a.qkv_dtype == KDA_DTYPE_F32 : ROWS == kRows32;
    const bool g32 = ROWS == kRowsAny ? a.g_dtype == KDA_DTYPE_F32 : ROWS != kRows16;
    uint32_t raw_q[8], raw_k[8], raw_g[8], raw_b[1], raw_v[C];
    uint32_t b_shift;
    // 8 consecutive elements held raw: 16-bit ones two a word (kRowsAny: one a word)
    auto fetch8 = [](const void* p, int64_t i, bool f32, uint32_t (&w)[8]) {
        if constexpr (ROWS != kRowsAny) {
            const uint4* x = reinterpret_cast<const uint4*>(static_cast<const char*>(p) + (f32 ? 4 : 2) * i);
            const uint4 lo = x[0];
            w[0] = lo.x; w[1] = lo.y; w[2] = lo.z; w[3] = lo.w;
            if (f32) {
                const uint4 hi = x[1];
                w[4] = hi.x; w[5] = hi.y; w[6] = hi.z; w[7] = hi.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                w[j] = f32 ? static_cast<const uint32_t*>(p)[i + j] : static_cast<const uint16_t*>(p)[i + j];
        }
    };
    // (one branch on the type for all eight)
    auto decode8 = [](const uint32_t (&w)[8], int dtype, bool f32, float (&x)[8]) {
        auto half = [&](int j) {
            return static_cast<uint16_t>(ROWS != kRowsAny ? w[j / 2] >> (16 * (j % 2)) : w[j]);
        };
        if (f32) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = __uint_as_float(w[j]);
        } else if (dtype == KDA_DTYPE_F16) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = static_cast<float>(__builtin_bit_cast(_Float16, half(j)));
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = bf16_bits_to_f32(half(j));
        }
    };
    auto fetch = [&](int64_t t0) {
        const int64_t ts = t0 + (stager ? st : 0), t = ts < T ? ts : T - 1;
        fetch8(a.q, b * a.q_stride[0] + t * a.q_stride[1] + h * a.q_stride[2] + sc, q32, raw_q);
        fetch8(a.k, b * a.k_stride[0] + t * a.k_stride[1] + h * a.k_stride[2] + sc, q32, raw_k);
        fetch8(a.g, b * a.g_stride[0] + t * a.g_stride[1] + h * a.g_stride[2] + sc, g32, raw_g);
        const RawElem rb = load_raw_elem(a.beta, b * a.beta_stride[0] + t * a.beta_stride[1] + h * a.beta_stride[2],
                                         a.beta_dtype);
        raw_b[0] = rb.word;
        b_shift = rb.shift;
        const int64_t tw = t0 + (rg < G ? rg : 0), tv = tw < T ? tw : T - 1;
        const int64_t i = b * a.v_stride[0] + tv * a.v_stride[1] + h * a.v_stride[2] + col0;
#pragma unroll
        for (int c = 0; c < C; ++c)
            raw_v[c] = q32 ? static_cast<const uint32_t*>(a.v)[i + c] : static_cast<const uint16_t*>(a.v)[i + c];
    };
    float gcoef[8], gbias[8];
    if (gate.a_log) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            gcoef[j] = expf(gate.a_log[h * K + sc + j]);
            gbias[j] = gate.dt_bias[h * K + sc + j] * kLog2e;
        }
    }

    fetch(0);

    float S[R][C];
    const bool s_vec = a.state_in_dtype == KDA_DTYPE_F32 && (reinterpret_cast<uintptr_t>(a.state_in) & 15) == 0;
    typedef float fc __attribute__((ext_vector_type(C)));
#pragma unroll
    for (int e = 0; e < R; ++e) {
        if (a.state_in == nullptr) {
#pragma unroll
            for (int c = 0; c < C; ++c) S[e][c] = 0.f;
        } else if (s_vec) {
            const fc x = *reinterpret_cast<const fc*>(static_cast<const float*>(a.state_in) + sbase + row(e) * V);
#pragma unroll
            for (int c = 0; c < C; ++c) S[e][c] = x[c];
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) S[e][c] = load_elem(a.state_in, sbase + row(e) * V + c, a.state_in_dtype);
        }
    }

    float* ckh = ckpt ? ckpt + (b * H + h) * ((T + 31) / 32) * ckpt_record(K, V) : nullptr;
    const float scale = a.scale;
    // the lane's outputs of the group at t0 (token t0 + rg)
    float oc[C];
    auto put_out = [&](int64_t t0) {
        if (rg < G && t0 + rg < T) {
            const int64_t io = ((b * T + t0 + rg) * H + h) * V + col0;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                float o = oc[c];
                if (a.clamp_fp16_out && a.qkv_dtype == KDA_DTYPE_F16) o = clamp_fp16_safe(o);
                store_elem(a.o, io + c, a.qkv_dtype, o);
            }
        }
    };
    int buf = 0;
    for (int64_t t0 = 0; t0 < T; t0 += G, buf ^= 1) {
        use_here(raw_q);
        use_here(raw_k);
        use_here(raw_g);
        use_here(raw_b);
        use_here(raw_v);
        // the group before this one: stored here and not at its end, where the
        // wait for the loads above would have been one for these stores too
        if (t0 > 0) put_out(t0 - G);
        if (stager) {
            float q[8], k[8], al[8], qk = 0.f;
            decode8(raw_q, a.qkv_dtype, q32, q);
            decode8(raw_k, a.qkv_dtype, q32, k);
            decode8(raw_g, a.g_dtype, g32, al);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                q[j] *= scale;
                qk = fmaf(q[j], k[j], qk);
            }
            if (gate.a_log) {
#pragma unroll
                for (int j = 0; j < 8; ++j) al[j] = gate_decay(fmaf(al[j], kLog2e, gbias[j]), gcoef[j]);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) al[j] = fast_exp(al[j]);
            }
#pragma unroll
            for (int j = 0; j < 8; j += RV) {
                fv x, y, z;
#pragma unroll
                for (int i = 0; i < RV; ++i) {
                    x[i] = q[j + i];
                    y[i] = k[j + i];
                    z[i] = al[j + i];
                }
                s_q[buf * G + st][(sc + j) / RV] = x;
                s_k[buf * G + st][(sc + j) / RV] = y;
                s_a[buf * G + st][(sc + j) / RV] = z;
            }
            qk = lanes_sum<TPR>(qk);             // over the token's staging threads
            if (sc == 0) {
                const float bt = decode_elem(RawElem{raw_b[0], b_shift}, a.beta_dtype);
                s_b[buf * G + st] = f2{gate.a_log ? sigmoid_f(bt) : bt, qk};
            }
        }
        float v[C];                              // of token rg
#pragma unroll
        for (int c = 0; c < C; ++c)
            v[c] = q32 ? __uint_as_float(raw_v[c])
                       : (a.qkv_dtype == KDA_DTYPE_F16
                              ? static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(raw_v[c])))
                              : bf16_bits_to_f32(static_cast<uint16_t>(raw_v[c])));
        fetch(t0 + G);
        __syncthreads();
        if (ckh && t0 % 32 == 0) {
            float* rec = ckh + (t0 / 32) * ckpt_record(K, V) + col0;
#pragma unroll
            for (int e = 0; e < R; ++e)
#pragma unroll
                for (int c = 0; c < C; ++c) rec[row(e) * V + c] = S[e][c];
        }

        const int n = T - t0 < G ? static_cast<int>(T - t0) : G;
        struct Tok {
            fv q[NP], k[NP], al[NP];
            f2 b_qk;
        };
        Tok ta, tb;
        auto read = [&](Tok& x, int i) {
            const int w = buf * G + i;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                x.al[p] = s_a[w][16 * p + rg];
                x.k[p] = s_k[w][16 * p + rg];
                x.q[p] = s_q[w][16 * p + rg];
            }
            x.b_qk = s_b[w];
        };
        read(ta, 0);
        // token i of the group, the j-th of its four (whose v sits in row
        // group j); the next token's operands are requested first
        auto step = [&](auto jc, int i, const Tok& x, Tok& next) {
            constexpr int J = decltype(jc)::value;
            read(next, i + 1);
            __builtin_amdgcn_sched_barrier(0);
            float u[C], r[C];
#pragma unroll
            for (int c = 0; c < C; ++c) u[c] = r[c] = 0.f;
#pragma unroll
            for (int e = 0; e < R; ++e) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    S[e][c] *= x.al[e / RV][e % RV];
                    u[c] = fmaf(S[e][c], x.k[e / RV][e % RV], u[c]);
                    r[c] = fmaf(S[e][c], x.q[e / RV][e % RV], r[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) u[c] = row16_sum(u[c]);
#pragma unroll
            for (int c = 0; c < C; ++c) r[c] = row16_sum(r[c]);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float d = x.b_qk[0] * (row16_bcast<J>(v[c]) - u[c]);
#pragma unroll
                for (int e = 0; e < R; ++e) S[e][c] = fmaf(x.k[e / RV][e % RV], d, S[e][c]);
                const float o = fmaf(x.b_qk[1], d, r[c]);
                oc[c] = rg == i ? o : oc[c];
            }
        };
        auto next4 = [&]() {
#pragma unroll
            for (int c = 0; c < C; ++c) v[c] = row16_down4(v[c]);
        };
        using J0 = std::integral_constant<int, 0>;
        using J1 = std::integral_constant<int, 1>;
        using J2 = std::integral_constant<int, 2>;
        using J3 = std::integral_constant<int, 3>;
        int i = 0;
        for (; i + 4 <= n; i += 4) {
            step(J0{}, i, ta, tb);
            step(J1{}, i + 1, tb, ta);
            step(J2{}, i + 2, ta, tb);
            step(J3{}, i + 3, tb, ta);
            next4();
        }
        if (i < n) step(J0{}, i, ta, tb);
        if (i + 1 < n) step(J1{}, i + 1, tb, ta);
        if (i + 2 < n) step(J2{}, i + 2, ta, tb);
    }
    put_out(T - 1 - (T - 1) % G);

    const bool o_vec = a.state_out_dtype == KDA_DTYPE_F32 && (reinterpret_cast<uintptr_t>(a.state_out) & 15) == 0;
#pragma unroll
    for (int e = 0; e < R; ++e) {
        if (o_vec) {
            fc x;
#pragma unroll
            for (int c = 0; c < C; ++c) x[c] = S[e][c];
            *reinterpret_cast<fc*>(static_cast<float*>(a.state_out) + sbase + row(e) * V) = x;
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) store_elem(a.state_out, sbase + row(e) * V + c, a.state_out_dtype, S[e][c]);
        }
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// How recurrent_seq_kernel may fetch the rows of q, k and g.
Rows seq_rows(const kda_fwd_args& a) {
    auto aligned = [&](const void* p, const int64_t (&st)[3], int dtype) {
        const int64_t es = dtype == KDA_DTYPE_F32 ? 4 : 2;
        return aligned16(p) && (a.B == 1 || st[0] * es % 16 == 0) && (a.T == 1 || st[1] * es % 16 == 0) &&
               (a.H == 1 || st[2] * es % 16 == 0);
    };
    if (!aligned(a.q, a.q_stride, a.qkv_dtype) || !aligned(a.k, a.k_stride, a.qkv_dtype) ||
        !aligned(a.g, a.g_stride, a.g_dtype))
        return kRowsAny;
    const bool q32 = a.qkv_dtype == KDA_DTYPE_F32, g32 = a.g_dtype == KDA_DTYPE_F32;
    return q32 ? (g32 ? kRows32 : kRowsAny) : (g32 ? kRowsMixed : kRows16);
}

template <int K, int C>
int launch_seq_c(const kda_fwd_args& a, hipStream_t stream, const kda_gate_args& gate, float* ckpt) {
    const dim3 grid(static_cast<unsigned>(a.B * a.H * (a.V / (16 * C)))), block(256);
    switch (seq_rows(a)) {
        case kRows16:
            hipLaunchKernelGGL((recurrent_seq_kernel<K, C, kRows16>), grid, block, 0, stream, a, gate, ckpt);
            break;
        case kRowsMixed:
            hipLaunchKernelGGL((recurrent_seq_kernel<K, C, kRowsMixed>), grid, block, 0, stream, a, gate, ckpt);
            break;
        case kRows32:
            hipLaunchKernelGGL((recurrent_seq_kernel<K, C, kRows32>), grid, block, 0, stream, a, gate, ckpt);
            break;
        default:
            hipLaunchKernelGGL((recurrent_seq_kernel<K, C, kRowsAny>), grid, block, 0, stream, a, gate, ckpt);
    }
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

template <int K, int NW, int CPL>
int launch_k_nw(const kda_fwd_args& a, hipStream_t stream, const kda_gate_args& gate) {
    const dim3 grid(static_cast<unsigned>(a.B * a.H * (a.V / (4 * CPL * NW)))), block(64 * NW);
    const bool vec = (a.V & 3) == 0 && a.state_out_dtype == KDA_DTYPE_F32 && aligned16(a.state_out) &&
                     (a.state_in == nullptr || (a.state_in_dtype == KDA_DTYPE_F32 && aligned16(a.state_in)));
    if (vec)
        hipLaunchKernelGGL((recurrent_kernel<K, NW, CPL, true>), grid, block, 0, stream, a, gate);
    else
        hipLaunchKernelGGL((recurrent_kernel<K, NW, CPL, false>), grid, block, 0, stream, a, gate);
    return hipGetLastError() == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}

// Columns per workgroup of a span, 16 C: the narrowest that keeps the
// workgroups within what runs side by side.  us at K = V = 128, C = 1 / 2 / 4:
// 256 workgroups of C = 1 (B=2 H=16 T=1024, fp32) 191 / 260 / 433; 512 (B=4,
// T=37) 16.8 / 15.6 / 22.0; 1024 (B=8, T=300) 150 / 117 / 133; 2048 (B=16,
// T=200) 175 / 151 / 144; 4096 (B=32, T=100) 178 / 155 / 141.
template <int K>
int launch_seq(const kda_fwd_args& a, hipStream_t stream, const kda_gate_args& gate, float* ckpt) {
    const int64_t wgs = a.B * a.H * (a.V / 16);
    if (wgs > 1024 && a.V % 64 == 0) return launch_seq_c<K, 4>(a, stream, gate, ckpt);
    if (wgs > 256 && a.V % 32 == 0) return launch_seq_c<K, 2>(a, stream, gate, ckpt);
    return launch_seq_c<K, 1>(a, stream, gate, ckpt);
}

// Spans of smaller states (cols = B H V) whose tokens are faster one at a time:
// 2 tokens of many columns, whose chains already fill the chip; up to four of more
// workgroups of 32 columns than run side by side (V no multiple of 64); and K =
// 256, whose span kernel holds 8 tokens a group.  us, one at a time / span kernel,
// fp16: T=2 K=V=128, 8192 columns 6.6 / 6.2, 16384 7.4 / 8.2, 32768 8.9 / 10.5;
// K=V=64, 16384 5.8 / 5.9, 24576 6.1 / 6.6, T=3 7.5 / 7.0; K=V=32, 24576 5.6 /
// 5.6, 32768 5.7 / 6.3; K=64 V=32, 32768, T=2 6.4 / 9.4, T=4 9.3 / 10.0, T=6 12.1
// / 10.7, at 24576 T=3 7.5 / 7.1; K=128 V=32, 16384, T=3 9.2 / 8.5, 24576, T=3
// 10.3 / 12.5, T=4 12.3 / 12.9, T=6 16.4 / 14.0; K=256 V=64, 8192, T=2 8.0 / 8.8, T=3 10.0 /
// 9.2, 16384, T=4 13.7 / 13.2 (fp32 13.5 / 14.2), T=6 17.3 / 14.2, 24576, T=6
// 21.9 / 24.9.
template <int K>
bool one_by_one(int64_t T, int64_t V, int64_t cols) {
    if (K == 256) return cols > 16384 || (cols > 8192 && T <= 4) || (cols > 4096 && T == 2);
    if (T == 2) return cols > (K == 128 ? 8192 : 16384);
    return K >= 64 && V % 64 != 0 && cols > (K == 128 ? 16384 : 24576) && T <= 4;
}

template <int K>
int launch_k(const kda_fwd_args& a, hipStream_t stream, const kda_gate_args& gate, float* ckpt) {
    // A single token, and 2 to 7 tokens of a state large enough to be bound by
    // its own read and write (B=64 H=16 K=V=128, 64 MiB: T=2 26 us against 37
    // in the span kernel, T=4 33 / 40, T=8 41 / 41; B=16: T=2 11.5 / 11.2, T=4
    // 17 / 12), run one token at a time over wide column tiles.
    const int64_t cols = a.B * a.H * a.V;
    const bool wide = cols > 64 * 512 || one_by_one<K>(a.T, a.V, cols);
    if (ckpt != nullptr || (a.T > 1 && (a.T >= 8 || !wide))) return launch_seq<K>(a, stream, gate, ckpt);
    // K <= 128: one wave a workgroup, of 64 columns (K = 128: 32 rows x 4
    // columns a lane, 2 waves a SIMD: the 2048 waves of a B=64 H=16 V=128 step
    // are all resident at once), 32 or 16.  A narrower wave's chain is
    // shorter, a wider one has more of the state in flight.  us a step at
    // H=16 K=V=128, 64 / 32 / 16 columns: B=1 5.3 / 4.3 / 4.0, B=8 6.0 / 5.3 /
    // 5.2, B=16 8.9 / 8.6 / 10.6, B=32 14.2 / 13.1 / 23.0, B=48 18.8 / 19.5 /
    // 33.1, B=64 22.9 / 27.8 / 44.0; K=V=64, 32 / 16: B=1 3.5 / 3.4, B=16 4.1 /
    // 4.1, B=64 7.8 / 11.1.  K 256: 16 columns a wave (K / 16 rows a lane).
    if constexpr (K <= 128) {
        if (cols <= 64 * 256 || a.V % 32 != 0) return launch_k_nw<K, 1, 4>(a, stream, gate);
        if constexpr (K == 128) {
            if (cols > 64 * 1024 && a.V % 64 == 0) return launch_k_nw<K, 1, 16>(a, stream, gate);
        }
        return launch_k_nw<K, 1, 8>(a, stream, gate);
    }
    if (a.V % 64 == 0) return launch_k_nw<K, 4, 4>(a, stream, gate);
    if (a.V % 32 == 0) return launch_k_nw<K, 2, 4>(a, stream, gate);
    return launch_k_nw<K, 1, 4>(a, stream, gate);
}

}  // namespace

bool recurrent_supported(int64_t K, int64_t V) {
    if (!(K == 32 || K == 64 || K == 128 || K == 256)) return false;
    return V % 16 == 0;
}

int recurrent_launch(const kda_fwd_args& a, hipStream_t stream, const kda_gate_args* gate_p, float* ckpt) {
    const kda_gate_args gate = gate_p ? *gate_p : kda_gate_args{nullptr, nullptr};
    switch (a.K) {
        case 32: return launch_k<32>(a, stream, gate, ckpt);
        case 64: return launch_k<64>(a, stream, gate, ckpt);
        case 128: return launch_k<128>(a, stream, gate, ckpt);
        case 256: return launch_k<256>(a, stream, gate, ckpt);
        default: return KDA_ERR_UNSUPPORTED;
    }
}

}  // namespace kda
