// kda_short.hip -- sequences of at most 16 tokens at D = 32 or 64: the whole
// recurrence, and its whole adjoint, of one (b, h) in one wave, straight from
// the op's inputs to its outputs.
//
// What bounds them: HBM.  A sequence of 8 tokens at D = 64 reads 4 to 5 KB and
// writes 1 KB of o and a 16 KB state.  The chunked kernels pad such a sequence
// to a 64-row chunk, write its factors (41 KB) and states (24 KB) for the next
// kernel and run five of them: the time-only scan of 1568 x 12 sequences of 8
// tokens took 913 us forward and 1890 us backward on them.  Here 101 us forward
// (433 MB, 4.3 TB/s, the 308 MB of final states most of it) and 87 us backward
// without states (231 MB, 2.7 TB/s; 200 VGPRs, two waves a SIMD).
//
// One wave per sequence, four waves of a workgroup side by side with their own
// LDS and no workgroup barrier.  The sequence is one block of at most 16 rows:
//     A_kk, A_qk   e^{a_t - a_s} pair by pair (a: cumsum of g), exact at any decay
//                  and any sign of g -- at most 136 pairs, so no anchors
//     V' = (I + diag(beta) A_kk)^-1 beta (V - e^a K S0),  O = e^a Q S0 + A_qk V'
//     S  = S0 e^G + (e^{G - a} K)^T V'
// Two lane maps alternate through LDS rows of D + 4 floats: lane = channel for
// everything per (t, d) (the solves are T dependent rows of one FMA per lane),
// lane = pair (t, s) for the dot products over channels.  Products with a state
// run on the fp32 MFMA (16x16x4): nothing is rounded below fp32 between the
// inputs and the outputs, for bf16 operands too.
#include "kda_internal.h"

namespace kda {

namespace {

__device__ __forceinline__ float uniform(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr float LOG2E = 1.44269504088896340736f;
// A token's g below this, less the sum of its channel's positive g, is taken as
// that floor: a weight across the token is then at most e^-110, zero in fp32,
// with either value, and the cumsums of the tokens after it keep their precision.
constexpr float G_MIN = -110.f;

// The wave's TT x D tile of a [B, T, H, D] tensor as 16-byte vectors, rows past
// T zero: vector c (row c / CPR) on lane c % 64.
template <int D, int TT, typename E>
struct Rows {
    static constexpr int EPV = 16 / (int)sizeof(E), CPR = D / EPV, N = TT * CPR, NV = (N + 63) / 64;
    uint4 r[NV];
    __device__ __forceinline__ void load(const E* base, size_t ld, int T) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * 64 + lane_id(), row = c / CPR;
            r[i] = make_uint4(0u, 0u, 0u, 0u);
            if (row < T) r[i] = *reinterpret_cast<const uint4*>(base + (size_t)row * ld + (c % CPR) * EPV);
        }
    }
    __device__ __forceinline__ void put(float* lds) const {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * 64 + lane_id(), row = c / CPR;
            if (N % 64 != 0 && c >= N) break;
            float4* p = reinterpret_cast<float4*>(lds + row * (D + 4) + (c % CPR) * EPV);
            if constexpr (sizeof(E) == 4) {
                p[0] = make_float4(__uint_as_float(r[i].x), __uint_as_float(r[i].y), __uint_as_float(r[i].z),
                                   __uint_as_float(r[i].w));
            } else {
                p[0] = make_float4(bf_lo(r[i].x), bf_hi(r[i].x), bf_lo(r[i].y), bf_hi(r[i].y));
                p[1] = make_float4(bf_lo(r[i].z), bf_hi(r[i].z), bf_lo(r[i].w), bf_hi(r[i].w));
            }
        }
    }
};

// LDS rows to the rows t < T of a [B, T, H, D] tensor
template <int D, int TT, typename E>
__device__ __forceinline__ void rows_out(const float* lds, E* base, size_t ld, int T) {
    using R = Rows<D, TT, E>;
#pragma unroll
    for (int i = 0; i < R::NV; ++i) {
        const int c = i * 64 + lane_id(), row = c / R::CPR, col = (c % R::CPR) * R::EPV;
        if (row >= T) continue;
        const float4* p = reinterpret_cast<const float4*>(lds + row * (D + 4) + col);
        uint4 o;
        if constexpr (sizeof(E) == 4) {
            o = __builtin_bit_cast(uint4, p[0]);
        } else {
            const float4 x = p[0], y = p[1];
            o = make_uint4(pack2bf(x.x, x.y), pack2bf(x.z, x.w), pack2bf(y.x, y.y), pack2bf(y.z, y.w));
        }
        *reinterpret_cast<uint4*>(base + (size_t)row * ld + col) = o;
    }
}

// dot products of the rows of LDS tiles, lane = pair: X[t].Y[s] summed over the
// channels for s <= t, by 8 x 8 blocks (t = 8 bi + lane / 8, s = 8 bj + lane % 8)
template <int TT> struct Pairs {
    static constexpr int NBK = TT == 8 ? 1 : 3;
    __device__ static __forceinline__ int t(int b) { return (b > 0 ? 8 : 0) + (lane_id() >> 3); }
    __device__ static __forceinline__ int s(int b) { return (b > 1 ? 8 : 0) + (lane_id() & 7); }
};

__device__ __forceinline__ float dot4(float4 a, float4 b, float c) {
    return fmaf(a.x, b.x, fmaf(a.y, b.y, fmaf(a.z, b.z, fmaf(a.w, b.w, c))));
}

// A_kk (s < t) and A_qk (s <= t) from the rows Q, K and a (in log2 units),
// zeros elsewhere, into TT x TT tiles of row stride TT + 4
template <int D, int TT>
__device__ __forceinline__ void decay_pairs(const float* Q, const float* K, const float* A, float* akk, float* aqk) {
    using P = Pairs<TT>;
    constexpr int LD = D + 4, LA = TT + 4;
    float sk[P::NBK] = {}, sq[P::NBK] = {};
#pragma unroll 2
    for (int d = 0; d < D; d += 4) {
#pragma unroll
        for (int b = 0; b < P::NBK; ++b) {
            const int t = P::t(b) * LD + d, s = P::s(b) * LD + d;
            const float4 kt = *reinterpret_cast<const float4*>(K + t), qt = *reinterpret_cast<const float4*>(Q + t);
            const float4 at = *reinterpret_cast<const float4*>(A + t), as = *reinterpret_cast<const float4*>(A + s);
            float4 x = *reinterpret_cast<const float4*>(K + s);
            x.x *= __builtin_amdgcn_exp2f(at.x - as.x);
            x.y *= __builtin_amdgcn_exp2f(at.y - as.y);
            x.z *= __builtin_amdgcn_exp2f(at.z - as.z);
            x.w *= __builtin_amdgcn_exp2f(at.w - as.w);
            sk[b] = dot4(kt, x, sk[b]);
            sq[b] = dot4(qt, x, sq[b]);
        }
    }
#pragma unroll
    for (int b = 0; b < P::NBK; ++b) {
        const int t = P::t(b), s = P::s(b);
        akk[t * LA + s] = s < t ? sk[b] : 0.f;
        aqk[t * LA + s] = s <= t ? sq[b] : 0.f;
    }
}

// row t of a TT x TT tile, the first n entries (uniform addresses)
template <int TT>
__device__ __forceinline__ void tile_row(const float* tile, int t, int n, float (&r)[TT]) {
#pragma unroll
    for (int s = 0; s < TT; s += 4)
        if (s < n) {
            const float4 x = *reinterpret_cast<const float4*>(tile + t * (TT + 4) + s);
            r[s] = x.x; r[s + 1] = x.y; r[s + 2] = x.z; r[s + 3] = x.w;
        }
}

// The sum over the channels of each LDS row: every lane gets row lane / PARTS's
template <int D, int TT>
__device__ __forceinline__ float row_sums(const float* lds) {
    constexpr int PARTS = 64 / TT, W = D / PARTS;
    const float* p = lds + (lane_id() / PARTS) * (D + 4) + (lane_id() % PARTS) * W;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < W; c += 4) {
        const float4 x = *reinterpret_cast<const float4*>(p + c);
        s += (x.x + x.y) + (x.z + x.w);
    }
#pragma unroll
    for (int m = 1; m < PARTS; m <<= 1) s += __shfl_xor(s, m, 64);
    return s;
}

// acc[n] (rows t = 4 g4 + e, columns 16 n + l % 16) += X M with X the LDS rows
// and M[k][c] = S[c][k] of the row-major D x D state S in memory
template <int D, int TT>
__device__ __forceinline__ void rows_times_St(const float* X, const float* __restrict__ S, f32x4 (&acc)[D / 16]) {
    const int r = lane_id() & 15, g4 = lane_id() >> 4;
#pragma unroll
    for (int m = 0; m < D / 16; ++m) {
        const float4 x = *reinterpret_cast<const float4*>(X + (r & (TT - 1)) * (D + 4) + 16 * m + 4 * g4);
#pragma unroll
        for (int n = 0; n < D / 16; ++n) {
            const float4 s = *reinterpret_cast<const float4*>(S + (size_t)(16 * n + r) * D + 16 * m + 4 * g4);
            acc[n] = mfma_f32(x.x, s.x, acc[n]);
            acc[n] = mfma_f32(x.y, s.y, acc[n]);
            acc[n] = mfma_f32(x.z, s.z, acc[n]);
            acc[n] = mfma_f32(x.w, s.w, acc[n]);
        }
    }
}

// as rows_times_St with M = S: acc[n][t][c] += sum_k X[t][k] S[k][c]
template <int D, int TT>
__device__ __forceinline__ void rows_times_S(const float* X, const float* __restrict__ S, f32x4 (&acc)[D / 16]) {
    const int r = lane_id() & 15, g4 = lane_id() >> 4;
#pragma unroll
    for (int m = 0; m < D / 16; ++m) {
        const float4 x = *reinterpret_cast<const float4*>(X + (r & (TT - 1)) * (D + 4) + 16 * m + 4 * g4);
#pragma unroll
        for (int n = 0; n < D / 16; ++n) {
            const float* s = S + (size_t)(16 * m + 4 * g4) * D + 16 * n + r;
            acc[n] = mfma_f32(x.x, s[0], acc[n]);
            acc[n] = mfma_f32(x.y, s[D], acc[n]);
            acc[n] = mfma_f32(x.z, s[2 * D], acc[n]);
            acc[n] = mfma_f32(x.w, s[3 * D], acc[n]);
        }
    }
}

// accumulator tiles to LDS rows t < TT
template <int D, int TT>
__device__ __forceinline__ void acc_rows(const f32x4 (&acc)[D / 16], float* lds) {
    const int r = lane_id() & 15, g4 = lane_id() >> 4;
    if (TT < 16 && g4 >= TT / 4) return;
#pragma unroll
    for (int n = 0; n < D / 16; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[(4 * g4 + e) * (D + 4) + 16 * n + r] = acc[n][e];
}

template <int N> __device__ __forceinline__ void clear(f32x4 (&acc)[N]) {
#pragma unroll
    for (int n = 0; n < N; ++n) acc[n] = zero4();
}

// out[i][j] = in[i][j] eG[j] (in null: zero) + sum_t (X0[t][j] Y0[t][i] - X1[t][j] Y1[t][i]),
// row-major D x D in memory; X1 null: one product.  y1s scales the rows of Y1.
template <int D, int TT>
__device__ __forceinline__ void state_out(const float* __restrict__ in, const float* eG, const float* X0,
                                          const float* Y0, const float* X1, const float* Y1, const float* y1s,
                                          float* __restrict__ out) {
    const int r = lane_id() & 15, g4 = lane_id() >> 4;
    constexpr int LD = D + 4, KS = TT / 4;
#pragma unroll
    for (int m = 0; m < D / 16; ++m) {
        float x0[KS], x1[KS];
#pragma unroll
        for (int p = 0; p < KS; ++p) {
            x0[p] = X0[(4 * p + g4) * LD + 16 * m + r];
            x1[p] = X1 ? -X1[(4 * p + g4) * LD + 16 * m + r] : 0.f;
        }
        const float4 e = *reinterpret_cast<const float4*>(eG + 16 * m + 4 * g4);
#pragma unroll
        for (int n = 0; n < D / 16; ++n) {
            const size_t off = (size_t)(16 * n + r) * D + 16 * m + 4 * g4;
            f32x4 acc = zero4();
            if (in) {
                const float4 s = *reinterpret_cast<const float4*>(in + off);
                acc = f32x4{s.x * e.x, s.y * e.y, s.z * e.z, s.w * e.w};
            }
#pragma unroll
            for (int p = 0; p < KS; ++p) {
                acc = mfma_f32(x0[p], Y0[(4 * p + g4) * LD + 16 * n + r], acc);
                if (X1) acc = mfma_f32(x1[p], y1s[4 * p + g4] * Y1[(4 * p + g4) * LD + 16 * n + r], acc);
            }
            *reinterpret_cast<f32x4*>(out + off) = acc;
        }
    }
}

template <int D, int TT> struct ShortLds {
    static constexpr int ROWS = TT * (D + 4), TILE = TT * (TT + 4);
    float r[4][ROWS];
    float akk[TILE], aqk[TILE];
    float eG[D], beta[16];
};

// lane = channel: the in-block cumsum of g in log2 units, one decay per channel
// or per head; rows past T add nothing
template <int D, int TT, typename GT>
__device__ __forceinline__ void cumsum_g(const GT* __restrict__ g, size_t grow, int H, int T, int h, const float* lds,
                                         int ch, float (&a)[TT]) {
    float c = 0.f;
    float gh = 0.f;
    if constexpr (std::is_same<GT, GHead>::value) {
        const float* gp = reinterpret_cast<const float*>(g);
        if (lane_id() < T) gh = gp[(grow + lane_id()) * H + h];
    }
    float floor = G_MIN;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        a[t] = std::is_same<GT, GHead>::value ? uniform(gh, t) : lds[t * (D + 4) + ch];
        floor -= fmaxf(a[t], 0.f);
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        c += a[t] < floor ? floor : a[t];   // keeps a NaN
        a[t] = c * LOG2E;
    }
}

// the storage type of a per-channel g's rows (GHead has none: loaded apart)
template <typename GT> struct GStore { using type = GT; };
template <> struct GStore<GHead> { using type = float; };

template <int D, int TT, typename ST, typename GT>
__global__ __launch_bounds__(256) void kda_short_fwd_kernel(ShortArgs a) {
    constexpr int LD = D + 4;
    constexpr bool HEAD = std::is_same<GT, GHead>::value;
    using GE = typename GStore<GT>::type;
    __shared__ ShortLds<D, TT> sm[4];
    const int l = lane_id(), ch = l & (D - 1);
    const int seq = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (seq >= a.BH) return;   // no workgroup barrier below
    ShortLds<D, TT>& L = sm[threadIdx.x >> 6];
    const int b = seq / a.H, h = seq % a.H, T = a.T;
    const size_t row0 = (size_t)b * T, ld = (size_t)a.H * D, base = row0 * ld + (size_t)h * D;

    Rows<D, TT, ST> rq, rk, rv;
    Rows<D, TT, GE> rg;
    rq.load(static_cast<const ST*>(a.q) + base, ld, T);
    rk.load(static_cast<const ST*>(a.k) + base, ld, T);
    if constexpr (!HEAD) rg.load(static_cast<const GE*>(a.g) + base, ld, T);
    rv.load(static_cast<const ST*>(a.v) + base, ld, T);
    const float bl = l < T ? ld1(static_cast<const ST*>(a.beta) + (row0 + l) * a.H + h) : 0.f;
    rq.put(L.r[0]);
    rk.put(L.r[1]);
    if constexpr (!HEAD) rg.put(L.r[2]);
    rv.put(L.r[3]);
    wave_sync();
    float ac[TT];
    cumsum_g<D, TT, GT>(static_cast<const GT*>(a.g), row0, a.H, T, h, L.r[2], ch, ac);
    wave_sync();
#pragma unroll
    for (int t = 0; t < TT; ++t) L.r[2][t * LD + ch] = ac[t];
    wave_sync();
    decay_pairs<D, TT>(L.r[0], L.r[1], L.r[2], L.akk, L.aqk);
    wave_sync();

    // e^a Q, e^a K, e^{G - a} K over the rows of q, k and a; e^G
    const float* s0 = a.s0 ? a.s0 + (size_t)seq * D * D : nullptr;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const float kv = L.r[1][t * LD + ch];
        if (s0) {
            const float e = __builtin_amdgcn_exp2f(ac[t]);
            L.r[0][t * LD + ch] *= e;
            L.r[1][t * LD + ch] = kv * e;
        }
        L.r[2][t * LD + ch] = kv * __builtin_amdgcn_exp2f(ac[TT - 1] - ac[t]);
    }
    if (l < D) L.eG[ch] = __builtin_amdgcn_exp2f(ac[TT - 1]);
    wave_sync();
    float vp[TT], o[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        vp[t] = L.r[3][t * LD + ch];
        o[t] = 0.f;
    }
    if (s0) {
        f32x4 ak[D / 16], aq[D / 16];
        clear(ak);
        clear(aq);
        rows_times_St<D, TT>(L.r[1], s0, ak);
        rows_times_St<D, TT>(L.r[0], s0, aq);
        wave_sync();
        acc_rows<D, TT>(ak, L.r[1]);
        acc_rows<D, TT>(aq, L.r[0]);
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            vp[t] -= L.r[1][t * LD + ch];
            o[t] = L.r[0][t * LD + ch];
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        float ck[TT], cq[TT];
        tile_row<TT>(L.akk, t, t, ck);
        tile_row<TT>(L.aqk, t, t + 1, cq);
        float x = vp[t];
#pragma unroll
        for (int s = 0; s < TT; ++s)
            if (s < t) x = fmaf(-ck[s], vp[s], x);
        vp[t] = uniform(bl, t) * x;
#pragma unroll
        for (int s = 0; s < TT; ++s)
            if (s <= t) o[t] = fmaf(cq[s], vp[s], o[t]);
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        L.r[3][t * LD + ch] = vp[t];
        // what is stored: the norm below reads it as the backward will
        L.r[0][t * LD + ch] = sizeof(ST) == 2 ? bf2f(f2bf(o[t])) : o[t];
        if (a.y) L.r[1][t * LD + ch] = L.r[0][t * LD + ch] * L.r[0][t * LD + ch];
    }
    wave_sync();
    rows_out<D, TT, ST>(L.r[0], static_cast<ST*>(a.o) + base, ld, T);
    if (a.y) {
        // the layer's output norm: y = o rsqrt(mean_d o^2 + eps) w sigmoid(z)
        constexpr int PARTS = 64 / TT;
        const float rs = rsqrtf(row_sums<D, TT>(L.r[1]) * (1.f / D) + a.eps);
        const float w = a.nw[ch];
        const ST* z = static_cast<const ST*>(a.z) + row0 * a.ld_z + (size_t)h * D + ch;
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t)
            if (t < T)
                L.r[0][t * LD + ch] = L.r[0][t * LD + ch] * uniform(rs, t * PARTS) * w * sigm(ld1(z + (size_t)t * a.ld_z));
        wave_sync();
        rows_out<D, TT, ST>(L.r[0], static_cast<ST*>(a.y) + row0 * a.ld_y + (size_t)h * D, (size_t)a.ld_y, T);
    }
    if (a.s_final)
        state_out<D, TT>(s0, L.eG, L.r[2], L.r[3], nullptr, nullptr, nullptr, a.s_final + (size_t)seq * D * D);
}

// The adjoint, recomputing the forward from the inputs.  With Y = (I + L)^-T dV',
// X = V - e^a K S0 - A_kk V' (V' = beta X):
//     dV' = A_qk^T dO + Kb dS,  dR = beta Y = dv,  dbeta = Y . X
//     P_qk = dO V'^T (s <= t),  P_kk = -beta Y V'^T (s < t)
//     dQp = dO S0^T, dKp = -dR S0^T, dKb = V' dS^T, dS0 = e^G dS + Qp^T dO - Kp^T dR
// then dq, dk and da pair by pair, lane = channel; each pair's share of da is
// one value, added to a_t and taken from a_s, and dg is its reverse cumsum.
template <int D, int TT, typename ST, typename GT>
__global__ __launch_bounds__(256) void kda_short_bwd_kernel(ShortArgs a) {
    constexpr int LD = D + 4, LA = TT + 4, PARTS = 64 / TT;
    constexpr bool HEAD = std::is_same<GT, GHead>::value;
    using GE = typename GStore<GT>::type;
    using P = Pairs<TT>;
    __shared__ ShortLds<D, TT> sm[4];
    const int l = lane_id(), ch = l & (D - 1);
    const int seq = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (seq >= a.BH) return;   // no workgroup barrier below
    ShortLds<D, TT>& L = sm[threadIdx.x >> 6];
    const int b = seq / a.H, h = seq % a.H, T = a.T;
    const size_t row0 = (size_t)b * T, ld = (size_t)a.H * D, base = row0 * ld + (size_t)h * D;
    const size_t so = (size_t)seq * D * D;

    Rows<D, TT, ST> rq, rk, rv, rd;
    Rows<D, TT, GE> rg;
    rq.load(static_cast<const ST*>(a.q) + base, ld, T);
    rk.load(static_cast<const ST*>(a.k) + base, ld, T);
    if constexpr (!HEAD) rg.load(static_cast<const GE*>(a.g) + base, ld, T);
    rv.load(static_cast<const ST*>(a.v) + base, ld, T);
    rd.load(static_cast<const ST*>(a.dout) + base, ld, T);
    const float bl = l < T ? ld1(static_cast<const ST*>(a.beta) + (row0 + l) * a.H + h) : 0.f;
    if (l < 16) L.beta[l] = bl;
    rq.put(L.r[0]);
    rk.put(L.r[1]);
    if constexpr (!HEAD) rg.put(L.r[2]);
    rv.put(L.r[3]);
    wave_sync();
    float ac[TT], q[TT], k[TT], x[TT], vp[TT];
    cumsum_g<D, TT, GT>(static_cast<const GT*>(a.g), row0, a.H, T, h, L.r[2], ch, ac);
    wave_sync();
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        L.r[2][t * LD + ch] = ac[t];
        q[t] = L.r[0][t * LD + ch];
        k[t] = L.r[1][t * LD + ch];
        x[t] = L.r[3][t * LD + ch];
    }
    if (l < D) L.eG[ch] = __builtin_amdgcn_exp2f(ac[TT - 1]);
    wave_sync();
    decay_pairs<D, TT>(L.r[0], L.r[1], L.r[2], L.akk, L.aqk);
    wave_sync();
    // dO takes k's rows
    rd.put(L.r[1]);
    const float* s0 = a.s0 ? a.s0 + so : nullptr;
    const float* dsf = a.dsf ? a.dsf + so : nullptr;
    if (s0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) L.r[0][t * LD + ch] = k[t] * __builtin_amdgcn_exp2f(ac[t]);
        wave_sync();
        f32x4 acc[D / 16];
        clear(acc);
        rows_times_St<D, TT>(L.r[0], s0, acc);
        wave_sync();
        acc_rows<D, TT>(acc, L.r[0]);
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) x[t] -= L.r[0][t * LD + ch];
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        float ck[TT];
        tile_row<TT>(L.akk, t, t, ck);
#pragma unroll
        for (int s = 0; s < TT; ++s)
            if (s < t) x[t] = fmaf(-ck[s], vp[s], x[t]);
        vp[t] = uniform(bl, t) * x[t];
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < TT; ++t) L.r[3][t * LD + ch] = vp[t];
    float y[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) y[t] = 0.f;
    if (dsf) {
#pragma unroll
        for (int t = 0; t < TT; ++t) L.r[0][t * LD + ch] = k[t] * __builtin_amdgcn_exp2f(ac[TT - 1] - ac[t]);
        wave_sync();
        f32x4 acc[D / 16];
        clear(acc);
        rows_times_St<D, TT>(L.r[0], dsf, acc);
        wave_sync();
        acc_rows<D, TT>(acc, L.r[0]);
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) y[t] = L.r[0][t * LD + ch];
    }
    wave_sync();
    // rows from the last: y += A_qk[r]^T dO_r reaches the rows t <= r, and the
    // solved row r leaves the rows t < r
#pragma unroll
    for (int r = TT - 1; r >= 0; --r) {
        float cq[TT];
        tile_row<TT>(L.aqk, r, r + 1, cq);
        const float d = L.r[1][r * LD + ch];
#pragma unroll
        for (int t = 0; t < TT; ++t)
            if (t <= r) y[t] = fmaf(cq[t], d, y[t]);
    }
#pragma unroll
    for (int r = TT - 1; r > 0; --r) {
        float ck[TT];
        tile_row<TT>(L.akk, r, r, ck);
        const float by = -uniform(bl, r) * y[r];
#pragma unroll
        for (int t = 0; t < TT; ++t)
            if (t < r) y[t] = fmaf(ck[t], by, y[t]);
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        L.r[2][t * LD + ch] = y[t];
        L.r[0][t * LD + ch] = y[t] * x[t];
    }
    wave_sync();
    {
        const float db = row_sums<D, TT>(L.r[0]);
        const int t = l / PARTS;
        if (l % PARTS == 0 && t < T) st1(static_cast<ST*>(a.dbeta) + (row0 + t) * a.H + h, db);
        // P_qk and P_kk over the tiles
        float pq[P::NBK] = {}, pk[P::NBK] = {};
#pragma unroll 2
        for (int d = 0; d < D; d += 4) {
#pragma unroll
            for (int bk = 0; bk < P::NBK; ++bk) {
                const int tt = P::t(bk) * LD + d;
                const float4 v4 = *reinterpret_cast<const float4*>(L.r[3] + P::s(bk) * LD + d);
                pq[bk] = dot4(*reinterpret_cast<const float4*>(L.r[1] + tt), v4, pq[bk]);
                pk[bk] = dot4(*reinterpret_cast<const float4*>(L.r[2] + tt), v4, pk[bk]);
            }
        }
        wave_sync();
#pragma unroll
        for (int bk = 0; bk < P::NBK; ++bk) {
            const int tt = P::t(bk), s = P::s(bk);
            L.aqk[tt * LA + s] = s <= tt ? pq[bk] : 0.f;
            L.akk[tt * LA + s] = s < tt ? -L.beta[tt] * pk[bk] : 0.f;
        }
    }
    // the state's share of dq, dk, da
    float dq[TT], dk[TT], da[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) dq[t] = dk[t] = da[t] = 0.f;
    if (s0) {
        f32x4 acc[D / 16];
        clear(acc);
        rows_times_S<D, TT>(L.r[1], s0, acc);
        wave_sync();
        acc_rows<D, TT>(acc, L.r[0]);
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            dq[t] = __builtin_amdgcn_exp2f(ac[t]) * L.r[0][t * LD + ch];
            da[t] = q[t] * dq[t];
        }
        clear(acc);
        rows_times_S<D, TT>(L.r[2], s0, acc);
        wave_sync();
        acc_rows<D, TT>(acc, L.r[0]);
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            dk[t] = -uniform(bl, t) * __builtin_amdgcn_exp2f(ac[t]) * L.r[0][t * LD + ch];
            da[t] = fmaf(k[t], dk[t], da[t]);
        }
    }
    if (dsf) {
        f32x4 acc[D / 16];
        clear(acc);
        rows_times_S<D, TT>(L.r[3], dsf, acc);
        wave_sync();
        acc_rows<D, TT>(acc, L.r[0]);
        wave_sync();
        float dG = 0.f;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const float e = __builtin_amdgcn_exp2f(ac[TT - 1] - ac[t]) * L.r[0][t * LD + ch];
            dk[t] += e;
            da[t] = fmaf(-k[t], e, da[t]);
            dG = fmaf(k[t], e, dG);
        }
        if (s0) {
            // e^G_j sum_i dS[i][j] S0[i][j], the lane's channel j: coalesced over the lanes
            float s = 0.f;
            for (int i = 0; i < D; ++i) s = fmaf(dsf[(size_t)i * D + ch], s0[(size_t)i * D + ch], s);
            dG = fmaf(__builtin_amdgcn_exp2f(ac[TT - 1]), s, dG);
        }
        da[TT - 1] += dG;
    }
    if (a.ds0) {
        wave_sync();
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const float e = __builtin_amdgcn_exp2f(ac[t]);
            L.r[0][t * LD + ch] = q[t] * e;
            L.r[3][t * LD + ch] = k[t] * e;
        }
        wave_sync();
        state_out<D, TT>(dsf, L.eG, L.r[0], L.r[1], L.r[3], L.r[2], L.beta, a.ds0 + so);
    }
    wave_sync();
    // the pairs: c = e^{a_t - a_s}
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        float cq[TT], ck[TT];
        tile_row<TT>(L.aqk, t, t + 1, cq);
        tile_row<TT>(L.akk, t, t, ck);
#pragma unroll
        for (int s = 0; s < TT; ++s)
            if (s < t) {
                const float c = __builtin_amdgcn_exp2f(ac[t] - ac[s]), xk = c * k[s];
                dq[t] = fmaf(cq[s], xk, dq[t]);
                dk[t] = fmaf(ck[s], xk, dk[t]);
                const float z = c * fmaf(ck[s], k[t], cq[s] * q[t]);
                dk[s] += z;
                const float w = z * k[s];
                da[t] += w;
                da[s] -= w;
            }
        dq[t] = fmaf(cq[t], k[t], dq[t]);
        dk[t] = fmaf(cq[t], q[t], dk[t]);
    }
    float c = 0.f;
    wave_sync();
#pragma unroll
    for (int t = TT - 1; t >= 0; --t) {
        c += da[t];
        L.r[0][t * LD + ch] = dq[t];
        L.r[1][t * LD + ch] = dk[t];
        L.r[3][t * LD + ch] = uniform(bl, t) * y[t];
        L.r[2][t * LD + ch] = c;
    }
    wave_sync();
    rows_out<D, TT, ST>(L.r[0], static_cast<ST*>(a.dq) + base, ld, T);
    rows_out<D, TT, ST>(L.r[1], static_cast<ST*>(a.dk) + base, ld, T);
    rows_out<D, TT, ST>(L.r[3], static_cast<ST*>(a.dv) + base, ld, T);
    if constexpr (HEAD) {
        const float s = row_sums<D, TT>(L.r[2]);
        const int t = l / PARTS;
        if (l % PARTS == 0 && t < T) static_cast<float*>(a.dg)[(row0 + t) * a.H + h] = s;
    } else {
        rows_out<D, TT, GE>(L.r[2], static_cast<GE*>(a.dg) + base, ld, T);
    }
}

template <int D, int TT, typename ST, typename GT>
hipError_t launch_t(const ShortArgs& a, bool bwd, hipStream_t st) {
    const dim3 grid((unsigned)((a.BH + 3) / 4)), block(256);
    if (bwd)
        hipLaunchKernelGGL((kda_short_bwd_kernel<D, TT, ST, GT>), grid, block, 0, st, a);
    else
        hipLaunchKernelGGL((kda_short_fwd_kernel<D, TT, ST, GT>), grid, block, 0, st, a);
    return hipGetLastError();
}

template <int D, int TT>
hipError_t launch_d(const ShortArgs& a, int in_bf16, int g_kind, bool bwd, hipStream_t st) {
    if (in_bf16) {
        if (g_kind == 2) return launch_t<D, TT, uint16_t, GHead>(a, bwd, st);
        return g_kind == 1 ? launch_t<D, TT, uint16_t, uint16_t>(a, bwd, st)
                           : launch_t<D, TT, uint16_t, float>(a, bwd, st);
    }
    if (g_kind == 2) return hipErrorInvalidValue;
    return g_kind == 1 ? launch_t<D, TT, float, uint16_t>(a, bwd, st) : launch_t<D, TT, float, float>(a, bwd, st);
}

}  // namespace

// Whether a shape runs here.  Up to 8 tokens, at D = 32 and for fp32 operands
// one wave is never behind the chunk kernels (measured from 6 to 6144
// sequences, with and without states; 6144 bf16 sequences of 8 tokens at
// D = 64: 31 against 287 us forward, 169 against 594 us backward).  bf16 at
// D = 64 with 9 to 16 tokens: a wave's state products take as long as the chunk
// kernels' one round of workgroups, so those keep what fits one round of the
// 256 CUs (96 sequences with states: 32.9 against 27.8 us backward; 768: 36.8
// against 82.9).  The forward and the backward of a pair have to agree, so only
// the shape and the operand type decide.
bool short_sequences(int T, int D, int in_bf16, int BH) {
    if (T > SHORT_MAX_T || (D != 32 && D != 64)) return false;
    return T <= 8 || D == 32 || !in_bf16 || BH > 256;
}

hipError_t launch_short(const ShortArgs& a, int D, int in_bf16, int g_kind, bool bwd, hipStream_t st) {
    if (!short_sequences(a.T, D, in_bf16, a.BH)) return hipErrorInvalidValue;
    if (D == 32)
        return a.T <= 8 ? launch_d<32, 8>(a, in_bf16, g_kind, bwd, st) : launch_d<32, 16>(a, in_bf16, g_kind, bwd, st);
    return a.T <= 8 ? launch_d<64, 8>(a, in_bf16, g_kind, bwd, st) : launch_d<64, 16>(a, in_bf16, g_kind, bwd, st);
}

}  // namespace kda
