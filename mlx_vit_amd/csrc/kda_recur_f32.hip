// kda_recur_f32.hip -- the sequential recurrences for fp32 operands: the forward,
// the chunk-start state recompute and the reverse state carry (the equations of
// kda_recur.hip), split-bf16 products accurate to fp32.
//
// What bounds them: the chain over the chunks, and in it the CU's vector-memory
// path, which brings a workgroup its chunk's slabs (72 KB a step forward at
// D = 64) at about 26 KB per us; a second operand set in registers (loads two
// chunks ahead) or all of a phase's LDS reads at once changed nothing.  The
// design before (one 256-thread workgroup per (b, h), the slabs staged in one
// LDS set, every wave splitting every operand for its own columns: 30 fragment
// splits and 61 KB of LDS reads per wave and step, the next chunk's loads waited
// for) took 4.6 us a chunk forward.  Here
//   - a workgroup owns 16 CT state columns (32; D / 32 workgroups per (b, h)),
//     and wave w the rows: token block w & 3 of V', O and dV', dk block w of the
//     state.  A wave splits only its own rows of each operand (8 fragments at
//     D = 64), which it loads straight from global memory into registers a
//     chunk ahead; no slab passes through LDS;
//   - the B operands -- the state and V' (dS, dO and dV') -- pass between the
//     waves through LDS already split into bf16 hi and lo planes, as the MFMA
//     reads them;
//   - two barriers a step, which leave the loads and stores in flight;
//   - the backward's two recurrences are independent and share one launch.
// B2 H6 T1568 D64: forward 117 -> 64 us, state recompute and reverse carry 75 +
// 129 -> 61 us together; B2 H8 T1568 D128: forward 660 -> 141 us, the other two
// 151 + 209 -> 129 us.
#include "kda_internal.h"

namespace kda {

namespace {

template <int D> struct F32Geom {
    static constexpr int NT = D / BS, NW = NT > NB ? NT : NB, NTH = 64 * NW;
};

// one 16-row block of an fp32 A operand with K columns, as loaded: the lane's
// row l % 16, k-slots as ldfrag
template <int K> struct ARows {
    float4 x[K / 32][2];
    __device__ __forceinline__ void load(const float* __restrict__ base, int ld) {
        const float* p = base + (size_t)(lane_id() & 15) * ld + 4 * (lane_id() >> 4);
#pragma unroll
        for (int ks = 0; ks < K / 32; ++ks) {
            x[ks][0] = *reinterpret_cast<const float4*>(p + 32 * ks);
            x[ks][1] = *reinterpret_cast<const float4*>(p + 32 * ks + 16);
        }
    }
    __device__ __forceinline__ Frag8 frag(int ks) const {
        const float v[8] = {x[ks][0].x, x[ks][0].y, x[ks][0].z, x[ks][0].w,
                            x[ks][1].x, x[ks][1].y, x[ks][1].z, x[ks][1].w};
        return frag_from_f32<3>(v);
    }
};

// A B operand of COLS columns and K rows as bf16 hi and lo planes, k contiguous
template <int COLS, int K> struct Planes {
    static constexpr int LD = K + 8;
    uint16_t h[COLS][LD], l[COLS][LD];
    // an accumulator tile: rows k0 + 4 g4 + e of column c0 + l % 16
    __device__ __forceinline__ void put(int c0, int k0, const f32x4& v) {
        const int c = c0 + (lane_id() & 15), k = k0 + 4 * (lane_id() >> 4);
        const uint32_t a = pack2bf(v[0], v[1]), b = pack2bf(v[2], v[3]);
        *reinterpret_cast<uint2*>(&h[c][k]) = make_uint2(a, b);
        *reinterpret_cast<uint2*>(&l[c][k]) = make_uint2(pack2bf_rest(v[0], v[1], a), pack2bf_rest(v[2], v[3], b));
    }
    __device__ __forceinline__ Frag8 frag(int c0, int k0) const {
        const int c = c0 + (lane_id() & 15), k = k0 + 4 * (lane_id() >> 4);
        const uint2 a = *reinterpret_cast<const uint2*>(&h[c][k]), b = *reinterpret_cast<const uint2*>(&h[c][k + 16]);
        const uint2 x = *reinterpret_cast<const uint2*>(&l[c][k]), y = *reinterpret_cast<const uint2*>(&l[c][k + 16]);
        Frag8 f;
        f.h = __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
        f.l = __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
        return f;
    }
};

template <int D, int CT> struct F32Lds {
    Planes<16 * CT, D> s;    // the state (dS)
    Planes<16 * CT, C> v;    // V' (-dV')
    Planes<16 * CT, C> o;    // dO (reverse carry only)
};

// MODE 0: O and the final state (EPI: and the layer's gated norm of O; whole
// rows, CT = D / 16).  MODE 1: the chunk-start states h and V'.
template <int D, int MODE, int CT, bool EPI>
__device__ __forceinline__ void recur_f32_body(const RecurArgs& a, F32Lds<D, CT>& L, int wgi) {
    using G = F32Geom<D>;
    constexpr int NT = G::NT, CS = NT / CT, WC = G::NW / NB, CTV = CT / WC;
    static_assert(!EPI || (CS == 1 && WC == 1), "the fused norm needs whole output rows in a wave");
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane_id() & 15, g4 = lane_id() >> 4;
    const int m = w & (NB - 1), v0 = 16 * CTV * (w / NB);   // the wave's token block and first column of V', O
    const int bh = wgi / CS, c0 = (wgi - bh * CS) * 16 * CT, b = bh / a.H, hd = bh - b * a.H;
    const bool has = w < NT;                                // the wave owns dk block w of the state
    const int mt = has ? w : 0;
    const size_t ch0 = (size_t)bh * a.nc;
    const float* gW = static_cast<const float*>(a.W) + ch0 * C * D + BS * m * D;
    const float* gU = static_cast<const float*>(a.U) + ch0 * C * D + (BS * m + 4 * g4) * D + c0 + v0 + r16;
    const float* gQp = static_cast<const float*>(a.Qp) + (MODE == 0 ? ch0 * C * D + BS * m * D : 0);
    const float* gKbT = static_cast<const float*>(a.KbT) + ch0 * C * D + BS * mt * C;
    const float* gAqk = static_cast<const float*>(a.Aqk) + (MODE == 0 ? ch0 * C * C + BS * m * C : 0);
    const float* gEg = a.eG + ch0 * D + BS * mt + 4 * g4;

    f32x4 S[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        S[j] = zero4();
        if (has && a.s0)
            S[j] = *reinterpret_cast<const f32x4*>(a.s0 + ((size_t)bh * D + c0 + 16 * j + r16) * D + BS * mt + 4 * g4);
        if (has) L.s.put(16 * j, BS * mt, S[j]);
    }
    struct Ops {
        ARows<D> W, Q;
        ARows<C> K, A;
        f32x4 U[CTV], eg;
    };
    Ops p;   // each part reloaded for the next chunk once it is used
    auto load_wu = [&](int n) __attribute__((always_inline)) {
        p.W.load(gW + (size_t)n * C * D, D);
#pragma unroll
        for (int j = 0; j < CTV; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) p.U[j][e] = gU[(size_t)n * C * D + e * D + 16 * j];
    };
    auto load_k = [&](int n) __attribute__((always_inline)) {
        p.K.load(gKbT + (size_t)n * C * D, C);
        p.eg = *reinterpret_cast<const f32x4*>(gEg + (size_t)n * D);
    };
    load_wu(0);
    load_k(0);
    if constexpr (MODE == 0) {
        p.Q.load(gQp, D);
        p.A.load(gAqk, C);
    }
    // more: another chunk follows, whose operands are loaded as this one's are used.
    // The last chunk is a copy of its own: its loads again cost 64 x 64 tokens x 12
    // x 64 73.6 us of forward against 65, a branch around them 4 us of 95 at 25 chunks
    auto step = [&](int n, auto more_c) __attribute__((always_inline)) {
        constexpr bool more = decltype(more_c)::value;
        const int nx = n + 1;
        // the norm's gate values of this chunk's rows (past T the last one's), used at
        // the step's end: loaded there they made every step wait (2 x 1568 x 6 x 64 with
        // the norm 208 -> 172 us)
        const int t0 = n * C + BS * m + 4 * g4;
        float z[4][CTV];
        if constexpr (EPI)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float* zp = static_cast<const float*>(a.z) +
                                  ((size_t)b * a.T + min(t0 + e, a.T - 1)) * a.ld_z + (size_t)hd * D + r16;
#pragma unroll
                for (int j = 0; j < CTV; ++j) z[e][j] = zp[16 * j];
            }
        lds_barrier();                         // the state's planes
        Frag8 Bs[CTV][D / 32];
#pragma unroll
        for (int j = 0; j < CTV; ++j)
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) Bs[j][ks] = L.s.frag(v0 + 16 * j, 32 * ks);
        // V' = U - W S
        f32x4 vp[CTV];
#pragma unroll
        for (int j = 0; j < CTV; ++j) vp[j] = zero4();
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            const Frag8 A = p.W.frag(ks);
#pragma unroll
            for (int j = 0; j < CTV; ++j) vp[j] = mma<3>(A, Bs[j][ks], vp[j]);
        }
#pragma unroll
        for (int j = 0; j < CTV; ++j) {
            vp[j] = p.U[j] - vp[j];
            L.v.put(v0 + 16 * j, BS * m, vp[j]);
        }
        if constexpr (more) load_wu(nx);
        if constexpr (MODE == 1) {
            float* h = static_cast<float*>(a.h) + (ch0 + n) * D * D + (BS * mt + 4 * g4) * D + c0 + r16;
            float* V = static_cast<float*>(a.Vp) + (ch0 + n) * C * D + (BS * m + 4 * g4) * D + c0 + v0 + r16;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (has)
#pragma unroll
                    for (int j = 0; j < CT; ++j) h[e * D + 16 * j] = S[j][e];
#pragma unroll
                for (int j = 0; j < CTV; ++j) V[e * D + 16 * j] = vp[j][e];
            }
        }
        f32x4 O[CTV];
        if constexpr (MODE == 0) {
#pragma unroll
            for (int j = 0; j < CTV; ++j) O[j] = zero4();
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
                const Frag8 A = p.Q.frag(ks);
#pragma unroll
                for (int j = 0; j < CTV; ++j) O[j] = mma<3>(A, Bs[j][ks], O[j]);
            }
            if constexpr (more) p.Q.load(gQp + (size_t)nx * C * D, D);
        }
        lds_barrier();                         // V' planes; every wave has read the state's
        Frag8 Bv[CT][C / 32];
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) Bv[j][ks] = L.v.frag(16 * j, 32 * ks);
        __builtin_amdgcn_sched_barrier(0);     // one LDS round trip for all of them
        // S <- e^G S + Kb^T V'
        if (has) {
#pragma unroll
            for (int j = 0; j < CT; ++j) S[j] = S[j] * p.eg;
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) {
                const Frag8 A = p.K.frag(ks);
#pragma unroll
                for (int j = 0; j < CT; ++j) S[j] = mma<3>(A, Bv[j][ks], S[j]);
            }
#pragma unroll
            for (int j = 0; j < CT; ++j) L.s.put(16 * j, BS * mt, S[j]);
            if constexpr (more) load_k(nx);
        }
        if constexpr (MODE == 0) {
            // O = Qp S + A_qk V' (A_qk lower triangular)
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) {
                if (2 * ks > m) continue;
                const Frag8 A = p.A.frag(ks);
#pragma unroll
                for (int j = 0; j < CTV; ++j)
                    O[j] = mma<3>(A, WC == 1 ? Bv[j][ks] : L.v.frag(v0 + 16 * j, 32 * ks), O[j]);
            }
            if constexpr (more) p.A.load(gAqk + (size_t)nx * C * C, C);
            const size_t row = (size_t)b * a.T + t0;
            float* o = static_cast<float*>(a.o) + (row * a.H + hd) * D + c0 + v0 + r16;
            const size_t rs = (size_t)a.H * D;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float rn = 0.f;
                if constexpr (EPI) {
                    float ss = 0.f;
#pragma unroll
                    for (int j = 0; j < CTV; ++j) ss = fmaf(O[j][e], O[j][e], ss);
#pragma unroll
                    for (int x = 1; x < 16; x <<= 1) ss += __shfl_xor(ss, x, 64);
                    rn = rsqrtf(ss * (1.f / D) + a.eps);
                }
                if (t0 + e < a.T)
#pragma unroll
                    for (int j = 0; j < CTV; ++j) {
                        o[e * rs + 16 * j] = O[j][e];
                        if constexpr (EPI) {
                            const int c = 16 * j + r16;
                            static_cast<float*>(a.y)[(row + e) * a.ld_y + (size_t)hd * D + c] =
                                O[j][e] * rn * a.nw[c] * sigm(z[e][j]);
                        }
                    }
            }
        }
    };
    for (int n = 0; n < a.nc - 1; ++n) step(n, std::true_type{});
    step(a.nc - 1, std::false_type{});
    if (MODE == 0 && has && a.s_final)
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *reinterpret_cast<f32x4*>(a.s_final + ((size_t)bh * D + c0 + 16 * j + r16) * D + BS * mt + 4 * g4) = S[j];
}

// dV' = A_qk^T dO + Kb dS;  dS <- e^G dS + Qp^T dO - W^T dV', from the last chunk
template <int D, int CT>
__device__ __forceinline__ void dh_f32_body(const DhArgs& a, F32Lds<D, CT>& L, int wgi) {
    using G = F32Geom<D>;
    constexpr int NT = G::NT, CS = NT / CT, WC = G::NW / NB, CTV = CT / WC;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane_id() & 15, g4 = lane_id() >> 4;
    const int m = w & (NB - 1), v0 = 16 * CTV * (w / NB);
    const int bh = wgi / CS, c0 = (wgi - bh * CS) * 16 * CT, b = bh / a.H, hd = bh - b * a.H;
    const bool has = w < NT;
    const int mt = has ? w : 0;
    const size_t ch0 = (size_t)bh * a.nc;
    const float* gA = static_cast<const float*>(a.AqkT) + ch0 * C * C + BS * m * C;
    const float* gKb = static_cast<const float*>(a.Kb) + ch0 * C * D + BS * m * D;
    const float* gQ = static_cast<const float*>(a.QpT) + ch0 * C * D + BS * mt * C;
    const float* gW = static_cast<const float*>(a.WT) + ch0 * C * D + BS * mt * C;
    const float* gEg = a.eG + ch0 * D + BS * mt + 4 * g4;
    const float* gO = static_cast<const float*>(a.dout);
    const size_t rs = (size_t)a.H * D;

    f32x4 S[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        S[j] = zero4();
        if (has && a.dsf)
            S[j] = *reinterpret_cast<const f32x4*>(a.dsf + ((size_t)bh * D + c0 + 16 * j + r16) * D + BS * mt + 4 * g4);
        if (has) L.s.put(16 * j, BS * mt, S[j]);
    }
    struct Ops {
        ARows<C> A, Q, W;
        ARows<D> K;
        f32x4 dO[CTV], eg;   // dO of the chunk before the operands'
    };
    Ops p;   // each part reloaded for the next chunk once it is used
    // rows past T are read from the last one and zeroed where they are used
    auto load_do = [&](int n) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = min(n * C + BS * m + 4 * g4 + e, a.T - 1);
            const float* x = gO + (((size_t)b * a.T + t) * a.H + hd) * D + c0 + v0 + r16;
#pragma unroll
            for (int j = 0; j < CTV; ++j) p.dO[j][e] = x[16 * j];
        }
    };
    auto put_do = [&](int n) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CTV; ++j) {
            f32x4 x = p.dO[j];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n * C + BS * m + 4 * g4 + e >= a.T) x[e] = 0.f;
            L.o.put(v0 + 16 * j, BS * m, x);
        }
    };
    int n = a.nc - 1;
    load_do(n);
    p.A.load(gA + (size_t)n * C * C, C);
    p.K.load(gKb + (size_t)n * C * D, D);
    p.Q.load(gQ + (size_t)n * C * D, C);
    p.eg = *reinterpret_cast<const f32x4*>(gEg + (size_t)n * D);
    p.W.load(gW + (size_t)n * C * D, C);
    put_do(n);
    load_do(max(n - 1, 0));
    auto step = [&](int n, auto more_c) __attribute__((always_inline)) {   // as in the forward
        constexpr bool more = decltype(more_c)::value;
        const int nx = n - 1;
        lds_barrier();                         // the planes of dS and dO
        if (has) {
            float* dh = static_cast<float*>(a.dh) + (ch0 + n) * D * D + (BS * mt + 4 * g4) * D + c0 + r16;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < CT; ++j) dh[e * D + 16 * j] = S[j][e];
        }
        Frag8 Bo[CT][C / 32], Bs[CTV][D / 32];
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) Bo[j][ks] = L.o.frag(16 * j, 32 * ks);
#pragma unroll
        for (int j = 0; j < CTV; ++j)
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) Bs[j][ks] = L.s.frag(v0 + 16 * j, 32 * ks);
        __builtin_amdgcn_sched_barrier(0);     // one LDS round trip for all of them
        f32x4 dv[CTV];
#pragma unroll
        for (int j = 0; j < CTV; ++j) dv[j] = zero4();
        // A_qk^T is upper triangular
#pragma unroll
        for (int ks = 0; ks < C / 32; ++ks) {
            if (2 * ks + 1 < m) continue;
            const Frag8 A = p.A.frag(ks);
#pragma unroll
            for (int j = 0; j < CTV; ++j)
                dv[j] = mma<3>(A, WC == 1 ? Bo[j][ks] : L.o.frag(v0 + 16 * j, 32 * ks), dv[j]);
        }
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            const Frag8 A = p.K.frag(ks);
#pragma unroll
            for (int j = 0; j < CTV; ++j) dv[j] = mma<3>(A, Bs[j][ks], dv[j]);
        }
#pragma unroll
        for (int j = 0; j < CTV; ++j) L.v.put(v0 + 16 * j, BS * m, -dv[j]);
        if constexpr (more) {
            p.A.load(gA + (size_t)nx * C * C, C);
            p.K.load(gKb + (size_t)nx * C * D, D);
        }
        float* dV = static_cast<float*>(a.dVp) + (ch0 + n) * C * D + (BS * m + 4 * g4) * D + c0 + v0 + r16;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < CTV; ++j) dV[e * D + 16 * j] = dv[j][e];
        if (has) {
#pragma unroll
            for (int j = 0; j < CT; ++j) S[j] = S[j] * p.eg;
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) {
                const Frag8 A = p.Q.frag(ks);
#pragma unroll
                for (int j = 0; j < CT; ++j) S[j] = mma<3>(A, Bo[j][ks], S[j]);
            }
            if constexpr (more) {
                p.Q.load(gQ + (size_t)nx * C * D, C);
                p.eg = *reinterpret_cast<const f32x4*>(gEg + (size_t)nx * D);
            }
        }
        lds_barrier();                         // -dV' planes; every wave has read those of dS and dO
        if constexpr (more) {
            put_do(nx);
            load_do(max(nx - 1, 0));
        }
        if (has) {
            Frag8 Bv[CT][C / 32];
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int ks = 0; ks < C / 32; ++ks) Bv[j][ks] = L.v.frag(16 * j, 32 * ks);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < C / 32; ++ks) {
                const Frag8 A = p.W.frag(ks);
#pragma unroll
                for (int j = 0; j < CT; ++j) S[j] = mma<3>(A, Bv[j][ks], S[j]);
            }
#pragma unroll
            for (int j = 0; j < CT; ++j) L.s.put(16 * j, BS * mt, S[j]);
            if constexpr (more) p.W.load(gW + (size_t)nx * C * D, C);
        }
    };
    for (; n > 0; --n) step(n, std::true_type{});
    step(0, std::false_type{});
    if (has && a.ds0)
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *reinterpret_cast<f32x4*>(a.ds0 + ((size_t)bh * D + c0 + 16 * j + r16) * D + BS * mt + 4 * g4) = S[j];
}

template <int D, int CT, bool EPI>
__global__ __launch_bounds__(F32Geom<D>::NTH) void kda_recur_f32_kernel(const RecurArgs a) {
    __shared__ __align__(16) F32Lds<D, CT> L;
    recur_f32_body<D, 0, CT, EPI>(a, L, blockIdx.x);
}

// The state recompute (workgroups 0 .. BH CS - 1) beside the reverse carry (the
// next BH CS): neither reads what the other writes
template <int D, int CT>
__global__ __launch_bounds__(F32Geom<D>::NTH) void kda_states_dh_f32_kernel(const RecurArgs ra, const DhArgs da) {
    __shared__ __align__(16) F32Lds<D, CT> L;
    const int nrec = ra.BH * (D / BS / CT);
    if ((int)blockIdx.x < nrec)
        recur_f32_body<D, 1, CT, false>(ra, L, blockIdx.x);
    else
        dh_f32_body<D, CT>(da, L, blockIdx.x - nrec);
}

constexpr int F32_CT = 2;   // column tiles per workgroup
// Whether the forward at D = 64 takes one workgroup per (b, h) instead of two, which
// read every operand twice: where two would be more than the CUs, and for single
// chunks earlier.  One against two: 96 x 64 tokens 19.4 / 20.5 us, 128 x 64 19.7 /
// 22.4, 192 x 64 21.1 / 26.3, 192 x 256 59.7 / 65.1; but 48 x 64 19.2 / 18.2, 128 x 256
// 46.1 / 44.7, 12 x 1568 112 / 90.
static bool whole_rows(int BH, int nc) { return BH >= (nc == 1 ? 96 : 129); }

template <int D> hipError_t recur_f32_t(const RecurArgs& a, hipStream_t st) {
    constexpr int NT = D / BS, NTH = F32Geom<D>::NTH;
    if (a.y) {
        if constexpr (D <= 64)
            hipLaunchKernelGGL((kda_recur_f32_kernel<D, NT, true>), dim3(a.BH), dim3(NTH), 0, st, a);
        else
            return hipErrorInvalidValue;
    } else if (D == 64 && whole_rows(a.BH, a.nc)) {
        if constexpr (D == 64) hipLaunchKernelGGL((kda_recur_f32_kernel<D, NT, false>), dim3(a.BH), dim3(NTH), 0, st, a);
    } else {
        hipLaunchKernelGGL((kda_recur_f32_kernel<D, F32_CT, false>), dim3(a.BH * (NT / F32_CT)), dim3(NTH), 0, st, a);
    }
    return hipGetLastError();
}

template <int D> hipError_t states_dh_f32_t(const RecurArgs& ra, const DhArgs& da, hipStream_t st) {
    hipLaunchKernelGGL((kda_states_dh_f32_kernel<D, F32_CT>), dim3(2 * ra.BH * (D / BS / F32_CT)),
                       dim3(F32Geom<D>::NTH), 0, st, ra, da);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_recur_f32(const RecurArgs& a, int D, hipStream_t st) {
    if (D == 32) return recur_f32_t<32>(a, st);
    if (D == 64) return recur_f32_t<64>(a, st);
    if (D == 128) return recur_f32_t<128>(a, st);
    return hipErrorInvalidValue;
}

hipError_t launch_states_dh_f32(const RecurArgs& ra, const DhArgs& da, int D, hipStream_t st) {
    if (ra.BH != da.BH || !ra.Vp || !ra.KbT || !da.AqkT || !da.QpT || !da.WT || !da.Kb) return hipErrorInvalidValue;
    if (D == 32) return states_dh_f32_t<32>(ra, da, st);
    if (D == 64) return states_dh_f32_t<64>(ra, da, st);
    if (D == 128) return states_dh_f32_t<128>(ra, da, st);
    return hipErrorInvalidValue;
}

}  // namespace kda
