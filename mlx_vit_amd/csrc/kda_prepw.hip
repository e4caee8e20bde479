// kda_prepw.hip -- the forward prep of bf16 operands at D = 64 and 128.
//
// Same chunk algebra and outputs as kda_prep_kernel (kda_fwd.hip; nope_gdn_mlx.py:
// 2400-2472, 1319-1334, 1141-1207), in 80 KB of LDS at D = 128 so that two 8-wave
// workgroups share a CU: one chunk's loads and stores run beside another's
// products and solve.  With a chunk's every array in LDS (133 KB, one 16-wave
// workgroup a CU) each barrier left the CU idle.  At D = 64 two share it as
// before (the registers' limit), with two phases and their LDS passes fewer.
// (At D = 128 up to 192 chunks, at most one a CU, stay with the sixteen-wave
// kernel: PREP16_CHUNKS in kda_fwd.hip.)
// What is kept out of LDS:
//   - the in-block cumsums a of g: a thread loads q, k and g of the same (token,
//     8 channels), so the operands k e^{a}, q e^{a}, k e^{b} form in registers;
//     only the block totals pass through LDS.  Chunks with strong blocks lay
//     raw q, k and a over the regions written later;
//   - v: in registers until the products have read K_r, then in its place;
//   - A_kk: the off-diagonal tiles go from the accumulators to the split
//     operands of the solve, the diagonal ones to the rows their inverses take.
// Before -> after: 32768 x 16 x 128 411 -> 333 us (1.14 GB read and written, 2.8 ->
// 3.4 TB/s against 5.2 for a copy); 8 x 1568 x 8 x 96 at the layer's initial decay
// 103 -> 81 us; 8 x 1568 x 12 x 64 55 -> 48 us, at that decay 68 -> 62 us.  Left:
// the vector instructions of the operand conversions, at the 128 registers two
// workgroups allow (three at D = 64, 80 registers: 80 us).
#include "kda_internal.h"

namespace kda {

namespace {

constexpr int PW_NTH = 512, PW_LDT = C + 8, PW_SPR = 2 * BS + 8, PW_SPB = BS * PW_SPR;

template <int D>
struct PrepWLds {
    static constexpr int LDK = D + 8;
    uint16_t ql[C][LDK];   // raw q (strong chunks), then q e^{a}; U at the end
    uint16_t kr[C][LDK];   // raw k (strong chunks), then k e^{b}, then v
    union {
        struct {
            uint16_t kl[C][LDK];    // k e^{a}; W at the end
            uint16_t aqk[C][PW_LDT];   // A_qk on its way out
            uint16_t spl[6][PW_SPB];   // split -beta A_kk of the blocks below the diagonal
        };
        float g[C][D + 4];   // a, strong chunks only, before kl is written
    };
    float fac[14][D];          // factor tables, rows FAC_*
    float tii[NB][BS][BS + 4];    // block totals of g; A_kk's diagonal tiles; their inverses, then split
    float beta[C];
    int fl[PW_NTH / 64];          // decay flags per wave
};
static_assert(sizeof(PrepWLds<128>) <= 80 * 1024, "two workgroups a CU");

// the value of lane 15 of the lane's row of 16
__device__ __forceinline__ float row16_last(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x15F, 0xf, 0xf, false));
}

}  // namespace

template <int D, typename TG>
__global__ __launch_bounds__(PW_NTH, 4) void kda_prepw_kernel(const PrepArgs a) {
    using ST = uint16_t;
    constexpr int NTH = PW_NTH, NW = NTH / 64, NT = D / BS, LDK = D + 8, LDT = PW_LDT, PREC = 1, SPR = PW_SPR;
    constexpr bool GH = std::is_same<TG, GHead>::value;   // one fp32 decay per (b, t, h)
    using TGE = typename std::conditional<GH, float, TG>::type;
    static_assert(NW == 2 * NB && (2 * NT) % NW == 0, "two waves a row block; whole column tiles of [K | V] a wave");
    __shared__ __align__(16) PrepWLds<D> s;

    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, r16 = l & 15, g4 = l >> 4;
    __builtin_assume(w >= 0 && w < NW);
    const int ch = blockIdx.x, bh = ch / a.nc, n = ch - bh * a.nc;
    const int b = bh / a.H, h = bh - b * a.H;
    const int t0 = n * C, valid = min(C, a.T - t0);
    // dio: the channels of a q, k, v, g row (a multiple of 8; the rest read as zero)
    const int dio = (D == 128 && a.dio > 0) ? a.dio : D;
    const size_t rs = (size_t)a.H * dio;
    const size_t base = ((size_t)b * a.T + t0) * rs + (size_t)h * dio;
    const size_t bbase = ((size_t)b * a.T + t0) * a.H + h;
    const size_t cCD = (size_t)ch * C * D, cCC = (size_t)ch * C * C;
    ST* oW = static_cast<ST*>(a.W);
    ST* oU = static_cast<ST*>(a.U);
    ST* oQp = static_cast<ST*>(a.Qp);
    ST* oQpT = static_cast<ST*>(a.QpT);
    ST* oKb = static_cast<ST*>(a.Kb);
    ST* oKbT = static_cast<ST*>(a.KbT);
    ST* oWT = static_cast<ST*>(a.WT);
    ST* oAqk = static_cast<ST*>(a.Aqk);
    ST* oAqkT = static_cast<ST*>(a.AqkT);
    float* const oAkk = a.Akk;
    float* const oTii = a.Tii;
    auto pk4 = [](const float* x) __attribute__((always_inline)) {
        return make_uint2(pack2bf(x[0], x[1]), pack2bf(x[2], x[3]));
    };

    // ---------------- load ----------------
    // wave w: rows of block w / 2, lane row r16 of it, the 8-channel groups
    // 4 (w % 2) + g4 and 8 more; rows past T and channels past dio are read from the
    // last valid ones and zeroed after
    constexpr int CP = D / 64, GE = 16 / (int)sizeof(TGE), GV = GH ? 1 : 8 / GE;
    const int blk = w >> 1, row = BS * blk + r16, c0 = 8 * (4 * (w & 1) + g4);
    uint4 qr[CP], kr[CP], gr[CP][GV];
    float gh = 0.f;
    {
        const size_t ro = base + (size_t)min(row, valid - 1) * rs;
        const ST* qp = static_cast<const ST*>(a.q) + ro;
        const ST* kp = static_cast<const ST*>(a.k) + ro;
        const TGE* gp = static_cast<const TGE*>(a.g) + ro;
        if constexpr (GH) gh = static_cast<const float*>(a.g)[bbase + (size_t)min(row, valid - 1) * a.H];
#pragma unroll
        for (int cp = 0; cp < CP; ++cp) {
            const int cc = min(c0 + 64 * cp, dio - 8);
            qr[cp] = *reinterpret_cast<const uint4*>(qp + cc);
            kr[cp] = *reinterpret_cast<const uint4*>(kp + cc);
            if constexpr (!GH)
#pragma unroll
                for (int u = 0; u < GV; ++u) gr[cp][u] = *reinterpret_cast<const uint4*>(gp + cc + GE * u);
        }
    }
    const float braw = ld1<ST>(static_cast<const ST*>(a.beta) + bbase + (size_t)min(tid, valid - 1) * a.H);
    Tile<ST, C, D, NTH> tv;
    tv.load(static_cast<const ST*>(a.v) + base, rs, valid, dio);

    // a, the inclusive cumsum of g over the block's rows (the 16 lanes of a DPP
    // row), the block totals, and the decay flags: bit 4 g > 0 or a NaN, bit i block
    // i's span beyond the guard, bit 5 + i one of its 4-row spans beyond its guard
    float* const sT = &s.tii[0][0][0];   // [NB][D]
    float at[CP][8];
    int fpos = 0, fspan = 0, fsub = 0;
#pragma unroll
    for (int cp = 0; cp < CP; ++cp) {
        const bool ok = row < valid && c0 + 64 * cp < dio;
        if (!ok) qr[cp] = kr[cp] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float x = gh;
            if constexpr (!GH) x = Vec16<TGE>{gr[cp][e / GE]}.get(e % GE);
            x = ok ? x : 0.f;
            if (!(x <= 0.f)) fpos = 1;
            at[cp][e] = row16_scan(x);
            const float prev = __int_as_float(
                __builtin_amdgcn_update_dpp(0, __float_as_int(at[cp][e]), 0x114, 0xf, 0xf, true));   // four rows back
            if (r16 == BS - 1 && !(-at[cp][e] <= SPAN_MAX)) fspan = 1;
            if ((r16 & 3) == 3 && !(prev - at[cp][e] <= SUB_SPAN_MAX)) fsub = 1;
        }
        if (r16 == BS - 1) {
            float4* p = reinterpret_cast<float4*>(sT + blk * D + c0 + 64 * cp);
            p[0] = make_float4(at[cp][0], at[cp][1], at[cp][2], at[cp][3]);
            p[1] = make_float4(at[cp][4], at[cp][5], at[cp][6], at[cp][7]);
        }
    }
    if (tid < C) s.beta[tid] = (tid < valid) ? braw : 0.f;
    {
        const int wm = (__ballot(fpos) ? 16 : 0) | (__ballot(fspan) ? 1 << blk : 0) | (__ballot(fsub) ? 32 << blk : 0);
        if (l == 0) s.fl[w] = wm;
    }
    __syncthreads();
    int dfl = 0;
#pragma unroll
    for (int u = 0; u < NW; ++u) dfl |= s.fl[u];
    dfl = __builtin_amdgcn_readfirstlane(dfl);

    // factor tables (FAC_* rows): exponents are sums of block totals
    {
        const int d = tid % D, r = __builtin_amdgcn_readfirstlane(tid / D);
        const float T0 = sT[d], T1 = sT[D + d], T2 = sT[2 * D + d], T3 = sT[3 * D + d], T12 = T1 + T2;
        for (int fr = r; fr < FAC_ONE; fr += NTH / D) {
            const float x = (fr == 0) ? T0 : (fr == 1) ? T0 + T1 : (fr == 2) ? (T0 + T1) + T2
                          : (fr == 3) ? T1 + (T2 + T3) : (fr == 4) ? T2 + T3 : (fr == 5) ? T3
                          : (fr == 6) ? T1 : (fr == 7) ? T2 : (fr == 8) ? T12
                          : fminf(-((fr == 9) ? T0 : (fr == 10) ? T1 : (fr == 11) ? T2 : T3), SPAN_MAX);
            s.fac[fr][d] = kexp<PREC>(x);
        }
        if (r == NTH / D - 1) s.fac[FAC_ONE][d] = 1.f;
        if (a.eG && tid < D) a.eG[(size_t)ch * D + d] = kexp<PREC>((T0 + T1) + (T2 + T3));
    }

    // lane (r, g) puts / gets A[r][4 g .. 4 g + 3] of a split block
    auto put_split = [&](uint16_t* p, const float* v) __attribute__((always_inline)) {
        const uint32_t h0 = pack2bf(v[0], v[1]), h1 = pack2bf(v[2], v[3]);
        *reinterpret_cast<uint2*>(p + r16 * SPR + 4 * g4) = make_uint2(h0, h1);
        *reinterpret_cast<uint2*>(p + r16 * SPR + BS + 4 * g4) =
            make_uint2(pack2bf_rest(v[0], v[1], h0), pack2bf_rest(v[2], v[3], h1));
    };
    auto get_split = [&](const uint16_t* p) __attribute__((always_inline)) {
        Frag4 f;
        f.h = __builtin_bit_cast(short4v, *reinterpret_cast<const uint2*>(p + r16 * SPR + 4 * g4));
        f.l = __builtin_bit_cast(short4v, *reinterpret_cast<const uint2*>(p + r16 * SPR + BS + 4 * g4));
        return f;
    };

    // From here to the solve the kernel is instantiated twice, chunks within the
    // span guard without the code of the others.
    auto middle = [&](auto strong_c) __attribute__((always_inline)) {
        constexpr bool STRONG = decltype(strong_c)::value;
        const bool unsafe = STRONG && (dfl & 16) != 0;           // g > 0 or NaN: every pair by itself
        const int pmask = (STRONG && !unsafe) ? (dfl & 15) : 0;  // diagonal blocks beyond the span guard
        const int qmask = pmask & (dfl >> 5);                    // ... whose 4-row sub-blocks also exceed it
        // strong chunks: the entries this thread forms from raw q, k (their LDS places
        // are still taken): all pairs (unsafe), or those of blocks in qmask
        constexpr int NPU = C * C / NTH, NPW = NB * BS * BS / NTH;
        float pak[NPU], paq[NPW];
        f32x4 P = zero4(), Q = zero4();   // wave w < NB: its block's sub-anchored tile
        if constexpr (STRONG) {
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                const int c = c0 + 64 * cp;
                *reinterpret_cast<uint4*>(&s.ql[row][c]) = qr[cp];
                *reinterpret_cast<uint4*>(&s.kr[row][c]) = kr[cp];
                *reinterpret_cast<float4*>(&s.g[row][c]) = make_float4(at[cp][0], at[cp][1], at[cp][2], at[cp][3]);
                *reinterpret_cast<float4*>(&s.g[row][c + 4]) = make_float4(at[cp][4], at[cp][5], at[cp][6], at[cp][7]);
            }
            __syncthreads();
            if (unsafe) {
#pragma unroll
                for (int it = 0; it < NPU; ++it) {
                    const int p = tid + NTH * it, t = p / C, sx = p - t * C;
                    float ak = 0.f, aq = 0.f;
                    if (sx <= t) {
#pragma unroll 1
                        for (int d = 0; d < D; ++d) {
                            const float ks =
                                ld1<ST>(&s.kr[sx][d]) * kexp<PREC>(chunk_gamma(s, t, d) - chunk_gamma(s, sx, d));
                            ak += ld1<ST>(&s.kr[t][d]) * ks;
                            aq += ld1<ST>(&s.ql[t][d]) * ks;
                        }
                    }
                    pak[it] = (sx < t) ? ak : 0.f;
                    if (oAkk) oAkk[cCC + (size_t)t * C + sx] = pak[it];
                    if (oAqk) st1<ST>(oAqk + cCC + (size_t)t * C + sx, aq);
                    if (oAqkT) st1<ST>(oAqkT + cCC + (size_t)sx * C + t, aq);
                }
            } else {
                if (((pmask & ~qmask) >> w) & 1) subanchor_tile<D, ST, PREC, true>(s, w, P, Q);
                if (qmask) {
                    const int nent = __popc(qmask) * BS * BS;
#pragma unroll
                    for (int it = 0; it < NPW; ++it) {
                        const int pp = tid + NTH * it;
                        pak[it] = paq[it] = 0.f;
                        if (pp < nent) {
                            const int kb = pp / (BS * BS), e = pp - kb * BS * BS;
                            int bq = 0;
                            for (int m = qmask, c = 0;; m &= m - 1, ++c)
                                if (c == kb) { bq = __ffs(m) - 1; break; }
                            const int t = BS * bq + e / BS, sx = BS * bq + e % BS;
                            float ak = 0.f, aq = 0.f;
                            if (sx <= t) {
#pragma unroll 2
                                for (int d = 0; d < D; ++d) {
                                    const float ks = ld1<ST>(&s.kr[sx][d]) * kexp<PREC>(s.g[t][d] - s.g[sx][d]);
                                    ak += ld1<ST>(&s.kr[t][d]) * ks;
                                    aq += ld1<ST>(&s.ql[t][d]) * ks;
                                }
                            }
                            pak[it] = (sx < t) ? ak : 0.f;
                            paq[it] = aq;
                        }
                    }
                }
            }
            __syncthreads();   // raw q, k, a are read: the operands take their place
        }

        // ---------------- K_l = K e^{a}, Q_l = Q e^{a}, K_r = K e^{b} ----------------
        float oql[CP][8], okb[CP][8];
#pragma unroll
        for (int cp = 0; cp < CP; ++cp) {
            const int c = c0 + 64 * cp;
            const Vec16<ST> qv{qr[cp]}, kv{kr[cp]};
            float okl[8], okr[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float bt = row16_last(at[cp][e]) - at[cp][e], el = kexp<PREC>(at[cp][e]), kf = kv.get(e);
                okl[e] = kf * el;
                oql[cp][e] = qv.get(e) * el;
                okr[e] = unsafe ? kf : kf * kexp<PREC>(bt);
                okb[cp][e] = okr[e];
                if (unsafe) {   // e^{G - gamma_t} in one exponent
                    float gsfx = bt;
                    for (int m = blk + 1; m < NB; ++m) gsfx += sT[m * D + c + e];
                    okb[cp][e] = kf * kexp<PREC>(gsfx);
                }
            }
            store_vec<ST>(&s.kl[row][c], okl);
            store_vec<ST>(&s.ql[row][c], oql[cp]);
            store_vec<ST>(&s.kr[row][c], okr);
        }
        __syncthreads();

        // Qp = Q_l e^{gamma_{16i-1}}, Kb = K_r e^{G - gamma_{16i+15}} (and, unsafe, their
        // transposes) from the thread's own values
        if (oQp || oKb || unsafe) {
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                const int c = c0 + 64 * cp;
                const float* fp = &s.fac[blk > 0 ? FAC_EP + blk - 1 : FAC_ONE][c];
                const float* fq = &s.fac[(blk < NB - 1 && !unsafe) ? FAC_EQ + blk : FAC_ONE][c];
                float xq[8], xk[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    xq[e] = oql[cp][e] * fp[e];
                    xk[e] = okb[cp][e] * fq[e];
                }
                if (oQp) store_vec<ST>(oQp + cCD + (size_t)row * D + c, xq);
                if (oKb) store_vec<ST>(oKb + cCD + (size_t)row * D + c, xk);
                if (unsafe) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (oKbT) st1<ST>(oKbT + cCD + (size_t)(c + e) * C + row, xk[e]);
                        if (oQpT) st1<ST>(oQpT + cCD + (size_t)(c + e) * C + row, xq[e]);
                    }
                }
            }
        }

        // ---------------- products: waves 0-3 the diagonal tiles, 4-7 the six below ----------------
        // Tiles are formed transposed (lane row t = r16, four consecutive s), so that
        // A_kk goes out, to the split operands and to the inverses as vectors; A_qk^T
        // from a product the other way round.
        if (!unsafe) {
            auto form_tile = [&](int i, int j, f32x4& PT, f32x4& QT, f32x4& QN) __attribute__((always_inline)) {
                const float* fsc = &s.fac[(j == i) ? FAC_FD + i : (j == i - 1) ? 0 : fac_f_row(i, j)][0];
                PT = QT = QN = zero4();
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks) {
                    const Frag8 Ak = ldfrag_c<PREC, ST>(&s.kl[0][0], LDK, BS * i, 32 * ks);
                    const Frag8 Aq = ldfrag_c<PREC, ST>(&s.ql[0][0], LDK, BS * i, 32 * ks);
                    const Frag8 Bk = (j == i - 1) ? ldfrag_c<PREC, ST>(&s.kr[0][0], LDK, BS * j, 32 * ks)
                                                  : ldfrag_c_scaled<PREC, ST>(&s.kr[0][0], LDK, BS * j, 32 * ks,
                                                                              fsc + 32 * ks);
                    PT = mma<PREC>(Bk, Ak, PT);
                    if (oAqk) QT = mma<PREC>(Bk, Aq, QT);
                    if (oAqkT) QN = mma<PREC>(Aq, Bk, QN);
                }
            };
            if (w < NB) {
                if (!((pmask >> w) & 1)) {
                    f32x4 PT, QT, QN;
                    form_tile(w, w, PT, QT, QN);
                    float p4[4], q4[4], n4[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        p4[e] = (4 * g4 + e < r16) ? PT[e] : 0.f;
                        q4[e] = (4 * g4 + e <= r16) ? QT[e] : 0.f;
                        n4[e] = (r16 <= 4 * g4 + e) ? QN[e] : 0.f;
                    }
                    *reinterpret_cast<float4*>(&s.tii[w][r16][4 * g4]) = make_float4(p4[0], p4[1], p4[2], p4[3]);
                    if (oAqk) *reinterpret_cast<uint2*>(&s.aqk[BS * w + r16][BS * w + 4 * g4]) = pk4(q4);
                    if (oAqkT)
                        *reinterpret_cast<uint2*>(oAqkT + cCC + (size_t)(BS * w + r16) * C + BS * w + 4 * g4) = pk4(n4);
                } else if (!((qmask >> w) & 1)) {
                    float n4[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        s.tii[w][4 * g4 + e][r16] = (r16 < 4 * g4 + e) ? P[e] : 0.f;
                        n4[e] = (r16 <= 4 * g4 + e) ? Q[e] : 0.f;
                        if (oAqk) st1<ST>(&s.aqk[BS * w + 4 * g4 + e][BS * w + r16], n4[e]);
                    }
                    if (oAqkT)
                        *reinterpret_cast<uint2*>(oAqkT + cCC + (size_t)(BS * w + r16) * C + BS * w + 4 * g4) = pk4(n4);
                }
            } else {
                constexpr int OFFD[6] = {1, 3, 4, 6, 7, 8};   // tile_ij indices of the blocks below the diagonal
                for (int o = w - NB; o < 6; o += NW - NB) {
                    int i, j;
                    tile_ij(OFFD[o], i, j);
                    f32x4 PT, QT, QN;
                    form_tile(i, j, PT, QT, QN);
                    const float br = -s.beta[BS * i + r16];
                    const float lv[4] = {br * PT[0], br * PT[1], br * PT[2], br * PT[3]};
                    put_split(&s.spl[pair_idx(i, j)][0], lv);
                    if (oAkk)
                        *reinterpret_cast<float4*>(oAkk + cCC + (size_t)(BS * i + r16) * C + BS * j + 4 * g4) =
                            make_float4(PT[0], PT[1], PT[2], PT[3]);
                    const float q4[4] = {QT[0], QT[1], QT[2], QT[3]}, n4[4] = {QN[0], QN[1], QN[2], QN[3]};
                    if (oAqk) *reinterpret_cast<uint2*>(&s.aqk[BS * i + r16][BS * j + 4 * g4]) = pk4(q4);
                    if (oAqkT)
                        *reinterpret_cast<uint2*>(oAqkT + cCC + (size_t)(BS * j + r16) * C + BS * i + 4 * g4) = pk4(n4);
                }
            }
            // the six tiles above the diagonal are zero
            if (tid < 6 * 64) {
                const int u = tid >> 6;
                const int i = (u < 3) ? 0 : (u < 5) ? 1 : 2;
                const int j = (u < 3) ? u + 1 : (u < 5) ? u - 1 : 3;
                const uint2 z = make_uint2(0u, 0u);
                if (oAqk) *reinterpret_cast<uint2*>(&s.aqk[BS * i + r16][BS * j + 4 * g4]) = z;
                if (oAkk)
                    *reinterpret_cast<float4*>(oAkk + cCC + (size_t)(BS * i + r16) * C + BS * j + 4 * g4) =
                        make_float4(0.f, 0.f, 0.f, 0.f);
                if (oAqkT) *reinterpret_cast<uint2*>(oAqkT + cCC + (size_t)(BS * j + r16) * C + BS * i + 4 * g4) = z;
            }
        }
        if constexpr (STRONG) {
            // the entries formed from raw q, k, from registers to their places
            if (unsafe) {
#pragma unroll
                for (int it = 0; it < NPU; ++it) {
                    const int p = tid + NTH * it, t = p / C, sx = p - t * C, i = t / BS, j = sx / BS;
                    if (i == j) s.tii[i][t % BS][sx % BS] = pak[it];
                    if (j < i) {
                        const float x = -s.beta[t] * pak[it];
                        uint16_t* sp = &s.spl[pair_idx(i, j)][(t % BS) * SPR + sx % BS];
                        const uint32_t hi = pack2bf(x, 0.f);
                        sp[0] = (uint16_t)hi;
                        sp[BS] = (uint16_t)pack2bf_rest(x, 0.f, hi);
                    }
                }
            } else if (qmask) {
                const int nent = __popc(qmask) * BS * BS;
#pragma unroll
                for (int it = 0; it < NPW; ++it) {
                    const int pp = tid + NTH * it;
                    if (pp < nent) {
                        const int kb = pp / (BS * BS), e = pp - kb * BS * BS;
                        int bq = 0;
                        for (int m = qmask, c = 0;; m &= m - 1, ++c)
                            if (c == kb) { bq = __ffs(m) - 1; break; }
                        const int t = BS * bq + e / BS, sx = BS * bq + e % BS;
                        s.tii[bq][e / BS][e % BS] = pak[it];
                        if (oAqk) st1<ST>(&s.aqk[t][sx], paq[it]);
                        if (oAqkT) st1<ST>(oAqkT + cCC + (size_t)sx * C + t, paq[it]);
                    }
                }
            }
            if (unsafe || qmask) __syncthreads();
        }
        // waves 0-3: the diagonal block out, inverted in place and split (the wave's own
        // LDS writes, read back in order)
        if (w < NB) {
            float (*tb)[BS + 4] = s.tii[w];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (oAkk && !unsafe)
                *reinterpret_cast<float4*>(oAkk + cCC + (size_t)(BS * w + r16) * C + BS * w + 4 * g4) =
                    *reinterpret_cast<const float4*>(&tb[r16][4 * g4]);
            float xq[4];
            block_inverse_reg<BS + 4>(&tb[0][0], s.beta + BS * w, xq);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int e = 0; e < 4; ++e) tb[4 * (l & 3) + e][l >> 2] = xq[e];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const float4 x = *reinterpret_cast<const float4*>(&tb[r16][4 * g4]);
            if (oTii)
                *reinterpret_cast<float4*>(oTii + (size_t)ch * NB * BS * BS + w * BS * BS + r16 * BS + 4 * g4) = x;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const float v4[4] = {x.x, x.y, x.z, x.w};
            put_split(reinterpret_cast<uint16_t*>(&tb[0][0]), v4);
        }
        // KbT, QpT: per 16 x 16 tile one MFMA forms X diag(scale), the scale split into
        // bf16 hi + lo halves of one K = 32 step: a lane gets four consecutive tokens
        // of a channel, as kda_prep_kernel does
        if (!unsafe) {
            constexpr int PBT = NB * NT / NW;
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                ST* out = o ? oQpT : oKbT;
                if (out == nullptr) continue;
                const ST* X = o ? &s.ql[0][0] : &s.kr[0][0];
                Frag4 A[PBT];
                float sv[PBT];
#pragma unroll
                for (int it = 0; it < PBT; ++it) {   // token block i, channel block j
                    const int tt = w + NW * it, i = tt / NT, j = tt % NT;
                    A[it] = ldfrag4<1, ST>(X, LDK, BS * i, BS * j);
                    sv[it] = o ? (i ? s.fac[FAC_EP + i - 1][BS * j + r16] : 1.f)
                              : (i < NB - 1 ? s.fac[FAC_EQ + i][BS * j + r16] : 1.f);
                }
#pragma unroll
                for (int it = 0; it < PBT; ++it) {
                    const int tt = w + NW * it, i = tt / NT, j = tt % NT;
                    const short hi = (short)f2bf(sv[it]), lo = (short)f2bf(sv[it] - bf2f((uint16_t)hi));
                    short4v bh4, bl4;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool dg = 4 * g4 + e == r16;
                        bh4[e] = dg ? hi : (short)0;
                        bl4[e] = dg ? lo : (short)0;
                    }
                    const f32x4 c =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(cat4(A[it].h, A[it].h), cat4(bh4, bl4), zero4(), 0, 0, 0);
                    const float c4[4] = {c[0], c[1], c[2], c[3]};
                    *reinterpret_cast<uint2*>(out + cCD + (size_t)(BS * j + r16) * C + BS * i + 4 * g4) = pk4(c4);
                }
            }
        }
        __syncthreads();   // K_r is read; A_qk, the inverses and the split blocks are written
        tv.store(&s.kr[0][0], LDK);
        if (oAqk && !unsafe) tile_out<ST, C, C, NTH>(&s.aqk[0][0], LDT, oAqk + cCC, C, C);
        __syncthreads();
    };
    if (dfl & 31)
        middle(std::true_type{});
    else
        middle(std::false_type{});

    // ---------------- block forward substitution: the wave's column tiles of [K_t | beta V] ----------------
    constexpr int TPW = 2 * NT / NW;
    f32x4 X[TPW][NB];
    Frag4 XB[TPW][NB - 1];   // X's split B fragments, formed once for the later blocks
    bool isK[TPW];
    int d0[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
        const int ct = w + NW * u;
        isK[u] = ct < NT;
        d0[u] = BS * (isK[u] ? ct : ct - NT);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        f32x4 Y[TPW];
        const float4 b4 = *reinterpret_cast<const float4*>(&s.beta[BS * i + 4 * g4]);
        const float bv[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int u = 0; u < TPW; ++u) {
            float cx[4];
            ld_col4(isK[u] ? &s.kl[0][0] : &s.kr[0][0], LDK, d0[u], BS * i, cx);
            const float fe = (i && isK[u]) ? s.fac[FAC_EP + (i ? i - 1 : 0)][d0[u] + r16] : 1.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) Y[u][e] = bv[e] * fe * cx[e];
        }
#pragma unroll
        for (int j = 0; j < i; ++j) {
            const Frag4 A = get_split(&s.spl[pair_idx(i, j)][0]);
#pragma unroll
            for (int u = 0; u < TPW; ++u) Y[u] = mma4f<3>(A, XB[u][j], Y[u]);
        }
        const Frag4 Tf = get_split(reinterpret_cast<const uint16_t*>(&s.tii[i][0][0]));
#pragma unroll
        for (int u = 0; u < TPW; ++u) {
            X[u][i] = mma4f<3>(Tf, accfrag4<3>(Y[u]), zero4());
            if (i < NB - 1) XB[u][i] = accfrag4<3>(X[u][i]);
        }
    }
    __syncthreads();
    // W -> kl, U -> ql (both read by now), stored coalesced; WT straight from the
    // accumulators
#pragma unroll
    for (int u = 0; u < TPW; ++u)
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            ST* o = isK[u] ? &s.kl[0][0] : &s.ql[0][0];
#pragma unroll
            for (int e = 0; e < 4; ++e) st1<ST>(o + (BS * i + 4 * g4 + e) * LDK + d0[u] + r16, X[u][i][e]);
            if (isK[u] && oWT) {
                const float x[4] = {X[u][i][0], X[u][i][1], X[u][i][2], X[u][i][3]};
                *reinterpret_cast<uint2*>(oWT + cCD + (size_t)(d0[u] + r16) * C + BS * i + 4 * g4) = pk4(x);
            }
        }
    __syncthreads();
    tile_out<ST, C, D, NTH>(&s.kl[0][0], LDK, oW + cCD, D, C);
    tile_out<ST, C, D, NTH>(&s.ql[0][0], LDK, oU + cCD, D, C);
}

hipError_t launch_prep_wide(const PrepArgs& a, int D, int g_kind, int nchunks, hipStream_t st) {
#define KDA_PREPW_CASE(DD, TG) hipLaunchKernelGGL((kda_prepw_kernel<DD, TG>), dim3(nchunks), dim3(PW_NTH), 0, st, a)
    if (D == 128 && g_kind == 1) KDA_PREPW_CASE(128, uint16_t);
    else if (D == 128 && g_kind == 0) KDA_PREPW_CASE(128, float);
    else if (D == 64 && g_kind == 1) KDA_PREPW_CASE(64, uint16_t);
    else if (D == 64 && g_kind == 0) KDA_PREPW_CASE(64, float);
    else if (D == 64 && g_kind == 2) KDA_PREPW_CASE(64, GHead);
    else return hipErrorInvalidValue;
#undef KDA_PREPW_CASE
    return hipGetLastError();
}

}  // namespace kda
