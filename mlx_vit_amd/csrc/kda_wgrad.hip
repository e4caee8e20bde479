// kda_wgrad.hip -- weight gradients of the layer's linear maps: for each
// problem dW[n][k] = sum_m dY[m][n] X[m][k] (bf16 operands and result, fp32
// sums over the tokens m) and, on request, the bias gradient sum_m dY[m][n];
// all of a layer's problems in one launch.  And the batched conversion copy
// (kda_layer_pack) that lays a layer's parameters out for its kernels, and the
// scalar decay's logarithm and its adjoint (kda_log_decay): 150528 values at 8 x
// 1568 x 12, one launch each instead of four element-wise ones of 4 to 5 us.
//
// What bounds it: the sum runs over the tokens (12544 at 8 clips) while the
// results are small (64 x 768 to 2448 x 768), so a tile per workgroup leaves
// most of the chip idle unless the sum is split: the library's kernels took
// 84 us for each 64 x 768 and 768 x 768 gradient (1.2 and 14.8 GFLOP) and 98 us
// for 2304 x 768.  Here the token range is split so that all the problems' 128 x
// 128 tiles together fill two workgroups per CU once, the fp32 partial tiles
// go to a workspace and a second launch adds them in a fixed order.  Both
// operands have the contracted index along their rows, so tiles go to LDS as
// they lie by DMA (32 tokens a step, four buffers, three steps ahead) and
// reach the MFMA through transposing reads; the swizzle gives the four rows x
// 32 bytes of a 16-lane read distinct banks.
#include "kda_internal.h"

namespace kda {

namespace {

constexpr int WT = 128;      // tile edge (n, and k unless the problem has at most 64 columns)
constexpr int WM = 32;       // tokens per step
constexpr int WSTAGES = 4;

struct WgProblem {
    const uint16_t *dy, *x;
    uint16_t *dw, *db;
    int64_t ld_dy, ld_x;
    int n, k, nt, kt;        // columns and tiles
    int blk0;                // first workgroup
    int narrow;              // k <= 64: 128 x 64 tiles
    size_t part0;            // first float of its partial sums, [split][n][k]
    size_t bpart0;           // and of the bias's, [split][n]
};
struct WgArgs {
    WgProblem p[WGRAD_MAX_PROBLEMS];
    int count, rows, splits, rows_per_split;   // rows_per_split: a multiple of WM
    float* part;
};

// byte offset of byte b of row r in a tile of RB-byte rows: the 16-byte chunk
// index is XORed so that rows r..r+3 (a 16-lane transposing read) and the two
// groups of rows that differ in bit 2 fall on different banks
template <int RB>
__device__ __forceinline__ int wswz(int r, int b) {
    const int key = (((r & 3) << 1) | ((r & 4) << 1)) & (RB / 16 - 1);
    return r * RB + (((b >> 4) ^ key) << 4) + (b & 15);
}

// operand fragment (16x16x32) of columns n0..n0+15 over the tile's 32 rows
template <int RB>
__device__ __forceinline__ bf16x8 wfrag(const char* tile, int n0) {
    const int l = lane_id(), j = l & 15, g = l >> 4, r = 4 * g + (j >> 2), b = 2 * (n0 + 4 * (j & 3));
    const short4v x = ld_tr4(reinterpret_cast<const uint16_t*>(tile + wswz<RB>(r, b)));
    const short4v y = ld_tr4(reinterpret_cast<const uint16_t*>(tile + wswz<RB>(r + 16, b)));
    return __builtin_bit_cast(bf16x8, short8v{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]});
}

// This wave's part of a WM x COLS tile's DMA: instruction i of NI fills 1 KB of
// the tile; the lane's row in the step and byte offset in the row (columns
// past the operand's last 16-byte chunk read that one: their results are not
// stored)
template <int COLS>
struct WgDma {
    static constexpr int RB = 2 * COLS, NI = WM * RB / 1024, PER = NI / 4;
    int row[PER];
    uint32_t off[PER], cb[PER];
    uint32_t ldb;
    __device__ __forceinline__ void init(int c0, int cols, int64_t ld, int w) {
        ldb = (uint32_t)(2 * ld);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int p = 1024 * (w + 4 * i) + 16 * lane_id(), r = p / RB, pc = (p % RB) >> 4;
            const int key = (((r & 3) << 1) | ((r & 4) << 1)) & (RB / 16 - 1);
            row[i] = r;
            cb[i] = 16u * (uint32_t)min(c0 / 8 + (pc ^ key), (cols - 1) / 8);
            off[i] = (uint32_t)r * ldb + cb[i];
        }
    }
    __device__ __forceinline__ void issue_full(const char* base, uint32_t lds, int w) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) dma16_s32(base, off[i], lds + 1024u * (uint32_t)(w + 4 * i));
    }
    // rows at or past `valid` read row valid - 1
    __device__ __forceinline__ void issue(const char* base, int valid, uint32_t lds, int w) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t o = valid >= WM ? off[i] : (uint32_t)min(row[i], valid - 1) * ldb + cb[i];
            dma16_s32(base, o, lds + 1024u * (uint32_t)(w + 4 * i));
        }
    }
};

template <int TK>
__device__ __forceinline__ void wgrad_tile(const WgArgs& a, const WgProblem& p, int nti, int kti, int split,
                                           char* lds) {
    constexpr int RBA = 2 * WT, RBX = 2 * TK, STAGE = WM * (RBA + RBX);
    // waves: 2 x 2 of 64 x 64, or 4 x 1 of 32 x 64
    constexpr int WN = TK == 128 ? 64 : 32, FN = WN / 16, FK = 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), r16 = l & 15, g4 = l >> 4;
    const int wn = TK == 128 ? (w >> 1) * 64 : w * 32, wk = TK == 128 ? (w & 1) * 64 : 0;
    const int n0 = nti * WT, k0 = kti * TK;
    const int m0 = split * a.rows_per_split, m1 = min(a.rows, m0 + a.rows_per_split);
    const int steps = (m1 - m0 + WM - 1) / WM;
    WgDma<WT> da;
    WgDma<TK> dx;
    da.init(n0, p.n, p.ld_dy, w);
    dx.init(k0, p.k, p.ld_x, w);
    constexpr int L = WgDma<WT>::PER + WgDma<TK>::PER;   // DMA instructions per wave and step
    const uint32_t base = lds_addr(lds);
    // gy, gx: the next step to issue
    const char* gy = reinterpret_cast<const char*>(p.dy) + (size_t)m0 * (2 * p.ld_dy);
    const char* gx = reinterpret_cast<const char*>(p.x) + (size_t)m0 * (2 * p.ld_x);
    const int64_t stepy = 2 * WM * p.ld_dy, stepx = 2 * WM * p.ld_x;
    auto issue = [&](int s) {
        const int valid = m1 - m0 - s * WM;
        const uint32_t st = base + (uint32_t)((s % WSTAGES) * STAGE);
        da.issue(gy, valid, st, w);
        dx.issue(gx, valid, st + WM * RBA, w);
        gy += stepy;
        gx += stepx;
    };
    for (int s = 0; s < min(steps, WSTAGES - 1); ++s) issue(s);

    f32x4 acc[FN][FK], accb[FN];
#pragma unroll
    for (int i = 0; i < FN; ++i) {
        accb[i] = zero4();
#pragma unroll
        for (int j = 0; j < FK; ++j) acc[i][j] = zero4();
    }
    const bool bias = p.db != nullptr && kti == 0 && wk == 0;
    const uint16_t one = 0x3f80;
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(one | (one << 16), one | (one << 16), one | (one << 16),
                                                              one | (one << 16)));
    auto compute = [&](const char* st) {
        bf16x8 fa[FN], fx[FK];
#pragma unroll
        for (int i = 0; i < FN; ++i) fa[i] = wfrag<RBA>(st, wn + 16 * i);
#pragma unroll
        for (int j = 0; j < FK; ++j) fx[j] = wfrag<RBX>(st + WM * RBA, wk + 16 * j);
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FK; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fx[j], acc[i][j], 0, 0, 0);
        if (bias) {
#pragma unroll
            for (int i = 0; i < FN; ++i) accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], ones, accb[i], 0, 0, 0);
        }
    };
    // Each step: this wave's share of step s has landed (the later steps' DMA
    // stays in flight), barrier -- so every wave's has, and every wave has read
    // step s - 1, whose buffer step s + 3 takes -- then issue and compute.
    // Groups of WSTAGES whole steps first: buffers at immediate offsets, no row
    // clamps (with these and the arguments re-read in the loop, 64 against 58 us
    // for 2444 x 768)
    int s = 0;
    for (; (s + 2 * WSTAGES - 1) * WM <= m1 - m0; s += WSTAGES) {
#pragma unroll
        for (int u = 0; u < WSTAGES; ++u) {
            dma_wait<(WSTAGES - 2) * L>();
            lds_barrier();
            const uint32_t dst = base + (uint32_t)(((u + WSTAGES - 1) % WSTAGES) * STAGE);
            da.issue_full(gy, dst, w);
            dx.issue_full(gx, dst + WM * RBA, w);
            gy += stepy;
            gx += stepx;
            compute(lds + u * STAGE);
        }
    }
    for (; s < steps; ++s) {
        dma_wait_chunks<L>(min(WSTAGES - 2, steps - 1 - s));
        lds_barrier();
        char* st = lds + (s % WSTAGES) * STAGE;
        const int valid = m1 - m0 - s * WM;
        if (valid < WM) {
            // the last step's rows past the end: zero in both operands
            for (int i = threadIdx.x; i < (WM - valid) * (RBA / 16); i += 256)
                *reinterpret_cast<uint4*>(st + valid * RBA + 16 * i) = make_uint4(0u, 0u, 0u, 0u);
            for (int i = threadIdx.x; i < (WM - valid) * (RBX / 16); i += 256)
                *reinterpret_cast<uint4*>(st + WM * RBA + valid * RBX + 16 * i) = make_uint4(0u, 0u, 0u, 0u);
            lds_barrier();
        }
        if (s + WSTAGES - 1 < steps) issue(s + WSTAGES - 1);
        compute(st);
    }
    const size_t nk = (size_t)p.n * p.k;
    float* part = a.part + p.part0 + (size_t)split * nk;
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = n0 + wn + 16 * i + 4 * g4 + e;
            if (n >= p.n) continue;
#pragma unroll
            for (int j = 0; j < FK; ++j) {
                const int k = k0 + wk + 16 * j + r16;
                if (k < p.k) {
                    if (a.splits == 1) p.dw[(size_t)n * p.k + k] = f2bf(acc[i][j][e]);
                    else part[(size_t)n * p.k + k] = acc[i][j][e];
                }
            }
            if (bias && r16 == 0) {
                if (a.splits == 1) p.db[n] = f2bf(accb[i][e]);
                else a.part[p.bpart0 + (size_t)split * p.n + n] = accb[i][e];
            }
        }
}

__global__ __launch_bounds__(256, 2) void kda_wgrad_kernel(const WgArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[WSTAGES * WM * 2 * (WT + WT)];
    // workgroups with equal blockIdx % 8 share an XCD's L2: each XCD gets a run of
    // consecutive tiles (of one split, mostly), so it reads an eighth of the
    // tiles' rows instead of all of them
    const int nb = (int)gridDim.x, xcd = (int)blockIdx.x % 8, q = nb / 8, rem = nb % 8;
    const int lb = xcd * q + min(xcd, rem) + (int)blockIdx.x / 8;
    int j = 0;
    while (j + 1 < a.count && lb >= a.p[j + 1].blk0) ++j;
    j = __builtin_amdgcn_readfirstlane(j);
    const WgProblem& p = a.p[j];
    const int b = lb - p.blk0, tiles = p.nt * p.kt, split = b / tiles, t = b - split * tiles;
    const int kti = t % p.kt, nti = t / p.kt;
    if (p.narrow)
        wgrad_tile<64>(a, p, nti, kti, split, lds);
    else
        wgrad_tile<128>(a, p, nti, kti, split, lds);
}

// the splits' partial sums in order, four columns a thread (k is a multiple of
// 8); then the biases
__global__ __launch_bounds__(256) void kda_wgrad_reduce_kernel(const WgArgs a, size_t total4) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total4; i += (size_t)gridDim.x * 256) {
        size_t e = i;
        int j = 0;
        for (; j + 1 < a.count; ++j) {
            const size_t c = ((size_t)a.p[j].n * a.p[j].k) / 4;
            if (e < c) break;
            e -= c;
        }
        const WgProblem& p = a.p[j];
        const size_t nk = (size_t)p.n * p.k;
        const float* src = a.part + p.part0 + 4 * e;
        float4 s = *reinterpret_cast<const float4*>(src);
        for (int q = 1; q < a.splits; ++q) {
            const float4 x = *reinterpret_cast<const float4*>(src + q * nk);
            s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
        }
        *reinterpret_cast<uint2*>(p.dw + 4 * e) = make_uint2(pack2bf(s.x, s.y), pack2bf(s.z, s.w));
    }
    for (int j = 0; j < a.count; ++j)
        if (a.p[j].db)
            for (int n = blockIdx.x * 256 + threadIdx.x; n < a.p[j].n; n += gridDim.x * 256) {
                float s = 0.f;
                for (int q = 0; q < a.splits; ++q) s += a.part[a.p[j].bpart0 + (size_t)q * a.p[j].n + n];
                a.p[j].db[n] = f2bf(s);
            }
}

// Tiles, splits and partial offsets.  The splits fill 2 workgroups on each of
// 256 CUs once where the rows allow at least 8 steps each (12544 rows of one
// layer: 168 tiles, 3 splits of 131 steps).
size_t plan(WgArgs& a) {
    int tiles = 0;
    for (int j = 0; j < a.count; ++j) {
        WgProblem& p = a.p[j];
        p.narrow = p.k <= 64;
        p.nt = (p.n + WT - 1) / WT;
        p.kt = p.narrow ? 1 : (p.k + WT - 1) / WT;
        tiles += p.nt * p.kt;
    }
    const int steps = (a.rows + WM - 1) / WM;
    const int s = std::max(1, std::min(512 / std::max(tiles, 1), steps / 8));
    a.rows_per_split = (steps + s - 1) / s * WM;
    a.splits = std::max(1, (a.rows + a.rows_per_split - 1) / a.rows_per_split);
    size_t f = 0;
    int blk = 0;
    for (int j = 0; j < a.count; ++j) {
        WgProblem& p = a.p[j];
        p.blk0 = blk;
        blk += p.nt * p.kt * a.splits;
        if (a.splits > 1) {
            p.part0 = f;
            f += (size_t)a.splits * p.n * p.k;
            p.bpart0 = f;
            if (p.db) f += (((size_t)a.splits * p.n) + 3) & ~(size_t)3;
        }
    }
    return f;
}

WgArgs to_args(const WgradProblem* q, int count, int rows) {
    WgArgs a = {};
    a.count = count;
    a.rows = rows;
    for (int j = 0; j < count; ++j) {
        WgProblem& p = a.p[j];
        p.dy = static_cast<const uint16_t*>(q[j].dy);
        p.x = static_cast<const uint16_t*>(q[j].x);
        p.dw = static_cast<uint16_t*>(q[j].dw);
        p.db = static_cast<uint16_t*>(q[j].db);
        p.ld_dy = q[j].ld_dy;
        p.ld_x = q[j].ld_x;
        p.n = (int)q[j].n;
        p.k = (int)q[j].k;
    }
    return a;
}

// g = max(log alpha, g_min), fp32, of a decay alpha (bf16 or fp32)
template <typename T>
__global__ __launch_bounds__(256) void kda_log_decay_kernel(const T* __restrict__ alpha, float* __restrict__ g, size_t n,
                                                            float g_min) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float x = logf(ld1<T>(alpha + i));
        g[i] = x < g_min ? g_min : x;   // keeps a NaN
    }
}

// its adjoint: d alpha = dg / alpha where log alpha >= g_min, else 0
template <typename T>
__global__ __launch_bounds__(256) void kda_log_decay_bwd_kernel(const T* __restrict__ alpha, const float* __restrict__ dg,
                                                                T* __restrict__ dalpha, size_t n, float g_min) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float a = ld1<T>(alpha + i);
        st1<T>(dalpha + i, (logf(a) >= g_min ? dg[i] : 0.f) / a);
    }
}

// job j owns workgroups [wg0[j], wg0[j + 1]), PACK_PER elements each
constexpr int PACK_PER = 4096;
struct PackArgs {
    PackJob j[PACK_MAX_JOBS];
    int wg0[PACK_MAX_JOBS + 1];
    int count;
};

__global__ __launch_bounds__(256) void kda_pack_kernel(const PackArgs a) {
    int j = 0;
    while (j + 1 < a.count && (int)blockIdx.x >= a.wg0[j + 1]) ++j;
    j = __builtin_amdgcn_readfirstlane(j);
    const PackJob& p = a.j[j];
    const int sd = (int)(p.dtypes & 255), dd = (int)(p.dtypes >> 8);
    const int64_t e0 = (int64_t)((int)blockIdx.x - a.wg0[j]) * PACK_PER, e1 = min(p.n, e0 + (int64_t)PACK_PER);
    const bool vec = (((uintptr_t)p.src | (uintptr_t)p.dst) & 15) == 0;
    if (sd == 1 && dd == 1) {
        const uint16_t* s = static_cast<const uint16_t*>(p.src);
        uint16_t* d = static_cast<uint16_t*>(p.dst);
        int64_t i = e0 + 8 * (int64_t)threadIdx.x;
        if (vec)
            for (; i + 8 <= e1; i += 8 * 256) *reinterpret_cast<uint4*>(d + i) = *reinterpret_cast<const uint4*>(s + i);
        for (; i < e1; i += 8 * 256)
            for (int c = 0; c < 8 && i + c < e1; ++c) d[i + c] = s[i + c];
        return;
    }
    for (int64_t i = e0 + threadIdx.x; i < e1; i += 256) {
        const float v = sd == 1 ? bf2f(static_cast<const uint16_t*>(p.src)[i]) : static_cast<const float*>(p.src)[i];
        if (dd == 1) static_cast<uint16_t*>(p.dst)[i] = f2bf(v);
        else static_cast<float*>(p.dst)[i] = v;
    }
}

}  // namespace

size_t wgrad_ws_floats(const WgradProblem* q, int count, int rows) {
    WgArgs a = to_args(q, count, rows);
    return plan(a);
}

hipError_t launch_wgrad(const WgradProblem* q, int count, int rows, float* part, hipStream_t st) {
    if (count < 1 || count > WGRAD_MAX_PROBLEMS) return hipErrorInvalidValue;
    WgArgs a = to_args(q, count, rows);
    plan(a);
    a.part = part;
    const WgProblem& last = a.p[count - 1];
    const unsigned blocks = (unsigned)(last.blk0 + last.nt * last.kt * a.splits);
    hipLaunchKernelGGL(kda_wgrad_kernel, dim3(blocks), dim3(256), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.splits == 1) return e;
    size_t total4 = 0;
    for (int j = 0; j < count; ++j) total4 += (size_t)a.p[j].n * a.p[j].k / 4;
    hipLaunchKernelGGL(kda_wgrad_reduce_kernel, dim3((unsigned)std::min<size_t>((total4 + 255) / 256, 2048)), dim3(256),
                       0, st, a, total4);
    return hipGetLastError();
}

hipError_t launch_log_decay(const void* alpha, float* g, const float* dg, void* dalpha, size_t n, float g_min,
                            int in_bf16, hipStream_t st) {
    const dim3 grid((unsigned)std::min<size_t>((n + 255) / 256, 2048)), block(256);
    if (dg) {
        if (in_bf16)
            hipLaunchKernelGGL((kda_log_decay_bwd_kernel<uint16_t>), grid, block, 0, st, static_cast<const uint16_t*>(alpha),
                               dg, static_cast<uint16_t*>(dalpha), n, g_min);
        else
            hipLaunchKernelGGL((kda_log_decay_bwd_kernel<float>), grid, block, 0, st, static_cast<const float*>(alpha), dg,
                               static_cast<float*>(dalpha), n, g_min);
    } else {
        if (in_bf16)
            hipLaunchKernelGGL((kda_log_decay_kernel<uint16_t>), grid, block, 0, st, static_cast<const uint16_t*>(alpha), g,
                               n, g_min);
        else
            hipLaunchKernelGGL((kda_log_decay_kernel<float>), grid, block, 0, st, static_cast<const float*>(alpha), g, n,
                               g_min);
    }
    return hipGetLastError();
}

hipError_t launch_pack(const PackJob* jobs, int count, hipStream_t st) {
    if (count < 0 || count > PACK_MAX_JOBS) return hipErrorInvalidValue;
    PackArgs a = {};
    int wg = 0;
    for (int j = 0; j < count; ++j) {
        if (jobs[j].n <= 0) continue;
        a.j[a.count] = jobs[j];
        a.wg0[a.count] = wg;
        wg += (int)((jobs[j].n + PACK_PER - 1) / PACK_PER);
        a.wg0[++a.count] = wg;
    }
    if (wg == 0) return hipSuccess;
    hipLaunchKernelGGL(kda_pack_kernel, dim3(wg), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace kda
