// Router pieces for prefill-sized calls: the dense query projection on the matrix cores, and the load statistics.
//
//   mortar_router_project_bf16   qv = x Wq^T (morph/model/routing.py:190-198) for bf16 x and fp32 Wq, at fp32 precision
//   mortar_router_stats          expert-load EMA and load-balance loss behind the gates (routing.py:262-284)
#include "mortar_device.h"
#include "mortar_internal.h"

namespace {

// qv[m, o] = sum_k x[m, k] * W[o, k], x bf16, W fp32, fp32 result.
//
// An fp32 weight is exactly the sum of three bf16 values (its top 8, next 8 and last 8 significant bits), so three bf16
// MFMAs on the same activation operand give exact products in fp32 accumulators: the arithmetic of an fp32 GEMM at three
// times the cost of a bf16 one instead of the sixteen times of the fp32 matrix instructions (4096 x 2048 x 2048: 81 us,
// 1270 TFLOP/s of the three terms, against 257 us through the library's fp32 GEMM with its conversion of x; the MFMAs
// alone take 60 us at the clocks the part holds under them).
//
// A workgroup of NW waves owns MT tokens x 16 NW outputs; a wave owns 16 outputs for all MT tokens, so that a weight is
// split once per workgroup: 44 vector instructions per 3 MT / 16 MFMAs, hidden behind the matrix pipe from 128 tokens up.
// Both operands travel in steps of 64 values through D buffers in LDS, copied asynchronously (global_load_lds, no registers)
// D - 1 steps ahead; storing the activations from registers instead cost 1000 of 5300 cycles per step.  One barrier per
// step.  Four consecutive lanes copy 64 contiguous bytes (in another order per lane group: `n`-dependent swizzles), so that
// the copies stay coalesced and the operand reads touch every bank once.
constexpr int RG_KS = 64;

__device__ __forceinline__ void split3(const float (&w)[8], u32x4_t (&p)[3]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t h[2], m[2], l[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = w[2 * q + e];
            h[e] = __builtin_bit_cast(uint32_t, v);
            const float r = v - __builtin_bit_cast(float, h[e] & 0xffff0000u);
            m[e] = __builtin_bit_cast(uint32_t, r);
            l[e] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, m[e] & 0xffff0000u));
        }
        // the high halves of two words side by side
        p[0][q] = __builtin_amdgcn_perm(h[1], h[0], 0x07060302u);
        p[1][q] = __builtin_amdgcn_perm(m[1], m[0], 0x07060302u);
        p[2][q] = __builtin_amdgcn_perm(l[1], l[0], 0x07060302u);
    }
}

template <int MT, int NW, int D>
__global__ void __launch_bounds__(NW * 64) router_gemm_kernel(const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, float *qv,
                                                              int64_t ldq, int n_ntiles) {
    constexpr int MI = MT / 16, FR = MI * 2, U = FR / NW, MG = MI < 4 ? MI : 4;
    constexpr int XB = MT * RG_KS * 2, WB = 16 * RG_KS * 4, BUF = XB + NW * WB;       // activations, then one block of weights per wave
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    // ids are dealt round-robin over the 8 XCDs: each takes a run of tiles, so that its L2 serves the x rows of few token tiles
    const int per_xcd = (int)((gridDim.x + 7) >> 3);
    const int id = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int n_mtiles = (M + MT - 1) / MT;
    if (id >= n_mtiles * n_ntiles) return;
    const int m0 = (id / n_ntiles) * MT, o0 = (id % n_ntiles) * (16 * NW) + wave * 16;

    // Activations: fragments (16 tokens x 32 values, 1 KB) wave + NW * i; slot l of a fragment holds 16-byte unit
    // (l & 3) ^ s(token) of token l / 4 (mortar_unit_swz).  Weights: row 4 i + l / 16, slot l & 15 of its 256 bytes holds unit (l & 15) ^ row.
    const uint16_t *xs[U];
    const float *ws[4];
    int kx[U], kw[4];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int f = wave + NW * i, t = lane >> 2, row = m0 + (f >> 1) * 16 + t;
        kx[i] = (f & 1) * 32 + ((lane & 3) ^ mortar_unit_swz(t)) * 8;
        xs[i] = x + (int64_t)(row < M ? row : M - 1) * ldx + kx[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * i + g;
        kw[i] = (n ^ r) * 4;
        ws[i] = W + (int64_t)(o0 + r < N ? o0 + r : N - 1) * K + kw[i];
    }
    const uint32_t rd = (uint32_t)(n * 64 + (g ^ mortar_unit_swz(n)) * 16);
    // K % 8 == 0: a unit is in the row or past its end as a whole; the ones past the end are cleared (last step only)
    auto stage = [&](int k0, int buf) {
        const bool part = k0 + RG_KS > K;
        unsigned char *xd = lds + buf * BUF + wave * 1024, *wd = lds + buf * BUF + XB + wave * WB;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (part && k0 + kx[i] >= K) *reinterpret_cast<u32x4_t *>(xd + i * NW * 1024 + lane * 16) = u32x4_t{0u, 0u, 0u, 0u};
            else mortar_load_to_lds((const MORTAR_GLOBAL char *)(xs[i] + k0), __builtin_amdgcn_readfirstlane(mortar_lds_addr(xd + i * NW * 1024)));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (part && k0 + kw[i] >= K) *reinterpret_cast<u32x4_t *>(wd + i * 1024 + lane * 16) = u32x4_t{0u, 0u, 0u, 0u};
            else mortar_load_to_lds((const MORTAR_GLOBAL char *)(ws[i] + k0), __builtin_amdgcn_readfirstlane(mortar_lds_addr(wd + i * 1024)));
        }
    };
    f32x4_t acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int b = 0; b < D - 1; ++b)
        if (b * RG_KS < K) stage(b * RG_KS, b);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += RG_KS) {
        const int kn = k0 + (D - 1) * RG_KS;
        if (kn < K) stage(kn, buf == 0 ? D - 1 : buf - 1);
        const unsigned char *cur = lds + buf * BUF;
        float w[2][8];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 v = *reinterpret_cast<const float4 *>(cur + XB + wave * WB + n * 256 + ((8 * h + 2 * g + j) ^ n) * 16);
                w[h][4 * j] = v.x; w[h][4 * j + 1] = v.y; w[h][4 * j + 2] = v.z; w[h][4 * j + 3] = v.w;
            }
        // groups of MG token fragments; the operands of the next group are read while the current one multiplies
        constexpr int NG = 2 * MI / MG;
        u32x4_t b[2][MG];
        auto operands = [&](int q) {
#pragma unroll
            for (int i = 0; i < MG; ++i)
                b[q & 1][i] = *reinterpret_cast<const u32x4_t *>(cur + ((q * MG % MI + i) * 2 + q * MG / MI) * 1024 + rd);
        };
        operands(0);
        u32x4_t p[3];
#pragma unroll
        for (int q = 0; q < NG; ++q) {
            if (q * MG % MI == 0) split3(w[q * MG / MI], p);
            if (q + 1 < NG) operands(q + 1);
#pragma unroll
            for (int t = 2; t >= 0; --t)                                      // small terms first
#pragma unroll
                for (int i = 0; i < MG; ++i) acc[q * MG % MI + i] = mortar_mfma(p[t], b[q & 1][i], acc[q * MG % MI + i]);
        }
        // The next step has landed: at most the copies of the D - 2 steps after it are still in flight.  (Every whole step
        // issues U + 4 copies per wave; a partial or missing one issues fewer, so the last steps wait for everything.)
        if (D > 2 && kn + RG_KS <= K) asm volatile("s_waitcnt vmcnt(%0)" ::"i"((D - 2) * (U + 4)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        buf = buf + 1 == D ? 0 : buf + 1;
    }
    const int o = o0 + 4 * g;
    if (o < N) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int m = m0 + i * 16 + n;
            if (m < M) *reinterpret_cast<f32x4_t *>(qv + (int64_t)m * ldq + o) = acc[i];
        }
    }
}

template <int MT, int NW, int D>
int launch_gemm(const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, float *qv, int64_t ldq, hipStream_t st) {
    constexpr int smem = D * (MT * RG_KS * 2 + NW * 16 * RG_KS * 4);
    static_assert(smem <= 160 * 1024, "LDS of a CU");
    static bool done = false;
    if (!done) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(router_gemm_kernel<MT, NW, D>), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "router projection: %s", hipGetErrorString(e));
        done = true;
    }
    const int nt = (N + 16 * NW - 1) / (16 * NW), mt = (M + MT - 1) / MT;
    const unsigned grid = (unsigned)(((int64_t)mt * nt + 7) / 8 * 8);
    hipLaunchKernelGGL((router_gemm_kernel<MT, NW, D>), dim3(grid), dim3(NW * 64), smem, st, x, M, K, ldx, W, N, qv, ldq, nt);
    return MORTAR_OK;
}

// The same product for fewer tokens, K <= 2048.  The kernel above gives a workgroup all of K, 32 steps behind a barrier each, and
// has too few workgroups; here the eight waves of a workgroup share K: 16 outputs per workgroup, wave w holds the three terms of
// 32 CH values of their rows in registers (one burst of loads, split once) and the workgroup's token tiles pass over them.
// Activations travel two tiles ahead through LDS regions that belong to one wave (no barrier), in copies of whole 64 CH-byte row
// pieces: operand loads straight from L2 (16 rows of 64 bytes at a power-of-two stride) took 2 us per tile.  The eight partial sums
// of a group of 64 tokens meet in LDS.  The high terms have accumulators of their own, four chains per tile: the error stays that
// of the wave-wide fp32 sums that this replaces.
// NORM (M <= 16, one tile): the rows are RMS-normalised on the way into the products.  The waves share the rows' scales (rms_* of
// mortar_device.h, the bits of rmsnorm_rows_kernel) while the weights are on their way, and the workgroups of the first outputs also
// write the rows to xn, for the products that follow the router.  (Figures: launch_router.)
constexpr int RS_TG = 4;                  // token tiles of 16 per group

template <int CH, bool NORM>
__global__ void __launch_bounds__(512) router_skinny_kernel(const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, const float *bias,
                                                            float *qv, int64_t ldq, const uint16_t *nw, float eps, uint16_t *xn) {
    constexpr int WU = 8 * CH, XU = 4 * CH, XT = 16 * XU * 16;      // 16-byte units of a row piece (weights, activations); bytes of a tile
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];       // 8 waves x 2 tiles (first the weights) | partial sums
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int o0 = blockIdx.x * 16, kw = wave * 32 * CH;
    unsigned char *own = lds + wave * 2 * XT;
    f32x4_t *part = reinterpret_cast<f32x4_t *>(lds + 16 * XT);
    // token tiles of this workgroup in order: tile t is tile t % RS_TG of its group t / RS_TG
    auto tile_row = [&](int t) { return ((int)blockIdx.y + t / RS_TG * (int)gridDim.y) * 16 * RS_TG + t % RS_TG * 16; };
    // Slot s of a tile (weights: of the 16 rows) holds unit (s % units) ^ row of row s / units: the operand reads then touch every bank
    // once.  K % 8 == 0: a unit lies in the row or past its end as a whole; past the end the row's first values are copied and
    // cleared after the read.
    auto x_src = [&](int t, int i) {
        const int s = i * 64 + lane, r = s / XU, k = kw + ((s % XU) ^ r) * 8, row = tile_row(t) + r;
        return x + (int64_t)(row < M ? row : M - 1) * ldx + (k < K ? k : 0);
    };
    auto x_copy = [&](int t) {
#pragma unroll
        for (int i = 0; i < CH; ++i)
            mortar_load_to_lds((const MORTAR_GLOBAL char *)x_src(t, i), __builtin_amdgcn_readfirstlane(mortar_lds_addr(own + (t & 1) * XT + i * 1024)));
    };
#pragma unroll
    for (int i = 0; i < 2 * CH; ++i) {
        const int s = i * 64 + lane, r = s / WU, k = kw + ((s % WU) ^ r) * 4, row = o0 + r;
        mortar_load_to_lds((const MORTAR_GLOBAL char *)(W + (int64_t)(row < N ? row : N - 1) * K + (k < K ? k : 0)),
                           __builtin_amdgcn_readfirstlane(mortar_lds_addr(own + i * 1024)));
    }
    u32x4_t x0[CH];                        // the first tile waits in registers: its LDS holds the weights
#pragma unroll
    for (int i = 0; i < CH; ++i) x0[i] = *reinterpret_cast<const u32x4_t *>(x_src(0, i));
    u32x4_t w8[NORM ? CH : 1];             // norm weights of this lane's operand pieces
    if constexpr (NORM) {
        const int nch = K / 8;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int k = kw + 32 * c + 8 * g;
            w8[c] = nw ? *reinterpret_cast<const u32x4_t *>(nw + (k < K ? k : 0)) : u32x4_t{0u, 0u, 0u, 0u};
        }
        float *scale = reinterpret_cast<float *>(part);
        if (wave < M) {                                             // rows wave, wave + 8
            u32x4_t u[2][CH / 2];
            const int m = wave, m1 = m + 8 < M ? m + 8 : m;
#pragma unroll
            for (int j = 0; j < CH / 2; ++j) {
                const int ch = lane + 64 * j < nch ? lane + 64 * j : nch - 1;
                u[0][j] = reinterpret_cast<const u32x4_t *>(x + (int64_t)m * ldx)[ch];
                u[1][j] = reinterpret_cast<const u32x4_t *>(x + (int64_t)m1 * ldx)[ch];
            }
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int j = 0; j < CH / 2; ++j)
                if (lane + 64 * j < nch) { s0 = rms_sumsq8(u[0][j], s0); s1 = rms_sumsq8(u[1][j], s1); }
            s0 = rms_scale(rms_wave_sum(s0), K, eps);
            s1 = rms_scale(rms_wave_sum(s1), K, eps);
            if (lane == 0) { scale[m] = s0; scale[m1] = s1; }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    u32x4_t p[CH][3];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float4 w = *reinterpret_cast<const float4 *>(own + (n * WU + ((8 * c + 2 * g + j) ^ n)) * 16);
            v[4 * j] = w.x; v[4 * j + 1] = w.y; v[4 * j + 2] = w.z; v[4 * j + 3] = w.w;
        }
        split3(v, p[c]);
        if (kw + 32 * c + 8 * g >= K) p[c][0] = p[c][1] = p[c][2] = u32x4_t{0u, 0u, 0u, 0u};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < CH; ++i) *reinterpret_cast<u32x4_t *>(own + i * 1024 + lane * 16) = x0[i];
    if (tile_row(1) < M) x_copy(1);
    float rms = 0.f;
    if constexpr (NORM) {
        __syncthreads();
        rms = reinterpret_cast<const float *>(part)[n < M ? n : 0];
        __syncthreads();                   // the partial sums go where the scales were
    }
    for (int t0 = 0; tile_row(t0) < M; t0 += RS_TG) {
        f32x4_t acc[RS_TG];
#pragma unroll
        for (int i = 0; i < RS_TG; ++i) {
            const int t = t0 + i;
            f32x4_t hi[4], lo = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) hi[c] = lo;
            if (tile_row(t) < M) {
                // tile t has landed: the copies of tile t + 1, where there is one, are all that may be in flight
                if (tile_row(t + 1) < M) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(CH) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                u32x4_t b[CH];
#pragma unroll
                for (int c = 0; c < CH; ++c) b[c] = *reinterpret_cast<const u32x4_t *>(own + (t & 1) * XT + (n * XU + ((4 * c + g) ^ n)) * 16);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (tile_row(t + 2) < M) x_copy(t + 2);
                if constexpr (NORM) {
                    const int m = tile_row(t) + n;
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        const int k = kw + 32 * c + 8 * g;
                        b[c] = rms_apply8(b[c], rms, w8[c], nw != nullptr);
                        if (blockIdx.x == 0 && m < M && k < K) *reinterpret_cast<u32x4_t *>(xn + (int64_t)m * K + k) = b[c];
                    }
                }
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    if (kw + 32 * c + 8 * g >= K) b[c] = u32x4_t{0u, 0u, 0u, 0u};
                    lo = mortar_mfma(p[c][2], b[c], lo);
                    hi[c & 3] = mortar_mfma(p[c][0], b[c], hi[c & 3]);
                    lo = mortar_mfma(p[c][1], b[c], lo);
                }
            }
            acc[i] = lo + ((hi[0] + hi[1]) + (hi[2] + hi[3]));
        }
#pragma unroll
        for (int i = 0; i < RS_TG; ++i) part[(wave * RS_TG + i) * 64 + lane] = acc[i];
        __syncthreads();
        if (wave < RS_TG) {                                   // wave i finishes tile i: a lane holds outputs o0 + 4 g .. + 3 of token n
            f32x4_t s = part[wave * 64 + lane];
#pragma unroll
            for (int k = 1; k < 8; ++k) s += part[(k * RS_TG + wave) * 64 + lane];
            const int m = tile_row(t0 + wave) + n, o = o0 + 4 * g;
            if (m < M && o < N) {
                if (bias) s += *reinterpret_cast<const f32x4_t *>(bias + o);
                *reinterpret_cast<f32x4_t *>(qv + (int64_t)m * ldq + o) = s;
            }
        }
        __syncthreads();
    }
}

// ---- load statistics -----------------------------------------------------------------------------------------------

constexpr int ST_ROWS = 64;          // tokens per workgroup of the first pass

// part[b][0][g] = sum of the gates, part[b][1][g] = active tokens, over the workgroup's rows (fixed order).  1024 threads:
// n <= 1024 columns x as many row slices as fit.
__global__ void __launch_bounds__(1024) router_stats_part_kernel(const float *gates, int64_t M, int n, float *part) {
    __shared__ float ps[1024], pa[1024];
    const int64_t r0 = (int64_t)blockIdx.x * ST_ROWS;
    const int rows = M - r0 < ST_ROWS ? (int)(M - r0) : ST_ROWS;
    const int slices = 1024 / n, c = threadIdx.x % n, sl = threadIdx.x / n;
    const float *p = gates + r0 * n + c;
    float s = 0.f, a = 0.f;
    if (sl < slices) {
#pragma unroll 16
        for (int r = sl; r < rows; r += slices) {
            const float v = p[(int64_t)r * n];
            s += v;
            a += v > 0.f ? 1.f : 0.f;
        }
    }
    ps[threadIdx.x] = s;
    pa[threadIdx.x] = a;
    __syncthreads();
    if (threadIdx.x < (unsigned)n) {
        for (int k = 1; k < slices; ++k) { s += ps[k * n + c]; a += pa[k * n + c]; }
        part[((int64_t)blockIdx.x * 2) * n + c] = s;
        part[((int64_t)blockIdx.x * 2 + 1) * n + c] = a;
    }
}

__device__ __forceinline__ double block_sum_f64(double v, double *red) {      // 1024 threads
    v = mortar_wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < 16; ++i) s += red[i];
    return s;
}

// One workgroup: 1024 threads = n <= 1024 columns x as many row slices as fit, then the EMA and the variance of the means.
__global__ void __launch_bounds__(1024) router_stats_final_kernel(const float *part, int nb, int64_t M, int n, float alpha, float beta, float coeff,
                                                                  float *ema, float *aux) {
    __shared__ float ps[1024], pa[1024];
    __shared__ double red[16];
    const int slices = 1024 / n, c = threadIdx.x % n, sl = threadIdx.x / n;
    float s = 0.f, a = 0.f;
    if (sl < slices) {
#pragma unroll 16
        for (int b = sl; b < nb; b += slices) {
            s += part[((int64_t)b * 2) * n + c];
            a += part[((int64_t)b * 2 + 1) * n + c];
        }
    }
    ps[threadIdx.x] = s;
    pa[threadIdx.x] = a;
    __syncthreads();
    double mean = 0.0;
    if (threadIdx.x < (unsigned)n) {
        for (int k = 1; k < slices; ++k) { s += ps[k * n + c]; a += pa[k * n + c]; }
        ema[c] = __builtin_fmaf(beta, a / (float)M, ema[c] * alpha);
        mean = (double)(s / (float)M);
    }
    const double avg = block_sum_f64(mean, red) / n;
    const double d = threadIdx.x < (unsigned)n ? mean - avg : 0.0;
    const double var = block_sum_f64(d * d, red);
    if (threadIdx.x == 0) *aux = coeff * (float)(var / (n - 1));               // n == 1: NaN, as torch.var has it
}

int check_launch(const char *what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "%s launch: %s", what, hipGetErrorString(e));
    return MORTAR_OK;
}

}  // namespace

namespace {
template <int CH, bool NORM>
int launch_skinny(dim3 grid, const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, const float *bias, float *qv, int64_t ldq,
                  const uint16_t *nw, float eps, uint16_t *xn, hipStream_t st) {
    constexpr int smem = 16 * (16 * 4 * CH * 16) + 8 * RS_TG * 1024;
    static_assert(smem <= 160 * 1024, "LDS of a CU");
    static bool done = false;
    if (!done) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(router_skinny_kernel<CH, NORM>), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "router projection: %s", hipGetErrorString(e));
        done = true;
    }
    hipLaunchKernelGGL((router_skinny_kernel<CH, NORM>), grid, dim3(512), smem, st, x, M, K, ldx, W, N, bias, qv, ldq, nw, eps, xn);
    return check_launch("router projection");
}
}  // namespace

// One workgroup per CU: 16 outputs each, the token groups of 64 dealt over what is left of the chip.
static int64_t skinny_rounds(int64_t M, int32_t d_out) {
    const int64_t groups = (M + 16 * RS_TG - 1) / (16 * RS_TG), gy = d_out > 4096 ? 1 : 256 / ((d_out + 15) / 16);
    return (groups + gy - 1) / gy;
}

int mortar_router_project_skinny(const uint16_t *x, int64_t M, int32_t d_in, int64_t ldx, const float *wq, int32_t d_out, const float *bias,
                                 float *qv, int64_t ldq, void *stream, const uint16_t *norm_w, float eps, uint16_t *xn) {
    const int nt = (d_out + 15) / 16;
    const int64_t groups = (M + 16 * RS_TG - 1) / (16 * RS_TG), rounds = skinny_rounds(M, d_out);
    const int64_t gy = (groups + rounds - 1) / rounds;
    const dim3 grid((unsigned)nt, (unsigned)gy);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (d_in <= 1024)
        return xn ? launch_skinny<4, true>(grid, x, (int)M, d_in, ldx, wq, d_out, bias, qv, ldq, norm_w, eps, xn, st)
                  : launch_skinny<4, false>(grid, x, (int)M, d_in, ldx, wq, d_out, bias, qv, ldq, nullptr, 0.f, nullptr, st);
    return xn ? launch_skinny<8, true>(grid, x, (int)M, d_in, ldx, wq, d_out, bias, qv, ldq, norm_w, eps, xn, st)
              : launch_skinny<8, false>(grid, x, (int)M, d_in, ldx, wq, d_out, bias, qv, ldq, nullptr, 0.f, nullptr, st);
}

extern "C" int mortar_router_project_bf16(const uint16_t *x, int64_t M, int32_t d_in, int64_t ldx, const float *wq, int32_t d_out, float *qv,
                                          int64_t ldq, void *stream) {
    if (!x || !wq || !qv) return mortar_fail(MORTAR_ERR_ARG, "router projection: null pointer");
    if (M <= 0 || M > (1 << 30) || d_in <= 0 || d_out <= 0 || d_in % 8 || d_out % 4 || ldx < d_in || ldx % 8 || ldq < d_out || ldq % 4)
        return mortar_fail(MORTAR_ERR_ARG, "router projection: M, d_in (a multiple of 8), d_out (of 4) and the leading dimensions must be positive and aligned");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(wq) | reinterpret_cast<uintptr_t>(qv)) & 15)
        return mortar_fail(MORTAR_ERR_ARG, "router projection: x, wq and qv must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Tokens per workgroup: the choice with the least rounds of workgroups x time of a round.  A round of 256 workgroups (one
    // per CU) of 128 outputs takes mt + 100 units (49 us at 128 tokens and 2048 inputs, 72 us at 256); the 64-token tile of 64
    // outputs fits a CU twice and takes 131 units alone, 164 with a neighbour.
    const int64_t nt8 = (d_out + 127) / 128, w64 = (M + 63) / 64 * ((d_out + 63) / 64);
    const int64_t c256 = ((M + 255) / 256 * nt8 + 255) / 256 * 356, c128 = ((M + 127) / 128 * nt8 + 255) / 256 * 228;
    const int64_t c64 = w64 <= 256 ? 131 : (w64 + 511) / 512 * 164;
    // The kernel that shares K takes 30 + 17 units per round of 64-token groups where a wave holds 256 values of K (6.5 + 3.7 us) and,
    // where it holds 128, 37 + 20 units of a K of 1024.  Against the tiles: 65 tokens x 2048 x 2048 27.4 -> 9.4 us, 300 28 -> 17,
    // 700 34 -> 28, 1000 35 against 36; at 1024 values 65 15.1 -> 5.8, 1000 16.1 -> 13.0, 2000 20 against 21.
    const int64_t rs = skinny_rounds(M, d_out);
    const int64_t csk = d_in > 2048 ? INT64_MAX : d_in > 1024 ? (30 + 17 * rs) * 2048 / d_in : (37 + 20 * rs) * 1024 / d_in;
    if (csk <= c64 && csk <= c128 && csk <= c256) return mortar_router_project_skinny(x, M, d_in, ldx, wq, d_out, nullptr, qv, ldq, stream);
    int rc;
    if (c256 <= c128 && c256 <= c64) rc = launch_gemm<256, 8, 2>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    else if (c128 <= c64) rc = launch_gemm<128, 8, 2>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    else rc = launch_gemm<64, 4, 3>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    if (rc) return rc;
    return check_launch("router projection");
}

extern "C" int64_t mortar_router_stats_workspace_bytes(int64_t M, int32_t n) {
    if (M <= 0 || n <= 0) return 0;
    return (M + ST_ROWS - 1) / ST_ROWS * 2 * n * (int64_t)sizeof(float);
}

extern "C" int mortar_router_stats(const float *gates, int64_t M, int32_t n, float alpha, float one_minus_alpha, float coeff, float *ema, float *aux,
                                   void *workspace, void *stream) {
    if (!gates || !ema || !aux || !workspace) return mortar_fail(MORTAR_ERR_ARG, "router stats: null pointer");
    if (M <= 0 || n <= 0 || M > ((int64_t)1 << 30)) return mortar_fail(MORTAR_ERR_ARG, "router stats: bad shape");
    if (n > 1024) return mortar_fail(MORTAR_ERR_LIMIT, "router stats: n=%d exceeds 1024 clusters", n);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int nb = (int)((M + ST_ROWS - 1) / ST_ROWS);
    float *part = static_cast<float *>(workspace);
    hipLaunchKernelGGL(router_stats_part_kernel, dim3((unsigned)nb), dim3(1024), 0, st, gates, M, n, part);
    hipLaunchKernelGGL(router_stats_final_kernel, dim3(1), dim3(1024), 0, st, part, nb, M, n, alpha, one_minus_alpha, coeff, ema, aux);
    return check_launch("router stats");
}
