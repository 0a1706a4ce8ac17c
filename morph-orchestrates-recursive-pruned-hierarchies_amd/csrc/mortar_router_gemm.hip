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
// times the cost of a bf16 one instead of the sixteen times of the fp32 matrix instructions (4096 x 2048 x 2048: 257 us
// through the library's fp32 GEMM with its conversion of x).
//
// A workgroup of NW waves owns MT tokens x 16 NW outputs; a wave owns 16 outputs for all MT tokens, so that a weight is
// loaded (straight from global memory in the MFMA operand order: 16 rows x 128 bytes per instruction) and split once per
// workgroup: 44 vector instructions per 3 MT / 16 MFMAs, hidden behind the matrix pipe from 128 tokens up.  The
// activations go through LDS in steps of 64 values, two buffers, one barrier per step; a fragment of 16 tokens x 32
// values is 1 KB in operand order, its 16-byte units swizzled (token ^ 4 * group) so that both the staging writes (4
// tokens x 4 units per 16 lanes) and the operand reads touch every bank once.
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

template <int MT, int NW>
__global__ void __launch_bounds__(NW * 64) router_gemm_kernel(const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, float *qv,
                                                              int64_t ldq, int n_ntiles) {
    constexpr int MI = MT / 16, FR = MI * 2, U = FR / NW, MG = MI < 8 ? MI : 8;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2][MT * RG_KS * 2];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    // ids are dealt round-robin over the 8 XCDs: each takes a run of tiles, so that its L2 serves the x rows of few token tiles
    const int per_xcd = (int)((gridDim.x + 7) >> 3);
    const int id = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int n_mtiles = (M + MT - 1) / MT;
    if (id >= n_mtiles * n_ntiles) return;
    const int m0 = (id / n_ntiles) * MT, o0 = (id % n_ntiles) * (16 * NW) + wave * 16;

    // staging role: fragment wave + NW * i, token lane >> 2, 16-byte unit lane & 3
    const uint16_t *xs[U];
    uint32_t dst[U];
    int ks[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int f = wave + NW * i, row = m0 + (f >> 1) * 16 + (lane >> 2), u = lane & 3;
        ks[i] = (f & 1) * 32 + u * 8;
        xs[i] = x + (int64_t)(row < M ? row : M - 1) * ldx + ks[i];
        dst[i] = (uint32_t)(f * 1024 + u * 256 + (((lane >> 2) ^ (4 * u)) * 16));
    }
    const int orow = o0 + n < N ? o0 + n : N - 1;
    const float *ws = W + (int64_t)orow * K + g * 8;
    const uint32_t rd = (uint32_t)(g * 256 + ((n ^ (4 * g)) * 16));

    u32x4_t xr[U];
    float4 wr[2][2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const bool in = k0 + ks[i] < K;                                   // K % 8 == 0: a unit is in or out as a whole
            xr[i] = *reinterpret_cast<const u32x4_t *>(xs[i] + (in ? k0 : -ks[i]));
            if (!in) xr[i] = u32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = k0 + h * 32 + g * 8 < K;
            const float4 *p = reinterpret_cast<const float4 *>(ws + (in ? k0 + h * 32 : -g * 8));
            wr[h][0] = p[0];
            wr[h][1] = p[1];
            if (!in) wr[h][0] = wr[h][1] = float4{0.f, 0.f, 0.f, 0.f};
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < U; ++i) *reinterpret_cast<u32x4_t *>(&lds[buf][dst[i]]) = xr[i];
    };
    f32x4_t acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    fetch(0);
    put(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += RG_KS) {
        float w[2][8];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                w[h][4 * j] = wr[h][j].x; w[h][4 * j + 1] = wr[h][j].y; w[h][4 * j + 2] = wr[h][j].z; w[h][4 * j + 3] = wr[h][j].w;
            }
        const bool more = k0 + RG_KS < K;
        if (more) fetch(k0 + RG_KS);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4_t p[3];
            split3(w[h], p);
#pragma unroll
            for (int i0 = 0; i0 < MI; i0 += MG) {
                u32x4_t b[MG];
#pragma unroll
                for (int i = 0; i < MG; ++i) b[i] = *reinterpret_cast<const u32x4_t *>(&lds[buf][((i0 + i) * 2 + h) * 1024 + rd]);
#pragma unroll
                for (int t = 2; t >= 0; --t)                                  // small terms first
#pragma unroll
                    for (int i = 0; i < MG; ++i) acc[i0 + i] = mortar_mfma(p[t], b[i], acc[i0 + i]);
            }
        }
        if (more) put(buf ^ 1);
        __syncthreads();
        buf ^= 1;
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

template <int MT, int NW>
void launch_gemm(const uint16_t *x, int M, int K, int64_t ldx, const float *W, int N, float *qv, int64_t ldq, hipStream_t st) {
    const int nt = (N + 16 * NW - 1) / (16 * NW), mt = (M + MT - 1) / MT;
    const unsigned grid = (unsigned)(((int64_t)mt * nt + 7) / 8 * 8);
    hipLaunchKernelGGL((router_gemm_kernel<MT, NW>), dim3(grid), dim3(NW * 64), 0, st, x, M, K, ldx, W, N, qv, ldq, nt);
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
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
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

extern "C" int mortar_router_project_bf16(const uint16_t *x, int64_t M, int32_t d_in, int64_t ldx, const float *wq, int32_t d_out, float *qv,
                                          int64_t ldq, void *stream) {
    if (!x || !wq || !qv) return mortar_fail(MORTAR_ERR_ARG, "router projection: null pointer");
    if (M <= 0 || M > (1 << 30) || d_in <= 0 || d_out <= 0 || d_in % 8 || d_out % 4 || ldx < d_in || ldx % 8 || ldq < d_out || ldq % 4)
        return mortar_fail(MORTAR_ERR_ARG, "router projection: M, d_in (a multiple of 8), d_out (of 4) and the leading dimensions must be positive and aligned");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(wq) | reinterpret_cast<uintptr_t>(qv)) & 15)
        return mortar_fail(MORTAR_ERR_ARG, "router projection: x, wq and qv must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Tokens per workgroup: the choice with the least rounds of 256 workgroups (one per CU) x work of a workgroup; a
    // workgroup costs its tokens plus the split of its weights, which weighs about 40 tokens.
    const int64_t nt8 = (d_out + 127) / 128;
    auto cost = [&](int mt) { return (((M + mt - 1) / mt * nt8 + 255) / 256) * (mt + 40); };
    const int64_t c256 = cost(256), c128 = cost(128), c64 = cost(64);
    if (c256 <= c128 && c256 <= c64) launch_gemm<256, 8>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    else if (c128 <= c64) launch_gemm<128, 8>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    else if ((M + 63) / 64 * nt8 > 128) launch_gemm<64, 8>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);
    else launch_gemm<64, 4>(x, (int)M, d_in, ldx, wq, d_out, qv, ldq, st);      // few tiles: half the outputs per workgroup, twice the workgroups
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
