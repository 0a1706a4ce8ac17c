// Device-side re-pack: ternarise block values and rewrite a matrix's code and scale arrays in place.
//
// The reference ternarises carved blocks in torch (deploy_quant.py:81-95 for the deploy pack,
// block_sparse.py:909-919 on every QAT forward: scale = mean|w|, q = sign(w/s) * (|w/s| > threshold)) and keeps the
// transposed topology for the dX product as index arrays over the same data (stk matrix.py:107-125).  Here the
// topology of a pack (columns, offsets, octet positions) is fixed once on the host, and this kernel refreshes the
// values: a wavefront reads four blocks (optionally other blocks, transposed: the dX pack), forms the scale, and writes the row
// dwords into `codes`, the octet stream and its 4-bit copy.
#include <hip/hip_runtime.h>

#include "mortar_device.h"
#include "mortar_internal.h"

#include <type_traits>

namespace {

constexpr int PARTIALS = 256;           // workgroups of the |w| reduction; the workspace holds one double each

// sum |w| over all values -> partial[blockIdx] (fixed order: the result does not depend on timing).  n is a multiple
// of 256 (whole blocks) and the array is 16-byte aligned, so every thread reads 16-byte pieces.
struct AbsSumArgs {
    const void *values;
    double *partial;
    int64_t n;
    int f32;
};
constexpr int MAX_JOBS = 4;
struct AbsSumJobs { AbsSumArgs job[MAX_JOBS]; };

__device__ __forceinline__ void abs_sum(const void *values, int64_t n, int f32, double *partial) {
    __shared__ double wsum[4];
    double s = 0.0;
    const int per = f32 ? 4 : 8;                                     // values per 16-byte piece
    const uint4 *v = reinterpret_cast<const uint4 *>(values);
    auto add = [&](uint4 q) {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (f32) {
                s += (double)fabsf(__uint_as_float(w[e]));
            } else {
                s += (double)fabsf(__uint_as_float(w[e] << 16));
                s += (double)fabsf(__uint_as_float(w[e] & 0xffff0000u));
            }
        }
    };
    // eight pieces in flight per thread: with one wave per SIMD, a load per turn of the loop waits out its latency
    constexpr int64_t STEP = (int64_t)PARTIALS * 256;
    const int64_t m = n / per;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < m; i += 8 * STEP) {
        uint4 q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = v[i + u * STEP < m ? i + u * STEP : i];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i + u * STEP < m) add(q[u]);
    }
    s = mortar_wave_sum(s);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}
__global__ __launch_bounds__(256) void abs_sum_kernel(AbsSumJobs a) {
    const AbsSumArgs &j = a.job[blockIdx.y];
    abs_sum(j.values, j.n, j.f32, j.partial);
}

__global__ void clear_status_kernel(int32_t *status) {
    if (threadIdx.x < 2) status[threadIdx.x] = 0;
}

struct RequantArgs {
    uint32_t *codes, *sdup, *codes_o, *sd_o, *codes4_o;
    const void *values;
    const int32_t *pos, *src_block;
    const float *scale_in;
    float *scale_out;
    int32_t *status;
    const double *partial;
    int32_t nnz, f32, transpose, mode;
    float threshold;
    float ternary_tol;      // > 0: with a given scale, flag values that are neither 0 nor +-s within this relative bound
};

// The smallest float c > 0 with RN(c / s) > threshold, so that |w / s| > threshold is |w| >= c without a division per value (the
// rounded quotient does not fall as w grows).  Lane l tries the float l - 32 steps from threshold * s; false when the change does not lie
// between those (a quotient that underflows), and the caller divides.
__device__ __forceinline__ bool code_cut(float s, float threshold, int lane, float &cut) {
    const int b = (int)__float_as_uint(threshold * s) + lane - 32;
    const float c = __uint_as_float(b > 0 ? (uint32_t)b : 0u);
    const uint64_t above = __ballot(c / s > threshold);
    cut = __shfl(c, above ? __builtin_ctzll(above) : 0);
    return above != 0 && (above & 1) == 0 && (above & (above + (above & -above))) == 0 && (above >> 63) != 0;
}

// mode 0: one scale per matrix from the partial sums, 1: one per block, 2: scale_in[0], 3: scale_in[source block].
// A wavefront takes four blocks, a lane one row of one of them: 32 or 64 bytes of values in, and one dword for each of the arrays out.
// One wave per block with the quotients of four values per lane was bound by its vector instructions (gate_up and down at
// 2048 x 5632 and 25 %, both orientations: 12.5 us on average): a row is encoded by one comparison per value, and a transposed
// block is turned as 16 x 16 two-bit codes in registers, four exchanges between the 16 lanes of a block (now 6.6 us).
__device__ __forceinline__ void requant(const RequantArgs &a, int block) {
    const int lane = threadIdx.x & 63, n = lane & 15;
    const int j0 = (block * 4 + (threadIdx.x >> 6)) * 4, j = j0 + (lane >> 4);
    if (j0 >= a.nnz) return;
    const bool on = j < a.nnz;
    const int jc = on ? j : a.nnz - 1;
    const int src = a.src_block ? a.src_block[jc] : jc;
    const int P = a.pos[jc];
    float w[16];
    if (a.f32) {
        const float4 *v = reinterpret_cast<const float4 *>(a.values) + (int64_t)src * 64 + n * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float4 x = v[e];
            w[4 * e] = x.x; w[4 * e + 1] = x.y; w[4 * e + 2] = x.z; w[4 * e + 3] = x.w;
        }
    } else {
        const uint4 *v = reinterpret_cast<const uint4 *>(a.values) + (int64_t)src * 32 + n * 2;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint4 x = v[e];
            const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w[8 * e + 2 * k] = __uint_as_float(u[k] << 16);
                w[8 * e + 2 * k + 1] = __uint_as_float(u[k] & 0xffff0000u);
            }
        }
    }
    float s;
    if (a.mode == 0) {
        const double t = mortar_wave_sum((a.partial[lane] + a.partial[lane + 64]) + (a.partial[lane + 128] + a.partial[lane + 192]));
        s = fmaxf((float)(t / ((double)a.nnz * 256.0)), 1e-8f);
    } else if (a.mode == 1) {
        double t[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            t[q] = ((double)fabsf(w[4 * q]) + (double)fabsf(w[4 * q + 1])) + ((double)fabsf(w[4 * q + 2]) + (double)fabsf(w[4 * q + 3]));
            t[q] += mortar_row_xor<8>(t[q]);
            t[q] += mortar_row_xor<4>(t[q]);
            t[q] += mortar_row_xor<2>(t[q]);
            t[q] += mortar_row_xor<1>(t[q]);
        }
        s = fmaxf((float)(((t[0] + t[2]) + (t[1] + t[3])) * (1.0 / 256.0)), 1e-6f);
    } else {
        s = a.scale_in[a.mode == 2 ? 0 : src];
    }
    // scale pattern: bf16(s) one exponent step down, in both halves (0 zeroes the block)
    uint32_t u = __float_as_uint(s);
    uint32_t sb = (u & 0x7fffffffu) > 0x7f800000u ? 0x7fc0u : ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
    uint32_t sd = 0;
    if ((sb & 0x7fffu) != 0) {
        const uint32_t e8 = (sb >> 7) & 0xffu;
        if (e8 < 27 || e8 > 227) {
            if (on && n == 0 && a.status) a.status[0] = 1;
        } else {
            const uint32_t adj = sb - 0x0400u;
            sd = adj | (adj << 16);
        }
    }
    if (a.ternary_tol > 0.f && a.status) {
        // every value must be 0 or +-s up to the bound (a bf16 cast of +-s(1 + rounding) may land one step beside bf16(s))
        bool bad = false;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float m = fabsf(w[e]);
            bad = bad || !(m <= a.ternary_tol * s || fabsf(m - s) <= a.ternary_tol * s);
        }
        if (on && bad) a.status[1] = 1;
    }
    // two bits per value in column order: 1 = +, 3 = -
    uint32_t row = 0;
    float cut;
    const uint32_t flip = u & 0x80000000u;                       // a given scale may be negative
    if (!(a.mode & 1) && code_cut(fabsf(s), a.threshold, lane, cut)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t enc = 1u | ((__float_as_uint(w[e]) ^ flip) >> 30 & 2u);
            row |= (fabsf(w[e]) >= cut ? enc : 0u) << (2 * e);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float wn = w[e] / s;
            row |= (fabsf(wn) > a.threshold && wn != 0.f ? (wn < 0.f ? 3u : 1u) : 0u) << (2 * e);
        }
    }
    if (sd == 0) row = 0;
    if (a.transpose) {                                  // 16 x 16 codes across the 16 lanes of the block
        auto turn = [&](auto distance, int bits, uint32_t low) {        // swaps the off-diagonal halves of every 2 o x 2 o square
            constexpr int o = decltype(distance)::value;
            const uint32_t other = mortar_row_xor<o>(row);
            row = (n & o) ? (row & ~low) | ((other & ~low) >> bits) : (row & low) | ((other & low) << bits);
        };
        turn(std::integral_constant<int, 8>{}, 16, 0x0000ffffu);
        turn(std::integral_constant<int, 4>{}, 8, 0x00ff00ffu);
        turn(std::integral_constant<int, 2>{}, 4, 0x0f0f0f0fu);
        turn(std::integral_constant<int, 1>{}, 2, 0x33333333u);
    }
    // device order of a row: column c < 8 in field 2 c + 1, column c >= 8 in field 2 (c - 8)
    auto spread = [](uint32_t x) {
        x = (x | (x << 8)) & 0x00ff00ffu;
        x = (x | (x << 4)) & 0x0f0f0f0fu;
        return (x | (x << 2)) & 0x33333333u;
    };
    row = (spread(row & 0xffffu) << 2) | spread(row >> 16);
    if (!on) return;
    a.codes[(int64_t)j * 16 + n] = row;
    a.codes_o[(int64_t)(P >> 2) * 64 + n * 4 + (P & 3)] = row;
    if (a.codes4_o) {
        const int64_t o4 = (((int64_t)(P >> 3) * 4 + 2 * ((P >> 2) & 1)) * 16 + n) * 4 + (P & 3);
        a.codes4_o[o4] = row & 0xCCCCCCCCu;
        a.codes4_o[o4 + 64] = (row << 2) & 0xCCCCCCCCu;
    }
    if (n == 0) {
        a.sdup[j] = sd;
        a.sd_o[P] = sd;
        if (a.scale_out) a.scale_out[(a.mode == 0 || a.mode == 2) ? 0 : j] = s;
    }
}

// Several matrices in one launch (a training step re-packs two and their transposes, launches of 4 to 11 us each that the latency of a
// few dependent loads bounds: 2 + 4 launches 36 us, one of each kind 17 us at 2048 x 5632 and 25 %): workgroups [first[i], first[i + 1]) take the blocks of job i.
struct RequantJobs {
    RequantArgs job[MAX_JOBS];
    int first[MAX_JOBS + 1];
};
__global__ __launch_bounds__(256) void requant_kernel(RequantJobs a) {
    int i = 0;
#pragma unroll
    for (int k = 1; k < MAX_JOBS; ++k) i += (int)blockIdx.x >= a.first[k];
    requant(a.job[i], (int)blockIdx.x - a.first[i]);
}

// Fills one job from a matrix; the scale comes from `partial` (mode 0) until the caller says otherwise.
RequantArgs requant_args(const mortar_bcsr_t *W, const void *values, int32_t f32, const int32_t *pos, const int32_t *src_block,
                         int32_t transpose, float threshold, int32_t *status, const void *partial) {
    RequantArgs a{};
    a.codes = const_cast<uint32_t *>(W->codes);
    a.sdup = const_cast<uint32_t *>(W->sdup);
    a.codes_o = const_cast<uint32_t *>(W->codes_o);
    a.sd_o = const_cast<uint32_t *>(W->sd_o);
    a.codes4_o = const_cast<uint32_t *>(W->codes4_o);
    a.values = values;
    a.pos = pos;
    a.src_block = src_block;
    a.status = status;
    a.partial = static_cast<const double *>(partial);
    a.nnz = W->nnz;
    a.f32 = f32;
    a.transpose = transpose;
    a.threshold = threshold;
    return a;
}

// Launches the |w| sums of `ns` value arrays and the re-pack of `n` matrices.
int launch_requant(const AbsSumJobs &sums, int ns, RequantJobs &jobs, int n, hipStream_t st) {
    if (ns > 0) hipLaunchKernelGGL(abs_sum_kernel, dim3(PARTIALS, ns), dim3(256), 0, st, sums);
    jobs.first[0] = 0;
    for (int i = 0; i < MAX_JOBS; ++i) {
        if (i < n) jobs.first[i + 1] = jobs.first[i] + (jobs.job[i].nnz + 15) / 16;
        else jobs.first[i + 1] = INT32_MAX;
    }
    hipLaunchKernelGGL(requant_kernel, dim3(jobs.first[n]), dim3(256), 0, st, jobs);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "requantize: %s", hipGetErrorString(e));
    return MORTAR_OK;
}

int check_requant(const mortar_bcsr_t *W, const void *values, const int32_t *pos, float threshold) {
    if (!W || !values || !pos) return mortar_fail(MORTAR_ERR_ARG, "requantize: null pointer");
    if (!W->codes || !W->sdup || !W->codes_o || !W->sd_o || W->nnz <= 0) return mortar_fail(MORTAR_ERR_ARG, "requantize: incomplete matrix");
    if (!(threshold >= 0.f)) return mortar_fail(MORTAR_ERR_ARG, "requantize: threshold must be >= 0");
    if (reinterpret_cast<uintptr_t>(values) & 15) return mortar_fail(MORTAR_ERR_ARG, "requantize: values must be 16-byte aligned");
    return MORTAR_OK;
}

// Overwrites out[0..ndw) with quiet-NaN patterns (0x7FC07FC0: NaN as two bf16 and as one fp32) when a status word is set.
// Every thread reads the two words; the usual case (both 0) ends after that one load.
__global__ __launch_bounds__(256) void poison_kernel(uint32_t *out, int64_t ndw, const int32_t *status) {
    if ((status[0] | status[1]) == 0) return;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < ndw; i += (int64_t)gridDim.x * 256) out[i] = 0x7FC07FC0u;
}

}  // namespace

extern "C" int mortar_poison_on_status(void *out, int64_t bytes, const int32_t *status, void *stream) {
    if (!out || !status) return mortar_fail(MORTAR_ERR_ARG, "poison_on_status: null pointer");
    if (bytes < 0 || (bytes & 3) || (reinterpret_cast<uintptr_t>(out) & 3))
        return mortar_fail(MORTAR_ERR_ARG, "poison_on_status: out must be 4-byte aligned and a multiple of 4 bytes long");
    if (bytes == 0) return MORTAR_OK;
    const int64_t ndw = bytes / 4;
    const int grid = (int)(ndw / 256 < 1 ? 1 : (ndw / 256 > 1024 ? 1024 : ndw / 256));
    hipLaunchKernelGGL(poison_kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<uint32_t *>(out), ndw, status);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "poison_on_status: %s", hipGetErrorString(e));
    return MORTAR_OK;
}

extern "C" int64_t mortar_requantize_workspace_bytes(void) { return (int64_t)PARTIALS * sizeof(double); }

extern "C" int mortar_requantize(const mortar_bcsr_t *W, const void *values, int32_t values_f32, const int32_t *pos,
                                 const int32_t *src_block, int32_t transpose, int32_t scale_mode, float threshold,
                                 const float *scale_in, float *scale_out, int32_t *status, int32_t flags,
                                 float ternary_tol, void *workspace, void *stream) {
    const int rc = check_requant(W, values, pos, threshold);
    if (rc) return rc;
    if (scale_mode < 0 || scale_mode > 3) return mortar_fail(MORTAR_ERR_ARG, "requantize: scale_mode %d not in 0..3", scale_mode);
    if (scale_mode >= 2 && !scale_in) return mortar_fail(MORTAR_ERR_ARG, "requantize: scale_mode %d needs scale_in", scale_mode);
    if (scale_mode == 0 && !workspace) return mortar_fail(MORTAR_ERR_ARG, "requantize: scale_mode 0 needs the workspace");
    if (flags & ~1) return mortar_fail(MORTAR_ERR_ARG, "requantize: unknown flags 0x%x", flags);
    if (!(ternary_tol >= 0.f) || (ternary_tol > 0.f && (scale_mode < 2 || !status)))
        return mortar_fail(MORTAR_ERR_ARG, "requantize: ternary_tol needs a given scale (scale_mode 2 or 3) and a status word");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (status && !(flags & 1)) hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(64), 0, st, status);
    AbsSumJobs sums{};
    sums.job[0] = {values, static_cast<double *>(workspace), (int64_t)W->nnz * 256, values_f32};
    RequantJobs jobs{};
    RequantArgs &a = jobs.job[0] = requant_args(W, values, values_f32, pos, src_block, transpose, threshold, status, workspace);
    a.scale_in = scale_in;
    a.scale_out = scale_out;
    a.mode = scale_mode;
    a.ternary_tol = ternary_tol;
    return launch_requant(sums, scale_mode == 0, jobs, 1, st);
}

extern "C" int mortar_requantize_pairs(const mortar_repack_t *m, int32_t n, void *stream) {
    if (!m || n < 1 || 2 * n > MAX_JOBS) return mortar_fail(MORTAR_ERR_ARG, "requantize_pairs: 1 to %d matrices", MAX_JOBS / 2);
    AbsSumJobs sums{};
    RequantJobs jobs{};
    int nj = 0;
    for (int i = 0; i < n; ++i) {
        int rc = check_requant(m[i].W, m[i].values, m[i].pos, m[i].threshold);
        if (rc == MORTAR_OK && m[i].Wt) rc = check_requant(m[i].Wt, m[i].values, m[i].pos_t, m[i].threshold);
        if (rc) return rc;
        if (!m[i].workspace || (m[i].Wt && (!m[i].src_t || m[i].Wt->nnz != m[i].W->nnz)))
            return mortar_fail(MORTAR_ERR_ARG, "requantize_pairs: matrix %d: workspace missing, or W^T does not match W", i);
        for (int k = 0; k < i; ++k) {        // both sums are under way at once
            const int64_t apart = static_cast<const char *>(m[i].workspace) - static_cast<const char *>(m[k].workspace);
            if (apart < mortar_requantize_workspace_bytes() && -apart < mortar_requantize_workspace_bytes())
                return mortar_fail(MORTAR_ERR_ARG, "requantize_pairs: matrices %d and %d share a workspace", k, i);
        }
        sums.job[i] = {m[i].values, static_cast<double *>(m[i].workspace), (int64_t)m[i].W->nnz * 256, m[i].values_f32};
        jobs.job[nj] = requant_args(m[i].W, m[i].values, m[i].values_f32, m[i].pos, nullptr, 0, m[i].threshold, m[i].status, m[i].workspace);
        jobs.job[nj++].scale_out = m[i].scale_out;
        if (m[i].Wt)
            jobs.job[nj++] = requant_args(m[i].Wt, m[i].values, m[i].values_f32, m[i].pos_t, m[i].src_t, 1, m[i].threshold, m[i].status_t, m[i].workspace);
    }
    return launch_requant(sums, n, jobs, nj, static_cast<hipStream_t>(stream));
}
