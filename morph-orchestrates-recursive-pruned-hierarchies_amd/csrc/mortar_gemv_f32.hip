// Decode GEMV in the reference engine's arithmetic on a matrix with one scale, in ONE launch.
//
// mortar_gemv (morph/kernels/triton/fused_decode_step.py:1341-1459, 1502-1547): fp32 activations, exact +-x / 0 products, fp32
// sums, the fp32 scale after the sum, SwiGLU and gates in fp32.  The part-split decode kernel of mortar_spmm_core.h with
// another prologue and epilogue: an fp32 activation is split exactly into three bf16 terms while the tile is staged (row
// term * T + t of the tile is a term of token t), the blocks are contracted as +-2 / 0, and the epilogue adds the three sums
// of a token (columns of the accumulator, two lane exchanges), scales, and applies SwiGLU and gates.
// Three launches per product (split, SpMM on 3 B rows, combine) took 11.9 us of GPU time and 16 us of host time at 8 rows of
// the 2048 -> 11264 matrix; what they moved through memory between them is now in LDS and registers.  Where this form makes many
// rounds of workgroups (wide K, many rows) the three launches stay the faster one: mortar_gemv_f32_one_better.
#include "mortar_spmm_core.h"

namespace {

struct GemvOneArgs {
    const float *x, *scale, *gates;
    float *y;
    const int32_t *row_act, *col_act;
    int64_t ldx, ldy, ldg, ldr, ldc;
    int swiglu_x;
};

__device__ __forceinline__ float sigmoid_f32(float g) { return 1.0f / (1.0f + __expf(-g)); }

// T tokens per tile (3 T rows of 16 MFMA columns), PW waves share the parts of a unit, UW units per workgroup.  CS > 0: PW is CS times
// the number of parts and each wave takes a run of a part's octets, for launches that would leave half of the chip idle: latency bounds
// these, a wave's chain of batches first, so it is cut.  At d_model 2048, density 0.25, us, the whole parts against the cut ones: SwiGLU
// form 1 row 5.01 -> 4.32, 8 rows 5.32 -> 5.18; plain product over 5632 inputs 4.86 -> 3.91, 8 rows 6.85 -> 6.13.  A third of that is the
// grid of two dimensions and the staging without integer divisions, which the launches with whole parts share.
template <int T, int NACC, int PW, int UW, int CS>
__global__ void __launch_bounds__(PW * UW * 64) gemv_f32_one_kernel(const SpmmParams p0, const GemvOneArgs a) {
    constexpr int MT = 3 * T, WAVES = PW * UW, THREADS = WAVES * 64, CW = CS > 0 ? CS : 1;
    const SpmmView p = mortar_view(p0);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint4 *lx = reinterpret_cast<uint4 *>(smem);
    f32x4_t *red = reinterpret_cast<f32x4_t *>(smem + tile_bytes(MT, p.Cb));          // [WAVES][NACC][64]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4, bsel = g >> 1, hsel = g & 1;
    const int mt = blockIdx.y, sp = blockIdx.x;
    const int t0 = mt * T, nt = p.M - t0 < T ? p.M - t0 : T;                           // p.M counts tokens here
    const int ug = wave / PW, wq = wave % PW, pos = sp * UW + ug;
    const bool valid = pos < p.n_units;
    const int nparts = p.nseg * NACC;
    MortarBatch first;
    const int q0 = wq / CW;
    int d0 = 0, d1 = 0, dnb = 0;
    if (valid && q0 < nparts) {          // the first weights are on their way before the tile is staged
        const u32x4_t d = mortar_part_desc_scalar<NACC>(p, pos, q0);
        d0 = (int)d[0]; d1 = (int)d[1]; dnb = (int)d[2];
        if (CS > 0) {
            const int no = d1 - d0, c = wq % CW, lo = no * c / CW, hi = no * (c + 1) / CW;
            dnb = dnb - 8 * lo < 8 * (hi - lo) ? dnb - 8 * lo : 8 * (hi - lo);
            d1 = d0 + hi; d0 += lo;
        }
        if (d0 < d1) mortar_load_batch<CODE_UNIFORM>(p, first, d0, d1, n, bsel, hsel);
    }
    // what the epilogue reads besides the sums, requested early: the lane's gate and row flags (token n)
    const int tok = t0 + n;
    const bool mine = valid && n < nt;
    float gate = 1.f;
    int on_a = 1, on_b = 1;
    if (mine) {
        if (NACC == 2 && a.gates) gate = a.gates[(int64_t)tok * a.ldg + (pos * 16 + 4 * g) / p.cluster_size];
        if (a.row_act) {
            on_a = a.row_act[(int64_t)tok * a.ldr + pos];
            if (NACC == 2) on_b = a.row_act[(int64_t)tok * a.ldr + p.n_units + pos];
        }
    }
    const float scale = a.scale[0];

    // stage: item = (token, 8 consecutive inputs)
    const int K = p.Cb * 16, nch = K / 8;
    for (int i0 = tid; i0 < nt * nch; i0 += 4 * THREADS) {
        float4 q[4][2];
        int off[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * THREADS;
            if (i >= nt * nch) break;
            int t = 0;
#pragma unroll
            for (int k = 1; k < T; ++k) t += i >= k * nch;               // i / nch without the forty instructions of a division
            const int c = i - t * nch;
            const float4 *src = reinterpret_cast<const float4 *>(a.x + (int64_t)(t0 + t) * a.ldx + c * 8);
            q[u][0] = src[0];
            q[u][1] = src[1];
            if (a.swiglu_x) {
                const float4 u0 = src[K / 4], u1 = src[K / 4 + 1];
                float4 &f = q[u][0], &h = q[u][1];
                f = float4{f.x * sigmoid_f32(f.x) * u0.x, f.y * sigmoid_f32(f.y) * u0.y, f.z * sigmoid_f32(f.z) * u0.z, f.w * sigmoid_f32(f.w) * u0.w};
                h = float4{h.x * sigmoid_f32(h.x) * u1.x, h.y * sigmoid_f32(h.y) * u1.y, h.z * sigmoid_f32(h.z) * u1.z, h.w * sigmoid_f32(h.w) * u1.w};
            }
            if (a.col_act && a.col_act[(int64_t)(t0 + t) * a.ldc + (c >> 1)] == 0) q[u][0] = q[u][1] = float4{0.f, 0.f, 0.f, 0.f};
            off[u] = (c >> 1) * (MT * 32) + t * 32 + (c & 1) * 16;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i0 + u * THREADS >= nt * nch) break;
            const float v[8] = {q[u][0].x, q[u][0].y, q[u][0].z, q[u][0].w, q[u][1].x, q[u][1].y, q[u][1].z, q[u][1].w};
            u32x4_t hi, mid, lo;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                hi[k] = bf16_pack2(v[2 * k], v[2 * k + 1]);
                const float r0 = v[2 * k] - bf16_to_f32(hi[k] & 0xffffu), r1 = v[2 * k + 1] - bf16_to_f32(hi[k] >> 16);
                mid[k] = bf16_pack2(r0, r1);
                lo[k] = bf16_pack2(r0 - bf16_to_f32(mid[k] & 0xffffu), r1 - bf16_to_f32(mid[k] >> 16));
            }
            *reinterpret_cast<u32x4_t *>(smem + off[u]) = hi;
            *reinterpret_cast<u32x4_t *>(smem + off[u] + T * 32) = mid;
            *reinterpret_cast<u32x4_t *>(smem + off[u] + 2 * T * 32) = lo;
        }
    }
    __syncthreads();
    // a unit whose rows are off, or whose gate is zero, for every token of the tile multiplies nothing
    const bool work = valid && __ballot(mine && gate != 0.f && (on_a != 0 || (NACC == 2 && on_b != 0))) != 0ull;

    f32x4_t acc[NACC][1];
#pragma unroll
    for (int b = 0; b < NACC; ++b) acc[b][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t tk[1] = {(uint32_t)n};
    if constexpr (CS > 0) {
        if (work && d0 < d1)
            mortar_row_part<1, MT, false, CODE_UNIFORM>(p, lx, first, d0, d1, dnb, (uint32_t)(hsel * 16 + n * 32) + (uint32_t)(q0 / NACC * p.seg_cb) * (uint32_t)(MT * 32),
                                                        tk, 1, n, bsel, hsel, acc[0]);
        red[wave * 64 + lane] = acc[0][0];
        __syncthreads();
        if (wq != 0) return;
        acc[0][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < PW; ++w) acc[w / CW % NACC][0] += red[(wave + w) * 64 + lane];
    } else if (work) {
        for (int sg = 0; sg < p.nseg; ++sg) {
            const uint32_t xo = (uint32_t)(hsel * 16 + n * 32) + (uint32_t)(sg * p.seg_cb) * (uint32_t)(MT * 32);
#pragma unroll
            for (int b = 0; b < NACC; ++b) {
                const int q = sg * NACC + b;
                if (q % PW != wq) continue;
                int g0 = d0, g1 = d1, nb = dnb;
                if (q != wq) {
                    const u32x4_t dq = mortar_part_desc<NACC>(p, pos, sg, b);
                    g0 = __builtin_amdgcn_readfirstlane((int)dq[0]); g1 = __builtin_amdgcn_readfirstlane((int)dq[1]);
                    nb = __builtin_amdgcn_readfirstlane((int)dq[2]);
                }
                if (g0 >= g1) continue;
                if (q != wq) mortar_load_batch<CODE_UNIFORM>(p, first, g0, g1, n, bsel, hsel);
                mortar_row_part<1, MT, false, CODE_UNIFORM>(p, lx, first, g0, g1, nb, xo, tk, 1, n, bsel, hsel, acc[b]);
            }
        }
    }
    if (PW > 1 && CS == 0) {
#pragma unroll
        for (int b = 0; b < NACC; ++b) red[(wave * NACC + b) * 64 + lane] = acc[b][0];
        __syncthreads();
        if (wq != 0) return;
#pragma unroll
        for (int w = 1; w < PW; ++w)
#pragma unroll
            for (int b = 0; b < NACC; ++b) acc[b][0] += red[((wave + w) * NACC + b) * 64 + lane];
    }
    if (!valid) return;
    // columns n, n + T and n + 2 T of the accumulator are the three terms of token n
    f32x4_t r[NACC];
#pragma unroll
    for (int b = 0; b < NACC; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float m = __shfl(acc[b][0][v], lane + T, 64), l = __shfl(acc[b][0][v], lane + 2 * T, 64);
            r[b][v] = scale * (0.5f * ((acc[b][0][v] + m) + l));
        }
    if (!mine) return;
    if (!on_a) r[0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (NACC == 2) {
        if (!on_b) r[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            r[0][v] = r[0][v] * sigmoid_f32(r[0][v]) * r[1][v];
            if (a.gates) r[0][v] *= gate;
        }
    }
    *reinterpret_cast<f32x4_t *>(a.y + (int64_t)tok * a.ldy + pos * 16 + 4 * g) = r[0];
}

int one_lds(int t, int nacc, int pw, int Cb) { return tile_bytes(3 * t, Cb) + (pw > 1 ? pw * 4 * nacc * 1024 : 0); }

struct OneShape { int t, pw; };        // tokens per tile (0: none fits), waves per unit

OneShape one_shape(const mortar_bcsr_t *W, int mode, int B) {
    const int seg = W->seg_cb < W->Cb ? W->seg_cb : W->Cb, nacc = mode + 1, nparts = (W->Cb + seg - 1) / seg * nacc;
    // waves per unit: a divisor of the part count where there is one (as the bf16 part-split launches)
    const int pw = nparts == 1 ? 1 : nparts % 4 == 0 ? 4 : nparts % 3 == 0 ? 3 : nparts % 2 == 0 ? 2 : (nparts + 3) / 4 < (nparts + 2) / 3 ? 4 : 3;
    // tokens per tile: all of them where they fit (at most five: 15 of the MFMA's 16 columns), else the most that LDS takes
    int t = 0;
    for (int c : {1, 2, 4, 5})
        if (one_lds(c, nacc, pw, W->Cb) <= 160 * 1024) { t = c; if (c >= B) break; }
    return {t, pw};
}

template <int T, int NACC, int PW, int UW, int CS>
int launch_one(SpmmParams &p, const GemvOneArgs &a, hipStream_t st) {
    const int smem = tile_bytes(3 * T, p.Cb) + (PW > 1 ? PW * UW * (CS > 0 ? 1 : NACC) * 1024 : 0);
    static bool done = false;
    int rc = mortar_allow_big_lds(gemv_f32_one_kernel<T, NACC, PW, UW, CS>, done);
    if (rc) return rc;
    p.n_mtiles = (p.M + T - 1) / T;
    p.n_split = (p.n_units + UW - 1) / UW;
    if ((rc = mortar_launch_check(p.n_split, p.n_mtiles))) return rc;
    hipLaunchKernelGGL((gemv_f32_one_kernel<T, NACC, PW, UW, CS>), dim3((unsigned)p.n_split, (unsigned)p.n_mtiles), dim3(PW * UW * 64), smem, st, p, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "gemv_f32 launch: %s", hipGetErrorString(e));
    return MORTAR_OK;
}

// Few units: as many waves per unit as the part-split launches of mortar_smallm_chunk.hip take, in workgroups of one or two units while
// they are one round of the chip.  -1: no such form, or no need of one.
template <int T, int NACC>
int launch_chunk(SpmmParams &p, const GemvOneArgs &a, hipStream_t st) {
    const int nparts = p.nseg * NACC;
    for (int uw : {1, 2}) {
        if ((int64_t)((p.M + T - 1) / T) * ((p.n_units + uw - 1) / uw) > 256) continue;
        for (int cs : {4, 2}) {
            const int pw = nparts * cs;
            if ((cs == 4 && p.avg_octets < 4) || tile_bytes(3 * T, p.Cb) + pw * uw * 1024 > 160 * 1024) continue;
            switch (uw * 1000 + pw * 10 + cs) {
                case 1082: return launch_one<T, NACC, 8, 1, 2>(p, a, st);
                case 1084: return launch_one<T, NACC, 8, 1, 4>(p, a, st);
                case 1122: return launch_one<T, NACC, 12, 1, 2>(p, a, st);
                case 1124: return launch_one<T, NACC, 12, 1, 4>(p, a, st);
                case 2042: return launch_one<T, NACC, 4, 2, 2>(p, a, st);
                case 2044: return launch_one<T, NACC, 4, 2, 4>(p, a, st);
                case 2062: return launch_one<T, NACC, 6, 2, 2>(p, a, st);
                case 2082: return launch_one<T, NACC, 8, 2, 2>(p, a, st);
                case 2084: return launch_one<T, NACC, 8, 2, 4>(p, a, st);
            }
        }
    }
    return -1;
}

template <int T, int NACC>
int launch_pw(int pw, SpmmParams &p, const GemvOneArgs &a, hipStream_t st) {
    const int rc = launch_chunk<T, NACC>(p, a, st);
    if (rc >= 0) return rc;
    switch (pw) {
        case 1: return launch_one<T, NACC, 1, 4, 0>(p, a, st);
        case 2: return launch_one<T, NACC, 2, 4, 0>(p, a, st);
        case 3: return launch_one<T, NACC, 3, 4, 0>(p, a, st);
    }
    return launch_one<T, NACC, 4, 4, 0>(p, a, st);
}

template <int NACC>
int launch_t(int t, int pw, SpmmParams &p, const GemvOneArgs &a, hipStream_t st) {
    // The plain product takes the smallest tile that still is one round of the chip: a workgroup stages its tokens' fp32 values of all K,
    // which costs more than the weights read by another tile (5632 inputs, 2048 outputs, 4 rows in tiles of 4 / 2 / 1 tokens 5.8 / 4.3 / - us,
    // 8 rows 6.1 / 4.7 / -; 4096 inputs, 1536 outputs, 4 rows 5.1 / 4.1).  The SwiGLU form reads twice the weights of a narrower tile:
    // d_model 1536, 4 rows 4.6 -> 4.2 at density 0.25, but 2 rows at 0.5 4.1 -> 4.7.
    if (NACC == 1) {
        int rc = t > 1 ? launch_chunk<1, NACC>(p, a, st) : -1;
        if (rc < 0 && t > 2) rc = launch_chunk<2, NACC>(p, a, st);
        if (rc >= 0) return rc;
    }
    switch (t) {
        case 1: return launch_pw<1, NACC>(pw, p, a, st);
        case 2: return launch_pw<2, NACC>(pw, p, a, st);
        case 4: return launch_pw<4, NACC>(pw, p, a, st);
    }
    return launch_pw<5, NACC>(pw, p, a, st);
}

}  // namespace

// Every workgroup stages its tile of all K again, and few tokens fit one where K is wide: a round of workgroups costs 5 us (as
// many per CU as LDS holds), while the three launches of mortar_gemv_f32 grow slowly with the rows.  They meet at three rounds
// for the SwiGLU form (d_model 3072, 24 rows: 16.0 against 15.6 us, 64 rows 35 against 22; 4096, 16 rows 17.9 against 21.4, 64 rows
// 51 against 33) and at four for the plain product (11008 inputs, 32 rows: 26.8 against 31.2, 64 rows 50 against 32.5; 22016 inputs,
// 8 rows 26.5 against 31.6, 64 rows 192 against 50).
extern "C" int mortar_gemv_f32_one_better(const mortar_bcsr_t *W, int32_t mode, int32_t B) {
    if (!W || W->Rb <= 0 || W->Cb <= 0 || W->seg_cb <= 0 || B <= 0 || B > 64 || (mode != 0 && mode != 1)) return 0;
    const OneShape s = one_shape(W, mode, B);
    if (s.t == 0) return 0;
    const int units = mode == 0 ? W->Rb : W->Rb / 2, lds = one_lds(s.t, mode + 1, s.pw, W->Cb);
    const int by_lds = 160 * 1024 / lds, by_waves = 32 / (4 * s.pw), per_cu = by_lds < by_waves ? by_lds : by_waves;
    const int64_t wgs = (int64_t)((B + s.t - 1) / s.t) * ((units + 3) / 4), rounds = (wgs + 256 * per_cu - 1) / (256 * per_cu);
    return rounds <= (mode == 0 ? 4 : 3);
}

extern "C" int mortar_gemv_f32_one(const mortar_bcsr_t *W, const float *scale, int32_t mode, int32_t swiglu_x, const float *x, int32_t B,
                                   int64_t ldx, float *y, int64_t ldy, const float *gates, int32_t n_clusters, int64_t ldg,
                                   const int32_t *row_act, int64_t ldr, const int32_t *col_act, int64_t ldc, void *stream) {
    if (!W || !W->row_desc || !W->codes_o || !W->col_o || !scale || !x || !y) return mortar_fail(MORTAR_ERR_ARG, "gemv_f32_one: null pointer");
    if (B <= 0 || B > 64) return mortar_fail(MORTAR_ERR_LIMIT, "gemv_f32_one: B=%d outside 1..64", B);
    if (mode != 0 && mode != 1) return mortar_fail(MORTAR_ERR_ARG, "gemv_f32_one: mode must be 0 or 1");
    if (W->Rb <= 0 || W->Cb <= 0 || W->nnz <= 0 || W->seg_cb <= 0 || (mode == 1 && (W->Rb & 1)))
        return mortar_fail(MORTAR_ERR_ARG, "gemv_f32_one: bad matrix");
    const int too_large = mortar_check_octets(W);
    if (too_large) return too_large;
    const int64_t nout = mode == 0 ? (int64_t)W->Rb * 16 : (int64_t)W->Rb * 8, need = (int64_t)W->Cb * 16 * (swiglu_x ? 2 : 1);
    if (ldx < need || (B > 1 && ldx % 4) || ldy < nout || ldy % 4 || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15))
        return mortar_fail(MORTAR_ERR_ARG, "gemv_f32_one: bad leading dimension or alignment (rows 16-byte aligned)");
    if (gates && (mode != 1 || n_clusters <= 0 || nout % n_clusters || (nout / n_clusters) % 4))
        return mortar_fail(MORTAR_ERR_ARG, "gemv_f32_one: gates need mode 1 and d_ff / n_clusters a whole multiple of 4");
    SpmmParams p{};
    p.row_desc = reinterpret_cast<const u32x4_t *>(W->row_desc);
    p.codes_o = reinterpret_cast<const u32x4_t *>(W->codes_o);
    p.sd_o = reinterpret_cast<const u32x4_t *>(W->sd_o);
    p.col_o = reinterpret_cast<const u32x4_t *>(W->col_o);
    p.seg_cb = W->seg_cb < W->Cb ? W->seg_cb : W->Cb;
    p.nseg = (W->Cb + p.seg_cb - 1) / p.seg_cb;
    p.Rb = W->Rb; p.Cb = W->Cb; p.M = B;
    p.avg_octets = (int)(((int64_t)W->nnz + 8 * (int64_t)W->Rb * p.nseg - 1) / (8 * (int64_t)W->Rb * p.nseg));
    p.n_units = mode == 0 ? W->Rb : W->Rb / 2;
    p.n_clusters = 1; p.cluster_size = gates ? (int)(nout / n_clusters) : 1 << 30;
    const OneShape sh = one_shape(W, mode, B);
    if (sh.t == 0) return MORTAR_NO_KERNEL;
    const GemvOneArgs a{x, scale, gates, y, row_act, col_act, ldx, ldy, ldg, ldr, ldc, swiglu_x != 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    return mode == 0 ? launch_t<1>(sh.t, sh.pw, p, a, st) : launch_t<2>(sh.t, sh.pw, p, a, st);
}
