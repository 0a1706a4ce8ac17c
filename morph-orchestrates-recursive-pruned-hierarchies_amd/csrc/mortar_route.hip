// ReMoE gating tail, active-token compaction, decode gather flags and RMSNorm.
//
//   mortar_remoe_gates   TileRouter.forward steps 5-8 (morph/model/routing.py:232-284; single-token
//                        form morph/kernels/triton/fused_router.py:88-97)
//   mortar_remoe_route   per (token tile, cluster) compacted list of active tokens (wavefront ballot)
//   mortar_route_flags   morph/kernels/triton/fused_decode_step.py:1883-1927
//   mortar_rmsnorm_bf16  morph/model/attention.py:133-141
#include "mortar_device.h"
#include "mortar_internal.h"

#include <type_traits>

namespace {

constexpr int MAXPL_LIMIT = 16;   // logits per lane -> n <= 1024

__device__ __forceinline__ uint32_t order_key(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);   // unsigned order == float order (-0 < +0)
}
__device__ __forceinline__ float key_to_float(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __builtin_bit_cast(float, u);
}

__device__ __forceinline__ float wave_sum(float v) { return mortar_wave_sum(v); }

// Sum over the wavefront with DPP adds only (no LDS crossbar): quads, half rows, rows, then the row broadcasts; the total
// arrives in the last row and is read from lane 63.  Adds in another order than wave_sum, so not for results that have
// to match a kernel built on wave_sum bit for bit.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_f32(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROW_MASK, 0xf, false));
}
__device__ __forceinline__ float wave_sum_dpp(float v) {
    v += dpp_f32<0xB1, 0xf>(v);     // quad_perm [1,0,3,2]
    v += dpp_f32<0x4E, 0xf>(v);     // quad_perm [2,3,0,1]
    v += dpp_f32<0x141, 0xf>(v);    // row_half_mirror
    v += dpp_f32<0x140, 0xf>(v);    // row_mirror
    v += dpp_f32<0x142, 0xa>(v);    // row_bcast:15 into rows 1 and 3
    v += dpp_f32<0x143, 0xc>(v);    // row_bcast:31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Gating tail of one token on one wavefront.  The k-th largest logit is found exactly by an MSB-first radix
// select on order-preserving keys: for each bit the wave counts the keys >= the candidate prefix (ballots and scalar
// counts: with four waves to a SIMD the vector ALU is what is short; 17.6 -> 12.9 us with the sort below, 4096 tokens x 352 groups).  Ties need no special care: the result is a VALUE, and the gate rule is `logit > kth`.
// `lp` may point to global memory or LDS; gates / active are this token's output rows.
template <int MAXPL>      // logits per lane this instantiation holds: n <= 64 * MAXPL
__device__ __forceinline__ void remoe_gates_wave(const float *lp, int n, int k, float *gates, uint8_t *active, int lane) {
    float v[MAXPL];
    uint32_t key[MAXPL];
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
        const int idx = i * 64 + lane;
        v[i] = idx < n ? lp[idx] : 0.f;
        key[i] = idx < n ? order_key(v[i] == 0.f ? 0.f : v[i]) : 0u;   // -0 and +0 compare equal, as in topk
    }
    float kth = 0.f;
    const bool thresh = k < n;
    if (thresh && MAXPL == 1 && n <= 32) {
        // few groups: every lane counts the keys above its own and those not below it; the k-th largest is where k lies between
        int above = 0, from = 0;
        for (int j = 0; j < n; ++j) {
            const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)key[0], j);
            above += o > key[0] ? 1 : 0;
            from += o >= key[0] ? 1 : 0;
        }
        const uint64_t at = __ballot(lane < n && above < k && k <= from);
        kth = key_to_float((uint32_t)__builtin_amdgcn_readlane((int)key[0], __builtin_ctzll(at)));
    } else if (thresh) {
        // [prefix, prefix + 2^(bit+1)) is the bucket that holds the k-th largest key: c_lo keys are >= its lower end, c_hi keys
        // >= its upper end.  Once the bucket holds ONE key that key is the answer and the remaining bits need no counting
        // (distinct logits get there after about log2(n) + the exponent bits they share; exact ties walk all 32 bits).
        uint32_t prefix = 0;
        int c_lo = 64 * MAXPL, c_hi = 0, bit = 31;
        for (; bit >= 0 && c_lo - c_hi > 1; --bit) {
            const uint32_t cand = prefix | (1u << bit);
            int c = 0;
#pragma unroll
            for (int i = 0; i < MAXPL; ++i) c += (int)__popcll(__ballot(key[i] >= cand));            // padding keys are 0 < cand
            if (c >= k) { prefix = cand; c_lo = c; } else { c_hi = c; }
        }
        if (bit >= 0) {                       // left early: the bucket's one key (bits 0..bit of it were never looked at)
            uint32_t m = 0;
#pragma unroll
            for (int i = 0; i < MAXPL; ++i) m = (key[i] >> (bit + 1)) == (prefix >> (bit + 1)) && key[i] > m ? key[i] : m;
            prefix = mortar_wave_reduce(m, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
        }
        kth = key_to_float(prefix);
    }
    float g0[MAXPL];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
        const int idx = i * 64 + lane;
        float d = thresh ? v[i] - kth : v[i];
        d = d > 0.f ? d : (d != d ? d : 0.f);     // relu that lets NaN through, as torch.relu does
        g0[i] = idx < n ? d : 0.f;
        s += g0[i];
    }
    s = wave_sum(s);
    s = s < 1e-6f ? 1e-6f : s;                     // clamp(min=1e-6)
    const float t = (float)k / s;
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
        const int idx = i * 64 + lane;
        if (idx < n) {
            const float gv = g0[i] * t;
            gates[idx] = gv;
            if (active) active[idx] = gv > 0.f;
        }
    }
}

template <int MAXPL>
__global__ void __launch_bounds__(256) remoe_gates_kernel(const float *logits, int64_t M, int n, int k,
                                                           float *gates, uint8_t *active) {
    const int64_t tok = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tok >= M) return;
    remoe_gates_wave<MAXPL>(logits + tok * n, n, k, gates + tok * n, active ? active + tok * n : nullptr, threadIdx.x & 63);
}

// ---- decode-side router front end (TileRouter.forward steps 1-4 in front of the gating tail) -------------------
// Launch 1: qv[b, o] = sum_i x[b, i] * Wq[o, i] + iter_vec[o].  One wavefront per output row o; the row of Wq is
// read once per group of TB tokens (16-byte loads, fp32), x comes from L2.
template <int TB, bool XF32>
__global__ void __launch_bounds__(256) router_project_kernel(const void *xv, int B, int d, int64_t ldx, const float *wq,
                                                              const float *iter_vec, float *qv) {
    const int lane = threadIdx.x & 63;
    const int o = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (o >= d) return;
    const float4 *wr = reinterpret_cast<const float4 *>(wq + (int64_t)o * d);
    const float bias = iter_vec ? iter_vec[o] : 0.f;
    const int n4 = d / 4;
    for (int b0 = 0; b0 < B; b0 += TB) {
        float acc[TB];
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[t] = 0.f;
        // four 16-byte loads of the weight row in flight per lane (the row is read from HBM exactly once per token
        // group; the loop is latency-bound otherwise)
        for (int i0 = lane; i0 < n4; i0 += 256) {
            float4 w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i4 = i0 + 64 * u;
                w[u] = i4 < n4 ? wr[i4] : float4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i4 = i0 + 64 * u < n4 ? i0 + 64 * u : n4 - 1;
#pragma unroll
                for (int t = 0; t < TB; ++t) {
                    const int b = b0 + t < B ? b0 + t : B - 1;
                    float x0, x1, x2, x3;
                    if (XF32) {
                        const float4 xx = reinterpret_cast<const float4 *>(static_cast<const float *>(xv) + (int64_t)b * ldx)[i4];
                        x0 = xx.x; x1 = xx.y; x2 = xx.z; x3 = xx.w;
                    } else {
                        const uint2 xx = reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(xv) + (int64_t)b * ldx)[i4];
                        x0 = __builtin_bit_cast(float, xx.x << 16); x1 = __builtin_bit_cast(float, xx.x & 0xffff0000u);
                        x2 = __builtin_bit_cast(float, xx.y << 16); x3 = __builtin_bit_cast(float, xx.y & 0xffff0000u);
                    }
                    acc[t] = __builtin_fmaf(x3, w[u].w, __builtin_fmaf(x2, w[u].z, __builtin_fmaf(x1, w[u].y, __builtin_fmaf(x0, w[u].x, acc[t]))));
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            const float s = wave_sum(acc[t]);
            if (lane == 0 && b0 + t < B) qv[(int64_t)(b0 + t) * d + o] = s + bias;
        }
    }
}

// The projection of 1 to TB <= 4 bf16 rows with the RMSNorm before it, d <= 2048: wave w of every workgroup normalises row w into LDS
// (rms_* of mortar_device.h: the bits of rmsnorm_rows_kernel) while the weight rows are on their way, the first workgroup also writes
// the rows to xn for the products.  A launch of its own for the norm is a chain of 3.4 us with one wave per row.  Same products and
// order of sums as router_project_kernel.  (Figures: launch_router.)
template <int TB>
__global__ void __launch_bounds__(256) router_norm_project_kernel(const uint16_t *x, int B, int d, int64_t ldx, const uint16_t *nw, float eps, uint16_t *xn,
                                                                  const float *wq, const float *iter_vec, float *qv) {
    extern __shared__ __attribute__((aligned(16))) float sm[];       // bf16 [TB][d]
    u32x4_t *xs = reinterpret_cast<u32x4_t *>(sm);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int o = blockIdx.x * 4 + wave, n4 = d / 4, nch = d / 8;       // d % 8 == 0: every wave has an output
    const bool norm = wave < B && wave < TB;
    u32x4_t u[4], w8[4];
    if (norm) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ch = lane + 64 * j < nch ? lane + 64 * j : nch - 1;
            u[j] = reinterpret_cast<const u32x4_t *>(x + wave * ldx)[ch];
            w8[j] = nw ? reinterpret_cast<const u32x4_t *>(nw)[ch] : u32x4_t{0u, 0u, 0u, 0u};
        }
    }
    float4 w[8];
    const float4 *wr = reinterpret_cast<const float4 *>(wq + (int64_t)o * d);
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = lane + 64 * j < n4 ? wr[lane + 64 * j] : float4{0.f, 0.f, 0.f, 0.f};
    const float bias = iter_vec ? iter_vec[o] : 0.f;
    if (norm) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < nch) ss = rms_sumsq8(u[j], ss);
        const float r = rms_scale(rms_wave_sum(ss), d, eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ch = lane + 64 * j;
            if (ch < nch) {
                const u32x4_t v = rms_apply8(u[j], r, w8[j], nw != nullptr);
                xs[wave * nch + ch] = v;
                if (blockIdx.x == 0) reinterpret_cast<u32x4_t *>(xn + (int64_t)wave * d)[ch] = v;
            }
        }
    }
    __syncthreads();
    float acc[TB];
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[t] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int i4 = lane + 64 * j < n4 ? lane + 64 * j : n4 - 1;
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            const uint2 xx = reinterpret_cast<const uint2 *>(xs)[(t < B ? t : B - 1) * n4 + i4];
            acc[t] = __builtin_fmaf(__builtin_bit_cast(float, xx.y & 0xffff0000u), w[j].w, __builtin_fmaf(__builtin_bit_cast(float, xx.y << 16), w[j].z,
                     __builtin_fmaf(__builtin_bit_cast(float, xx.x & 0xffff0000u), w[j].y, __builtin_fmaf(__builtin_bit_cast(float, xx.x << 16), w[j].x, acc[t]))));
        }
    }
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        const float s = wave_sum(acc[t]);
        if (lane == 0 && t < B) qv[(int64_t)t * d + o] = s + bias;
    }
}

__device__ __forceinline__ float block_sum256(float v, float *red) {      // red: 4 floats of LDS; all 256 threads call
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// Descending sort of 64 * KPL keys held KPL per lane (element lane * KPL + r in register r), KPL a power of two or three times one: a
// bitonic sort whose runs start at KPL keys instead of one.  Every lane sorts its own; then runs of L lanes alternate in direction and are
// merged, by exchanges between lanes (half-wave and row swaps, DPP: no LDS) and a merge inside the lane.  A bitonic sequence of any even
// length falls into two bitonic halves, so a lane's KPL need not be a power of two.  Lanes of ascending runs hold inverted keys, so that
// no comparison inside a lane needs a select.  What counts is the number of instructions, with four waves to a SIMD: 361 keys in 6 per lane
// 520 of them, where 512 padded ones in 8 per lane took 1000: router_rank_kernel at 4096
// tokens 17.6 -> 14.2 us, a routed decode step of one row with 128 clusters (144 keys, 4 per lane) 21.7 -> 19.0.
__device__ __forceinline__ void sort_cx(uint32_t &a, uint32_t &b) {
    const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
    a = hi;
    b = lo;
}
template <int N, int O, int KPL>
__device__ __forceinline__ void sort_three(uint32_t (&key)[KPL]) {
    sort_cx(key[O], key[O + 1]);
    sort_cx(key[O + 1], key[O + 2]);
    sort_cx(key[O], key[O + 1]);
}
template <int N, int O, int KPL>
__device__ __forceinline__ void sort_merge(uint32_t (&key)[KPL]) {          // key[O .. O + N) bitonic
    if constexpr (N == 3) sort_three<N, O>(key);
    else if constexpr (N > 1) {
#pragma unroll
        for (int i = 0; i < N / 2; ++i) sort_cx(key[O + i], key[O + N / 2 + i]);
        sort_merge<N / 2, O>(key);
        sort_merge<N / 2, O + N / 2>(key);
    }
}
template <int N, int O, int KPL>
__device__ __forceinline__ void sort_lane(uint32_t (&key)[KPL]) {
    if constexpr (N == 3) sort_three<N, O>(key);
    else if constexpr (N > 1) {
        sort_lane<N / 2, O>(key);
        sort_lane<N / 2, O + N / 2>(key);
#pragma unroll
        for (int i = 0; i < N / 2; ++i) sort_cx(key[O + i], key[O + N - 1 - i]);
        sort_merge<N / 2, O>(key);
        sort_merge<N / 2, O + N / 2>(key);
    }
}
template <int LJ, int KPL>
__device__ __forceinline__ void sort_exchange(uint32_t (&key)[KPL], int lane) {      // the larger key to the lane with bit LJ clear
    if constexpr (LJ >= 16) {
        // the swap brings two keys' partners to the same lane, a second one takes the results back
#pragma unroll
        for (int r = 0; r < KPL; r += 2) {
            const auto s = LJ == 32 ? __builtin_amdgcn_permlane32_swap(key[r], key[r + 1], false, false)
                                    : __builtin_amdgcn_permlane16_swap(key[r], key[r + 1], false, false);
            uint32_t hi = s[0], lo = s[1];
            sort_cx(hi, lo);
            const auto t = LJ == 32 ? __builtin_amdgcn_permlane32_swap(hi, lo, false, false) : __builtin_amdgcn_permlane16_swap(hi, lo, false, false);
            key[r] = t[0];
            key[r + 1] = t[1];
        }
    } else {
#pragma unroll
        for (int r = 0; r < KPL; ++r) {
            const uint32_t a = key[r], o = mortar_row_xor<LJ>(a);
            const uint32_t hi = a > o ? a : o, lo = a > o ? o : a;
            key[r] = (lane & LJ) == 0 ? hi : lo;
        }
    }
}
template <int L, int KPL>
__device__ __forceinline__ void sort_runs(uint32_t (&key)[KPL], int lane) {          // runs of L lanes from runs of L / 2
    const bool was_up = (lane & (L / 2)) != 0, up = L < 64 && (lane & L) != 0;
    const uint32_t flip = was_up != up ? ~0u : 0u;
#pragma unroll
    for (int r = 0; r < KPL; ++r) key[r] ^= flip;
    if constexpr (L >= 64) sort_exchange<32>(key, lane);
    if constexpr (L >= 32) sort_exchange<16>(key, lane);
    if constexpr (L >= 16) sort_exchange<8>(key, lane);
    if constexpr (L >= 8) sort_exchange<4>(key, lane);
    if constexpr (L >= 4) sort_exchange<2>(key, lane);
    sort_exchange<1>(key, lane);
    sort_merge<KPL, 0>(key);
    if constexpr (L < 64) sort_runs<L * 2>(key, lane);
}
template <int KPL>
__device__ __forceinline__ void wave_sort_desc(uint32_t (&key)[KPL], int lane) {
    static_assert(KPL % 2 == 0, "exchanges of two keys");
    const uint32_t flip = (lane & 1) ? ~0u : 0u;
#pragma unroll
    for (int r = 0; r < KPL; ++r) key[r] ^= flip;
    sort_lane<KPL, 0>(key);
    sort_runs<2>(key, lane);
}

// The n largest of the P = nsk * nsk product scores of one token in descending order (+ bias) -> lgt[0 .. n), on one wave.
template <int KPL>
__device__ __attribute__((noinline)) void ranked_logits(const float *sct, int nsk, int P, const float *bias, int n, float *lgt,
                                              float *logits_row, int lane) {
    uint32_t key[KPL];
    int ia = lane * KPL / nsk, ib = lane * KPL - ia * nsk;      // product i = ia * nsk + ib
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        const int i = lane * KPL + r;
        uint32_t kk = 0u;                                    // padding: the smallest key
        if (i < P) {
            const uint32_t u = __float_as_uint(sct[ia] + sct[nsk + ib]);
            kk = (u & 0x80000000u) ? ~u : (u | 0x80000000u);   // NaN ranks above +inf, as torch.topk has it
        }
        key[r] = kk;
        if (++ib == nsk) { ib = 0; ++ia; }
    }
    wave_sort_desc<KPL>(key, lane);
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        const int g = lane * KPL + r;
        if (g < n) {
            const float l = __uint_as_float((key[r] & 0x80000000u) ? (key[r] & 0x7fffffffu) : ~key[r]) + bias[g];
            lgt[g] = l;
            if (logits_row) logits_row[g] = l;
        }
    }
}

__device__ __forceinline__ void rank_products(const float *sct, int nsk, int P, const float *bias, int n, float *lgt, float *logits_row, int lane) {
    if (P <= 128) ranked_logits<2>(sct, nsk, P, bias, n, lgt, logits_row, lane);
    else if (P <= 256) ranked_logits<4>(sct, nsk, P, bias, n, lgt, logits_row, lane);
    else if (P <= 384) ranked_logits<6>(sct, nsk, P, bias, n, lgt, logits_row, lane);
    else if (P <= 512) ranked_logits<8>(sct, nsk, P, bias, n, lgt, logits_row, lane);
    else ranked_logits<16>(sct, nsk, P, bias, n, lgt, logits_row, lane);           // P <= 1024
}

// Launch 2, one workgroup per token: LayerNorm(qv) -> sub-key scores of the two query halves -> product-key logits
// (+ group bias) -> gating tail.  P = nsk * nsk products map to the n groups one to one (P == n), wrap (P < n), or are
// ranked and the n largest kept (P > n).
// PRE > 0 (d <= 2048; PRE = sub-key rows per wave: 2 for nsk <= 4, 10 for nsk <= 20): every parameter a thread needs
// (LayerNorm weights, its slices of the sub-key rows of its wave) is fetched into registers before the first reduction,
// so the kernel pays one memory round trip instead of one per phase and key row.
template <int MAXPL, int PRE>
__global__ void __launch_bounds__(256) router_tail_kernel(const float *qv, int d, int64_t ldq, const float *iter_vec, const float *ln_w, const float *ln_b,
                                                           float ln_eps, const float *ka, const float *kb, int nsk,
                                                           const float *bias, int n, int k, float *logits_out,
                                                           float *gates, uint8_t *active) {
    extern __shared__ __attribute__((aligned(16))) float sm[];       // qn[d] | s[2 * nsk] | logits[n] | red[4] | sort keys
    float *qn = sm, *sc = sm + d, *lg = sc + 2 * nsk, *red = lg + n;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *q = qv + (int64_t)b * ldq;
    const int d2 = d / 2, n4 = d2 / 4;          // d % 8 == 0: both halves are whole float4 runs
    constexpr int QE = 8, DPW = PRE > 0 ? PRE : 1, KU = 4;      // PRE: entries per thread, sub-key dots per wave, float4 per lane and dot
    float qe[QE], lw[QE], lbv[QE];
    float4 kreg[DPW][KU];
    if (PRE) {
#pragma unroll
        for (int j = 0; j < QE; ++j) {
            const int i = tid + 256 * j, ic = i < d ? i : d - 1;
            qe[j] = q[ic]; lw[j] = ln_w[ic]; lbv[j] = ln_b[ic];
        }
        float iv[QE];
#pragma unroll
        for (int j = 0; j < QE; ++j) iv[j] = 0.f;
        if (iter_vec) {
#pragma unroll
            for (int j = 0; j < QE; ++j) iv[j] = iter_vec[tid + 256 * j < d ? tid + 256 * j : d - 1];
        }
#pragma unroll
        for (int cc = 0; cc < DPW; ++cc) {
            int c = wave + 4 * cc;
            c = c < 2 * nsk ? c : 2 * nsk - 1;
            const float4 *kr = reinterpret_cast<const float4 *>(c < nsk ? ka + (int64_t)c * d2 : kb + (int64_t)(c - nsk) * d2);
#pragma unroll
            for (int u = 0; u < KU; ++u) kreg[cc][u] = lane + 64 * u < n4 ? kr[lane + 64 * u] : float4{0.f, 0.f, 0.f, 0.f};
        }
        if (iter_vec) {
#pragma unroll
            for (int j = 0; j < QE; ++j) qe[j] += iv[j];
        }
    }
    float s = 0.f;
    if (PRE) {
#pragma unroll
        for (int j = 0; j < QE; ++j) s += tid + 256 * j < d ? qe[j] : 0.f;
    } else {
        for (int i = tid; i < d; i += 256) { const float t = iter_vec ? q[i] + iter_vec[i] : q[i]; qn[i] = t; s += t; }      // a thread re-reads its own entries
    }
    const float mean = block_sum256(s, red) / (float)d;
    float v = 0.f;
    if (PRE) {
#pragma unroll
        for (int j = 0; j < QE; ++j) { const float c = tid + 256 * j < d ? qe[j] - mean : 0.f; v = __builtin_fmaf(c, c, v); }
    } else {
        for (int i = tid; i < d; i += 256) { const float c = qn[i] - mean; v = __builtin_fmaf(c, c, v); }
    }
    const float rstd = 1.0f / sqrtf(block_sum256(v, red) / (float)d + ln_eps);
    if (PRE) {
#pragma unroll
        for (int j = 0; j < QE; ++j)
            if (tid + 256 * j < d) qn[tid + 256 * j] = (qe[j] - mean) * rstd * lw[j] + lbv[j];
    } else {
        for (int i = tid; i < d; i += 256) qn[i] = (qn[i] - mean) * rstd * ln_w[i] + ln_b[i];
    }
    __syncthreads();
    if (PRE) {
#pragma unroll
        for (int cc = 0; cc < DPW; ++cc) {
            const int c = wave + 4 * cc;
            const float4 *qh = reinterpret_cast<const float4 *>(c < nsk ? qn : qn + d2);
            float a = 0.f;
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const float4 qq = qh[lane + 64 * u < n4 ? lane + 64 * u : n4 - 1];
                a = __builtin_fmaf(qq.w, kreg[cc][u].w, __builtin_fmaf(qq.z, kreg[cc][u].z, __builtin_fmaf(qq.y, kreg[cc][u].y, __builtin_fmaf(qq.x, kreg[cc][u].x, a))));
            }
            a = wave_sum(a);
            if (lane == 0 && c < 2 * nsk) sc[c] = a;
        }
    } else {
        for (int c = wave; c < 2 * nsk; c += 4) {
            const float4 *kr = reinterpret_cast<const float4 *>(c < nsk ? ka + (int64_t)c * d2 : kb + (int64_t)(c - nsk) * d2);
            const float4 *qh = reinterpret_cast<const float4 *>(c < nsk ? qn : qn + d2);
            float a = 0.f;
            for (int i0 = lane; i0 < n4; i0 += 256) {
                float4 kv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) kv[u] = i0 + 64 * u < n4 ? kr[i0 + 64 * u] : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float4 qq = qh[i0 + 64 * u < n4 ? i0 + 64 * u : n4 - 1];
                    a = __builtin_fmaf(qq.w, kv[u].w, __builtin_fmaf(qq.z, kv[u].z, __builtin_fmaf(qq.y, kv[u].y, __builtin_fmaf(qq.x, kv[u].x, a))));
                }
            }
            a = wave_sum(a);
            if (lane == 0) sc[c] = a;
        }
    }
    __syncthreads();
    const int P = nsk * nsk;
    if (P > n) {
        // more product keys than groups: the group logits are the n largest product scores in descending order
        // (torch.topk(product_scores, n).values, morph/model/routing.py:212-222).  Bitonic sort of order-preserving
        // integer keys (NaN ranks above +inf, as torch.topk has it), padded with the smallest key: in one wave's registers
        // up to 1024 products, through LDS by the whole workgroup beyond.
        if (P <= 1024) {           // one wave ranks them in its registers (no LDS traffic, no barrier per step)
            float *lrow = logits_out ? logits_out + (int64_t)b * n : nullptr;
            if (wave == 0) rank_products(sc, nsk, P, bias, n, lg, lrow, lane);
        } else {
            uint32_t *sk = reinterpret_cast<uint32_t *>(red + 4);
            int P2 = 1;
            while (P2 < P) P2 <<= 1;
            for (int i = tid; i < P2; i += 256) {
                uint32_t key = 0u;
                if (i < P) {
                    const uint32_t u = __float_as_uint(sc[i / nsk] + sc[nsk + i % nsk]);
                    key = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
                }
                sk[i] = key;
            }
            __syncthreads();
            for (int k2 = 2; k2 <= P2; k2 <<= 1) {
                for (int j = k2 >> 1; j > 0; j >>= 1) {
                    for (int t = tid; t < P2 / 2; t += 256) {
                        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), l = i | j;
                        const uint32_t a = sk[i], c = sk[l];
                        const bool desc = (i & k2) == 0;
                        if (desc ? a < c : a > c) { sk[i] = c; sk[l] = a; }
                    }
                    __syncthreads();
                }
            }
            for (int g = tid; g < n; g += 256) {
                const uint32_t key = sk[g];
                const float l = __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key) + bias[g];
                lg[g] = l;
                if (logits_out) logits_out[(int64_t)b * n + g] = l;
            }
        }
    } else {
        for (int g = tid; g < n; g += 256) {
            const int pr = g % P;
            const float l = (sc[pr / nsk] + sc[nsk + pr % nsk]) + bias[g];
            lg[g] = l;
            if (logits_out) logits_out[(int64_t)b * n + g] = l;
        }
    }
    __syncthreads();
    if (wave == 0)
        remoe_gates_wave<MAXPL>(lg, n, k, gates + (int64_t)b * n, active ? active + (int64_t)b * n : nullptr, lane);
}

// ---- router tail for prefill-sized calls (TileRouter.forward steps 2-8 behind a library GEMM for the projection) ----

// A workgroup of four waves takes groups of up to TT = 4 tokens (a loop over its share of the groups), so the sub-key
// rows are read from L2 once per group instead of once per token.
//   1. LayerNorm by the whole workgroup: every thread holds its float4 pieces of all rows of the group, the iteration
//      vector and the LayerNorm parameters from ONE round of loads; the sums meet through LDS; normalised rows -> LDS.
//   2. the 2 * nsk sub-key dot products, one key row per wave at a time against all tokens of the group; the next row's
//      piece is requested before the current one is multiplied.
//   3. per token (one wave each): product-key logits (+ bias) -> LDS, ranked first when nsk^2 > n (a bitonic network
//      in the wave's registers), then the gating tail.
// Same arithmetic as router_tail_kernel; the sums are ordered differently.  A group is a chain of latencies (about 3 us of
// loads, 2 us of LayerNorm, 1.3 us per key row and wave, 2-10 us of logits and gating), so throughput comes from the
// groups in flight: three workgroups per CU (two for rows wider than 4096 values) at this register count, with the
// sort kept out of line (inlined, its registers add to the whole kernel's).
constexpr int TAIL_TT = 4;

template <int MAXPL, int J>      // J: float4 pieces of a row per thread (d <= 1024 * J); tokens per group tt = min(4, 8 / J)
__global__ void __launch_bounds__(256, J == 8 ? 2 : 3) router_tail_group_kernel(const float *qv, int64_t N, int d, int64_t ldq, const float *iter_vec,
                                                                 const float *ln_w, const float *ln_b, float ln_eps,
                                                                 const float *ka, const float *kb, int nsk, const float *bias,
                                                                 int n, int k, int tt, float *logits_out, float *gates,
                                                                 uint8_t *active) {
    extern __shared__ __attribute__((aligned(16))) float sm[];       // qn[tt][d] | sc[tt][2 nsk] | lg[tt][n] | red[16]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int d2 = d / 2, d4 = d / 4, n4 = d2 / 4;
    const int P = nsk * nsk;
    float *qn = sm, *sc = qn + (size_t)tt * d, *lg = sc + tt * 2 * nsk, *red = lg + (size_t)tt * n;
    const float4 *iv4 = reinterpret_cast<const float4 *>(iter_vec);
    const float4 *lw4 = reinterpret_cast<const float4 *>(ln_w), *lb4 = reinterpret_cast<const float4 *>(ln_b);
    const float4 zero4 = float4{0.f, 0.f, 0.f, 0.f};
    for (int64_t g0 = (int64_t)blockIdx.x * tt; g0 < N; g0 += (int64_t)gridDim.x * tt) {
        const int nt = N - g0 < tt ? (int)(N - g0) : tt;
        {
            // LayerNorm of the group's tokens by the whole workgroup: thread tid holds the float4 pieces tid + 256 * j of every
            // token (tt * pieces <= 8), so all rows, the iteration vector and the LayerNorm parameters are one round of
            // loads; sums meet through LDS (red: [4 waves][4 tokens]).
            constexpr int TT = 8 / J < TAIL_TT ? 8 / J : TAIL_TT, E = TT * J;
            float4 v[E], w[J], b[J];
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const int i = tid + 256 * jj, ic = i < d4 ? i : d4 - 1;
                if (J < 4) {              // wide rows fetch the LayerNorm parameters when they are used (registers)
                    w[jj] = lw4[ic];
                    b[jj] = lb4[ic];
                }
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const bool on = t < nt && i < d4;
                    float4 a = reinterpret_cast<const float4 *>(qv + (g0 + (t < nt ? t : 0)) * ldq)[ic];
                    if (iter_vec) { const float4 c = iv4[ic]; a.x += c.x; a.y += c.y; a.z += c.z; a.w += c.w; }
                    v[t * J + jj] = on ? a : zero4;
                }
            }
            float s[TT], mean[TT], rstd[TT];
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                s[t] = 0.f;
#pragma unroll
                for (int jj = 0; jj < J; ++jj) { const float4 a = v[t * J + jj]; s[t] += (a.x + a.y) + (a.z + a.w); }
                const float a = wave_sum_dpp(s[t]);
                if (lane == 0) red[wave * TAIL_TT + t] = a;
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < TT; ++t) mean[t] = (red[t] + red[TAIL_TT + t] + red[2 * TAIL_TT + t] + red[3 * TAIL_TT + t]) / (float)d;
            __syncthreads();
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                s[t] = 0.f;
#pragma unroll
                for (int jj = 0; jj < J; ++jj) {
                    if (tid + 256 * jj < d4) {
                        const float4 q = v[t * J + jj];
                        const float a = q.x - mean[t], c = q.y - mean[t], f = q.z - mean[t], h = q.w - mean[t];
                        s[t] = __builtin_fmaf(h, h, __builtin_fmaf(f, f, __builtin_fmaf(c, c, __builtin_fmaf(a, a, s[t]))));
                    }
                }
                const float a = wave_sum_dpp(s[t]);
                if (lane == 0) red[wave * TAIL_TT + t] = a;
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                rstd[t] = 1.0f / sqrtf((red[t] + red[TAIL_TT + t] + red[2 * TAIL_TT + t] + red[3 * TAIL_TT + t]) / (float)d + ln_eps);
#pragma unroll
                for (int jj = 0; jj < J; ++jj) {
                    const int i = tid + 256 * jj;
                    if (J >= 4) {
                        w[jj] = lw4[i < d4 ? i : d4 - 1];
                        b[jj] = lb4[i < d4 ? i : d4 - 1];
                    }
                    if (t < nt && i < d4) {
                        const float4 q = v[t * J + jj];
                        const float m = mean[t], r = rstd[t];
                        reinterpret_cast<float4 *>(qn + (size_t)t * d)[i] =
                            float4{(q.x - m) * r * w[jj].x + b[jj].x, (q.y - m) * r * w[jj].y + b[jj].y,
                                   (q.z - m) * r * w[jj].z + b[jj].z, (q.w - m) * r * w[jj].w + b[jj].w};
                    }
                }
            }
        }
        __syncthreads();
        {
            // items of this wave: (key row c = wave + 4 * row, piece of 256 float4); the next item's piece is loaded first
            const int chunks = (n4 + 255) / 256;
            const int rows = (2 * nsk - wave + 3) / 4;
            const int items = rows * chunks;
            auto load_item = [&](int it, float4 (&kv)[4]) {
                const int itc = it < items ? it : items - 1;
                const int c = wave + 4 * (itc / chunks), i0 = lane + 256 * (itc % chunks);
                const float4 *kr = reinterpret_cast<const float4 *>(c < nsk ? ka + (int64_t)c * d2 : kb + (int64_t)(c - nsk) * d2);
#pragma unroll
                for (int u = 0; u < 4; ++u) kv[u] = kr[i0 + 64 * u < n4 ? i0 + 64 * u : n4 - 1];
            };
            float4 kv[4];
            if (items > 0) load_item(0, kv);
            float acc[TAIL_TT];
#pragma unroll
            for (int t = 0; t < TAIL_TT; ++t) acc[t] = 0.f;
            for (int it = 0; it < items; ++it) {
                float4 kn[4];
                load_item(it + 1, kn);
                const int c = wave + 4 * (it / chunks), i0 = lane + 256 * (it % chunks);
                const int off4 = c < nsk ? 0 : n4;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i0 + 64 * u >= n4) kv[u] = zero4;
#pragma unroll
                for (int t = 0; t < TAIL_TT; ++t) {
                    if (t < nt) {
                        const float4 *qh = reinterpret_cast<const float4 *>(qn + (size_t)t * d) + off4;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float4 qq = qh[i0 + 64 * u < n4 ? i0 + 64 * u : n4 - 1];
                            acc[t] = __builtin_fmaf(qq.w, kv[u].w, __builtin_fmaf(qq.z, kv[u].z, __builtin_fmaf(qq.y, kv[u].y, __builtin_fmaf(qq.x, kv[u].x, acc[t]))));
                        }
                    }
                }
                if (it % chunks == chunks - 1) {
#pragma unroll
                    for (int t = 0; t < TAIL_TT; ++t) {
                        const float a = wave_sum_dpp(acc[t]);
                        if (lane == 0 && t < nt) sc[t * 2 * nsk + c] = a;
                        acc[t] = 0.f;
                    }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) kv[u] = kn[u];
            }
        }
        __syncthreads();
        if (wave < nt) {                             // tt <= 4: one token per wave, nothing shared between waves from here on
            const int t = wave;
            const float *sct = sc + t * 2 * nsk;
            float *lgt = lg + (size_t)t * n;
            float *lrow = logits_out ? logits_out + (g0 + t) * n : nullptr;
            if (P > n) {
                // more product keys than groups: the n largest product scores in descending order (routing.py:212-222)
                rank_products(sct, nsk, P, bias, n, lgt, lrow, lane);        // the host admits P <= 1024
            } else {
                for (int g = lane; g < n; g += 64) {
                    const int pr = g % P;
                    const float l = (sct[pr / nsk] + sct[nsk + pr % nsk]) + bias[g];
                    lgt[g] = l;
                    if (lrow) lrow[g] = l;
                }
            }
            // the wave reads logits that other lanes of it wrote: LDS serves a wave's accesses in order, the fence keeps
            // the compiler from moving the reads up
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            remoe_gates_wave<MAXPL>(lgt, n, k, gates + (g0 + t) * n, active ? active + (g0 + t) * n : nullptr, lane);
        }
        __syncthreads();
    }
}

// ---- the same tail in two launches (rows of up to 4096 values, up to 32 sub-keys) --------------------------------------
// The group kernel above is one chain of latencies per 4 tokens (loads, LayerNorm, key rows one after another, then a sort
// per wave with the other phases waiting): 62 us for 4096 tokens x 352 groups, 20 us of it bandwidth or arithmetic.  Cut in
// two, each half fills the chip on its own terms:
//   router_scores_kernel   16 tokens per workgroup; the 2 nsk dot products per token run on the fp32 matrix instructions
//                          (16 keys x 16 tokens), so the key rows are read once per 16 tokens and no product needs a wave
//                          reduction.  Wave w takes every fourth 16-value chunk of query half w / 4; a lane holds 4 values
//                          of one token per chunk in registers from the one read of the row to the products.
//   router_rank_kernel     one wave per token: logits (ranked when there are more products than groups), gating tail.
// The scores travel in the token's own row of `gates` (2 nsk <= n), which the second kernel reads before it writes it.
__device__ __forceinline__ float rows_sum(float v) {             // over the four 16-lane rows: lanes ^ 16, then ^ 32
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int KT, int CH>     // key tiles of 16 per half, chunks of 16 values per wave
__global__ void __launch_bounds__(512) router_scores_kernel(const float *qv, int64_t N, int d, int64_t ldq, const float *iter_vec,
                                                             const float *ln_w, const float *ln_b, float ln_eps, const float *ka,
                                                             const float *kb, int nsk, int n, float *scores) {
    __shared__ float red[2][8][16];
    __shared__ __attribute__((aligned(16))) f32x4_t part[8][KT][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tok = lane & 15, g = lane >> 4, half = wave >> 2, sub = wave & 3;
    const int d2 = d / 2;
    const int64_t t0 = (int64_t)blockIdx.x * 16;
    const int64_t row = t0 + tok < N ? t0 + tok : N - 1;
    const float4 zero4 = float4{0.f, 0.f, 0.f, 0.f};
    const float *q = qv + row * ldq + half * d2, *iv = iter_vec ? iter_vec + half * d2 : nullptr;
    // chunk j of this wave: values 16 (sub + 4 j) + 4 g .. + 3 of the half (d2 % 4 == 0: in or out as a whole)
    auto at = [&](int j) { return 16 * (sub + 4 * j) + 4 * g; };
    float4 v[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const int i = at(j) < d2 ? at(j) : 0;
        v[j] = *reinterpret_cast<const float4 *>(q + i);
    }
    const float *lw = ln_w + half * d2, *lb = ln_b + half * d2;
    const float *kr[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) kr[t] = (half ? kb : ka) + (int64_t)(t * 16 + tok < nsk ? t * 16 + tok : nsk - 1) * d2;
    // LayerNorm parameters and key pieces are fetched PF chunks ahead of their products, the first before the statistics
    constexpr int PF = 4;
    float4 pw[PF], pb[PF], pk[PF][KT];
    auto fetch = [&](int j) {
        const int i = at(j) < d2 ? at(j) : 0;
        pw[j % PF] = *reinterpret_cast<const float4 *>(lw + i);
        pb[j % PF] = *reinterpret_cast<const float4 *>(lb + i);
#pragma unroll
        for (int t = 0; t < KT; ++t) pk[j % PF][t] = *reinterpret_cast<const float4 *>(kr[t] + i);
    };
#pragma unroll
    for (int j = 0; j < PF; ++j) fetch(j);
    float s = 0.f;
    if (iv) {                        // eight loads in flight (one test per chunk made each wait for the one before)
#pragma unroll
        for (int j0 = 0; j0 < CH; j0 += 8) {
            float4 c[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) c[j] = *reinterpret_cast<const float4 *>(iv + (at(j0 + j) < d2 ? at(j0 + j) : 0));
#pragma unroll
            for (int j = 0; j < 8; ++j) { v[j0 + j].x += c[j].x; v[j0 + j].y += c[j].y; v[j0 + j].z += c[j].z; v[j0 + j].w += c[j].w; }
        }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        if (at(j) >= d2) v[j] = zero4;
        s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
    }
    s = rows_sum(s);
    if (g == 0) red[0][wave][tok] = s;
    __syncthreads();
    float mean = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) mean += red[0][w][tok];
    mean /= (float)d;
    s = 0.f;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        if (at(j) < d2) {
            const float a = v[j].x - mean, b = v[j].y - mean, c = v[j].z - mean, e = v[j].w - mean;
            s = __builtin_fmaf(e, e, __builtin_fmaf(c, c, __builtin_fmaf(b, b, __builtin_fmaf(a, a, s))));
        }
    }
    s = rows_sum(s);
    if (g == 0) red[1][wave][tok] = s;
    __syncthreads();
    float var = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) var += red[1][w][tok];
    const float rstd = 1.0f / sqrtf(var / (float)d + ln_eps);
    f32x4_t acc[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const bool in = at(j) < d2;
        const float4 w = pw[j % PF], b = pb[j % PF];
        float4 kk[KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) kk[t] = pk[j % PF][t];
        if (j + PF < CH) fetch(j + PF);
        float4 x = v[j];
        x = float4{(x.x - mean) * rstd * w.x + b.x, (x.y - mean) * rstd * w.y + b.y, (x.z - mean) * rstd * w.z + b.z, (x.w - mean) * rstd * w.w + b.w};
        if (!in) x = zero4;
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const float4 k = kk[t];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.x, x.x, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.y, x.y, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.z, x.z, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.w, x.w, acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < KT; ++t) part[wave][t][lane] = acc[t];
    __syncthreads();
    // the four waves of a half meet; wave 4 half + t (t < KT) finishes key tile t: lane (token, g) holds keys 16 t + 4 g + e
    if (sub < KT && t0 + tok < N) {
        const f32x4_t a = (part[half * 4][sub][lane] + part[half * 4 + 1][sub][lane]) + (part[half * 4 + 2][sub][lane] + part[half * 4 + 3][sub][lane]);
        float *o = scores + (t0 + tok) * n + half * nsk;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (sub * 16 + 4 * g + e < nsk) o[sub * 16 + 4 * g + e] = a[e];
    }
}

template <int MAXPL>
__global__ void __launch_bounds__(256) router_rank_kernel(int64_t N, int nsk, const float *bias, int n, int k, float *logits_out, float *gates,
                                                           uint8_t *active) {
    extern __shared__ __attribute__((aligned(16))) float sm[];       // per wave: sc[2 nsk] | lg[n]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t tok = (int64_t)blockIdx.x * 4 + wave;
    if (tok >= N) return;
    float *sct = sm + wave * (2 * nsk + n), *lgt = sct + 2 * nsk, *lrow = logits_out ? logits_out + tok * n : nullptr;
    float *grow = gates + tok * n;
    const int P = nsk * nsk;
    if (lane < 2 * nsk) sct[lane] = grow[lane];
    auto wave_fence = [] {                   // LDS serves a wave's accesses in order; this keeps the compiler from moving them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    wave_fence();
    if (P > n) {
        rank_products(sct, nsk, P, bias, n, lgt, lrow, lane);
    } else {
        for (int g = lane; g < n; g += 64) {
            const int pr = g % P;
            const float l = (sct[pr / nsk] + sct[nsk + pr % nsk]) + bias[g];
            lgt[g] = l;
            if (lrow) lrow[g] = l;
        }
    }
    wave_fence();
    remoe_gates_wave<MAXPL>(lgt, n, k, grow, active ? active + tok * n : nullptr, lane);
}

// Workgroup = (token tile, chunk of 64 clusters).  The tile's active bytes for the chunk are staged in LDS
// with coalesced reads; then every wave compacts whole clusters: lanes = tokens, ballot -> prefix popcount.
__global__ void __launch_bounds__(256) remoe_route_kernel(const uint8_t *active, int64_t M, int n, int tile,
                                                           int32_t *tok_cnt, uint8_t *tok_list) {
    __shared__ uint8_t a[256][64 + 4];
    const int t = blockIdx.x, cc = blockIdx.y * 64;
    const int ncl = (n - cc) < 64 ? (n - cc) : 64;
    const int64_t m0 = (int64_t)t * tile;
    for (int i = threadIdx.x; i < tile * 64; i += 256) {
        const int r = i >> 6, c = i & 63;
        const int64_t m = m0 + r;
        a[r][c] = (m < M && c < ncl) ? active[m * n + cc + c] : 0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = wave; c < ncl; c += 4) {
        const int64_t e = (int64_t)t * n + cc + c;
        int base = 0;
        for (int r0 = 0; r0 < tile; r0 += 64) {
            const int r = r0 + lane;
            const bool on = r < tile && a[r][c] != 0;
            const unsigned long long mask = __ballot(on);
            const int pos = base + __popcll(mask & ((1ull << lane) - 1ull));
            if (on) tok_list[e * tile + pos] = (uint8_t)r;
            base += __popcll(mask);
        }
        if (lane == 0) tok_cnt[e] = base;
    }
}

__global__ void __launch_bounds__(256) route_flags_kernel(const float *gates, int64_t B, int ncls, int64_t ldg,
                                                           int d_ff, int32_t *row_act, int64_t ldr,
                                                           int32_t *col_act, int64_t ldc) {
    const int nc = d_ff / 16, cls = d_ff / ncls;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= B * nc) return;
    const int64_t b = i / nc;
    const int r = (int)(i % nc);
    const int lo = (r * 16) / cls, hi = (r * 16 + 15) / cls;
    const int f = (gates[b * ldg + lo] > 0.f) || (gates[b * ldg + hi] > 0.f);
    if (col_act) col_act[b * ldc + r] = f;
    if (row_act) {
        row_act[b * ldr + r] = f;
        row_act[b * ldr + nc + r] = f;
    }
}

// One wavefront per row, in 16-byte units, with the summation order and rounding steps of the fused form in
// the gate_up staging (rms_* in mortar_device.h): both give the same bits.
// A call of few rows is a chain of latencies.  CU > 0: rows of at most 64 CU units stay in registers, everything requested at once; the loops
// below are a round trip per 64 units, twice.  us (graph replay), the loops -> this: 16 rows of 2048 / 4096 / 8192 values 3.6 -> 2.7, 5.2 -> 3.4, 8.9 ->
// 5.0; 16384 rows, which run at the rate of memory, 28 -> 21, 58 -> 41, 145 -> 100, 12000 rows of 512 6.5 -> 6.4.
template <int CU>
__global__ void __launch_bounds__(256) rmsnorm_rows_kernel(const uint16_t *x, int64_t M, int d, int64_t ldx,
                                                            const uint16_t *w, float eps, uint16_t *y, int64_t ldy) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= M) return;
    const u32x4_t *xp = reinterpret_cast<const u32x4_t *>(x + row * ldx);
    const u32x4_t *wp = reinterpret_cast<const u32x4_t *>(w);
    u32x4_t *yp = reinterpret_cast<u32x4_t *>(y + row * ldy);
    const int nch = d / 8;
    float ss = 0.f;
    if constexpr (CU > 0) {
        u32x4_t u[CU], w8[CU];
#pragma unroll
        for (int j = 0; j < CU; ++j) u[j] = xp[lane + 64 * j < nch ? lane + 64 * j : nch - 1];
#pragma unroll
        for (int j = 0; j < CU; ++j) w8[j] = w ? wp[lane + 64 * j < nch ? lane + 64 * j : nch - 1] : u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < CU; ++j)
            if (lane + 64 * j < nch) ss = rms_sumsq8(u[j], ss);
        const float r = rms_scale(rms_wave_sum(ss), d, eps);
#pragma unroll
        for (int j = 0; j < CU; ++j)
            if (lane + 64 * j < nch) yp[lane + 64 * j] = rms_apply8(u[j], r, w8[j], w != nullptr);
        return;
    }
    for (int ch = lane; ch < nch; ch += 64) ss = rms_sumsq8(xp[ch], ss);
    const float r = rms_scale(rms_wave_sum(ss), d, eps);
    for (int ch = lane; ch < nch; ch += 64)
        yp[ch] = rms_apply8(xp[ch], r, w ? wp[ch] : u32x4_t{0u, 0u, 0u, 0u}, w != nullptr);
}

// Any d / alignment: element-wise (its sums are ordered differently; no fused counterpart exists for such rows).
__global__ void __launch_bounds__(256) rmsnorm_kernel(const uint16_t *x, int64_t M, int d, int64_t ldx,
                                                       const uint16_t *w, float eps, uint16_t *y, int64_t ldy) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const uint16_t *xp = x + row * ldx;
    float s = 0.f;
    for (int i = threadIdx.x; i < d; i += 256) {
        const float v = bf16_to_f32(xp[i]);
        s += v * v;
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float tot = red[0] + red[1] + red[2] + red[3];
    const float r = 1.0f / sqrtf(tot / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256) {
        float v = bf16r(bf16_to_f32(xp[i]) * r);
        if (w) v = bf16r(v * bf16_to_f32(w[i]));
        y[row * ldy + i] = (uint16_t)bf16_bits_rne(v);
    }
}

int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "%s launch: %s", what, hipGetErrorString(e));
    return MORTAR_OK;
}

}  // namespace

extern "C" int mortar_remoe_gates(const float *logits, int64_t M, int32_t n, int32_t k, float *gates,
                                  uint8_t *active, void *stream) {
    if (!logits || !gates) return mortar_fail(MORTAR_ERR_ARG, "remoe_gates: null pointer");
    if (M <= 0 || n <= 0 || k <= 0) return mortar_fail(MORTAR_ERR_ARG, "remoe_gates: M, n, k must be positive");
    if (n > 64 * MAXPL_LIMIT) return mortar_fail(MORTAR_ERR_LIMIT, "remoe_gates: n=%d exceeds %d clusters", n, 64 * MAXPL_LIMIT);
    const dim3 grid((unsigned)((M + 3) / 4)), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int npl = (n + 63) / 64;
    if (npl <= 1) hipLaunchKernelGGL(remoe_gates_kernel<1>, grid, block, 0, st, logits, M, n, k, gates, active);
    else if (npl <= 2) hipLaunchKernelGGL(remoe_gates_kernel<2>, grid, block, 0, st, logits, M, n, k, gates, active);
    else if (npl <= 4) hipLaunchKernelGGL(remoe_gates_kernel<4>, grid, block, 0, st, logits, M, n, k, gates, active);
    else if (npl <= 6) hipLaunchKernelGGL(remoe_gates_kernel<6>, grid, block, 0, st, logits, M, n, k, gates, active);
    else if (npl <= 8) hipLaunchKernelGGL(remoe_gates_kernel<8>, grid, block, 0, st, logits, M, n, k, gates, active);
    else hipLaunchKernelGGL(remoe_gates_kernel<16>, grid, block, 0, st, logits, M, n, k, gates, active);
    return check_launch("remoe_gates");
}

// One workgroup per token.
static int launch_tail(const float *qv, int64_t N, int32_t d, int64_t ldq, const float *iter_vec, const float *ln_w, const float *ln_b, float ln_eps,
                       const float *ka, const float *kb, int32_t nsk, const float *bias, int32_t n, int32_t k, float *logits_out, float *gates,
                       uint8_t *active, hipStream_t st) {
    size_t sort_keys = 0;                          // nsk^2 > n: room for the product scores, padded to a power of two
    if ((int64_t)nsk * nsk > n) { sort_keys = 1; while (sort_keys < (size_t)nsk * nsk) sort_keys <<= 1; }
    const size_t smem = (size_t)(d + 2 * nsk + n + 4 + sort_keys) * sizeof(float);
    const dim3 tg((unsigned)N), blk(256);
    const int npl = (n + 63) / 64;
    const int pre = d > 2048 ? 0 : nsk <= 4 ? 2 : nsk <= 20 ? 10 : 0;      // sub-key dots per wave with their rows in registers
#define MORTAR_TAILP(PL, PR) hipLaunchKernelGGL((router_tail_kernel<PL, PR>), tg, blk, smem, st, qv, d, ldq, iter_vec, ln_w, ln_b, ln_eps, \
                                               ka, kb, nsk, bias, n, k, logits_out, gates, active)
#define MORTAR_TAIL(PL) do { if (pre == 2) MORTAR_TAILP(PL, 2); else if (pre == 10) MORTAR_TAILP(PL, 10); else MORTAR_TAILP(PL, 0); } while (0)
    if (npl <= 1) MORTAR_TAIL(1);
    else if (npl <= 2) MORTAR_TAIL(2);
    else if (npl <= 4) MORTAR_TAIL(4);
    else if (npl <= 6) MORTAR_TAIL(6);
    else if (npl <= 8) MORTAR_TAIL(8);
    else MORTAR_TAIL(16);
#undef MORTAR_TAILP
#undef MORTAR_TAIL
    return check_launch("router tail");
}

// xn: the rows of x (bf16) are RMS-normalised on the way in and written there; null: they are taken as they are.
static int launch_router(const void *x, bool x_is_f32, int64_t B, int32_t d, int64_t ldx, const uint16_t *norm_w, float norm_eps, uint16_t *xn,
                         const float *wq, const float *iter_vec, const float *ln_w, const float *ln_b, float ln_eps, const float *ka, const float *kb,
                         int32_t nsk, const float *bias, int32_t n, int32_t k, float *qv, float *logits_out, float *gates, uint8_t *active, void *stream) {
    if (!x || !wq || !ln_w || !ln_b || !ka || !kb || !bias || !qv || !gates)
        return mortar_fail(MORTAR_ERR_ARG, "router: null pointer");
    if (B <= 0 || B > 64) return mortar_fail(MORTAR_ERR_LIMIT, "router: the fused front end serves 1..64 tokens (got %lld)", (long long)B);
    if (d <= 0 || d % 8 || d > 8192 || ldx < d || ldx % (x_is_f32 ? 4 : 8))
        return mortar_fail(MORTAR_ERR_ARG, "router: d must be a multiple of 8 up to 8192 and ldx >= d, 16-byte aligned rows");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(wq) | reinterpret_cast<uintptr_t>(ka) | reinterpret_cast<uintptr_t>(kb)) & 15)
        return mortar_fail(MORTAR_ERR_ARG, "router: x, wq, ka and kb must be 16-byte aligned");
    if (n <= 0 || k <= 0 || nsk <= 0) return mortar_fail(MORTAR_ERR_ARG, "router: n, k, nsk must be positive");
    if (n > 64 * MAXPL_LIMIT) return mortar_fail(MORTAR_ERR_LIMIT, "router: n=%d exceeds %d clusters", n, 64 * MAXPL_LIMIT);
    if ((int64_t)nsk * nsk > 2048)
        return mortar_fail(MORTAR_ERR_LIMIT, "router: %d x %d product keys exceed the 2048 the fused front end ranks", nsk, nsk);
    if (xn) {       // one workgroup writes xn while the others still read the rows and the norm's weights
        const auto apart = [xn, B, d](const uint16_t *p, int64_t values) { return !p || p + values <= xn || xn + B * d <= p; };
        if (!apart(static_cast<const uint16_t *>(x), (B - 1) * ldx + d) || !apart(norm_w, d))
            return mortar_fail(MORTAR_ERR_ARG, "norm_router: xn overlaps x or norm_w");
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 pg((unsigned)((d + 3) / 4)), blk(256);
    // From 5 bf16 tokens up the projection runs on the matrix cores (2048 x 2048, with the tail: 5 tokens 13.6 -> 12.0 us, 16 19.5 -> 12.4,
    // 64 46 -> 15.6; 4 tokens 11.0 against 11.8); fp32 activations, wider rows and fewer tokens take one wave per output.
    const bool aligned = ((reinterpret_cast<uintptr_t>(qv) | reinterpret_cast<uintptr_t>(iter_vec)) & 15) == 0;
    const uint16_t *xb = static_cast<const uint16_t *>(x);
    int rc;
    // The norm inside the projection, whole routed step with a launch of its own against it, d_model 2048: 4 rows 25.7 -> 22.5 us, 8 26.2 -> 25.5,
    // 16 28.1 -> 27.1; 1024, 16 rows 20.8 -> 20.2.  A second tile of tokens loses: 24 rows 31.4 -> 33.0, 1024 21.4 -> 22.0.
    if (xn && (d > 2048 || B > 16 || (B > 4 && !aligned) || ((reinterpret_cast<uintptr_t>(xn) | reinterpret_cast<uintptr_t>(norm_w)) & 15))) {
        if ((rc = mortar_rmsnorm_bf16(xb, B, d, ldx, norm_w, norm_eps, xn, d, stream))) return rc;
        x = xb = xn; ldx = d; xn = nullptr;
        if (reinterpret_cast<uintptr_t>(x) & 15) return mortar_fail(MORTAR_ERR_ARG, "router: xn must be 16-byte aligned");
    }
    if (!x_is_f32 && B > 4 && d <= 2048 && aligned) {
        rc = mortar_router_project_skinny(xb, B, d, ldx, wq, d, iter_vec, qv, d, stream, norm_w, norm_eps, xn);
    } else if (xn) {
        const int smem = (B == 1 ? 1 : 4) * d * 2;
        if (B == 1) hipLaunchKernelGGL(router_norm_project_kernel<1>, pg, blk, smem, st, xb, (int)B, d, ldx, norm_w, norm_eps, xn, wq, iter_vec, qv);
        else hipLaunchKernelGGL(router_norm_project_kernel<4>, pg, blk, smem, st, xb, (int)B, d, ldx, norm_w, norm_eps, xn, wq, iter_vec, qv);
        rc = check_launch("router projection");
    } else {
#define MORTAR_PROJ(TB, F) hipLaunchKernelGGL((router_project_kernel<TB, F>), pg, blk, 0, st, x, (int)B, d, ldx, wq, iter_vec, qv)
        if (x_is_f32) { if (B == 1) MORTAR_PROJ(1, true); else if (B <= 4) MORTAR_PROJ(4, true); else if (B <= 8) MORTAR_PROJ(8, true); else MORTAR_PROJ(16, true); }
        else { if (B == 1) MORTAR_PROJ(1, false); else if (B <= 4) MORTAR_PROJ(4, false); else if (B <= 8) MORTAR_PROJ(8, false); else MORTAR_PROJ(16, false); }
#undef MORTAR_PROJ
        rc = check_launch("router projection");
    }
    if (rc) return rc;
    return launch_tail(qv, B, d, d, nullptr, ln_w, ln_b, ln_eps, ka, kb, nsk, bias, n, k, logits_out, gates, active, st);
}

extern "C" int mortar_router_bf16(const void *x, int32_t x_is_f32, int64_t B, int32_t d, int64_t ldx, const float *wq,
                                  const float *iter_vec, const float *ln_w, const float *ln_b, float ln_eps,
                                  const float *ka, const float *kb, int32_t nsk, const float *bias, int32_t n,
                                  int32_t k, float *qv, float *logits_out, float *gates, uint8_t *active,
                                  void *stream) {
    return launch_router(x, x_is_f32 != 0, B, d, ldx, nullptr, 0.f, nullptr, wq, iter_vec, ln_w, ln_b, ln_eps, ka, kb, nsk, bias, n, k, qv, logits_out,
                         gates, active, stream);
}

extern "C" int mortar_norm_router_bf16(const uint16_t *x, int64_t B, int32_t d, int64_t ldx, const uint16_t *norm_w, float norm_eps, uint16_t *xn,
                                       const float *wq, const float *iter_vec, const float *ln_w, const float *ln_b, float ln_eps,
                                       const float *ka, const float *kb, int32_t nsk, const float *bias, int32_t n, int32_t k, float *qv,
                                       float *logits_out, float *gates, uint8_t *active, void *stream) {
    if (!xn) return mortar_fail(MORTAR_ERR_ARG, "norm_router: null pointer");
    return launch_router(x, false, B, d, ldx, norm_w, norm_eps, xn, wq, iter_vec, ln_w, ln_b, ln_eps, ka, kb, nsk, bias, n, k, qv, logits_out, gates,
                         active, stream);
}

extern "C" int mortar_router_tail_f32(const float *qv, int64_t N, int32_t d, int64_t ldq, const float *iter_vec,
                                      const float *ln_w, const float *ln_b, float ln_eps, const float *ka, const float *kb,
                                      int32_t nsk, const float *bias, int32_t n, int32_t k, float *logits_out, float *gates,
                                      uint8_t *active, void *stream) {
    if (!qv || !ln_w || !ln_b || !ka || !kb || !bias || !gates) return mortar_fail(MORTAR_ERR_ARG, "router tail: null pointer");
    if (N <= 0 || N > ((int64_t)1 << 31) / (n > 0 ? n : 1)) return mortar_fail(MORTAR_ERR_ARG, "router tail: N=%lld out of range", (long long)N);
    if (d <= 0 || d % 8 || d > 8192 || ldq < d || ldq % 4)
        return mortar_fail(MORTAR_ERR_ARG, "router tail: d must be a multiple of 8 up to 8192 and ldq >= d, 16-byte aligned rows");
    if ((reinterpret_cast<uintptr_t>(qv) | reinterpret_cast<uintptr_t>(iter_vec) | reinterpret_cast<uintptr_t>(ln_w) |
         reinterpret_cast<uintptr_t>(ln_b) | reinterpret_cast<uintptr_t>(ka) | reinterpret_cast<uintptr_t>(kb)) & 15)
        return mortar_fail(MORTAR_ERR_ARG, "router tail: qv, iter_vec, ln_w, ln_b, ka and kb must be 16-byte aligned");
    if (n <= 0 || k <= 0 || nsk <= 0) return mortar_fail(MORTAR_ERR_ARG, "router tail: n, k, nsk must be positive");
    if (n > 64 * MAXPL_LIMIT) return mortar_fail(MORTAR_ERR_LIMIT, "router tail: n=%d exceeds %d clusters", n, 64 * MAXPL_LIMIT);
    if ((int64_t)nsk * nsk > n && (int64_t)nsk * nsk > 1024)
        return mortar_fail(MORTAR_ERR_LIMIT, "router tail: %d x %d product keys for %d groups exceed the 1024 the kernel ranks", nsk, nsk, n);
    hipStream_t st = static_cast<hipStream_t>(stream);
    // One workgroup per token, its sub-key rows in registers, while that is one round of the chip: a chain of 6 to 16 us against the
    // 12 to 25 us of the launches below, whatever the number of tokens (65 tokens, 2048 values: 19 x 19 keys for 352 groups 24.5 ->
    // 15.5 us, 4 x 4 for 16 16.1 -> 6.5; 512: 24.9 -> 17.6; 700: 25.3 against 27.7; 2000 with 4 x 4: 17.4 -> 12.6).
    if (d <= 2048 && (nsk <= 4 ? N <= 2048 : nsk <= 20 && N <= 512))
        return launch_tail(qv, N, d, ldq, iter_vec, ln_w, ln_b, ln_eps, ka, kb, nsk, bias, n, k, logits_out, gates, active, st);
    if (d <= 4096 && nsk <= 32 && 2 * nsk <= n) {      // two launches; wider rows, more keys or fewer groups than scores: one
        const dim3 sg((unsigned)((N + 15) / 16)), rg((unsigned)((N + 3) / 4));
        const int ch = (d / 2 + 63) / 64;
#define MORTAR_SCORES(KT, CH) hipLaunchKernelGGL((router_scores_kernel<KT, CH>), sg, dim3(512), 0, st, qv, N, d, ldq, iter_vec, ln_w, ln_b, ln_eps, \
                                                 ka, kb, nsk, n, gates)
#define MORTAR_SCORESK(KT) do { if (ch <= 8) MORTAR_SCORES(KT, 8); else if (ch <= 16) MORTAR_SCORES(KT, 16); else MORTAR_SCORES(KT, 32); } while (0)
        if (nsk <= 16) MORTAR_SCORESK(1);
        else MORTAR_SCORESK(2);
#undef MORTAR_SCORESK
#undef MORTAR_SCORES
        const size_t rs = (size_t)4 * (2 * nsk + n) * sizeof(float);
        const int pl = (n + 63) / 64;
#define MORTAR_RANK(PL) hipLaunchKernelGGL((router_rank_kernel<PL>), rg, dim3(256), rs, st, N, nsk, bias, n, k, logits_out, gates, active)
        if (pl <= 1) MORTAR_RANK(1);
        else if (pl <= 2) MORTAR_RANK(2);
        else if (pl <= 4) MORTAR_RANK(4);
        else if (pl <= 6) MORTAR_RANK(6);
        else MORTAR_RANK(16);
#undef MORTAR_RANK
        return check_launch("router tail");
    }
    // a thread holds J float4 pieces of every row of its group (J = 1, 2, 4 or 8 for d <= 1024 J) and tt = min(4, 8 / J)
    // tokens share a group, so the normalised rows take at most 32 KB of LDS
    const int J = d <= 1024 ? 1 : d <= 2048 ? 2 : d <= 4096 ? 4 : 8;
    const int tt = 8 / J < TAIL_TT ? 8 / J : TAIL_TT;
    const size_t smem = ((size_t)tt * d + (size_t)tt * 2 * nsk + (size_t)tt * n + 16) * sizeof(float);
    const int64_t groups = (N + tt - 1) / tt;
    const dim3 grid((unsigned)(groups < 3072 ? groups : 3072)), blk(256);
    const int npl = (n + 63) / 64;
#define MORTAR_TAILG(PL, JJ) hipLaunchKernelGGL((router_tail_group_kernel<PL, JJ>), grid, blk, smem, st, qv, N, d, ldq, iter_vec, ln_w, \
                                               ln_b, ln_eps, ka, kb, nsk, bias, n, k, tt, logits_out, gates, active)
#define MORTAR_TAILJ(PL) do { if (J == 1) MORTAR_TAILG(PL, 1); else if (J == 2) MORTAR_TAILG(PL, 2); else if (J == 4) MORTAR_TAILG(PL, 4); \
                              else MORTAR_TAILG(PL, 8); } while (0)
    if (npl <= 2) MORTAR_TAILJ(2);
    else if (npl <= 6) MORTAR_TAILJ(6);
    else MORTAR_TAILJ(16);
#undef MORTAR_TAILJ
#undef MORTAR_TAILG
    return check_launch("router tail");
}

extern "C" int mortar_remoe_route(const uint8_t *active, int64_t M, int32_t n, int32_t tile, int32_t *tok_cnt,
                                  uint8_t *tok_list, void *stream) {
    if (!active || !tok_cnt || !tok_list) return mortar_fail(MORTAR_ERR_ARG, "remoe_route: null pointer");
    if (M <= 0 || n <= 0) return mortar_fail(MORTAR_ERR_ARG, "remoe_route: M and n must be positive");
    if (tile <= 0 || tile > 256 || (tile % 16 && tile != 4)) return mortar_fail(MORTAR_ERR_LIMIT, "remoe_route: tile must be 4 or a multiple of 16, at most 256");
    const unsigned nt = (unsigned)((M + tile - 1) / tile);
    hipLaunchKernelGGL(remoe_route_kernel, dim3(nt, (unsigned)((n + 63) / 64)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), active, M, n, tile, tok_cnt, tok_list);
    return check_launch("remoe_route");
}

extern "C" int mortar_route_flags(const float *gates, int64_t B, int32_t n_clusters, int64_t ldg, int32_t d_ff,
                                  int32_t *row_act, int64_t ldr, int32_t *col_act, int64_t ldc, void *stream) {
    if (!gates || (!row_act && !col_act)) return mortar_fail(MORTAR_ERR_ARG, "route_flags: null pointer");
    if (B <= 0 || n_clusters <= 0 || d_ff <= 0 || d_ff % 16 || d_ff % n_clusters)
        return mortar_fail(MORTAR_ERR_ARG, "route_flags: d_ff must be a multiple of 16 and of n_clusters");
    const int64_t total = B * (d_ff / 16);
    hipLaunchKernelGGL(route_flags_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), gates, B, n_clusters, ldg, d_ff, row_act, ldr, col_act, ldc);
    return check_launch("route_flags");
}

extern "C" int mortar_rmsnorm_bf16(const uint16_t *x, int64_t M, int32_t d, int64_t ldx, const uint16_t *w,
                                   float eps, uint16_t *y, int64_t ldy, void *stream) {
    if (!x || !y) return mortar_fail(MORTAR_ERR_ARG, "rmsnorm: null pointer");
    if (M <= 0 || d <= 0 || ldx < d || ldy < d) return mortar_fail(MORTAR_ERR_ARG, "rmsnorm: bad shape");
    const bool units = d % 8 == 0 && ldx % 8 == 0 && ldy % 8 == 0 &&
                       ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
    if (units) {
        // few rows: a workgroup each
        const int rpw = M <= 1024 ? 1 : 4;
        // The loops where they are still the faster form: calls of 12 to 17 MB, whose waves all fit the chip at once, of rows that fill their registers.
        // us, loops against registers: 8192 rows of 1024 values 7.6 against 8.0, 4096 of 2048 8.1 against 8.4.  Beside the range: 3000 rows of 2048 6.7 against
        // 6.5, 6000 10.8 against 9.5, 10000 of 1024 8.8 against 8.3; 1536 values, 4096 rows 6.5 either way; 1792 values, 5000 rows 9.1 against 8.7.
        const bool loops = (d == 1024 || d == 2048) && M * d > (6 << 20) && M * d < (17 << 19);
        const auto kern = loops ? rmsnorm_rows_kernel<0> : d <= 512 ? rmsnorm_rows_kernel<1> : d <= 1024 ? rmsnorm_rows_kernel<2> : d <= 2048 ? rmsnorm_rows_kernel<4> : d <= 4096 ? rmsnorm_rows_kernel<8>
                        : d <= 8192 ? rmsnorm_rows_kernel<16> : rmsnorm_rows_kernel<0>;
        hipLaunchKernelGGL(kern, dim3((unsigned)((M + rpw - 1) / rpw)), dim3(64 * rpw), 0, static_cast<hipStream_t>(stream),
                           x, M, d, ldx, w, eps, y, ldy);
    } else
        hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)M), dim3(256), 0, static_cast<hipStream_t>(stream), x, M, d,
                           ldx, w, eps, y, ldy);
    return check_launch("rmsnorm");
}
