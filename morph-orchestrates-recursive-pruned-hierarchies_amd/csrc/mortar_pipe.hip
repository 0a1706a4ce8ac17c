// Calls of 65 to some hundred rows on a matrix of several K segments, and decode calls of wide `down` matrices (mortar_smallm_pipe), also with
// the POST write: 16-token tiles, the segments through two LDS buffers.
//
// The K-segmented kernel stages a segment behind a barrier pair and its small tiles then wait for their first weight batch: with the few
// workgroups that some hundred rows make, every segment paid both round trips (`down` of d_model 2048 at 200 rows: 11 us, of which the
// products are 2).  Here the next segment's activations are in flight, in registers, while a segment is multiplied; they are stored into
// the other buffer behind one barrier per segment, and the first weight batch is requested in front of it.  A unit is spread over up to
// four waves (whole octets each) as far as the workgroups stay within one round of the chip.
//
// us per launch (graph replay), before -> now: `down` of d_model 1536 at 150 / 500 rows 8.4 -> 6.7, 10.2 -> 9.1, of 2048 at 65 / 200 / 500 rows
// 9.0 -> 8.1, 11.1 -> 9.1, 13.3 -> 11.9, of 3072 at 100 rows 18.2 -> 11.0, of 4096 at 65 / 200 rows 18.6 -> 13.4, 24.9 -> 19.8; gate_up of 3072 at
// 65..128 rows 13.1..14.1 -> 11.6..11.8.  Two units per wave, for more rows, were slower than the kernels that serve them (3072, 400 rows: 21.6
// against 25.4).
#include "mortar_spmm_core.h"

#include <type_traits>

namespace {

constexpr int PIPE_WAVES = 16, PIPE_MT = 16;
constexpr int PIPE_KQ = 5;        // 16-byte pieces per lane of a segment's tile: 16 waves x 5 x 2 block-columns >= the widest segment (155)

// NACC rows per unit (1 plain, 2 gate/up).  PW waves per unit: one wave takes all its rows, two or four take a row, or a run of a row's
// octets, each.  MASKED: x is zero where the input mask is (plain products).  HC: the results go into the POST write (kernels of their own: its code in the
// epilogue of the others cost them 0.05 to 0.15 us).
template <int NACC, bool MASKED, int PW, int CODE, bool HC>
__global__ void __launch_bounds__(PIPE_WAVES * 64) mortar_pipe_kernel(const SpmmParams p0) {
    constexpr int UW = PIPE_WAVES / PW, RW = PW == 1 ? NACC : 1, CS = PW == 1 ? 1 : PW / NACC;
    static_assert(PW == 1 || PW % NACC == 0, "a wave takes a unit, a row or a run of a row's octets");
    SpmmView p = mortar_view(p0);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int buf_bytes = tile_bytes(PIPE_MT, p.seg_cb);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4, bsel = g >> 1, hsel = g & 1;
    // xcd_map: the workgroups that share a token tile run on one XCD, whose L2 then holds it once (mortar_resident_kernel)
    const int wg = p.xcd_map ? (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    if (wg >= p.n_mtiles * p.n_split) return;
    const int mt = wg / p.n_split, m0 = mt * PIPE_MT;
    const int ug = wave / PW, wq = wave % PW, a0 = PW == 1 ? 0 : wq / CS, c = wq % CS;
    const int pos = (wg - mt * p.n_split) * UW + ug;
    const bool on = pos < p.n_units;
    const uint32_t lane_xo = (uint32_t)(hsel * 16 + n * 32);
    const uint32_t tk[1] = {(uint32_t)n};

    // a wave instruction stages 16 rows x 64 bytes (two block-columns) of x
    const int rlast = (p.M - m0 < PIPE_MT ? p.M - m0 : PIPE_MT) - 1, row = lane >> 2;
    const MORTAR_GLOBAL char *xr = p.x + (int64_t)(m0 + (row < rlast ? row : rlast)) * p.ldx * 2;
    u32x4_t v[PIPE_KQ];
    auto fetch = [&](int c0, int ncb) {
#pragma unroll
        for (int k = 0; k < PIPE_KQ; ++k) {
            const int u = (wave + k * PIPE_WAVES) * 4 + (lane & 3);
            const int uc = c0 * 2 + (u < 2 * ncb ? u : 2 * ncb - 1);
            v[k] = *(const MORTAR_GLOBAL u32x4_t *)(xr + (uint32_t)uc * 16u);
            if (MASKED && p.active[(int64_t)(m0 + (row < rlast ? row : rlast)) * p.n_clusters + uc * 8 / p.cluster_size] == 0) v[k] = u32x4_t{0u, 0u, 0u, 0u};
        }
    };
    auto put = [&](unsigned char *lb, int ncb) {
#pragma unroll
        for (int k = 0; k < PIPE_KQ; ++k) {
            const int u = (wave + k * PIPE_WAVES) * 4 + (lane & 3);
            if (row <= rlast && u < 2 * ncb) *reinterpret_cast<u32x4_t *>(lb + (uint32_t)(u >> 1) * (PIPE_MT * 32) + row * 32 + (u & 1) * 16) = v[k];
        }
    };
    auto width = [&](int sg) { return p.Cb - sg * p.seg_cb < p.seg_cb ? p.Cb - sg * p.seg_cb : p.seg_cb; };

    f32x4_t acc[RW][1];
#pragma unroll
    for (int a = 0; a < RW; ++a) acc[a][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Parts of a segment: a = row of the unit.  Descriptors are requested one segment ahead.
    u32x4_t dn[RW];
    int unit = -1;
    auto descriptors = [&](int sg) {
#pragma unroll
        for (int a = 0; a < RW; ++a) dn[a] = mortar_part_desc<NACC>(p, pos, sg, a0 + a);
    };
    descriptors(0);
    fetch(0, width(0));
    mortar_resolve_scale<CODE>(p);

    auto segment = [&](int sg, auto last) {
        constexpr bool LAST = decltype(last)::value;
        unsigned char *lb = smem + (sg & 1) * buf_bytes;
        int g0[RW], g1[RW], nb[RW];
#pragma unroll
        for (int a = 0; a < RW; ++a) {
            int s = on ? __builtin_amdgcn_readfirstlane((int)dn[a][0]) : 0, e = on ? __builtin_amdgcn_readfirstlane((int)dn[a][1]) : 0;
            int b = __builtin_amdgcn_readfirstlane((int)dn[a][2]);
            if (a == 0) unit = on ? __builtin_amdgcn_readfirstlane((int)dn[a][3]) : -1;
            if (CS > 1) {
                const int no = e - s, lo = no * c / CS, hi = no * (c + 1) / CS;
                b = b - 8 * lo < 8 * (hi - lo) ? b - 8 * lo : 8 * (hi - lo);
                e = s + hi; s += lo;
            }
            g0[a] = s; g1[a] = e; nb[a] = s < e ? b : 0;
        }
        // First batches are requested one part ahead, the first part's in front of the barrier, always and in a fixed order (an empty part
        // reads octet 0), as in the K-segmented kernel.  (Requesting it a segment ahead instead was 1 to 4 % slower.)
        constexpr int FIRST = 8 * RES_GROUPS;
        auto first_batch = [&](MortarBatch &bb, int a) {
            const bool any = g0[a] < g1[a];
            mortar_load_batch<CODE>(p, bb, any ? g0[a] : 0, any ? g1[a] : 1, n, bsel, hsel);
        };
        MortarBatch bq;
        first_batch(bq, 0);
        if (!LAST) descriptors(sg + 1);
        put(lb, width(sg));
        __syncthreads();
        if (!LAST) fetch((sg + 1) * p.seg_cb, width(sg + 1));
#pragma unroll
        for (int a = 0; a < RW; ++a) {
            MortarBatch bn;
            if (a + 1 < RW) first_batch(bn, a + 1);
            const uint4 *lx = reinterpret_cast<const uint4 *>(lb);
            mortar_row_part<1, PIPE_MT, false, CODE, true>(p, lx, bq, g0[a], g1[a], nb[a] < FIRST ? nb[a] : FIRST, lane_xo, tk, 1, n, bsel, hsel, acc[a]);
            if (nb[a] > FIRST) {
                MortarBatch bt;
                mortar_load_batch<CODE>(p, bt, g0[a] + RES_GROUPS, g1[a], n, bsel, hsel);
                mortar_row_part<1, PIPE_MT, false, CODE>(p, lx, bt, g0[a] + RES_GROUPS, g1[a], nb[a] - FIRST, lane_xo, tk, 1, n, bsel, hsel, acc[a]);
            }
            if (a + 1 < RW) bq = bn;
        }
    };
    for (int sg = 0; sg + 1 < p.nseg; ++sg) segment(sg, std::false_type{});
    segment(p.nseg - 1, std::true_type{});

    const bool has_gates = p.gates != nullptr;
    if constexpr (PW > 1) {           // the partial sums of a unit meet where the tiles were
        f32x4_t *red = reinterpret_cast<f32x4_t *>(smem);
        __syncthreads();
        red[wave * 64 + lane] = acc[0][0];
        __syncthreads();
        if (wq != 0 || unit < 0) return;
        f32x4_t s[NACC][1];
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            s[a][0] = red[(wave + a * CS) * 64 + lane];
#pragma unroll
            for (int w = 1; w < CS; ++w) s[a][0] += red[(wave + a * CS + w) * 64 + lane];
        }
        mortar_store_tile<1, NACC, CODE, HC>(p, unit, m0, tk, PIPE_MT, n, g, has_gates, s[0], s[NACC - 1]);
    } else if (unit >= 0) {
        mortar_store_tile<1, NACC, CODE, HC>(p, unit, m0, tk, PIPE_MT, n, g, has_gates, acc[0], acc[RW - 1]);
    }
}

template <int NACC, bool MASKED, int PW, int CODE, bool HC = false>
int launch(SpmmParams &p, hipStream_t st) {
    const int smem = 2 * tile_bytes(PIPE_MT, p.seg_cb) > PIPE_WAVES * 1024 ? 2 * tile_bytes(PIPE_MT, p.seg_cb) : PIPE_WAVES * 1024;
    if (p.seg_cb > PIPE_KQ * PIPE_WAVES * 2 || smem > 160 * 1024) return mortar_fail(MORTAR_ERR_LIMIT, "segment of %d block-columns does not fit", p.seg_cb);
    static bool attr_done = false;
    auto kern = mortar_pipe_kernel<NACC, MASKED, PW, CODE, HC>;
    int rc = mortar_allow_big_lds(kern, attr_done);
    if (rc) return rc;
    p.n_mtiles = (p.M + PIPE_MT - 1) / PIPE_MT;
    p.n_split = (p.n_units + PIPE_WAVES / PW - 1) / (PIPE_WAVES / PW);
    int64_t grid = mortar_grid_width(p, 1);
    // Without the renumbering ids go round the XCDs, and with it the units: an XCD reads an eighth of the weights and all of x.  With it, all of
    // the weights and an eighth of x.  The lines cross where x is about twice the weights (`down`, 300 rows at d_model 2048: 11.3 us either
    // way; 400 rows 13.3 against 11.5; d_model 4096, 100 rows 13.6 against 16.9).
    if ((int64_t)p.M * p.Cb * 32 < 2 * (int64_t)p.Rb * p.nseg * p.avg_octets * 1088) {
        p.xcd_map = 0;
        grid = (int64_t)p.n_mtiles * p.n_split;
    }
    if ((rc = mortar_launch_check(grid, 1))) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(PIPE_WAVES * 64), smem, st, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MORTAR_OK : mortar_fail(MORTAR_ERR_HIP, "spmm launch: %s", hipGetErrorString(e));
}

template <int NACC, bool MASKED, int CODE>
int launch_waves(int pw, SpmmParams &p, hipStream_t st) {
    if constexpr (NACC == 1) {
        if (p.hc_h)
            return pw == 4 ? launch<1, MASKED, 4, CODE, true>(p, st) : pw == 2 ? launch<1, MASKED, 2, CODE, true>(p, st) : launch<1, MASKED, 1, CODE, true>(p, st);
    }
    return pw == 4 ? launch<NACC, MASKED, 4, CODE>(p, st) : pw == 2 ? launch<NACC, MASKED, 2, CODE>(p, st) : launch<NACC, MASKED, 1, CODE>(p, st);
}

template <int CODE>
int launch_kind(int kind, int pw, SpmmParams &p, hipStream_t st) {
    return kind == 1 ? launch_waves<2, false, CODE>(pw, p, st) : kind == 3 ? launch_waves<1, true, CODE>(pw, p, st) : launch_waves<1, false, CODE>(pw, p, st);
}

}  // namespace

int mortar_pipe_launch(int kind, int code, SpmmParams &p, hipStream_t st) {
    if (kind == 2 || p.M > MLP_SEPARATE_MAX_ROWS || p.nseg < 2 || 2 * tile_bytes(PIPE_MT, p.seg_cb) > 160 * 1024) return -1;
    const int64_t tiles = (p.M + PIPE_MT - 1) / PIPE_MT;
    // Plain products whose 8- or 16-token tiles of all K make few workgroups run those (`down` of d_model 1024 at 100 / 200 / 500 rows: 5.2 / 5.5 /
    // 6.3 us against 6.3 / 6.4 / 7.0 here; of 1536 at 65 rows 6.0 against 6.5, at 100 rows 6.9 against 6.5).
    if (kind != 1 && p.M <= MORTAR_PARTSPLIT_MAX && (p.M + 7) / 8 * (int64_t)((p.n_units + 7) / 8) <= 128) return -1;
    if (mortar_wide_tile_better(kind, p)) return -1;
    for (int pw : {4, 2, 1}) {
        const int units = PIPE_WAVES / pw;
        if (tiles * ((p.n_units + units - 1) / units) > 256) continue;
        switch (code) {
            case CODE_4BIT | CODE_UNIFORM: return launch_kind<CODE_4BIT | CODE_UNIFORM>(kind, pw, p, st);
            case CODE_4BIT: return launch_kind<CODE_4BIT>(kind, pw, p, st);
            default: return launch_kind<CODE_2BIT>(kind, pw, p, st);
        }
    }
    return -1;
}
