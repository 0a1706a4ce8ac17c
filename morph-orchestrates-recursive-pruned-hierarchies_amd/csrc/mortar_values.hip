// Block-sparse product over stored bf16 block VALUES: y = x W^T with W given as the reference's BCSR arrays
// (mortar_data [nnz,16,16], mortar_offsets, mortar_column_indices), whatever values the blocks hold.
//
// This is the arithmetic of the reference's stk_dds operator itself (morph/sparse/stk/backend/custom_ops.py:35-56,
// kernel triton_kernels.py:170-230 with trans_B: bf16 operands, fp32 accumulation, bf16 store), which multiplies any
// bf16 data.  The ternary kernels of this library stream 2- and 4-bit codes and therefore serve ternary blocks only; this
// kernel is the general form behind the operator-level drop-in.  It needs no unpacking at all: a block row of 16 values
// is 32 contiguous bytes, so the lane that holds row n, column half h of a block pair in the MFMA's A operand fetches
// exactly its 16 bytes with one global load.
#include "mortar_spmm_core.h"

#include <cstdint>

namespace {

constexpr int VAL_WAVES = 16;                        // all of K in one tile
constexpr int VAL_CW = 12, VAL_LOADERS = 4;          // wider K: consumer and loader waves
constexpr int VAL_SEG_CB = 38;                       // block-columns of a fine K segment: two buffers of 64 tokens fit LDS

struct ValArgs {
    const int32_t *row_ptr;     // [Rb + 1]
    const int32_t *seg_ptr;     // [Rb, nfine + 1]: first block of row r in fine K segment s (mortar_segment_ptr_host); null for one segment
    const int16_t *col;         // [nnz]
    const uint16_t *data;       // [nnz, 16, 16] bf16
    const uint16_t *x;
    uint16_t *y;
    int64_t ldx, ldy;
    int M, Rb, Cb, nnz;
    int seg_cb, nfine;          // fine K segments of seg_cb block-columns
    int sub;                    // fine segments that one LDS segment holds
    int n_split, per;           // workgroups that share a token tile; block-rows of one of them
    int unit;                   // all of K in one tile: block-rows that a wave draws at a time (1 or 2)
};

// Tile layout in LDS: [pair of block-columns][token][64 bytes].  A wave instruction copies 16 tokens x 64 bytes straight from
// global memory (asynchronously, no registers; four lanes read 64 contiguous bytes).  The four 16-byte units of a token are
// stored in the order unit ^ s(token / 4), s = 0, 3, 2, 1 (mortar_unit_swz): the lanes that LDS serves together then touch
// every bank once.  The byte address
// of (column c, half h, token n) is enc(c) ^ lane with enc(c) = (c / 2) * MT * 64 + (c & 1) * 32 and a lane constant.
template <int MT>
__device__ __forceinline__ int val_enc(int c) { return (c >> 1) * (MT * 64) + (c & 1) * 32; }

// Copies block-columns [c0, c0 + ncb) of the tile at token m0 into `dst`, as loader `w` of `nw`.  Tokens past M repeat the last
// one, a missing second column of the last pair repeats the first: both feed results that are never stored or never read.
template <int MT>
__device__ __forceinline__ void val_copy(const ValArgs &a, unsigned char *dst, int m0, int c0, int ncb, int i, int lane) {
    constexpr int TG = MT / 16;
    const int t = lane >> 2, u = (lane & 3) ^ mortar_unit_swz(t);
    const int tg = i % TG, pr = i / TG;
    const int tok = m0 + tg * 16 + t;
    int c = 2 * pr + (u >> 1);
    c = c < ncb ? c : ncb - 1;
    const uint16_t *src = a.x + (int64_t)(tok < a.M ? tok : a.M - 1) * a.ldx + (int64_t)(c0 + c) * 16 + (u & 1) * 8;
    mortar_load_to_lds((const MORTAR_GLOBAL char *)src, __builtin_amdgcn_readfirstlane(mortar_lds_addr(dst + (pr * MT + tg * 16) * 64)));
}
template <int MT>
__device__ __forceinline__ void val_stage(const ValArgs &a, unsigned char *dst, int m0, int c0, int ncb, int w, int nw, int lane) {
    for (int i = w; i < (ncb + 1) / 2 * (MT / 16); i += nw) val_copy<MT>(a, dst, m0, c0, ncb, i, lane);
}

// Four block pairs of one block-row part in registers: values as MFMA operands, the columns on lanes 0..3 of every 16-lane row.
struct ValBatch {
    u32x4_t A[4];
    int col;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t val_rsrc(const void *base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// Blocks j, j + 1, ... of a part with `cnt` blocks left (more than 8: the first 8).  The loads are bounded buffer loads: base
// and bound are scalar, the lane offset a constant, and values past the part's end arrive as zeros - no address arithmetic and
// no selects on the vector ALU.  Columns past the end repeat the last one of the part (a zero times an operand of another column
// could be 0 x inf).  Nothing here touches a loaded value: the wait for it stands at the product.
__device__ __forceinline__ void val_fetch(const ValArgs &a, ValBatch &b, int j, int cnt, uint32_t lane_o, int lane_k) {
    j = j < a.nnz ? j : a.nnz - 1;
    const int last = cnt > 0 ? cnt - 1 : 0, k = lane_k < last ? lane_k : last;
    b.col = (int)__builtin_amdgcn_raw_buffer_load_b16(val_rsrc(a.col + j, 16), k * 2, 0, 0);
    const __amdgpu_buffer_rsrc_t r = val_rsrc(reinterpret_cast<const char *>(a.data) + (int64_t)j * 512, cnt > 0 ? (cnt < 8 ? cnt : 8) * 512 : 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) b.A[u] = __builtin_amdgcn_raw_buffer_load_b128(r, lane_o + u * 1024, 0, 0);
}

// The batch's pairs against the tile of columns c0 .. at `lb`; the operands of the next pair are read before the current one is
// multiplied.
template <int MT>
__device__ __forceinline__ void val_multiply(const unsigned char *lb, const ValBatch &b, int cnt, int c0, uint32_t lane_x, f32x4_t (&acc)[MT / 16]) {
    constexpr int MSUB = MT / 16;
    if (cnt <= 0) return;
    const uint32_t enc = (uint32_t)val_enc<MT>(b.col - c0);
    u32x4_t B[2][MSUB];
    auto operands = [&](int u) {
        const unsigned char *p = lb + (mortar_row_bcast(enc, u) ^ lane_x);
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) B[u & 1][ms] = *reinterpret_cast<const u32x4_t *>(p + ms * 1024);
    };
    operands(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (2 * u >= cnt) break;
        if (u < 3) operands(u + 1);
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) acc[ms] = mortar_mfma(b.A[u], B[u & 1][ms], acc[ms]);
    }
}

// Results of two consecutive block-rows, stored together: the lane groups exchange halves, so that a lane holds 8 consecutive
// features of one row and a token's 32 features are one 64-byte piece (one row at a time, 32-byte pieces, the stores alone
// bound the wide products).  Bounded buffer stores drop the tokens past M and, for the last row of an odd count, row b.
template <int MT>
struct ValOut {
    __amdgpu_buffer_rsrc_t r;
    uint32_t off[MT / 16], odd;
    __device__ __forceinline__ ValOut(const ValArgs &a, int m0, int n, int g) {
        const int nt = a.M - m0 < MT ? a.M - m0 : MT;
        r = val_rsrc(a.y + (int64_t)m0 * a.ldy, (int)((nt - 1) * a.ldy * 2 + a.Rb * 32));
        odd = g & 1;
#pragma unroll
        for (int ms = 0; ms < MT / 16; ++ms) {
            const int t = ms * 16 + n;
            off[ms] = t < nt ? (uint32_t)(t * a.ldy * 2) + odd * 32 + (g >> 1) * 16 : 0xfffffff0u;
        }
    }
    __device__ __forceinline__ void store(int row, bool both, const f32x4_t (&a0)[MT / 16], const f32x4_t (&a1)[MT / 16]) const {
#pragma unroll
        for (int ms = 0; ms < MT / 16; ++ms) {
            u32x4_t v;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const auto s = __builtin_amdgcn_permlane16_swap(bf16_pack2(a0[ms][2 * h], a0[ms][2 * h + 1]), bf16_pack2(a1[ms][2 * h], a1[ms][2 * h + 1]), false, false);
                v[h] = s[0];
                v[2 + h] = s[1];
            }
            // The row goes into the vector offset: behind a 16-byte store with a scalar offset the compiler may overwrite the data
            // registers in the next instruction, and gfx950 then stores the new values in the last lanes of a row (seen with
            // `v_mov_b32` there; with a scalar offset the compiler assumes that no wait state is needed).
            __builtin_amdgcn_raw_buffer_store_b128(v, r, (both || !odd) && off[ms] != 0xfffffff0u ? off[ms] + (uint32_t)row * 32 : 0xfffffff0u, 0, 0);
        }
    }
};

// A uniform index array as scalar loads.
__device__ __forceinline__ int val_idx(const int32_t *p, int i) {
    return ((const __attribute__((address_space(4))) int32_t *)p)[__builtin_amdgcn_readfirstlane(i)];
}

// All of K in one tile.  The waves draw block-rows (a.unit = 2: pairs of them) from a counter, so that rows of any length keep
// all of them busy; a wave's batches form one stream across rows, requested two ahead of their products.  Narrow K is bound by
// the results and the values together (16384 x 768 x 4096 at 25 %, 134 MB of results, a fill of which takes 21 us: 84 -> 51 us in a
// loop over the same buffers, 57 over six sets of them, 65..69 in the trace of a training step, 153 MB written there; rows one at a
// time took a quarter longer), wide K by the values from the L2, once per 32 tokens (4096 x 2048 x 11264: 102 -> 83 us, 18 TB/s of values).
template <int MT>
__global__ void __launch_bounds__(VAL_WAVES * 64) values_resident_kernel(const ValArgs a) {
    constexpr int MSUB = MT / 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    int *next_row = reinterpret_cast<int *>(smem + ((a.Cb + 1) / 2) * (MT * 64));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4, bsel = g >> 1, hsel = g & 1;
    const int mt = blockIdx.x / a.n_split, sp = blockIdx.x % a.n_split;
    const int m0 = mt * MT;
    const int r0 = sp * a.per, r1 = r0 + a.per < a.Rb ? r0 + a.per : a.Rb;
    const uint32_t lane_x = (uint32_t)(n * 64 + (hsel ^ mortar_unit_swz(n)) * 16);
    const uint32_t lane_o = (uint32_t)(bsel * 512 + n * 32 + hsel * 16);
    const int lane_k = 2 * (n & 3) + bsel;
    const ValOut<MT> out(a, m0, n, g);
    struct Unit { int r, p0, p1, p2; };                   // rows r and r + 1 (unit == 1: r alone): blocks p0 .. p1 and p1 .. p2
    auto load_unit = [&](int r) {
        Unit q{r, 0, 0, 0};
        if (r < r1) {
            q.p0 = val_idx(a.row_ptr, r);
            q.p1 = val_idx(a.row_ptr, r + 1);
            q.p2 = a.unit == 2 && r + 1 < r1 ? val_idx(a.row_ptr, r + 2) : q.p1;
        }
        return q;
    };
    Unit u = load_unit(r0 + a.unit * wave), v{r1, 0, 0, 0};
    // request cursor: part f of the sequence u row 0, u row 1, v row 0, v row 1; blocks fj .. fje
    int f = 0, fj = u.p0, fje = u.p1;
    auto request = [&](ValBatch &b) {
        val_fetch(a, b, fj, fje - fj, lane_o, lane_k);
        fj += 8;
        if (fj >= fje) {
            ++f;
            const int up1 = u.p1, up2 = u.p2, vp0 = v.p0, vp1 = v.p1, vp2 = v.p2;
            fj = f == 1 ? up1 : f == 2 ? vp0 : vp1;
            fje = f == 1 ? up2 : f == 2 ? vp1 : vp2;
        }
    };
    if (tid == 0) *next_row = r0 + a.unit * VAL_WAVES;
    val_stage<MT>(a, smem, m0, 0, a.Cb, wave, VAL_WAVES, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    auto draw = [&]() {
        int d = 0;
        if (lane == 0) d = atomicAdd(next_row, a.unit);
        return d;
    };
    if (u.r >= r1) return;
    v = load_unit(__builtin_amdgcn_readfirstlane(draw()));
    int drawn = draw();
    ValBatch b0, b1, b2;
    request(b0);
    request(b1);
    f32x4_t acc[MSUB], first[MSUB];
#pragma unroll
    for (int ms = 0; ms < MSUB; ++ms) acc[ms] = first[ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int k = 0, j = u.p0, je = u.p1;                       // part of u that is being multiplied
    // one batch; false when the wave's rows are done
    auto step = [&](const ValBatch &c, ValBatch &nx) {
        request(nx);
        val_multiply<MT>(smem, c, je - j, 0, lane_x, acc);
        j += 8;
        if (j < je) return true;
        if (k == 0) {
#pragma unroll
            for (int ms = 0; ms < MSUB; ++ms) {
                first[ms] = acc[ms];
                acc[ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
            k = 1; j = u.p1; je = u.p2;
            return true;
        }
        out.store(u.r, a.unit == 2 && u.r + 1 < r1, first, acc);
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) acc[ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        u = v;
        if (u.r >= r1) return false;
        f -= 2;
        k = 0; j = u.p0; je = u.p1;
        v = load_unit(__builtin_amdgcn_readfirstlane(drawn));
        if (f == 2) { fj = v.p0; fje = v.p1; }            // the cursor stands at the first part of a unit that was not known yet
        drawn = draw();
        return true;
    };
    while (step(b0, b2) && step(b1, b0) && step(b2, b1)) {}
}

// Wider K: segments through two LDS buffers, one barrier each.  Four loader waves copy the next segment while twelve multiply the
// current one: a wave's loads complete in order, so a wave that did both would wait for the copies (from beyond the L2) at its
// next weights.  A consumer keeps the accumulators of its UPW block-rows in registers over the segments.  The values (once per
// 64 tokens from the L2) and the operand reads from LDS bound it.  16384 x 4096 x 768 at 25 %: 91 -> 50 us in a loop over the same
// buffers, 62 over six sets of them, 61..72 in the trace of a training step.  Segments of 24 columns in three buffers took 6 % longer
// (short parts leave a batch half empty), batches requested two ahead 18 % (registers, moves).
template <int MT, int UPW>
__global__ void __launch_bounds__((VAL_CW + VAL_LOADERS) * 64) values_segmented_kernel(const ValArgs a) {
    constexpr int MSUB = MT / 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mt = blockIdx.x / a.n_split, sp = blockIdx.x % a.n_split;
    const int m0 = mt * MT;
    const int seg = a.seg_cb * a.sub, nseg = (a.Cb + seg - 1) / seg;
    const int buf_bytes = seg / 2 * (MT * 64);
    if (wave >= VAL_CW) {
        // segment sg is in its buffer at barrier sg; the other buffer was multiplied before that barrier
        for (int sg = 0; sg <= nseg; ++sg) {
            const int c0 = sg * seg, ncb = a.Cb - c0 < seg ? a.Cb - c0 : seg;
            if (sg < nseg) val_stage<MT>(a, smem + (sg & 1) * buf_bytes, m0, c0, ncb, wave - VAL_CW, VAL_LOADERS, lane);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        return;
    }
    const int n = lane & 15, g = lane >> 4, bsel = g >> 1, hsel = g & 1;
    const uint32_t lane_x = (uint32_t)(n * 64 + (hsel ^ mortar_unit_swz(n)) * 16);
    const uint32_t lane_o = (uint32_t)(bsel * 512 + n * 32 + hsel * 16);
    const int lane_k = 2 * (n & 3) + bsel;
    const int row0 = sp * a.per + wave * UPW;              // block-rows row0 + k
    f32x4_t acc[UPW][MSUB];
#pragma unroll
    for (int k = 0; k < UPW; ++k)
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) acc[k][ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // block range of row k in segment sg (empty for rows past the end)
    auto range = [&](int sg, int k, int &lo, int &hi) {
        const int r = row0 + k;
        const int e = (sg + 1) * a.sub < a.nfine ? (sg + 1) * a.sub : a.nfine;
        lo = hi = 0;
        if (r < a.Rb && sg < nseg) {
            lo = val_idx(a.seg_ptr, r * (a.nfine + 1) + sg * a.sub);
            hi = val_idx(a.seg_ptr, r * (a.nfine + 1) + e);
        }
    };
    // The parts (segment, row) are walked in order, each batch requested one ahead of its product.  lo / hi: the parts of this
    // segment and, last, the first one of the next.
    int lo[UPW + 1], hi[UPW + 1];
#pragma unroll
    for (int k = 0; k <= UPW; ++k) range(k / UPW, k % UPW, lo[k], hi[k]);
    ValBatch cur;
    val_fetch(a, cur, lo[0], hi[0] - lo[0], lane_o, lane_k);
    __syncthreads();
    for (int sg = 0; sg < nseg; ++sg) {
        const unsigned char *lb = smem + (sg & 1) * buf_bytes;
#pragma unroll
        for (int k = 0; k < UPW; ++k) {
            for (int j = lo[k];; j += 8) {
                const bool more = j + 8 < hi[k];
                const int nj = more ? j + 8 : lo[k + 1], ne = more ? hi[k] : hi[k + 1];
                ValBatch next;
                val_fetch(a, next, nj, ne - nj, lane_o, lane_k);
                val_multiply<MT>(lb, cur, hi[k] - j, sg * seg, lane_x, acc[k]);
                cur = next;
                if (!more) break;
            }
        }
        lo[0] = lo[UPW];
        hi[0] = hi[UPW];
#pragma unroll
        for (int k = 1; k <= UPW; ++k) range(sg + 1 + k / UPW, k % UPW, lo[k], hi[k]);
        __syncthreads();
    }
    const ValOut<MT> out(a, m0, n, g);
#pragma unroll
    for (int k = 0; k < UPW; k += 2)
        if (row0 + k < a.Rb) out.store(row0 + k, k + 1 < UPW && row0 + k + 1 < a.Rb, acc[k], acc[k + 1 < UPW ? k + 1 : k]);
}

__global__ void __launch_bounds__(256) values_zero_kernel(uint16_t *y, int64_t M, int n4, int64_t ldy) {      // a matrix without blocks
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < M * n4) *reinterpret_cast<u32x2_t *>(y + i / n4 * ldy + i % n4 * 4) = u32x2_t{0u, 0u};
}

// out[j] = in[src[j]]^T, one wavefront per block: the stored values in the block order of the transposed topology.
__global__ void __launch_bounds__(256) values_transpose_kernel(const uint2 *in, const int32_t *src, int nnz, uint32_t *out) {
    __shared__ uint16_t tile[4][16][18];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = blockIdx.x * 4 + wave;
    if (j >= nnz) return;
    const int r = lane >> 2, q = lane & 3;
    const uint2 v = in[(int64_t)src[j] * 64 + lane];
    tile[wave][4 * q][r] = (uint16_t)v.x;
    tile[wave][4 * q + 1][r] = (uint16_t)(v.x >> 16);
    tile[wave][4 * q + 2][r] = (uint16_t)v.y;
    tile[wave][4 * q + 3][r] = (uint16_t)(v.y >> 16);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t *t = reinterpret_cast<const uint32_t *>(&tile[wave][r][4 * q]);
    reinterpret_cast<uint2 *>(out)[(int64_t)j * 64 + lane] = uint2{t[0], t[1]};
}

template <typename K>
int val_launch(K kern, bool &done, const ValArgs &a, int64_t grid, int threads, int smem, hipStream_t st) {
    int rc = mortar_allow_big_lds(kern, done);
    if (rc) return rc;
    if ((rc = mortar_launch_check(grid, 1))) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), smem, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "dds_values launch: %s", hipGetErrorString(e));
    return MORTAR_OK;
}

template <int MT>
int launch_resident(ValArgs &a, hipStream_t st) {
    static bool done = false;
    const int tiles = (a.M + MT - 1) / MT, max_split = (a.Rb + VAL_WAVES - 1) / VAL_WAVES;
    int split = 256 / tiles;                 // about one workgroup per CU and round; every workgroup stages the whole tile
    split = split < 1 ? 1 : (split > max_split ? max_split : split);
    a.n_split = split;
    a.per = ((a.Rb + split - 1) / split + 1) & ~1;
    a.unit = a.per >= 4 * VAL_WAVES ? 2 : 1;              // pairs of rows (64-byte stores) while every wave has two of them
    return val_launch(values_resident_kernel<MT>, done, a, (int64_t)tiles * split, VAL_WAVES * 64, (a.Cb + 1) / 2 * (MT * 64) + 16, st);
}

template <int MT, int UPW>
int launch_segmented(ValArgs &a, hipStream_t st) {
    static bool done = false;
    a.per = VAL_CW * UPW;
    a.n_split = (a.Rb + a.per - 1) / a.per;
    a.sub = MT == 64 ? 1 : 2;
    return val_launch(values_segmented_kernel<MT, UPW>, done, a, (int64_t)((a.M + MT - 1) / MT) * a.n_split, (VAL_CW + VAL_LOADERS) * 64,
                      2 * (a.seg_cb * a.sub / 2 * (MT * 64)), st);
}

// A tile of all K: up to 156 block-columns (78 pairs) for 32 tokens, 78 for 64 (the row counter behind it is outside the tile's budget).
bool val_fits(int mt, int Cb) { return (Cb + 1) / 2 * (mt * 64) <= LDS_BUDGET; }

// The launch for the tokens of `a` (seg_cb and nfine are set).
int val_dispatch(ValArgs &a, hipStream_t st) {
    // the largest token tile of all K: a block's values are read from L2 once per tile
    if (a.nfine == 1) return val_fits(64, a.Cb) ? launch_resident<64>(a, st) : launch_resident<32>(a, st);
    // Tokens per tile and block-rows per wave: the choice with the least rounds of workgroups x (staging + rows), staging
    // weighing about three rows; a 64-token row costs 1.7 of a 32-token one (its values are fetched once for both halves).
    int best = 0;
    int64_t best_cost = INT64_MAX;
    const struct { int mt, upw, unit; } shape[5] = {{64, 4, 17}, {64, 2, 17}, {32, 4, 10}, {32, 2, 10}, {32, 1, 10}};
    for (int i = 0; i < 5; ++i) {
        const int64_t wgs = ((int64_t)a.M + shape[i].mt - 1) / shape[i].mt * ((a.Rb + VAL_CW * shape[i].upw - 1) / (VAL_CW * shape[i].upw));
        const int64_t cost = (wgs + 255) / 256 * (3 + shape[i].upw) * shape[i].unit;
        if (cost < best_cost) { best_cost = cost; best = i; }
    }
    switch (best) {
        case 0: return launch_segmented<64, 4>(a, st);
        case 1: return launch_segmented<64, 2>(a, st);
        case 2: return launch_segmented<32, 4>(a, st);
        case 3: return launch_segmented<32, 2>(a, st);
    }
    return launch_segmented<32, 1>(a, st);
}

}  // namespace

extern "C" int32_t mortar_values_seg_cb(int32_t Cb) {
    if (Cb <= 0) return 0;
    if (val_fits(32, Cb)) return Cb;
    return VAL_SEG_CB;
}

extern "C" int mortar_segment_ptr_host(const int32_t *row_ptr, const int16_t *col, int32_t Rb, int32_t Cb, int32_t seg_cb,
                                       int32_t *seg_ptr_out) {
    if (!row_ptr || !col || !seg_ptr_out || seg_cb <= 0) return mortar_fail(MORTAR_ERR_ARG, "segment_ptr: bad argument");
    const int rc = mortar_check_bcsr_host(row_ptr, col, Rb, Cb);
    if (rc) return rc;
    const int nseg = (Cb + seg_cb - 1) / seg_cb;
    for (int r = 0; r < Rb; ++r) {
        int j = row_ptr[r];
        for (int s = 0; s <= nseg; ++s) {
            while (j < row_ptr[r + 1] && col[j] < s * seg_cb) ++j;
            seg_ptr_out[(int64_t)r * (nseg + 1) + s] = s == nseg ? row_ptr[r + 1] : j;
        }
    }
    return MORTAR_OK;
}

extern "C" int mortar_dds_values_bf16(const int32_t *row_ptr, const int16_t *col, const int32_t *seg_ptr, const uint16_t *data,
                                      int32_t Rb, int32_t Cb, int64_t nnz, const uint16_t *x, int64_t M, int64_t ldx, uint16_t *y,
                                      int64_t ldy, void *stream) {
    if (!row_ptr || !col || !data || !x || !y) return mortar_fail(MORTAR_ERR_ARG, "dds_values: null pointer");
    if (Rb <= 0 || Cb <= 0 || nnz < 0 || nnz > 0x7fffffff) return mortar_fail(MORTAR_ERR_ARG, "dds_values: bad shape");
    if (M <= 0 || M > (1 << 30)) return mortar_fail(MORTAR_ERR_ARG, "dds_values: M=%lld out of range", (long long)M);
    if (ldx < (int64_t)Cb * 16 || ldx % 8 || ldy < (int64_t)Rb * 16 || ldy % 4)
        return mortar_fail(MORTAR_ERR_ARG, "dds_values: bad leading dimension (ldx %% 8 == 0, ldy %% 4 == 0)");
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(y) & 7) || (reinterpret_cast<uintptr_t>(data) & 15))
        return mortar_fail(MORTAR_ERR_ARG, "dds_values: x and data must be 16-byte and y 8-byte aligned");
    if (Rb >= 1 << 26) return mortar_fail(MORTAR_ERR_LIMIT, "dds_values: %d block-rows (a token's results are addressed with 31 bits)", Rb);
    const int seg_cb = mortar_values_seg_cb(Cb);
    const int nseg = (Cb + seg_cb - 1) / seg_cb;
    if (nseg > 1 && !seg_ptr) return mortar_fail(MORTAR_ERR_ARG, "dds_values: %d K segments need seg_ptr (mortar_segment_ptr_host)", nseg);
    if (nnz == 0) {
        const int n4 = Rb * 4;
        hipLaunchKernelGGL(values_zero_kernel, dim3((unsigned)((M * n4 + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), y, M, n4, ldy);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? MORTAR_OK : mortar_fail(MORTAR_ERR_HIP, "dds_values launch: %s", hipGetErrorString(e));
    }
    ValArgs a{};
    a.row_ptr = row_ptr; a.seg_ptr = seg_ptr; a.col = col; a.data = data; a.ldx = ldx; a.ldy = ldy;
    a.Rb = Rb; a.Cb = Cb; a.nnz = (int)nnz; a.seg_cb = seg_cb; a.nfine = nseg; a.sub = 1;
    // A tile's results are addressed with 31 bits from its first token: where 64 rows of y do not fit that (rows more than
    // 16.7 M values apart), as many tokens per launch as do.
    const int64_t reach = 1 + (0x7fffffff - (int64_t)Rb * 32) / (2 * ldy), step = reach >= 64 ? M : reach;
    for (int64_t m = 0; m < M; m += step) {
        a.x = x + m * ldx;
        a.y = y + m * ldy;
        a.M = (int)(M - m < step ? M - m : step);
        const int rc = val_dispatch(a, static_cast<hipStream_t>(stream));
        if (rc) return rc;
    }
    return MORTAR_OK;
}

extern "C" int mortar_transpose_blocks_bf16(const uint16_t *data, const int32_t *src_block, int64_t nnz, uint16_t *out, void *stream) {
    if (!data || !src_block || !out) return mortar_fail(MORTAR_ERR_ARG, "transpose_blocks: null pointer");
    if (nnz < 0 || nnz > 0x7fffffff || ((reinterpret_cast<uintptr_t>(data) | reinterpret_cast<uintptr_t>(out)) & 15))
        return mortar_fail(MORTAR_ERR_ARG, "transpose_blocks: nnz out of range or data not 16-byte aligned");
    if (nnz == 0) return MORTAR_OK;
    hipLaunchKernelGGL(values_transpose_kernel, dim3((unsigned)((nnz + 3) / 4)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<const uint2 *>(data), src_block, (int)nnz, reinterpret_cast<uint32_t *>(out));
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MORTAR_OK : mortar_fail(MORTAR_ERR_HIP, "transpose_blocks launch: %s", hipGetErrorString(e));
}
