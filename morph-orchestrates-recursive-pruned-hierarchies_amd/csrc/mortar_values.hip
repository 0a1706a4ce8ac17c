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
};

// Tile layout in LDS: [pair of block-columns][token][64 bytes].  A wave instruction copies 16 tokens x 64 bytes straight from
// global memory (asynchronously, no registers; four lanes read 64 contiguous bytes).  The four 16-byte units of a token are
// stored in the order unit ^ s(token / 4), s = 0, 3, 2, 1 (mortar_unit_swz): the lanes that LDS serves together then touch
// every bank once.  The byte address
// of (column c, half h, token n) is enc(c) ^ lane with enc(c) = (c / 2) * MT * 64 + (c & 1) * 32 and a lane constant.
template <int MT>
__device__ __forceinline__ int val_enc(int c) { return (c >> 1) * (MT * 64) + (c & 1) * 32; }

// Copies block-columns [c0, c0 + ncb) of the tile at token m0 into `dst`, as loader `w` of NW.  Tokens past M repeat the last
// one, a missing second column of the last pair repeats the first: both feed results that are never stored or never read.
// PACED: at most four copies of a loader are in flight.
template <int MT, int NW, bool PACED = false>
__device__ __forceinline__ void val_stage(const ValArgs &a, unsigned char *dst, int m0, int c0, int ncb, int w, int lane) {
    constexpr int TG = MT / 16, PS = NW / TG;              // a loader keeps its 16 tokens and walks over the pairs
    static_assert(NW % TG == 0, "loaders x token groups");
    const int t = lane >> 2, u = (lane & 3) ^ mortar_unit_swz(t), tg = w % TG;
    int tok = m0 + tg * 16 + t;
    tok = tok < a.M ? tok : a.M - 1;
    int pr = w / TG;
    const MORTAR_GLOBAL char *src = (const MORTAR_GLOBAL char *)(a.x + (int64_t)tok * a.ldx + (int64_t)c0 * 16 + u * 8) + pr * 64;
    uint32_t d = __builtin_amdgcn_readfirstlane(mortar_lds_addr(dst + (pr * MT + tg * 16) * 64));
    for (; 2 * pr + 1 < ncb; pr += PS) {
        mortar_load_to_lds(src, d);
        if (PACED) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
        src += PS * 64;
        d += PS * MT * 64;
    }
    if (2 * pr < ncb) mortar_load_to_lds(src - (u >> 1) * 32, d);
}

// Four block pairs of one block-row part in registers: values as MFMA operands, the columns on lanes 0..3 of every 16-lane row.
struct ValBatch {
    u32x4_t A[4];
    int col;
};
// Load instructions of a batch.  values_resident_kernel counts on them: val_fetch issues every one of them, whatever the batch holds, and whoever makes
// it leave one out lowers this (tests/test_isa_waits.py counts them in the compiled kernels).
constexpr int VAL_LOADS = sizeof(ValBatch::A) / 16 + 1;

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
    u32x4_t B[MSUB];
    auto operand = [&](int u, int ms) { return *reinterpret_cast<const u32x4_t *>(lb + (mortar_row_bcast(enc, u) ^ lane_x) + ms * 1024); };
#pragma unroll
    for (int ms = 0; ms < MSUB; ++ms) B[ms] = operand(0, ms);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (2 * u >= cnt) break;
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) {
            acc[ms] = mortar_mfma(b.A[u], B[ms], acc[ms]);
            if (u < 3) B[ms] = operand(u + 1, ms);
        }
    }
}

// Results of RU = 2 or 4 consecutive block-rows in bf16 pairs, as a lane holds them ([row][sub-tile]: features 4 g .. + 3 of token n),
// stored together.  Two rows: the lane groups exchange halves, so that a lane holds 8 consecutive features of one row and a token's
// 32 features are one 64-byte piece.  Four: the halves of a 16-lane row then trade their second and first pair of rows, so that an
// instruction stores 128-byte pieces of eight tokens.  Pieces matter where the rows of y lie a power of two apart, which puts the pieces
// of a wave on few memory channels (64 tokens x 8 KB per workgroup: 32-byte pieces 71..117 us for 134 MB, 64-byte ones 34..42, 128-byte
// ones 24, a fill 21).  Bounded buffer stores drop the tokens past M and the rows past the end (`rows` of the RU exist).  No scalar
// offset: behind a 16-byte store that has one the compiler may overwrite the data registers in the next instruction, and gfx950 then
// stores the new values in the last lanes of a row.
// NT: non-temporal, the values and the tiles stay in the L2.  Only pieces that are whole (val_whole_lines): the parts of one that straddles
// lines leave the L2 unmerged.
template <int MT, int RU, bool NT>
struct ValOut {
    static constexpr int TPI = RU == 4 ? 8 : 16;          // tokens per instruction
    __amdgpu_buffer_rsrc_t r;
    uint32_t off, ld;
    int slot, nt;                                         // row of the unit that this lane stores; tokens from its first one on
    __device__ __forceinline__ ValOut(const ValArgs &a, int m0, int n, int g) {
        const int tokens = a.M - m0 < MT ? a.M - m0 : MT, t = RU == 4 ? n & 7 : n;
        r = val_rsrc(a.y + (int64_t)m0 * a.ldy, (int)((tokens - 1) * a.ldy * 2 + a.Rb * 32));
        slot = (RU == 4 ? (n >> 3) * 2 : 0) + (g & 1);
        nt = tokens - t;
        ld = (uint32_t)(a.ldy * 2);
        off = (uint32_t)t * ld + slot * 32 + (g >> 1) * 16;
    }
    __device__ __forceinline__ void store(int row, int rows, const u32x2_t (&p)[RU][MT / 16]) const {
        const bool mine = slot < rows;
#pragma unroll
        for (int ms = 0; ms < MT / 16; ++ms) {
            u32x4_t v[RU / 2];
#pragma unroll
            for (int q = 0; q < RU / 2; ++q)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto s = __builtin_amdgcn_permlane16_swap(p[2 * q][ms][h], p[2 * q + 1][ms][h], false, false);
                    v[q][h] = s[0];
                    v[q][2 + h] = s[1];
                }
            if constexpr (RU == 4) {
                const bool up = slot >= 2;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t got = __builtin_amdgcn_mov_dpp(up ? v[0][i] : v[1][i], 0x128, 0xf, 0xf, true);        // row_ror:8
                    const uint32_t lo = up ? got : v[0][i], hi = up ? v[1][i] : got;
                    v[0][i] = lo;
                    v[1][i] = hi;
                }
            }
#pragma unroll
            for (int h = 0; h < RU / 2; ++h) {
                const int t0 = ms * 16 + h * TPI;
                __builtin_amdgcn_raw_buffer_store_b128(v[h], r, mine && t0 < nt ? off + (uint32_t)t0 * ld + (uint32_t)row * 32 : 0xfffffff0u, 0, NT ? 2 : 0);
            }
        }
    }
};
template <int MSUB>
__device__ __forceinline__ void val_pack(const f32x4_t (&acc)[MSUB], u32x2_t (&p)[MSUB]) {
#pragma unroll
    for (int ms = 0; ms < MSUB; ++ms) p[ms] = u32x2_t{bf16_pack2(acc[ms][0], acc[ms][1]), bf16_pack2(acc[ms][2], acc[ms][3])};
}

// A uniform index array as scalar loads.
__device__ __forceinline__ int val_idx(const int32_t *p, int i) {
    return ((const __attribute__((address_space(4))) int32_t *)p)[__builtin_amdgcn_readfirstlane(i)];
}

// All of K in one tile.  The waves draw units of RU consecutive block-rows from a counter, so that rows of any length keep all of them
// busy; a wave's batches form one stream across rows, requested two ahead of their products, the first two before the tile is waited
// for.  Narrow K is bound by the results and the values together: 16384 x 768 x 4096 at 25 % (134 MB of results, a fill of which takes
// 21 us) takes 52 us in a training step, 62 where several steps' buffers alternate and nothing of theirs is left in the last-level cache; stage and store
// alone are 33, the values alone 21, the products alone 25 (before the non-temporal 128-byte pieces: 59 us where these leave 50).  Wide K is bound by the values from the L2, once per 32 tokens (4096 x 2048 x 11264: 82 us).
template <int MT, int RU, bool NT>
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
    struct Unit { int r, p0, p1, p2, p3, p4; };           // rows r .. r + 3: blocks p0 .. p1, p1 .. p2, ... (none past the range's end)
    auto load_unit = [&](int r) {
        Unit q{r, 0, 0, 0, 0, 0};
        if (r < r1) {
            q.p0 = val_idx(a.row_ptr, r);
            q.p1 = val_idx(a.row_ptr, r + 1);
            q.p2 = val_idx(a.row_ptr, r + 2 < r1 ? r + 2 : r1);
            if (RU > 2) q.p3 = val_idx(a.row_ptr, r + 3 < r1 ? r + 3 : r1);
            if (RU > 2) q.p4 = val_idx(a.row_ptr, r + 4 < r1 ? r + 4 : r1);
        }
        return q;
    };
    Unit u = load_unit(r0 + RU * wave), v{r1, 0, 0, 0, 0, 0};
    // request cursor: part f of the sequence u row 0, ..., v row 0, ...; blocks fj .. fje
    int f = 0, fj = u.p0, fje = u.p1;
    auto part_end = [&](int i) {
        if (RU == 2) return i < 2 ? (i < 1 ? u.p1 : u.p2) : (i < 3 ? v.p1 : v.p2);
        return i < 4 ? (i < 2 ? (i < 1 ? u.p1 : u.p2) : (i < 3 ? u.p3 : u.p4)) : (i < 6 ? (i < 5 ? v.p1 : v.p2) : (i < 7 ? v.p3 : v.p4));
    };
    auto request = [&](ValBatch &b) {
        val_fetch(a, b, fj, fje - fj, lane_o, lane_k);
        fj += 8;
        if (fj >= fje) {
            ++f;
            fj = f == RU ? v.p0 : fje;                    // the rows of a unit follow each other
            fje = part_end(f);
        }
    };
    if (tid == 0) *next_row = r0 + RU * VAL_WAVES;
    val_stage<MT, VAL_WAVES>(a, smem, m0, 0, a.Cb, wave, lane);
    ValBatch b0, b1, b2;
    request(b0);                                          // within the first unit
    request(b1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * VAL_LOADS) : "memory");      // the tile has landed, the batches are on their way
    __syncthreads();
    auto draw = [&]() {
        int d = 0;
        if (lane == 0) d = atomicAdd(next_row, RU);
        return d;
    };
    if (u.r >= r1) return;
    v = load_unit(__builtin_amdgcn_readfirstlane(draw()));
    int drawn = draw();
    if (f == RU) { fj = v.p0; fje = v.p1; }
    f32x4_t acc[MSUB];
    u32x2_t done[RU][MSUB];                               // finished rows of the unit
#pragma unroll
    for (int ms = 0; ms < MSUB; ++ms) acc[ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int k = 0, j = u.p0, je = u.p1;                       // row of u that is being multiplied
    const ValOut<MT, RU, NT> out(a, m0, n, g);
    // one batch; false when the wave's rows are done
    auto step = [&](const ValBatch &c, ValBatch &nx) {
        request(nx);
        val_multiply<MT>(smem, c, je - j, 0, lane_x, acc);
        j += 8;
        if (j < je) return true;
#pragma unroll
        for (int q = 0; q < RU; ++q)
            if (q == k) val_pack<MSUB>(acc, done[q]);
#pragma unroll
        for (int ms = 0; ms < MSUB; ++ms) acc[ms] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (++k < RU) {
            j = je;
            je = part_end(k);
            return true;
        }
        out.store(u.r, r1 - u.r, done);
        u = v;
        if (u.r >= r1) return false;
        f -= RU;
        k = 0; j = u.p0; je = u.p1;
        v = load_unit(__builtin_amdgcn_readfirstlane(drawn));
        if (f == RU) { fj = v.p0; fje = v.p1; }           // the cursor stands at the first part of a unit that was not known yet
        drawn = draw();
        return true;
    };
    while (step(b0, b2) && step(b1, b0) && step(b2, b1)) {}
}

// Wider K: segments through two LDS buffers, one barrier each.  Four loader waves copy the next segment while twelve multiply the
// current one: a wave's loads complete in order, so a wave that did both would wait for the copies (from beyond the L2) at its
// next weights.  A consumer keeps the accumulators of its UPW block-rows in registers over the segments.  The values (once per
// 64 tokens from the L2) and the operand reads from LDS bound it.  16384 x 4096 x 768 at 25 %: 52 us in a training step, 61
// where several steps' buffers alternate (62 in a loop over its own before its results left in 128-byte non-temporal pieces, 56 now); the copies alone are 28,
// the values alone 28, the products alone 32.  Segments of 24 columns in three buffers took 6 % longer
// (short parts leave a batch half empty), batches requested two ahead 18 % (registers, moves).
template <int MT, int UPW, bool NT>
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
        // Segment sg is in its buffer at barrier sg; the other buffer was multiplied before that barrier.  The first segment comes as fast as it can, nobody
        // multiplies yet; copies of the others, all requested at once, stand in front of the values that the consumers wait for.  us, all at once -> four
        // of a loader in flight: 16384 x 4096 x 1024 at 12.5 / 25 / 50 % 78.5 -> 73.0, 104 -> 98.7, 145 -> 139, 1024 x 4096 x 768 at 25 % 14.9 -> 14.4; three in flight leave
        // calls of a few hundred tokens 2 % slower, two 10 %.
        for (int sg = 0; sg <= nseg; ++sg) {
            const int c0 = sg * seg, ncb = a.Cb - c0 < seg ? a.Cb - c0 : seg;
            if (sg == 0) val_stage<MT, VAL_LOADERS>(a, smem, m0, c0, ncb, wave - VAL_CW, lane);
            else if (sg < nseg) val_stage<MT, VAL_LOADERS, true>(a, smem + (sg & 1) * buf_bytes, m0, c0, ncb, wave - VAL_CW, lane);
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
    constexpr int RU = UPW < 4 ? 2 : 4;
    const ValOut<MT, RU, NT> out(a, m0, n, g);
#pragma unroll
    for (int k = 0; k < UPW; k += RU) {
        u32x2_t p[RU][MSUB];
#pragma unroll
        for (int q = 0; q < RU; ++q) val_pack<MSUB>(acc[k + q < UPW ? k + q : k], p[q]);
        const int rows = a.Rb - row0 - k;
        if (rows > 0) out.store(row0 + k, UPW < RU && rows > UPW ? UPW : rows, p);
    }
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

// Whether the pieces of `piece` bytes that a wave stores lie on lines, in every row of y: they may then be non-temporal.  us, plain -> non-temporal,
// 16384 tokens x 4096 features of 768 at 12.5 / 25 %: 39.7 -> 36.3, 53 -> 48; in rows of 4112 values 46 -> 101, 56 -> 106; with an elementwise
// kernel behind it that reads the result 83 -> 81, 97 -> 91, and 85 -> 130, 98 -> 136 for 4080 features.  16384 tokens x 768 features of 4096 58.9 -> 50.7
// (66.4 -> 64.7 with the reader), in rows of 772 values 58.4 -> 56.6.  Results of a few MB gain as well (2048 tokens x 4096 features 12.6 -> 11.2, with the
// reader 18.4 -> 18.1); of those between 30 and 70 MB some gain and some lose (8192 tokens x 2048 features of 768 19.8 -> 20.8, 30.3 -> 32.9).
bool val_whole_lines(const ValArgs &a, int piece) {
    return (reinterpret_cast<uintptr_t>(a.y) | (uintptr_t)(a.ldy * 2)) % (uintptr_t)piece == 0;
}

template <int MT, int RU, bool NT>
int launch_resident_form(const ValArgs &a, int64_t grid, hipStream_t st) {
    static bool done = false;
    return val_launch(values_resident_kernel<MT, RU, NT>, done, a, grid, VAL_WAVES * 64, (a.Cb + 1) / 2 * (MT * 64) + 16, st);
}

template <int MT>
int launch_resident(ValArgs &a, hipStream_t st) {
    const int tiles = (a.M + MT - 1) / MT, max_split = (a.Rb + VAL_WAVES - 1) / VAL_WAVES;
    int split = 256 / tiles;                 // about one workgroup per CU and round; every workgroup stages the whole tile
    split = split < 1 ? 1 : (split > max_split ? max_split : split);
    a.n_split = split;
    a.per = ((a.Rb + split - 1) / split + 3) & ~3;
    const int64_t grid = (int64_t)tiles * split;
    // 64-token tiles: four rows per unit while every wave has two such units, else two.  16384 x 768 x 4096 at 12.5 / 25 %: 37 / 51 us against 47 / 51 with
    // two rows, 8192 tokens 23 / 31 against 27 / 31; 4099 tokens (1.4 units of four per wave) 17.2 / 21.3 against 15.3 / 20.1, 300 tokens
    // 7.0 / 8.8 against 5.7 / 6.7.  (Few rows leave waves without a unit.  Half the workgroups instead: 24 to 128 rows, up to 1000 tokens, 5 to 40 % slower;
    // one row at a time: 17 to 33 rows of 12 blocks 2 to 5 % faster, 64 and more 8 to 13 % slower.)
    // 32-token tiles: always two.  Their units carry half the results and twice the values: [5632, 2048], 4096 tokens at 25 % 44.3 us against 46.4 with four
    // rows, with a reader behind it 59.6 against 63; [5632, 1280] 31.9 against 34.2, 47.5 against 50; equal at [4096, 1280].
    if constexpr (MT == 64) {
        if (a.per >= 8 * VAL_WAVES) return val_whole_lines(a, 128) ? launch_resident_form<MT, 4, true>(a, grid, st) : launch_resident_form<MT, 4, false>(a, grid, st);
    }
    return val_whole_lines(a, 64) ? launch_resident_form<MT, 2, true>(a, grid, st) : launch_resident_form<MT, 2, false>(a, grid, st);
}

template <int MT, int UPW, bool NT>
int launch_segmented_form(ValArgs &a, hipStream_t st) {
    static bool done = false;
    a.per = VAL_CW * UPW;
    a.n_split = (a.Rb + a.per - 1) / a.per;
    a.sub = MT == 64 ? 1 : 2;
    return val_launch(values_segmented_kernel<MT, UPW, NT>, done, a, (int64_t)((a.M + MT - 1) / MT) * a.n_split, (VAL_CW + VAL_LOADERS) * 64,
                      2 * (a.seg_cb * a.sub / 2 * (MT * 64)), st);
}

template <int MT, int UPW>
int launch_segmented(ValArgs &a, hipStream_t st) {
    if constexpr (UPW > 1) {                 // (one row's pieces are 32 bytes)
        if (val_whole_lines(a, 64)) return launch_segmented_form<MT, UPW, true>(a, st);
    }
    return launch_segmented_form<MT, UPW, false>(a, st);
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
