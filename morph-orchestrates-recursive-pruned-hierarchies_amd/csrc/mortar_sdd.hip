// Weight gradient on the carved topology: out[j] = a[:, rows of block j]^T @ b[:, columns of block j].
//
// Reference: stk_sdd_at_b (morph/sparse/stk/backend/custom_ops.py:78-96) -> _sdd_kernel
// (morph/sparse/stk/backend/triton_kernels.py): one 16x16 output tile per kept block, contracted over the M tokens,
// bf16 operands, fp32 accumulation, output in the operand dtype.
//
// Shape of the work: the contraction runs over tokens, so both MFMA operands need 8 tokens of ONE feature per lane
// while memory holds 16 features of ONE token per 32 bytes.  The slices are staged row-major with direct
// global->LDS loads (whole 128-byte lines: 4 block-columns of 8 tokens per instruction) and read back with the
// transposing LDS load (ds_read_b64_tr_b16): 16 lanes hand in the addresses of 4 token rows x 4 pieces of 4
// features and each lane gets 4 tokens of one feature.  A workgroup keeps the fp32 tiles of up to WAVES*NB blocks of
// a few consecutive block-rows in registers and walks the tokens in steps of 32; per step it stages the
// 32 x (columns of its K segment) slice of b once and the slice of a for its rows, into one of two buffers: the
// loads of the next step are in flight while the current one multiplies.  Workgroup ids are laid out per XCD (each
// has its own L2) as runs of (token range, row group) pairs with the K segments of a pair side by side, so that a
// slice of a is fetched from HBM once and a slice of b only by the XCDs that hold its token range.  Every token range
// writes its fp32 sums to its own slab of the workspace; a last pass adds the slabs in a fixed order and rounds to
// bf16, so results are reproducible.
//
// What bounds it: a kept block needs its own b tile per MFMA (no other block of the row shares it), 1 KB of LDS reads for 16
// cycles of the matrix core, and the two overlap only in part: three tile reads and two MFMAs per wavefront measured 298
// cycles beside 217 and 144 alone, two reads 231.  So a is read again only where the block-row changes, nothing but reads and
// MFMAs stands in the inner loop (a pair of slots never straddles two rows, addresses and copies are fixed over the steps),
// and the rest is the slabs.  Both launches, in a loop over the same operands: dW of 11264 x 2048 at 25 %, 4096 tokens 103 -> 84 us
// (89 over six sets of operands); 4096 x 768, 16384 tokens 68 -> 55 us (71); 2048 x 5632, 4096 tokens 65 -> 54 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <type_traits>
#include <utility>
#include <vector>

#include "mortar_device.h"
#include "mortar_internal.h"

namespace {

constexpr int SDD_WAVES = 16;
constexpr int SDD_NB_MAX = 22;                   // most blocks per wavefront (4 accumulator registers each)
constexpr int SDD_NB_SIZES[] = {8, 10, 12, 14, 16, 18, 20, 22};      // the kernels that are built
constexpr int SDD_RMAX = 32;                     // block-rows per workgroup (slice of a in LDS)
constexpr int SDD_SEG = 44;                      // block-columns per K segment (slice of b in LDS)
constexpr int SDD_TARGET_WGS = 256;              // workgroups wanted in flight (one per CU: two slice buffers each)
constexpr int SDD_NQ = SDD_SEG / 4;              // quads of block-columns per segment
constexpr int SDD_CS = 1024 + 32;                // LDS bytes per chunk = 8 tokens x 128 bytes (a quad's line) + skew
constexpr int SDD_QS = 4 * SDD_CS;               // LDS bytes per quad: 32 tokens
constexpr int SDD_BUF = (SDD_NQ + SDD_RMAX / 4) * SDD_QS;    // one buffer: the slice of b, then the slice of a
constexpr int SDD_STEP = 32;                     // tokens per step = K of one MFMA
constexpr int SDD_SLAB_BLOCKS = 140;             // blocks of one fp32 slab (written, read back) that cost one unit
constexpr int SDD_STAGE = ((SDD_NQ + SDD_RMAX / 4) * 4 + SDD_WAVES - 1) / SDD_WAVES;       // copy instructions of a wavefront per step

typedef short s16x4 __attribute__((ext_vector_type(4)));

struct SddArgs {
    const int32_t *plan;
    const uint16_t *a, *b;
    int64_t lda, ldb, M;
    float *acc;
    uint16_t *out;
    int32_t Cb, tsplit, steps_per_split, nsteps, nnz, per_xcd, n_wg, seg_cb;
};

// 8 tokens of one feature (= lane & 15) of the block-column (or block-row) whose first token sits at LDS address `tile`:
// group g = lane >> 4 gets tokens {8r + g} and {8r + 4 + g}, r = 0..3 - one token of each 8-token chunk per read, which
// spreads the 32 lanes served together over all banks.  Both operands use the same order, so the contraction is
// unchanged.  Written as inline assembly: the caller waits (lds_wait) where the operand is used, so that reads of later
// tiles stay in flight.
union SddTile {
    u32x2_t h[2];
    bf16x8_t v;
};
__device__ __forceinline__ void read_tr(SddTile &t, uint32_t addr) {
    asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:512" : "=&v"(t.h[0]), "=&v"(t.h[1]) : "v"(addr));
}
// The same if bit BIT of the (uniform) flags is set, else `t` stays.
template <int BIT>
__device__ __forceinline__ void read_tr_if(SddTile &t, uint32_t addr, uint32_t flags) {
    asm volatile("s_bitcmp1_b32 %3, %4\n\ts_cbranch_scc0 .Lsame%=\n\tds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:512\n.Lsame%=:"
                 : "+&v"(t.h[0]), "+&v"(t.h[1]) : "v"(addr), "s"(flags), "n"(BIT) : "scc");
}
// At most N reads may still be on their way afterwards.
template <int N>
__device__ __forceinline__ void lds_wait(SddTile &a, SddTile &b, SddTile &c) {
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(a.h[0]), "+v"(a.h[1]), "+v"(b.h[0]), "+v"(b.h[1]), "+v"(c.h[0]), "+v"(c.h[1]) : "n"(N));
}

// Asynchronous 16-byte-per-lane copy global -> LDS from a scalar base and a lane offset: lane l's 16 bytes land at
// lds_base + 16 * l.  The caller waits with s_waitcnt vmcnt(0) and a barrier before the destination is read.
__device__ __forceinline__ void load_to_lds_base(const char *base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(off), "s"(base) : "memory", "m0");
}

// Accumulator lane (og = lane >> 4, oc = lane & 15) holds rows 4 og .. 4 og + 3 of column oc; afterwards columns
// 4 (oc >> 2) .. + 3 of row 4 og + (oc & 3): a 4 x 4 transpose among the four lanes of a quad.
__device__ __forceinline__ f32x4_t quad_transpose(f32x4_t v, int lane) {
    const bool o1 = lane & 1, o2 = lane & 2;
    auto swap = [](float x, auto ctrl) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true)); };
    using xor1 = std::integral_constant<int, 0xB1>;        // quad_perm [1, 0, 3, 2]
    using xor2 = std::integral_constant<int, 0x4E>;        // quad_perm [2, 3, 0, 1]
    const float a = swap(o1 ? v[0] : v[1], xor1{}), b = swap(o1 ? v[2] : v[3], xor1{});
    v = f32x4_t{o1 ? a : v[0], o1 ? v[1] : a, o1 ? b : v[2], o1 ? v[3] : b};
    const float c = swap(o2 ? v[0] : v[2], xor2{}), d = swap(o2 ? v[1] : v[3], xor2{});
    return f32x4_t{o2 ? c : v[0], o2 ? d : v[1], o2 ? v[2] : c, o2 ? v[3] : d};
}
__device__ __forceinline__ void store_block(uint16_t *out, int64_t j, f32x4_t v, int lane) {
    const f32x4_t w = quad_transpose(v, lane);
    const int row = 4 * (lane >> 4) + (lane & 3), c = lane & 12;
    *reinterpret_cast<u32x2_t *>(out + j * 256 + row * 16 + c) = u32x2_t{bf16_pack2(w[0], w[1]), bf16_pack2(w[2], w[3])};
}

template <int... I, typename F>
__device__ __forceinline__ void sdd_unroll(std::integer_sequence<int, I...>, F f) { (f(std::integral_constant<int, I>{}), ...); }

// WIDE: 32 tokens of an operand do not fit a 32-bit offset (rows more than 2^26 values apart): 64-bit lane addresses.
template <int SDD_NB, bool WIDE>
__global__ __launch_bounds__(SDD_WAVES * 64) void sdd_kernel(SddArgs p) {
    constexpr int SDD_G = SDD_WAVES * SDD_NB;        // blocks per workgroup
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup -> (token range, row group, K segment).  Ids are dealt round-robin over the 8 XCDs, each with its own
    // L2.  The (token range, workgroup) items, workgroups in the plan's order (row groups of about the same rows side by
    // side over the K segments), are cut into 8 equal runs, one per XCD: the slice of a is then fetched from HBM once
    // (its nseg readers share an L2) and a slice of b only by the few XCDs that hold its token range.
    const int n_wg = p.n_wg;
    const int32_t *order = p.plan + 4 + n_wg * 4 + (int64_t)n_wg * SDD_G * 2;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int item = xcd * p.per_xcd + slot;
    if (slot >= p.per_xcd || item >= p.tsplit * n_wg) return;
    const int ts = item / n_wg;
    const int wg = order[item - ts * n_wg];
    const int32_t *desc = p.plan + 4 + wg * 4;
    const int row0 = desc[0], nrows = desc[1], seg = desc[2];
    const int seg_cb = p.seg_cb;
    const int c0 = seg * seg_cb;
    const int ncb = min(seg_cb, p.Cb - c0);
    const int nq = (ncb + 3) >> 2, nrq = (nrows + 3) >> 2;          // quads of block-columns / block-rows
    f32x4_t acc[SDD_NB];
#pragma unroll
    for (int b = 0; b < SDD_NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t tr_off = ((lane & 15) >> 2) * SDD_CS + (lane >> 4) * 128 + (lane & 3) * 8;
    // staging role of this lane inside one instruction: token 8c + (lane >> 3), 16-byte piece lane & 7 of the 128-byte line
    const int st_tok = lane >> 3, st_piece = lane & 7;
    const int s_begin = ts * p.steps_per_split, s_end = min(p.nsteps, s_begin + p.steps_per_split);

    // Staging: one wavefront instruction moves 8 tokens x one 128-byte line (4 block-columns, or 4 block-rows of a) into
    // 1 KB of contiguous LDS.  What an instruction reads and where it lands is fixed over the steps: a scalar base that
    // moves on by one step, a lane offset, an LDS address.  Columns and rows past the slice's end read its first one of
    // the quad (no block refers to them).
    const int n_copy = (nq + nrq) * 4;
    const char *base[SDD_STAGE];
    uint32_t voff[SDD_STAGE];
    int dst[SDD_STAGE];
#pragma unroll
    for (int k = 0; k < SDD_STAGE; ++k) {
        const int i = wave + k * SDD_WAVES, c = i & 3;
        const bool is_b = i < nq * 4;
        const int q = is_b ? i >> 2 : (i >> 2) - nq;
        const int piece = 4 * q + (st_piece >> 1) < (is_b ? ncb : nrows) ? st_piece : st_piece & 1;
        base[k] = is_b ? reinterpret_cast<const char *>(p.b + (int64_t)s_begin * SDD_STEP * p.ldb + (int64_t)(c0 + 4 * q) * 16)
                       : reinterpret_cast<const char *>(p.a + (int64_t)s_begin * SDD_STEP * p.lda + (int64_t)(row0 + 4 * q) * 16);
        voff[k] = (uint32_t)((WIDE ? 0 : (8 * c + st_tok) * (is_b ? p.ldb : p.lda) * 2) + piece * 16);
        dst[k] = (is_b ? q : SDD_NQ + q) * SDD_QS + c * SDD_CS;
    }
    // Stages step s (the steps come in order) into buffer `buf`.  Rows past M are not loaded: in the one partial step
    // they are cleared with plain stores (disjoint addresses from the loads).
    auto stage = [&](int s, int buf) {
        const int64_t left = p.M - (int64_t)s * SDD_STEP;
#pragma unroll
        for (int k = 0; k < SDD_STAGE; ++k) {
            const int i = wave + k * SDD_WAVES;
            if (i < n_copy) {
                char *d = smem + buf * SDD_BUF + dst[k];
                const uint32_t la = __builtin_amdgcn_readfirstlane(mortar_lds_addr(d));
                auto copy = [&]() {
                    if constexpr (WIDE) {
                        const int64_t row = (int64_t)(8 * (i & 3) + st_tok) * (i < nq * 4 ? p.ldb : p.lda) * 2;
                        mortar_load_to_lds((const MORTAR_GLOBAL char *)(base[k] + row + voff[k]), la);
                    } else {
                        load_to_lds_base(base[k], voff[k], la);
                    }
                };
                if (left >= SDD_STEP) copy();
                else if (8 * (i & 3) + st_tok < left) copy();
                else *reinterpret_cast<u32x4_t *>(d + lane * 16) = u32x4_t{0u, 0u, 0u, 0u};
                base[k] += (i < nq * 4 ? p.ldb : p.lda) * (2 * SDD_STEP);
            }
        }
    };

    if (s_begin < s_end) stage(s_begin, 0);
    // this wavefront's blocks: block index (-1 = none) and (row slot << 20 | LDS byte offset of the column's tile)
    const int32_t *ent_j = p.plan + 4 + n_wg * 4 + (int64_t)(wg * SDD_WAVES + wave) * SDD_NB;
    const int32_t *ent_o = ent_j + (int64_t)n_wg * SDD_G;
    const int my_j = lane < SDD_NB ? ent_j[lane] : -1;
    // slots come in pairs of one block-row: per pair one tile of a (read again only where the row changes), per slot one of b
    int bo[SDD_NB], ao[SDD_NB / 2];
#pragma unroll
    for (int b = 0; b < SDD_NB; ++b) {
        const int e = __builtin_amdgcn_readfirstlane(ent_o[b]), rs = e >> 20;
        bo[b] = e & 0xfffff;
        if (b % 2 == 0) ao[b / 2] = SDD_NQ * SDD_QS + (rs >> 2) * SDD_QS + (rs & 3) * 32;
    }
    uint32_t new_row = 0;                 // bit k: pair k is in another block-row than pair k - 1
#pragma unroll
    for (int k = 1; k < SDD_NB / 2; ++k) new_row |= (uint32_t)(ao[k] != ao[k - 1]) << k;
    new_row = __builtin_amdgcn_readfirstlane(new_row);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int buf = 0;
    for (int s = s_begin; s < s_end; ++s) {
        if (s + 1 < s_end) stage(s + 1, buf ^ 1);            // in flight while this step multiplies
        const char *cur = smem + buf * SDD_BUF;
        // b is read one pair of slots ahead of its MFMAs (an empty slot repeats a valid tile: its sum is never stored)
        const uint32_t at = mortar_lds_addr(cur) + tr_off;
        SddTile A, B[4];
        read_tr(A, at + ao[0]);
        read_tr(B[0], at + bo[0]);
        read_tr(B[1], at + bo[1]);
        sdd_unroll(std::make_integer_sequence<int, SDD_NB / 2>{}, [&](auto kc) {
            constexpr int k = decltype(kc)::value, c = 2 * (k & 1), n = c ^ 2;
            if constexpr (k + 1 < SDD_NB / 2) {
                read_tr(B[n], at + bo[2 * k + 2]);
                read_tr(B[n + 1], at + bo[2 * k + 3]);
                lds_wait<4>(A, B[c], B[c + 1]);
            } else {
                lds_wait<0>(A, B[c], B[c + 1]);
            }
            acc[2 * k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A.v, B[c].v, acc[2 * k], 0, 0, 0);
            acc[2 * k + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A.v, B[c + 1].v, acc[2 * k + 1], 0, 0, 0);
            if constexpr (k + 1 < SDD_NB / 2) read_tr_if<k + 1>(A, at + ao[k + 1], new_row);
        });
        __builtin_amdgcn_s_waitcnt(0);                       // the next step's slices have landed
        __syncthreads();                                     // ... for every wavefront, and this buffer is free again
        buf ^= 1;
    }
    // a slab keeps a block's sums in accumulator order (64 lanes x 16 bytes)
    float *part = p.acc + (int64_t)ts * p.nnz * 256;
#pragma unroll
    for (int b = 0; b < SDD_NB; ++b) {
        const int j = __builtin_amdgcn_readlane(my_j, b);
        if (j >= 0) {
            if (p.tsplit > 1) *reinterpret_cast<f32x4_t *>(part + (int64_t)j * 256 + lane * 4) = acc[b];
            else store_block(p.out, j, acc[b], lane);
        }
    }
}

__global__ __launch_bounds__(256) void sdd_zero_kernel(float *acc, int64_t n4) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n4) reinterpret_cast<f32x4_t *>(acc)[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// out = bf16(sum over the token ranges, in range order), one wavefront per block
__global__ __launch_bounds__(256) void sdd_round_kernel(const float *acc, uint16_t *out, int64_t n4, int tsplit) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n4) {
        f32x4_t v = reinterpret_cast<const f32x4_t *>(acc)[i];
        for (int t = 1; t < tsplit; ++t) v += reinterpret_cast<const f32x4_t *>(acc)[i + (int64_t)t * n4];
        store_block(out, i >> 6, v, threadIdx.x & 63);
    }
}

}  // namespace

// Workgroups of a plan with `nb` blocks per wavefront: per K segment, runs of consecutive block-rows holding at most
// 16 * nb blocks of the segment and at most SDD_RMAX rows.  A run is staged from a multiple of four block-rows, so that a copied 128-byte
// piece of a is a line and not parts of two (dW of 4096 x 768, 16384 tokens 70.5 -> 68.2 us, at density 0.5 and 8192 63.6 -> 61.8; 2048 x 5632,
// 4096 tokens 66.4 -> 65.1) - unless the rows of a are no whole lines ([5328, 1600], 6000 tokens at 12.5 % 48.6 -> 51.5) or the rows staged in
// addition make it many more runs: 53 for 51 of [8192, 1536], power-law rows of 12.5 %, 6000 tokens 70 -> 79, 68 for 66 of [11264, 2048] at 5 %, 2048 tokens
// 36.6 -> 33.5; the line is one in 32.
struct SddGroup { int row0, nrows, seg, blocks; std::vector<int32_t> j, o; };

static bool sdd_nb_built(int nb) {
    for (int v : SDD_NB_SIZES) if (v == nb) return true;
    return false;
}

static void sdd_segments(int Cb, int &nseg, int &seg_cb) {
    nseg = (Cb + SDD_SEG - 1) / SDD_SEG;
    seg_cb = ((Cb + nseg - 1) / nseg + 3) & ~3;                    // whole 128-byte lines
}

// First block of every row in every K segment, [Rb][nseg + 1].
struct SddRows { int nseg, seg_cb; std::vector<int32_t> at; };

static SddRows sdd_rows(const int32_t *row_ptr, const int16_t *col, int Rb, int Cb) {
    SddRows t;
    sdd_segments(Cb, t.nseg, t.seg_cb);
    t.at.resize((size_t)Rb * (t.nseg + 1));
    for (int r = 0; r < Rb; ++r) {
        int32_t *at = &t.at[(size_t)r * (t.nseg + 1)], j = row_ptr[r];
        const int32_t e = row_ptr[r + 1];
        for (int sg = 0; sg < t.nseg; ++sg) {
            at[sg] = j;
            while (j < e && col[j] < (sg + 1) * t.seg_cb) ++j;
        }
        at[t.nseg] = j;
    }
    return t;
}

static void sdd_groups_from(const SddRows &t, const int16_t *col, int Rb, int nb, bool fill, bool lines, std::vector<SddGroup> &wgs) {
    const int G = SDD_WAVES * nb;
    wgs.clear();
    for (int sg = 0; sg < t.nseg; ++sg) {
        SddGroup cur{0, 0, sg, 0, {}, {}};
        int held = 0;
        auto flush = [&]() {
            if (held) wgs.push_back(std::move(cur));
            cur = SddGroup{0, 0, sg, 0, {}, {}};
            held = 0;
        };
        for (int r = 0; r < Rb; ++r) {
            const int lo = t.at[(size_t)r * (t.nseg + 1) + sg], hi = t.at[(size_t)r * (t.nseg + 1) + sg + 1];
            if (hi == lo) continue;
            const int slots = (hi - lo + 1) & ~1;              // pairs of slots share a block-row
            if (held && (held + slots > G || r - cur.row0 + 1 > SDD_RMAX)) flush();
            if (!held) cur.row0 = lines ? r & ~3 : r;
            cur.nrows = r - cur.row0 + 1;
            cur.blocks += hi - lo;
            held += slots;
            if (!fill) continue;
            for (int j = lo; j < hi; ++j) {
                cur.j.push_back(j);
                const int cr = col[j] - sg * t.seg_cb;
                cur.o.push_back(((r - cur.row0) << 20) | ((cr >> 2) * SDD_QS + (cr & 3) * 32));
            }
            if (slots > hi - lo) {
                cur.j.push_back(-1);
                cur.o.push_back(cur.o.back());
            }
        }
        flush();
    }
}

static void sdd_groups(const SddRows &t, const int16_t *col, int Rb, int nb, bool fill, std::vector<SddGroup> &wgs) {
    sdd_groups_from(t, col, Rb, nb, false, false, wgs);
    bool lines = false;
    if (Rb % 4 == 0) {
        const size_t fewest = wgs.size();
        std::vector<SddGroup> whole;
        sdd_groups_from(t, col, Rb, nb, false, true, whole);
        lines = whole.size() * 32 <= fewest * 33;
        if (lines) wgs = std::move(whole);
    }
    if (fill) sdd_groups_from(t, col, Rb, nb, true, lines, wgs);
}

// Token ranges for M tokens over the n_wg workgroups of a plan with nb blocks per wavefront.  One workgroup runs per
// CU and the (range, workgroup) items are dealt evenly over the XCDs, so the launch takes
// ceil(items per XCD / CUs per XCD) rounds of ceil(steps / ranges) steps.  A step costs nb + 7 units (a block and wavefront
// one each, the barrier) plus a tenth per staged tile (block-rows + block-columns), a round 2.5 nb + 8 (the first slices, the
// stores); more than one range costs the pass that adds the slabs and, per range, a slab of fp32 sums to write and to read
// back.  A unit is 36 ns; the constants are a fit to 1022 launch times over six topologies, all group sizes, 1 to 16 ranges
// and 512 to 16384 tokens (6.5 % rms; the choice is within 2 % of the best on average).  The ranges are chosen for 60 staged
// tiles, whatever the plan; the returned cost of that choice counts the `tiles` given.
constexpr int SDD_TILES = 60;
static int64_t sdd_split(int32_t n_wg, int32_t nnz, int nb, int64_t M, int tiles, int &nsteps, int &steps_per_split, int &tsplit) {
    nsteps = (int)((M + SDD_STEP - 1) / SDD_STEP);
    auto cost = [&](int t, int tl) {
        const int sps = (nsteps + t - 1) / t, tt = (nsteps + sps - 1) / sps;
        const int64_t per_xcd = ((int64_t)n_wg * tt + 7) / 8;
        const int64_t rounds = (per_xcd + SDD_TARGET_WGS / 8 - 1) / (SDD_TARGET_WGS / 8);
        return rounds * (sps * (10 * nb + 70 + tl) + 25 * nb + 80) + (tt > 1 ? (int64_t)tt * nnz * 10 / SDD_SLAB_BLOCKS + 530 : 0);
    };
    int best = 1;
    if (nsteps > 0)
        for (int t = 2; t <= std::min(nsteps, 16); ++t)
            if (cost(t, SDD_TILES) < cost(best, SDD_TILES)) best = t;
    steps_per_split = std::max(1, (nsteps + best - 1) / best);
    tsplit = std::max(1, (nsteps + steps_per_split - 1) / steps_per_split);
    return nsteps > 0 ? cost(best, tiles) : 0;
}

// Blocks per wavefront for this topology at M tokens: the built size whose plan is cheapest by sdd_split's measure.
// Fewer blocks per workgroup mean more row groups, which fill the chip with fewer token ranges (fewer slabs), at the
// price of more staged bytes per block.
extern "C" int32_t mortar_sdd_blocks_per_wave_host(const int32_t *row_ptr, const int16_t *col, int32_t Rb, int32_t Cb, int64_t M) {
    const int rc = mortar_check_bcsr_host(row_ptr, col, Rb, Cb);
    if (rc) return rc;
    if (M < 0) return mortar_fail(MORTAR_ERR_ARG, "sdd_blocks_per_wave: M < 0");
    int best = SDD_NB_MAX;
    int64_t best_cost = INT64_MAX;
    const SddRows t = sdd_rows(row_ptr, col, Rb, Cb);
    for (int nb : SDD_NB_SIZES) {
        std::vector<SddGroup> wgs;
        int nsteps, sps, tsplit;
        sdd_groups(t, col, Rb, nb, false, wgs);
        int64_t rows = 0;
        for (const SddGroup &g : wgs) rows += g.nrows;
        const int tiles = t.seg_cb + (int)(rows / (int64_t)std::max<size_t>(1, wgs.size()));
        const int64_t cost = sdd_split((int32_t)wgs.size(), row_ptr[Rb], nb, M, tiles, nsteps, sps, tsplit);
        if (cost <= best_cost) { best_cost = cost; best = nb; }      // ties: the larger group (fewer staged bytes)
    }
    return best;
}

// Plan: {n_wg, seg_cb, nseg, offset of the launch order}, then per workgroup {first row, rows, segment, blocks}, then
// per (workgroup, wavefront, slot) the block index or -1, then per (workgroup, wavefront, slot)
// (row - first row) << 20 | LDS byte offset of the tile of (column - segment start); an empty slot repeats the
// workgroup's last block there; last the launch order: the workgroups (stored segment by segment) sorted by their
// position inside the segment, then by segment, so that row groups of about the same rows are neighbours.
extern "C" int64_t mortar_sdd_plan_host(const int32_t *row_ptr, const int16_t *col, int32_t Rb, int32_t Cb,
                                        int32_t blocks_per_wave, int32_t *plan_out, int64_t plan_words) {
    const int rc = mortar_check_bcsr_host(row_ptr, col, Rb, Cb);
    if (rc) return rc;
    if (!sdd_nb_built(blocks_per_wave))
        return mortar_fail(MORTAR_ERR_ARG, "sdd_plan: blocks_per_wave=%d is not a built size (8, 10, ... 22)", blocks_per_wave);
    const int SDD_G = SDD_WAVES * blocks_per_wave;
    std::vector<SddGroup> wgs;
    const SddRows t = sdd_rows(row_ptr, col, Rb, Cb);
    const int nseg = t.nseg, seg_cb = t.seg_cb;
    sdd_groups(t, col, Rb, blocks_per_wave, plan_out != nullptr, wgs);
    const int64_t n_wg = (int64_t)wgs.size();
    const int64_t tab = 4 + n_wg * 4 + n_wg * SDD_G * 2;          // word offset of the per-segment table
    const int64_t words = tab + n_wg;
    if (tab > INT32_MAX) return mortar_fail(MORTAR_ERR_LIMIT, "sdd_plan: plan too large");
    if (!plan_out) return words;
    if (plan_words < words) return mortar_fail(MORTAR_ERR_ARG, "sdd_plan: buffer holds %lld words, need %lld",
                                               (long long)plan_words, (long long)words);
    plan_out[0] = (int32_t)n_wg; plan_out[1] = seg_cb; plan_out[2] = nseg; plan_out[3] = (int32_t)tab;
    {
        std::vector<int> first(nseg + 1, 0);                       // first workgroup of every segment
        for (int64_t w = 0; w < n_wg; ++w) first[wgs[w].seg + 1] = (int)w + 1;
        for (int sg = 0; sg < nseg; ++sg) first[sg + 1] = std::max(first[sg + 1], first[sg]);
        int32_t *order = plan_out + tab;
        int64_t n = 0;
        for (int k = 0; n < n_wg; ++k)
            for (int sg = 0; sg < nseg; ++sg)
                if (first[sg] + k < first[sg + 1]) order[n++] = first[sg] + k;
    }
    int32_t *ent_j = plan_out + 4 + n_wg * 4, *ent_o = ent_j + n_wg * SDD_G;
    for (int64_t w = 0; w < n_wg; ++w) {
        int32_t *d = plan_out + 4 + w * 4;
        d[0] = wgs[w].row0; d[1] = wgs[w].nrows; d[2] = wgs[w].seg; d[3] = wgs[w].blocks;
        for (int i = 0; i < SDD_G; ++i) {
            const bool ok = i < (int)wgs[w].j.size();
            ent_j[w * SDD_G + i] = ok ? wgs[w].j[i] : -1;
            ent_o[w * SDD_G + i] = ok ? wgs[w].o[i] : wgs[w].o.back();
        }
    }
    return words;
}

extern "C" int64_t mortar_sdd_workspace_bytes(int32_t n_wg, int32_t nnz, int32_t blocks_per_wave, int64_t M) {
    if (n_wg <= 0 || nnz <= 0 || M < 0 || !sdd_nb_built(blocks_per_wave))
        return mortar_fail(MORTAR_ERR_ARG, "sdd_workspace_bytes: bad argument");
    int nsteps, sps, tsplit;
    sdd_split(n_wg, nnz, blocks_per_wave, M, SDD_TILES, nsteps, sps, tsplit);
    return (int64_t)tsplit * nnz * 256 * (int64_t)sizeof(float);
}

template <int NB, bool WIDE>
static hipError_t sdd_launch(const SddArgs &p, hipStream_t st) {
    static bool configured = false;
    const int smem = 2 * SDD_BUF;
    if (!configured) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(sdd_kernel<NB, WIDE>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return e;
        configured = true;
    }
    hipLaunchKernelGGL((sdd_kernel<NB, WIDE>), dim3((unsigned)(8 * p.per_xcd)), dim3(SDD_WAVES * 64), smem, st, p);
    return hipSuccess;
}

template <bool WIDE>
static hipError_t sdd_launch_nb(int nb, const SddArgs &p, hipStream_t st) {
    switch (nb) {
        case 8: return sdd_launch<8, WIDE>(p, st);
        case 10: return sdd_launch<10, WIDE>(p, st);
        case 12: return sdd_launch<12, WIDE>(p, st);
        case 14: return sdd_launch<14, WIDE>(p, st);
        case 16: return sdd_launch<16, WIDE>(p, st);
        case 18: return sdd_launch<18, WIDE>(p, st);
        case 20: return sdd_launch<20, WIDE>(p, st);
    }
    return sdd_launch<22, WIDE>(p, st);
}

extern "C" int mortar_sdd_bf16(const int32_t *plan, int32_t n_wg, int32_t blocks_per_wave,
                               int32_t Rb, int32_t Cb, int32_t nnz,
                               const uint16_t *a, int64_t lda, const uint16_t *b, int64_t ldb, int64_t M,
                               float *acc, uint16_t *out, void *stream) {
    if (!plan || !out || !acc || (M > 0 && (!a || !b))) return mortar_fail(MORTAR_ERR_ARG, "sdd: null pointer");
    if (n_wg <= 0 || Rb <= 0 || Cb <= 0 || nnz <= 0 || M < 0) return mortar_fail(MORTAR_ERR_ARG, "sdd: bad shape");
    if (!sdd_nb_built(blocks_per_wave))
        return mortar_fail(MORTAR_ERR_ARG, "sdd: blocks_per_wave=%d is not a built size (8, 10, ... 22)", blocks_per_wave);
    if (reinterpret_cast<uintptr_t>(out) & 15) return mortar_fail(MORTAR_ERR_ARG, "sdd: out must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (M == 0) {                                          // no tokens: the gradient is zero
        hipLaunchKernelGGL(sdd_zero_kernel, dim3((unsigned)(((int64_t)nnz * 32 + 255) / 256)), dim3(256), 0, st,
                           reinterpret_cast<float *>(out), (int64_t)nnz * 32);
        return MORTAR_OK;
    }
    if (lda < (int64_t)Rb * 16 || ldb < (int64_t)Cb * 16 || (lda & 7) || (ldb & 7) ||
        (reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15) ||
        (reinterpret_cast<uintptr_t>(acc) & 15))
        return mortar_fail(MORTAR_ERR_ARG, "sdd: operands need 16-byte aligned rows (leading dimensions multiples of 8)");
    const int64_t n4 = (int64_t)nnz * 64;
    SddArgs p;
    p.plan = plan; p.a = a; p.b = b; p.lda = lda; p.ldb = ldb; p.M = M; p.acc = acc; p.out = out;
    p.Cb = Cb; p.nnz = nnz; p.n_wg = n_wg;
    int nseg;
    sdd_segments(Cb, nseg, p.seg_cb);
    sdd_split(n_wg, nnz, blocks_per_wave, M, SDD_TILES, p.nsteps, p.steps_per_split, p.tsplit);
    p.per_xcd = (p.tsplit * n_wg + 7) / 8;
    hipError_t e = lda > (1 << 26) || ldb > (1 << 26) ? sdd_launch_nb<true>(blocks_per_wave, p, st) : sdd_launch_nb<false>(blocks_per_wave, p, st);
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    if (p.tsplit > 1)
        hipLaunchKernelGGL(sdd_round_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, acc, out, n4, p.tsplit);
    e = hipGetLastError();
    if (e != hipSuccess) return mortar_fail(MORTAR_ERR_HIP, "sdd: %s", hipGetErrorString(e));
    return MORTAR_OK;
}
