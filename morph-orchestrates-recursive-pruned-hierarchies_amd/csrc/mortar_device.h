// Device helpers shared by the gfx950 kernels: ternary block unpack, MFMA wrappers, bf16 rounding.
#ifndef MORTAR_DEVICE_H
#define MORTAR_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// Lane decomposition used by every MFMA kernel here (v_mfma_f32_16x16x32_bf16):
//   n = lane & 15   row of the A operand (output feature inside the block-row) / column of B (token)
//   g = lane >> 4   K group: the lane holds K slots 8g .. 8g+7
// One MFMA contracts two 16x16 blocks: bsel = g >> 1 picks the block, hsel = g & 1 its column half.
// The accumulator lane holds D[4g + v][n], v = 0..3: four consecutive output features of token n.

// 8 ternary codes -> 8 bf16 weights (+-bf16(scale) or 0) in four dwords.
// A row dword holds its 16 two-bit codes (bit 1 = negative, bit 0 = non-zero) interleaved: column c < 8 in slot
// 2c + 1, column c >= 8 in slot 2(c - 8).  `t` is the dword shifted left by 2*hsel, so that the lane's 8 columns
// sit in the odd slots: masked with 0xCCCCCCCC every nibble is {sign, non-zero, 0, 0}, which read as FP4 (E2M1) is
// -2, 0 or +2, and one hardware conversion per register (v_cvt_scalef32_pk_bf16_fp4, scale 1) gives the two bf16
// patterns 0xC000 / 0 / 0x4000 of a column pair.  Read as 16-bit floats those are -2, 0, +2 as well; `sd` holds
// the block scale's bf16 pattern minus one 16-bit-float exponent step in both halves, so one packed half multiply
// returns exactly +-scale or 0 in bf16 bits (a power-of-two product is exact; the host rejects scales whose
// pattern would leave the normal range).
// The 4-bit stream stores the nibbles themselves (byte i = {column 2i, column 2i + 1}): no shift, no mask.
__device__ __forceinline__ u32x4_t mortar_scale4(uint32_t nib, uint32_t sd) {
    const f16x2_t s = __builtin_bit_cast(f16x2_t, sd);
    u32x4_t r;
    r[0] = __builtin_bit_cast(uint32_t, s * __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, 1.0f, 0)));
    r[1] = __builtin_bit_cast(uint32_t, s * __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, 1.0f, 1)));
    r[2] = __builtin_bit_cast(uint32_t, s * __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, 1.0f, 2)));
    r[3] = __builtin_bit_cast(uint32_t, s * __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, 1.0f, 3)));
    return r;
}
__device__ __forceinline__ u32x4_t mortar_unpack8(uint32_t t, uint32_t sd) {
    return mortar_scale4(t & 0xCCCCCCCCu, sd);
}
// The conversions alone: bf16 +-2 cs / 0 for the eight nibbles, cs a power of two (matrices with one scale, applied after the sums).
__device__ __forceinline__ u32x4_t mortar_nib4(uint32_t nib, float cs = 1.0f) {
    u32x4_t r;
    r[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, cs, 0));
    r[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, cs, 1));
    r[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, cs, 2));
    r[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, cs, 3));
    return r;
}

__device__ __forceinline__ f32x4_t mortar_mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// fp32 -> bf16 (round to nearest even) through the hardware conversion (v_cvt_pk_bf16_f32).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pack2(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ uint32_t bf16_bits_rne(float f) { return bf16_pack2(f, 0.f) & 0xffffu; }
__device__ __forceinline__ float bf16_to_f32(uint32_t b) { return __builtin_bit_cast(float, b << 16); }
// f rounded to bf16, as a float: the conversion of (0, f) leaves the bf16 of f in the high half and zeros below it.
__device__ __forceinline__ float bf16r(float f) { return __builtin_bit_cast(float, bf16_pack2(0.f, f)); }

#define MORTAR_GLOBAL __attribute__((address_space(1)))

// Asynchronous 16-byte-per-lane copy global -> LDS (lane l's bytes land at lds_base + 16 * l): no registers, no
// address arithmetic beyond the source pointer.  The caller waits for the copies and at a barrier before the
// destination is read: with s_waitcnt vmcnt(0), or with the number of vector loads that are certain to have been issued behind the last copy.  (One wait state separates the write of M0 from its use as the LDS base.)
__device__ __forceinline__ void mortar_load_to_lds(const MORTAR_GLOBAL char *gsrc, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(gsrc) : "memory", "m0");
}
__device__ __forceinline__ uint32_t mortar_lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char *)p;
}

// Where 16-byte unit u of token n goes in an LDS tile of 64-byte token rows: position u ^ mortar_unit_swz(n).  A wave's
// ds_read_b128 is served in groups of 16 lanes {0-3, 12-15, 20-23, 24-27} and {4-11, 16-19, 28-31} (and the same 32 lanes
// up); with lanes = 16 tokens x 2 units each group then covers all 64 banks (8 of 12 cycles per read were conflicts with
// the plain order of tokens).
__device__ __forceinline__ int mortar_unit_swz(int n) { return (4 - (n >> 2)) & 3; }

// The value of lane (lane ^ X) within a row of 16 lanes, on the vector ALU.
template <int X>
__device__ __forceinline__ uint32_t mortar_row_xor(uint32_t v) {
    static_assert(X == 1 || X == 2 || X == 4 || X == 8, "distances within a row");
    if constexpr (X == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true);          // quad_perm [1,0,3,2]
    else if constexpr (X == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true);     // quad_perm [2,3,0,1]
    else if constexpr (X == 4)                                                                             // row_half_mirror (^ 7), quad_perm [3,2,1,0] (^ 3)
        return (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
    else return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true);                          // row_ror:8
}
template <int X>
__device__ __forceinline__ double mortar_row_xor(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)mortar_row_xor<X>((uint32_t)(u >> 32)) << 32 | mortar_row_xor<X>((uint32_t)u));
}
// op over the wavefront as a xor butterfly (distances 32, 16, 8, 4, 2, 1; every lane ends with the result), op commutative: half-wave and
// row swaps, then DPP.  The kernels that use it at a few rows are chains of latencies, and the six exchanges through the LDS crossbar were
// 0.3 us of each: the router's tail (four sums in a row) 5.8 -> 4.6 us, routed decode steps 7 % shorter over 60 shapes of 1 to 64 rows,
// gate_up with its norm 2 %.
template <typename Op>
__device__ __forceinline__ uint32_t mortar_wave_reduce(uint32_t v, Op op) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);        // the lower halves, the upper halves
    v = op(a[0], a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);        // the even rows, the odd rows
    v = op(b[0], b[1]);
    v = op(v, mortar_row_xor<8>(v));
    v = op(v, mortar_row_xor<4>(v));
    v = op(v, mortar_row_xor<2>(v));
    return op(v, mortar_row_xor<1>(v));
}
__device__ __forceinline__ float mortar_wave_sum(float v) {
    return __builtin_bit_cast(float, mortar_wave_reduce(__builtin_bit_cast(uint32_t, v), [](uint32_t a, uint32_t b) {
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b));
    }));
}
__device__ __forceinline__ double mortar_wave_sum(double v) {
    const auto halves = [&v](auto swap) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const auto l = swap((uint32_t)u), h = swap((uint32_t)(u >> 32));
        v = __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) + __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
    };
    halves([](uint32_t w) { return __builtin_amdgcn_permlane32_swap(w, w, false, false); });
    halves([](uint32_t w) { return __builtin_amdgcn_permlane16_swap(w, w, false, false); });
    v += mortar_row_xor<8>(v);
    v += mortar_row_xor<4>(v);
    v += mortar_row_xor<2>(v);
    return v + mortar_row_xor<1>(v);
}

// ---- RMSNorm pieces shared by the stand-alone kernel and the fused staging of gate_up, so that both round alike.
// A row is handled by one wavefront in 16-byte units (8 bf16): a lane adds the squares of its units in ascending
// unit order (fused multiply-adds, low half-word first), the lanes meet in a xor butterfly.
__device__ __forceinline__ float rms_sumsq8(u32x4_t u, float s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float lo = __builtin_bit_cast(float, u[j] << 16), hi = __builtin_bit_cast(float, u[j] & 0xffff0000u);
        s = __builtin_fmaf(lo, lo, s);
        s = __builtin_fmaf(hi, hi, s);
    }
    return s;
}
__device__ __forceinline__ float rms_wave_sum(float v) { return mortar_wave_sum(v); }
__device__ __forceinline__ float rms_scale(float sumsq, int d, float eps) { return 1.0f / sqrtf(sumsq / (float)d + eps); }
// bf16(bf16(x * r) * w) on 8 values; has_w = false leaves out the weight.
__device__ __forceinline__ u32x4_t rms_apply8(u32x4_t u, float r, u32x4_t w, bool has_w) {
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float lo = __builtin_bit_cast(float, u[j] << 16), hi = __builtin_bit_cast(float, u[j] & 0xffff0000u);
        uint32_t pk = bf16_pack2(lo * r, hi * r);
        if (has_w) {
            const float wl = __builtin_bit_cast(float, w[j] << 16), wh = __builtin_bit_cast(float, w[j] & 0xffff0000u);
            pk = bf16_pack2(__builtin_bit_cast(float, pk << 16) * wl, __builtin_bit_cast(float, pk & 0xffff0000u) * wh);
        }
        o[j] = pk;
    }
    return o;
}

// silu in fp32 from a bf16-rounded input; the result is rounded to bf16 by the caller, which absorbs the
// 1-ulp error of the hardware exp and reciprocal.
__device__ __forceinline__ float silu_f32(float g) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)); }

// SwiGLU epilogue for the four consecutive hidden features a lane holds: every intermediate is rounded to
// bf16 where the reference materialises a bf16 tensor (gate_up output, silu, product, gated product).
// `gate` is the router gate of these features (they lie in one cluster); pass has_gate = false for none.
__device__ __forceinline__ u32x2_t swiglu_pack4(f32x4_t g, f32x4_t u, bool has_gate, float gate) {
    // each value is rounded on its own (one conversion, no unpacking of a packed pair)
    float h[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) h[v] = bf16r(silu_f32(bf16r(g[v]))) * bf16r(u[v]);
    if (has_gate) {
        const float gb = bf16r(gate);
#pragma unroll
        for (int v = 0; v < 4; ++v) h[v] = bf16r(h[v]) * gb;
    }
    return u32x2_t{bf16_pack2(h[0], h[1]), bf16_pack2(h[2], h[3])};
}

#endif
