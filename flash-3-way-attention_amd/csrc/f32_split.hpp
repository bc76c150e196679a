// fp32 products on the bf16 matrix cores (gfx950), shared by the fp32 kernels.
//
// A float is the sum of three bf16 numbers, x = h + m + l: h is x rounded, m what that leaves, rounded, l the rest (three
// significands of eight bits hold all 24, down to 2^-109).  Of the nine products of two such sums six are formed, those of 2^-16 and more of
// the whole: what is left out is below 2^-24 of each product.  v_mfma_f32_32x32x16_bf16 takes 32 cycles for 16 k-slots and
// v_mfma_f32_32x32x2_f32 64 for two, so six products of the former cost 192 cycles where the latter costs 512, and a sum over
// 16 slots is rounded once per product instead of eight times.  Against 64 bits (32x32 tiles of N(0,1), 2-norm): a contraction
// over 64 is 1.44e-7 off on fp32 MFMAs, 1.10e-7 with the six products of each k-step in turn (products_of_step) and 0.50e-7
// with all the small ones ahead of the large ones (small_products, large_product); over 1024, 5.7e-7 and 4.9e-7.
//
// Operands that are infinite or above kSplitMax (h would be rounded to infinity and m, x - h, be no number): split8_any.  It gives
// an infinite one as (+-1, 0, +-infinity), of whose six products with a finite operand only l h is infinite, with the sign and the
// zero case of the fp32 product, and with an infinite one l h and h l; and a finite one h rounded toward zero.  split8 is for values
// that cannot be that large (probabilities), for a triple-dot backward's dS (an infinite one makes NaN of what it enters), and
// where a result is looked at for NaN and formed again (dps_f32_mfma.hip).  Small operands: bf16 ends at 2^-133 (these MFMAs take
// its subnormal numbers), so below 2^-109 (1.5e-33) l loses digits and below 2^-117 all of them.  Against 64 bits, the worst gradient of
// a triple-dot backward (T = 64, D = 64), whose dS lies some 2^-9 below dO: dO of 2^-105 3e-7 as at 1, 2^-109 1.2e-6, 2^-113 1.9e-5.
#pragma once
#include "mfma.hpp"

namespace tritt {

struct Split8 {
    bf16x8 h, m, l;
};
// x: anything whose elements 0 .. 7 are floats
template <typename X>
__device__ __forceinline__ Split8 split8(const X& x) {
    Split8 s;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const f32x2 v = {x[e], x[e + 1]};
        const bf16x2 h = __builtin_convertvector(v, bf16x2);
        const f32x2 r = {v[0] - (float)h[0], v[1] - (float)h[1]};
        const bf16x2 m = __builtin_convertvector(r, bf16x2);
        const f32x2 t = {r[0] - (float)m[0], r[1] - (float)m[1]};
        const bf16x2 l = __builtin_convertvector(t, bf16x2);
        s.h[e] = h[0]; s.h[e + 1] = h[1];
        s.m[e] = m[0]; s.m[e + 1] = m[1];
        s.l[e] = l[0]; s.l[e + 1] = l[1];
    }
    return s;
}
constexpr float kSplitMax = 0x1.fep127f;  // the largest bf16 number
template <typename X>
__device__ __forceinline__ float largest8(const X& x) {
    float most = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(x[e]));
    return most;
}
template <typename X>
__device__ __forceinline__ Split8 split8_any(const X& x) {
    Split8 s = split8(x);
    if (__builtin_expect(__any(largest8(x) > kSplitMax), 0)) {  // (a uniform branch: its body is placed out of the way)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (!(fabsf(x[e]) > kSplitMax)) continue;
            const bool infinite = fabsf(x[e]) == INFINITY;
            const float h = copysignf(infinite ? 1.f : kSplitMax, x[e]), r = infinite ? 0.f : x[e] - h;
            const __bf16 m = (__bf16)r;
            s.h[e] = (__bf16)h;
            s.m[e] = m;
            s.l[e] = (__bf16)(infinite ? x[e] : r - (float)m);
        }
    }
    return s;
}
template <bool ANY, typename X>
__device__ __forceinline__ Split8 split_value(const X& x) {
    if constexpr (ANY) return split8_any(x);
    else return split8(x);
}
__device__ __forceinline__ f32x16 small_products(const Split8& a, const Split8& b, f32x16 c) {
    using M = Mma<__bf16>;
    c = M::mma(a.l, b.h, c);
    c = M::mma(a.h, b.l, c);
    c = M::mma(a.m, b.m, c);
    c = M::mma(a.m, b.h, c);
    return M::mma(a.h, b.m, c);
}
__device__ __forceinline__ f32x16 large_product(const bf16x8& ah, const bf16x8& bh, f32x16 c) {
    return Mma<__bf16>::mma(ah, bh, c);
}
__device__ __forceinline__ f32x16 products_of_step(const Split8& a, const Split8& b, f32x16 c) {
    return large_product(a.h, b.h, small_products(a, b, c));
}

// A stage of 32 rows in LDS: three planes (h, m, l) of [32][D] bf16, rows dense, the 16-byte pieces of a row at piece ^
// split_swizzle(row).  Both reads below are then free of bank conflicts: a 16-byte read of the wave serves 16 lanes at a time,
// whose rows differ mod 16 here and must fall on distinct pieces mod 16 (256 bytes); an 8-byte transposed read serves 32
// lanes, four consecutive rows of 64 bytes each.
template <int D>
__device__ __forceinline__ constexpr int split_swizzle(int row) {
    if (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
    if (D == 64) return ((row & 2) << 1) | ((row >> 2) & 3);
    return (row >> 2) & 3;
}
template <int D>
constexpr int split_plane() {  // elements of a plane
    return 32 * D;
}
typedef __attribute__((ext_vector_type(4))) short s16x4;

// Operand "rows" of a score product, k-step ks: lane (n, g) gets columns 16 ks + 8 g .. + 7 of row key_of_row(n).
// `base` = split_row_base(lane) (elements); `tile` = the stage's h plane
template <int D>
__device__ __forceinline__ int split_row_base(int lane) {
    const int row = key_of_row(lane & 31), g = lane >> 5;
    return row * D + ((g ^ split_swizzle<D>(row)) * 8);
}
template <int D>
__device__ __forceinline__ Split8 split_rows(const __bf16* tile, int base, int ks) {
    const __bf16* at = tile + (base ^ (ks * 16));  // the piece's number is the low bits of base / 8, rows are powers of two
    return {*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + split_plane<D>()),
            *reinterpret_cast<const bf16x8*>(at + 2 * split_plane<D>())};
}
// Operand "columns" of a product over rows: lane (n, g) gets rows 16 half + 8 g .. + 7 of column 32 dt + n.  In every group
// of 16 lanes ds_read_b64_tr_b16 gives lane l elements l % 4 of what lanes l / 4, 4 + l / 4, 8 + l / 4 and 12 + l / 4 address,
// so lane i addresses row i / 4 and columns 4 (i % 4) .. + 3 of the group's 16; two reads for eight rows.
template <int D>
__device__ __forceinline__ int split_col_base(int lane) {
    const int i = lane & 15, row = 8 * (lane >> 5) + (i >> 2), piece = 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
    return row * D + ((piece ^ split_swizzle<D>(row)) * 8) + (i & 1) * 4;
}
template <int D>
__device__ __forceinline__ bf16x8 split_cols_plane(const __bf16* plane, int base, int half, int dt) {
    // four rows on, split_swizzle changes in its lowest bit; 16 rows on, not at all
    const int lo = base ^ (dt * 32), hi = lo ^ 8;
    const __bf16 *p = plane + half * 16 * D + lo, *q = plane + half * 16 * D + 4 * D + hi;
    const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)q);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
}
template <int D>
__device__ __forceinline__ Split8 split_cols(const __bf16* tile, int base, int half, int dt) {
    return {split_cols_plane<D>(tile, base, half, dt), split_cols_plane<D>(tile + split_plane<D>(), base, half, dt),
            split_cols_plane<D>(tile + 2 * split_plane<D>(), base, half, dt)};
}

}  // namespace tritt
