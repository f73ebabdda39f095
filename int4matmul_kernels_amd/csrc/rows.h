// What the few-row kernels share: their arguments, and the decode of eight codes of one column to the operand of
// v_mfma_f32_16x16x32_f16 (the 32 x 16 operand: lane group h of a wave holds chunk h, eight consecutive k, of a
// 32-row block; see skinny.hip).
#pragma once

#include "common.h"

namespace i4 {

// magic numbers (div_magic) of the divisors of the balanced launch's range arithmetic: K / 64, the group's units
struct BalancedMagics { uint32_t units, group_units; };

struct SkinnyArgs {
    h16* outs;
    const uint32_t* matrix;
    const uint32_t* mask;   // 16:32 sparse only
    const h16* x;
    const h16* scales;
    const h16* zeros;
    int R, K, S;
    int group_units;        // group size / 64
    int units_per_wave;
    int accumulate;         // 1: outs = fp16(fp32(outs) + product) (matvec semantics); 0: overwrite
    // split-K across workgroups (gridDim.z > 1; narrow matrices with a long K): each workgroup takes
    // `units_per_split` units, stores its fp32 partial tile to `part` and counts itself in; the last one
    // to arrive adds the partials up in split order and writes the strip
    int units_per_split;
    float* part;
    int* counters;
    // balanced launch of the few-row kernel (more strips than CUs): 256 workgroups share the strips' units
    // evenly, workgroup i takes [i q + i r / 256, (i + 1) q + (i + 1) r / 256) of strips x units, strip-major
    int bal_q, bal_r;
    BalancedMagics bal_magics;
    // launch with a fifth column per lane: the first `wide_wgs` workgroups take 80 columns, the others 64
    int wide_wgs;
};

template <int CW> struct Words;
template <> struct Words<4> { typedef u32x4 type; };
template <> struct Words<2> { typedef u32x2 type; };
template <> struct Words<1> { typedef uint32_t type; };

template <int CW>
__device__ __forceinline__ uint32_t word_of(const typename Words<CW>::type& v, int c) {
    if constexpr (CW == 1) return v;
    else return v[c];
}


// Per format: the k order of the 8 halves of an operand chunk, the offsets the
// magic-number decode leaves on the low / high half of operand register e, and
// the packed rows of a 32-row block.
//   int4: order 0,4,1,5,2,6,3,7; registers 0, 2 carry 1024 + q, registers 1, 3 carry 64 + q
//   int2: natural order, {1024 + q_even, 256 + q_odd};  int3: natural order, {1024 + q_even, 128 + q_odd}
template <int BITS, bool SPARSE = false> struct SkFmt;
template <> struct SkFmt<4, true> {
    static constexpr int ROWS = 2, LOADS = 6;            // per block: two words of codes and the mask word
    __device__ static constexpr int order(int e) { return (e >> 1) + 4 * (e & 1); }
    __device__ static constexpr uint32_t offs(int) { return 0u; }
};
template <> struct SkFmt<4> {
    static constexpr int ROWS = 4, LOADS = 2;            // packed rows per block, loads per lane and unit
    __device__ static constexpr int order(int e) { return (e >> 1) + 4 * (e & 1); }
    __device__ static constexpr uint32_t offs(int e) { return (e & 1) ? 0x54005400u : 0x64006400u; }
};
template <> struct SkFmt<2> {
    static constexpr int ROWS = 2, LOADS = 2;
    __device__ static constexpr int order(int e) { return e; }
    __device__ static constexpr uint32_t offs(int) { return 0x5C006400u; }
};
template <> struct SkFmt<3> {
    static constexpr int ROWS = 3, LOADS = 4;
    __device__ static constexpr int order(int e) { return e; }
    __device__ static constexpr uint32_t offs(int) { return 0x58006400u; }
};

// The 8 codes of one chunk (`f`: BITS bits apart, LSB first, garbage above) -> MFMA
// operand of magic numbers; m0/g0 (and m1/g1 for int4) are the format's mask and
// magic constants held in VGPRs.
template <int BITS>
__device__ __forceinline__ h16x8 magic_operand(uint32_t f, uint32_t m0, uint32_t m1, uint32_t g0, uint32_t g1) {
    u32x4 r;
    if constexpr (BITS == 4) {
        const uint32_t f8 = f >> 8;
        r = u32x4{(f & m0) | g0, (f & m1) | g1, (f8 & m0) | g0, (f8 & m1) | g1};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t u = f >> (2 * BITS * e);
            r[e] = (__builtin_amdgcn_perm(u, u, 0x01000100u) & m0) | g0;       // low 16 bits in both halves
        }
    }
    return bitcast<h16x8>(r);
}

// 16:32: `v` = the chunk's kept codes as consecutive nibbles, `sel` = the selectors of its mask byte
__device__ __forceinline__ u32x4 sparse_operand(uint32_t v, const u32x4& sel, uint32_t nib, uint32_t flag) {
    const uint32_t even = (v & nib) | flag, odd = ((v >> 4) & nib) | flag;
    return u32x4{__builtin_amdgcn_perm(odd, even, sel.x), __builtin_amdgcn_perm(odd, even, sel.y),
                 __builtin_amdgcn_perm(odd, even, sel.z), __builtin_amdgcn_perm(odd, even, sel.w)};
}

__device__ __forceinline__ h16x8 exact_operand_sparse(uint32_t v, uint32_t m8, h16 sc, h16 ze) {
    h16 row[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const bool kept = (m8 >> r) & 1u;
        row[r] = kept ? dequant_code<4>(v & 15u, sc, ze) : (h16)0.0f;
        v >>= kept ? 4 : 0;
    }
    h16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = row[SkFmt<4, true>::order(e)];
    return o;
}

// The chunk's 8 fp16 weights themselves, in the operand's k order, in either quantisation mode
// (the mode belongs to the lane's column and group), bit-exact with dequant_code and without a
// branch: from the magic-number pairs, P = the codes (offsets removed, exact) or +-2^e,
//     A = P + N (one rounding),  w = fma(A, B, C) (one rounding)
// with (N, B, C) = (-z, s, -0) for a linear group -- fp16(q - z), then fp16(. * s); adding -0
// changes no bit -- and (-0, -s, z) for an exponent group, the reference's single-rounded fma.
template <int BITS>
__device__ __forceinline__ h16x8 exact_operand(uint32_t f, uint32_t m0, uint32_t m1, uint32_t g0, uint32_t g1,
                                               h16 sc, h16 ze) {
    const u32x4 h = bitcast<u32x4>(magic_operand<BITS>(f, m0, m1, g0, g1));
    const bool expo = !(sc >= (h16)0.0f);
    const h16x2 minus0 = as_h2(0x80008000u), s2 = {sc, sc}, z2 = {ze, ze};
    const h16x2 N = expo ? minus0 : -z2, B = expo ? -s2 : s2, C = expo ? z2 : minus0;
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t offs = SkFmt<BITS>::offs(e);                    // {2^a, 2^b} as halves
        const h16x2 q = as_h2(h[e]) - as_h2(offs);                     // exact
        // the same offsets as integers, for the packed multiply: 2^(exponent field - 15)
        const uint32_t ints = off2(1u << (((offs >> 10) & 31u) - 15u), 1u << (((offs >> 26) & 31u) - 15u));
        const h16x2 P = expo ? as_h2(expo_operand<BITS>(h[e], ints)) : q;
        r[e] = as_u32(__builtin_elementwise_fma(P + N, B, C));
    }
    return bitcast<h16x8>(r);
}

// The chunk's codes as they are or, TWO_MODES and a negative (or NaN) scale, as +-2^e: both exact in fp16
template <int BITS, bool TWO_MODES>
__device__ __forceinline__ h16x8 plain_operand(uint32_t f, uint32_t m0, uint32_t m1, uint32_t g0, uint32_t g1, h16 sc) {
    const u32x4 h = bitcast<u32x4>(magic_operand<BITS>(f, m0, m1, g0, g1));
    const bool expo = TWO_MODES && !(sc >= (h16)0.0f);
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t offs = SkFmt<BITS>::offs(e);                    // {2^a, 2^b} as halves
        r[e] = as_u32(as_h2(h[e]) - as_h2(offs));
        if constexpr (TWO_MODES) {
            // the same offsets as integers, for the packed multiply: 2^(exponent field - 15)
            const uint32_t ints = off2(1u << (((offs >> 10) & 31u) - 15u), 1u << (((offs >> 26) & 31u) - 15u));
            r[e] = expo ? expo_operand<BITS>(h[e], ints) : r[e];
        }
    }
    return bitcast<h16x8>(r);
}

// the kernel whose waves share the staged states (csrc/wide.hip): false when its plan does not take the product
bool wide_rows(int bits, const SkinnyArgs& a, RowsCall call, void* workspace, size_t workspace_bytes, hipStream_t st);
size_t wide_workspace_bytes(int bits, int64_t R, int64_t K, int64_t S, bool sparse, int64_t group_units, RowsCall call);

}  // namespace i4
