// Quantized matrix-matrix product for gfx950:
//     outs[m, s] = fp16( sum_k fp32(x[m, k]) * fp32(w16[k, s]) )
// where w16 is the fp16 matrix the reference's unpack step builds (two fp16
// roundings per weight in linear mode, one fused multiply-add in exponent mode).
//
// Two kernels.  matmul_kernel_pipe (further down) is the fast one, for any number of
// rows and outputs whose columns fill at least two thirds of whole tiles;
// matmul_kernel takes everything else.  Common to both: one
// workgroup owns a tile of outs; per K step the packed weights of the tile are
// read from HBM once, decoded and dequantised to fp16 ONCE by the workgroup and
// stored to LDS in MFMA operand layout: 16-byte chunks
// of 8 consecutive k for one column, chunk (kc, n) at kc*BN + n, which both the
// writes (lanes along n) and the MFMA operand reads (lanes along n) touch
// without bank conflicts.  The states tile is stored row-major with an XOR
// swizzle of the chunk index so that row-contiguous writes and column-of-rows
// operand reads are both conflict-free.  Accumulation is fp32 in the MFMA
// accumulators.
//
// matmul_kernel walks K in steps of 64 with the global loads of step k+1 issued
// before the MFMA phase of step k (register prefetch) and two barriers per step.
//
// Workgroups are renumbered so that the 8 XCDs (each with its own L2) take
// disjoint column ranges of the weight matrix.
#include "common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace i4 {

constexpr int BK = 64;

// swizzle of the 16-byte chunk index inside a 128-byte row of the states tile
__device__ __forceinline__ int a_swz(int m) { return (m & 7) ^ ((m >> 3) & 1); }

struct MatmulArgs {
    h16* outs;
    const uint32_t* matrix;
    const uint32_t* mask;
    const h16* x;
    const h16* scales;
    const h16* zeros;
    int M, K, S;
    int group_units;        // group size / 64
    int tiles_m, tiles_n;
    int by_columns;         // pipelined kernel: 1 = an XCD walks its range of tile columns row by row
    // split-K (pipelined kernel, grids that would leave most of the GPU idle): `ksplit` workgroups
    // share a tile, each walks 1 / ksplit of the K steps and stores its fp32 partial tile to
    // `part`; the one that arrives last (`counters`, one per tile) adds them up in split order
    int ksplit;
    float* part;
    int* counters;
    // tiles (in grid order) before `split_from` are not split: a grid whose last round would fill
    // at most half of the GPU splits only the tiles of that round
    int split_from;
};

// Raw packed data of one (32-row block, column) cell
template <int BITS, bool SPARSE>
struct Cell {
    uint32_t w[SPARSE ? 2 : BITS];
    uint32_t m;
};

template <int BITS, bool SPARSE>
__device__ __forceinline__ void load_cell(Cell<BITS, SPARSE>& c, const MatmulArgs& a, int blk, int col) {
    constexpr int ROWS = SPARSE ? 2 : BITS;
    const int64_t S = a.S;
    const uint32_t* p = a.matrix + (int64_t)blk * ROWS * S + col;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) c.w[r] = p[r * S];
    c.m = SPARSE ? a.mask[(int64_t)blk * S + col] : 0xFFFFFFFFu;
}

// General cell decode: 32 fp16 weights = 4 chunks of 8, bit-exact with the
// reference decode, any format and either quantisation mode.
template <int BITS, bool SPARSE>
__device__ __forceinline__ void dequant_cell_generic(const Cell<BITS, SPARSE>& c, h16 sc, h16 ze, h16x8 out[4]) {
    uint32_t codes[32];
    if constexpr (SPARSE) {
        uint64_t v = (uint64_t)c.w[0] | ((uint64_t)c.w[1] << 32);
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const bool k = (c.m >> t) & 1u;
            codes[t] = (uint32_t)v & 0xFu;
            v >>= k ? 4 : 0;
        }
    } else if constexpr (BITS == 3) {
        const uint64_t lo = (uint64_t)c.w[0] | ((uint64_t)c.w[1] << 32);
        const uint64_t hi = (uint64_t)c.w[1] | ((uint64_t)c.w[2] << 32);
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const int pos = 3 * t;
            codes[t] = pos + 3 <= 64 ? (uint32_t)(lo >> pos) & 7u : (uint32_t)(hi >> (pos - 32)) & 7u;
        }
    } else {
        constexpr int PER = 32 / BITS;
#pragma unroll
        for (int i = 0; i < BITS; ++i) {
            uint32_t v = c.w[i];
#pragma unroll
            for (int j = 0; j < PER; ++j) { codes[i * PER + j] = v & ((1u << BITS) - 1u); v >>= BITS; }
        }
    }
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        h16 w = dequant_code<BITS>(codes[t], sc, ze);
        if (SPARSE && !((c.m >> t) & 1u)) w = (h16)0.0f;
        out[t >> 3][t & 7] = w;
    }
}

// ---- decodes of a chunk, 8 consecutive k of one column, bit-exact and in natural k order
// The coefficients of a column's group: {s, s}, {z, z} or what the decode makes of them.
// Linear mode: the reference's own two roundings, fp16(q - z), fp16(. * s).
struct LinearCoef {
    h16x2 s, z;
    __device__ __forceinline__ void set(h16x2 s2, h16x2 z2) { s = s2; z = z2; }
    __device__ __forceinline__ uint32_t weight(h16x2 q) const { return as_u32((q - z) * s); }
};
// Either mode, chosen per thread (a thread decodes whole columns, and the mode belongs to a (group, column)), without a branch:
//     A = P + N (one rounding),  w = fma(A, B, C) (one rounding)
// linear:   P = q, N = -z, B = s, C = -0:  fp16(q - z), then fp16(. * s) -- adding -0 changes nothing
// exponent: P = +-2^e, N = -0, B = -s, C = z:  the reference's single-rounded fma (matmul.cuh:127-136)
struct TwoModeCoef {
    uint32_t m;                                  // all ones in exponent mode (bit picks: a selection came out as a branch)
    h16x2 N, B, C;
    float scale;                                 // of the 8-bit floats: 2^9 for q, 1 for +-2^e
    __device__ __forceinline__ uint32_t pick(uint32_t e, uint32_t l) const { return (e & m) | (l & ~m); }
    __device__ __forceinline__ void set(h16x2 s2, h16x2 z2) {
        m = s2.x >= (h16)0.0f ? 0u : 0xFFFFFFFFu;
        N = as_h2(pick(0x80008000u, as_u32(z2) ^ 0x80008000u));
        B = as_h2(as_u32(s2) ^ (m & 0x80008000u));
        C = as_h2(pick(as_u32(z2), 0x80008000u));
        scale = bitcast<float>(pick(0x3F800000u, 0x44000000u));
    }
    __device__ __forceinline__ uint32_t weight(h16x2 P) const { return as_u32(__builtin_elementwise_fma(P + N, B, C)); }
    // four codes as bytes -> the 8-bit floats of q 2^-9 or +-2^e
    __device__ __forceinline__ uint32_t powers(uint32_t b) const {
        return pick(((b & 0x08080808u) << 4) | (((b & 0x07070707u) << 3) + 0x38383838u), b);
    }
};
// int2: the group's four weights, in either mode, are a v_perm table
struct Int2Coef {
    uint32_t T0, T1;
    __device__ __forceinline__ void set(h16x2 s2, h16x2 z2) {
        TwoModeCoef c;
        c.set(s2, z2);
        T0 = c.weight(as_h2(c.pick(0x40003C00u, 0x3C000000u)));
        T1 = c.weight(as_h2(c.pick(0xC000BC00u, 0x42004000u)));
    }
};
// int3: the eight values' upper bytes are one (their lower ones are 0)
struct Int3Coef : TwoModeCoef {
    uint32_t T0, T1;
    __device__ __forceinline__ void set(h16x2 s2, h16x2 z2) {
        TwoModeCoef::set(s2, z2);
        T0 = pick(0x4844403Cu, 0x42403C00u);
        T1 = pick(0xC8C4C0BCu, 0x47464544u);
    }
};
template <int BITS, bool TWO_MODES>
using Coef = std::conditional_t<BITS == 2, Int2Coef, std::conditional_t<BITS == 3, Int3Coef, std::conditional_t<TWO_MODES, TwoModeCoef, LinearCoef>>>;

// four codes of a word as bytes -> eight weights: a byte q < 16 is the 8-bit float q 2^-9
template <class C>
__device__ __forceinline__ h16x8 weights_of_bytes(uint32_t b03, uint32_t b47, const C& c) {
    float scale = 512.f;
    if constexpr (std::is_same_v<C, TwoModeCoef>) {
        b03 = c.powers(b03);
        b47 = c.powers(b47);
        scale = c.scale;
    }
    return bitcast<h16x8>(u32x4{c.weight(from_fp8<false>(b03, scale)), c.weight(from_fp8<true>(b03, scale)),
                                c.weight(from_fp8<false>(b47, scale)), c.weight(from_fp8<true>(b47, scale))});
}

// `bits`: the chunk's codes, LSB first, BITS bits apart (bits above 8 * BITS are ignored).  17 (int4), 17 (int2) and 24 (int3)
// instructions; with magic numbers and their removal 20, 24 and 24, and twice as many for either mode
template <int BITS, class C>
__device__ __forceinline__ h16x8 dequant_chunk(uint32_t bits, const C& c) {
    if constexpr (BITS == 4) {
        const uint32_t even = bits & 0x0F0F0F0Fu, odd = (bits >> 4) & 0x0F0F0F0Fu;
        return weights_of_bytes(__builtin_amdgcn_perm(odd, even, 0x05010400u), __builtin_amdgcn_perm(odd, even, 0x07030602u), c);
    } else if constexpr (BITS == 2) {
        const uint32_t v = (bits & 0xFFFFu) | (bits << 14);               // code 2 j at bit 4 j, code 2 j + 1 at 16 + 4 j
        u32x4 r;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            r[j] = __builtin_amdgcn_perm(c.T1, c.T0, __umul24((v >> (4 * j)) & 0x00030003u, 0x0202u) + 0x01000100u);
        return bitcast<h16x8>(r);
    } else {
        const uint32_t u = bits & 0xFFFFFFu;
        const uint32_t v = (u & 0xFFFFu) | ((u << 13) & 0xFFFF0000u);      // codes 0, 2, 4 at bits 0, 6, 12, codes 1, 3, 5 at 16, 22, 28
        const uint32_t y = u >> 10;                                       // code 6 at bit 8, code 7 at 11
        const uint32_t sel[4] = {v << 8, v << 2, v >> 4, (y << 13) | y};
        u32x4 r;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = c.weight(as_h2(__builtin_amdgcn_perm(c.T1, c.T0, (sel[j] & 0x07000700u) | 0x000C000Cu)));
        return bitcast<h16x8>(r);
    }
}

template <int BITS, bool SPARSE>
__device__ __forceinline__ void dequant_cell(const Cell<BITS, SPARSE>& c, h16 sc, h16 ze, h16x8 out[4]) {
    if constexpr (BITS == 4 && !SPARSE) {
        if (sc >= (h16)0.0f) {
            const LinearCoef co = {{sc, sc}, {ze, ze}};
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = dequant_chunk<4>(c.w[i], co);
            return;
        }
    }
    dequant_cell_generic<BITS, SPARSE>(c, sc, ze, out);
}

// T threads; thread t owns column t % BN of the weight tile and CPT of its
// (2 * BN / T) 32-row cells per K step.
template <int BITS, bool SPARSE, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void matmul_kernel(MatmulArgs a) {
    constexpr int WAVES_N = BN / WN, WAVES_M = BM / WM;
    constexpr int T = WAVES_M * WAVES_N * 64;
    constexpr int TM = WM / 32, TN = WN / 32;     // MFMA tiles per wave
    constexpr int A_CHUNKS = BM * 8 / T;          // 16-byte chunks of the states tile per thread
    constexpr int CPT = 2 * BN / T;               // weight cells per thread
    static_assert(BM * 8 % T == 0 && (T == BN || T == 2 * BN), "tile/thread mismatch");
    static_assert(CPT == 1 || CPT == 2, "one or two cells per thread");

    __shared__ __attribute__((aligned(16))) h16 As[BM * BK];
    __shared__ __attribute__((aligned(16))) h16 Bs[BK * BN];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;

    // XCD-aware renumbering: workgroup i runs on XCD i % 8; give each XCD a
    // contiguous range of column tiles and walk the row tiles fastest.
    int bid = blockIdx.x;
    const int total = a.tiles_m * a.tiles_n;
    {
        const int per_xcd = (total + 7) / 8;
        const int xcd = bid % 8, local = bid / 8;
        const int renum = xcd * per_xcd + local;
        if (total % 8 == 0) bid = renum;
    }
    const int tile_m = bid % a.tiles_m, tile_n = bid / a.tiles_m;
    const int m0 = tile_m * BM, s0 = tile_n * BN;
    const int64_t boff = blockIdx.z;
    const h16* x = a.x + boff * a.M * (int64_t)a.K;
    h16* outs = a.outs + boff * a.M * (int64_t)a.S;

    const int bn = t % BN, bhb0 = (t / BN) * CPT;
    const int bcol = min(s0 + bn, a.S - 1);

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    u32x4 areg[A_CHUNKS];
    Cell<BITS, SPARSE> cell[CPT];
    h16 sc, ze;

    auto load_tile = [&](int kt) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            const int c = t + T * i, m = c >> 3, kc = c & 7;
            const int row = min(m0 + m, a.M - 1);
            areg[i] = *reinterpret_cast<const u32x4*>(x + (int64_t)row * a.K + kt * BK + kc * 8);
        }
#pragma unroll
        for (int q = 0; q < CPT; ++q) load_cell<BITS, SPARSE>(cell[q], a, kt * 2 + bhb0 + q, bcol);
        const int64_t gofs = (int64_t)(kt / a.group_units) * a.S + bcol;
        sc = a.scales[gofs];
        ze = a.zeros[gofs];
    };

    const int ktiles = a.K / BK;
    load_tile(0);
    for (int kt = 0; kt < ktiles; ++kt) {
        // registers -> LDS
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            const int c = t + T * i, m = c >> 3, kc = c & 7;
            *reinterpret_cast<u32x4*>(&As[m * BK + ((kc ^ a_swz(m)) << 3)]) = areg[i];
        }
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            h16x8 w[4];
            dequant_cell<BITS, SPARSE>(cell[q], sc, ze, w);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<h16x8*>(&Bs[(((bhb0 + q) * 4 + e) * BN + bn) * 8]) = w[e];
        }
        __syncthreads();
        if (kt + 1 < ktiles) load_tile(kt + 1);

#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            const int kc = 2 * ks + (lane >> 5);
            h16x8 af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int m = wm0 + i * 32 + (lane & 31);
                af[i] = *reinterpret_cast<const h16x8*>(&As[m * BK + ((kc ^ a_swz(m)) << 3)]);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = wn0 + j * 32 + (lane & 31);
                bf[j] = *reinterpret_cast<const h16x8*>(&Bs[(kc * BN + n) * 8]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    // epilogue: accumulator register r of lane l is row 8*(r/4) + 4*(l/32) + r%4,
    // column l%32 of its 32x32 tile
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = s0 + wn0 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (row < a.M && col < a.S) outs[(int64_t)row * a.S + col] = (h16)acc[i][j][r];
            }
        }
}

// ---- the pipelined kernel: (TM * 32) x (NW * 64) tiles, 2 x NW waves of (TM * 16) x 64, K steps of 32.
//
// What bounds it is the power limit: at full load the clock falls to what the work of a K step allows, so energy per step counts,
// and beside it the step's length.  Hence
//  * v_mfma_f32_16x16x32_f16: a loop of nothing but MFMAs and their LDS reads, on all CUs and random data, does 1710 TFLOP/s where
//    32x32x16 ones do 1530 (a third less accumulator traffic per flop); at zeros, which cost no power, both do 2260;
//  * the states go from global memory straight to LDS, A_AHEAD steps ahead (six stages), which leaves the registers alone;
//  * decodes of 17 (int4, int2) and 24 (int3) instructions per chunk through the 8-bit float conversion and v_perm tables;
//  * scales and zeros are asked for once per pair of steps, int4's words of two columns in one load;
//  * the two halves of the workgroup run a step in opposite phases (PING): a SIMD holds a wave of each, one on the matrix
//    pipe, its decode in the shadow of its MFMAs, while the other does everything that touches the LDS or memory.  A wave's own
//    LDS stores between its MFMAs would hold these up (40 cycles each, on a step of 1024), and just before the barrier the
//    barrier; so what phase 1 stores at a step's start was decoded in the step before.  (1330 cycles a step with the
//    stores between the MFMAs, 1200 with those of the decode at its end, 1050 so, in a loop without global loads.)
// A tile of int4 or 16:32 that contains exponent-mode groups takes a second copy of the loop whose decode serves either mode;
// int2 and int3 have one decode for both.
//
// Measured, before (32x32x16 MFMAs, states through registers, magic-number decodes) / so, us: K=5120, S=20480, 2048 rows int4 398 /
// 346, int3 402 / 359, int2 394 / 337, 16:32 437 / 400, one group in 40 in exponent mode 464 / 369, int3 468 / 359; K=8192,
// S=28672, 4096 rows 1663 / 1430 (1.35 PFLOP/s); with the plan of the tiles below K=S=8192, 768 rows 146 / 107; K=20480, S=5120, 1024
// rows 265 / 206.
constexpr int PK = 32;            // K per step of the pipelined kernel

// 16:32 sparse int4.  `v` holds the (up to 8) kept codes of one 8-row chunk as
// consecutive nibbles, `m8` the chunk's mask bits.  A 256-entry table in LDS
// (8 words per mask byte: four words of per-half keep masks, two v_perm
// selectors) spreads the kept codes to their rows: the even / odd nibbles are
// separated into bytes, v_perm picks for every row the byte of its rank.  Dropped rows
// are cleared at the end, so they are exactly zero.
constexpr int SPARSE_LUT_WORDS = 256 * 8;

__device__ __forceinline__ void sparse_lut_entry(uint32_t e, uint32_t out[8]) {
    uint32_t sel[2] = {0, 0}, hm[4] = {0, 0, 0, 0};
    uint32_t rank = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const bool kept = (e >> i) & 1u;
        const uint32_t byte = kept ? ((rank & 1u) ? 4u + (rank >> 1) : (rank >> 1)) : 0x0Cu;
        sel[i >> 2] |= byte << (8 * (i & 3));
        if (kept) { hm[i >> 1] |= 0xFFFFu << (16 * (i & 1)); ++rank; }
    }
    out[0] = hm[0]; out[1] = hm[1]; out[2] = hm[2]; out[3] = hm[3];
    out[4] = sel[0]; out[5] = sel[1]; out[6] = 0; out[7] = 0;
}

template <class C>
__device__ __forceinline__ h16x8 dequant_chunk_sparse(uint32_t v, uint32_t m8, const uint32_t* lut, const C& c) {
    const u32x4 keep = *reinterpret_cast<const u32x4*>(lut + m8 * 8);
    const u32x2 sel = *reinterpret_cast<const u32x2*>(lut + m8 * 8 + 4);
    const uint32_t even = v & 0x0F0F0F0Fu, odd = (v >> 4) & 0x0F0F0F0Fu;
    const u32x4 r = bitcast<u32x4>(weights_of_bytes(__builtin_amdgcn_perm(odd, even, sel.x), __builtin_amdgcn_perm(odd, even, sel.y), c));
    return bitcast<h16x8>(r & keep);             // (dropped rows -> +0)
}

// Per-format constants of the pipelined kernel: packed rows per 32-row block and
// the number of packed words a thread loads per K step for its two chunks.
template <int BITS, bool SPARSE> struct PipeFmt;
template <> struct PipeFmt<4, false> { static constexpr int ROWS = 4, NWORDS = 2; };
template <> struct PipeFmt<3, false> { static constexpr int ROWS = 3, NWORDS = 2; };
template <> struct PipeFmt<2, false> { static constexpr int ROWS = 2, NWORDS = 1; };
template <> struct PipeFmt<4, true> { static constexpr int ROWS = 2, NWORDS = 2; };

constexpr int P_STAGES = 3, A_STAGES = 6;  // of the weights, of the states
constexpr int A_AHEAD = 5;                 // steps that the states are ahead
// immediate of s_waitcnt: at most so many vector memory and LDS operations outstanding
constexpr int wait_counts(int vm, int lgkm) { return (vm & 15) | 0x70 | lgkm << 8 | (vm >> 4) << 14; }

// Swizzle of the states stage: row m's 16-byte chunk c stands at c ^ pipe_swz(m).  A 16-byte LDS read is served in
// groups of lanes 0-3, 12-15, 20-27 and 4-11, 16-19, 28-31 (of each half wave); with lane = row + 16 chunk each group then
// touches all 64 banks once (247 bytes a cycle and CU; with (m >> 2) & 3, which suits 32 rows x 2 chunks, 127).
__device__ __forceinline__ int pipe_swz(int m) { return ((m >> 3) & 1) | (((m >> 1 ^ m >> 2) & 2)); }

// PING: the waves of the first half run phase 0, MFMAs first and then everything else; those of the second half phase 1,
// everything else first and the MFMAs last.  Without it all waves run phase 1.
template <int BITS, bool SPARSE, int TM, int NW, bool PING, bool SPLIT>
__device__ __forceinline__ void pipe_tile(const MatmulArgs& a, const int m0, const int s0, const h16* x,
                                          h16* outs, h16* const (&As)[A_STAGES], h16* Bs, uint32_t* lut, const int tile, const int split,
                                          const int nsplit) {
    constexpr int BM = TM * 32, BN = NW * 64, WM = TM * 16, WN = 64, TN = 4, T = 2 * NW * 64;
    constexpr int A_ROWS = T / 4;                                  // rows covered by one 16-byte load per thread
    constexpr int A_LOADS = (BM + A_ROWS - 1) / A_ROWS;            // such loads per thread and step (192 rows: the second half full)
    constexpr int B_STAGE = PK * BN;                               // halves per stage

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm0 = (wave / NW) * WM, wn0 = (wave % NW) * WN;

    // states stage: row m at m * 64 bytes, 16-byte chunk c of the row at c ^ pipe_swz(m).  Thread t fills position t % 4 of rows
    // t / 4 + A_ROWS * i (rows >= M re-read row M - 1 and are dropped at the store), from global memory straight to LDS.
    const int a_row = t >> 2, a_chunk = (t & 3) ^ pipe_swz(a_row);            // (rows + A_ROWS: same swizzle)
    // every global address is a buffer resource (the tile's rows of states; the whole
    // of the packed matrix, mask, scales, zeros) plus a per-lane 32-bit byte offset that
    // never changes plus a workgroup-uniform 32-bit offset that moves with the K step:
    // buffer loads add the three themselves, no address arithmetic is left to the VALU
    // (the launcher admits only shapes whose tensors stay below 2 GB: pipe_shape)
    constexpr int RSRC_FLAGS = 0x00020000;               // raw buffer, 32-bit data format
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(x + (int64_t)m0 * a.K), 0, min(a.M - m0, BM) * a.K * 2, RSRC_FLAGS);
    uint32_t a_off[A_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i)
        a_off[i] = (uint32_t)((min(a_row + A_ROWS * i, min(a.M - m0, BM) - 1) * a.K + a_chunk * 8) * 2);
    auto dma_a = [&](int stage, uint32_t step_off) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (__attribute__((address_space(3))) void*)&As[stage][i * A_ROWS * PK + wave * 512], 16,
                                                     a_off[i], step_off, 0, 0);
    };

    // weights: a thread decodes two chunks of 8 rows of every K step.
    // int4: word `row` of two adjacent columns, one 8-byte load; the others: column bn, rows 16 bhb .. 16 bhb + 15 of the
    // step's 32-row block: int2 word bhb; int3 words bhb, bhb + 1 (bits 48 bhb .. 48 bhb + 47 of the block's 96-bit stream); 16:32
    // sparse: both words and the mask word of the block.
    // Column 4 n + j of a wave's 64 stands at position 16 j + (n ^ 4 (j / 2)) of its row of chunks: an MFMA tile takes every fourth
    // column, so that the four tiles leave a lane with four adjacent columns of a row, an 8-byte store.  The fragment reads, 256 bytes
    // a cycle, and the stores of either mapping, 128 bytes of eight lanes a cycle, touch every bank once (with n ^ 8 the stores of
    // int4 met twice on every second one: 16 conflict cycles per wave and step).
    // (a last tile that is not full: the columns beyond the last repeat the last 64 and are not written)
    using F = PipeFmt<BITS, SPARSE>;
    constexpr int NWORDS = F::NWORDS;
    constexpr bool PAIR = BITS == 4 && !SPARSE;
    constexpr int W_LOADS = PAIR ? 1 : NWORDS + (SPARSE ? 1 : 0);
    const int bn = PAIR ? t % (BN / 2) * 2 : t % BN, bhb = PAIR ? t / (BN / 2) : t / BN;
    const int bcol = min(s0 + (bn & ~63), a.S - 64) + (PAIR ? bn & 63 : 4 * ((bn & 15) ^ (bn >> 3 & 4)) + (bn >> 4 & 3));
    int b_chunk[2];                                      // where the two chunks go (halves)
#pragma unroll
    for (int q = 0; q < 2; ++q)
        b_chunk[q] = 8 * (PAIR ? bhb * BN + (bn & ~63) + 16 * ((bn & 2) + q) + ((bn >> 2 & 15) ^ (bn << 1 & 4)) : (bhb * 2 + q) * BN + bn);
    struct Stage { uint32_t w[NWORDS]; uint32_t m; };
    // scale / zero travel as the aligned 32-bit word that holds the column's half
    // (sub-dword loads make the compiler wait for every outstanding load); `half_sel`
    // replicates the wanted half into both lanes of a packed register
    const uint32_t half_sel = (bcol & 1) ? 0x03020302u : 0x01000100u;
    uint32_t b_off[W_LOADS];
#pragma unroll
    for (int i = 0; i < (PAIR ? 1 : NWORDS); ++i)
        b_off[i] = (uint32_t)((((SPARSE ? 0 : bhb) + i) * a.S + bcol) * 4);
    const uint32_t m_off = (uint32_t)(bcol * 4);
    const uint32_t m_step = 4u * a.S;                    // bytes of one row of mask words
    const uint32_t sz_off = (uint32_t)((bcol & ~1) * 2);
    const uint32_t b_step = (uint32_t)(F::ROWS * 4) * a.S;   // bytes of packed weights per K step
    const uint32_t g_step = 2u * a.S;                    // bytes of one row of scales / zeros
    const int k_blocks = a.K / PK, n_groups = (k_blocks + a.group_units * 2 - 1) / (a.group_units * 2);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(a.matrix), 0, (int)(k_blocks * b_step), RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t m_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(SPARSE ? a.mask : a.matrix), 0, (int)(k_blocks * m_step), RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t sc_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(a.scales), 0, (int)(n_groups * g_step), RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t ze_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(a.zeros), 0, (int)(n_groups * g_step), RSRC_FLAGS);
    // cursor over K steps: byte offsets of the step's packed-weight rows, mask row and scale / zero row
    struct Cursor { uint32_t w, m, sz; int kt, left; };
    auto cursor_at = [&](int kt) {
        const int gu = a.group_units * 2, group = kt / gu;
        return Cursor{kt * b_step, SPARSE ? kt * m_step : 0u, group * g_step, kt, gu - kt % gu};
    };
    // scale and zero of the thread's column: of the pair of steps that is decoded, and as loaded for the next one (a group is
    // whole pairs of steps, and a workgroup starts with one)
    uint32_t next_s, next_z;
    auto load_b = [&](Stage& s, const Cursor& c, bool first_of_pair) {
        if constexpr (PAIR) {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, b_off[0], c.w, 0);
            s.w[0] = v.x;
            s.w[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < NWORDS; ++i) s.w[i] = __builtin_amdgcn_raw_buffer_load_b32(w_rsrc, b_off[i], c.w, 0);
        }
        if constexpr (SPARSE) s.m = __builtin_amdgcn_raw_buffer_load_b32(m_rsrc, m_off, c.m, 0);
        if (first_of_pair) {
            next_s = __builtin_amdgcn_raw_buffer_load_b32(sc_rsrc, sz_off, c.sz, 0);
            next_z = __builtin_amdgcn_raw_buffer_load_b32(ze_rsrc, sz_off, c.sz, 0);
        }
    };
    auto take_sz = [&](auto (&co)[PAIR ? 2 : 1]) {
#pragma unroll
        for (int q = 0; q < (PAIR ? 2 : 1); ++q) {
            const uint32_t sel = !PAIR ? half_sel : q ? 0x03020302u : 0x01000100u;
            co[q].set(as_h2(__builtin_amdgcn_perm(next_s, next_s, sel)), as_h2(__builtin_amdgcn_perm(next_z, next_z, sel)));
        }
    };
    // the 8 codes of the thread's chunk q (rows 16 bhb + 8 q .. + 7), LSB first
    const int i3_shift = 16 * bhb;
    auto chunk_bits = [&](const Stage& s, int q) -> uint32_t {
        if constexpr (BITS == 4) return s.w[q];
        else if constexpr (BITS == 2) return q ? s.w[0] >> 16 : s.w[0];
        else return (uint32_t)((((uint64_t)s.w[1] << 32) | s.w[0]) >> (i3_shift + 24 * q));
    };
    // 16:32 sparse: mask bits of chunk q and its kept codes as consecutive nibbles.
    // The codes of rows before the chunk are skipped by a right shift of 4 bits
    // each (done in two halves: the total can reach 64).
    auto sparse_chunk = [&](const Stage& s, int q, uint32_t& v, uint32_t& m8) {
        const uint32_t m16 = (s.m >> (16 * bhb)) & 0xFFFFu;
        uint32_t skip = bhb ? __builtin_popcount(s.m & 0xFFFFu) : 0;
        if (q) skip += __builtin_popcount(m16 & 0xFFu);
        m8 = (m16 >> (8 * q)) & 0xFFu;
        const uint64_t st = ((uint64_t)s.w[1] << 32) | s.w[0];
        v = (uint32_t)((st >> (2 * skip)) >> (2 * skip));
    };
    auto decode = [&](const Stage& st, const auto (&co)[PAIR ? 2 : 1], h16x8 (&w)[2]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const auto& c = co[PAIR ? q : 0];
            if constexpr (SPARSE) {
                uint32_t v, m8;
                sparse_chunk(st, q, v, m8);
                w[q] = dequant_chunk_sparse(v, m8, lut, c);
            } else {
                w[q] = dequant_chunk<BITS>(chunk_bits(st, q), c);
            }
        }
    };
    auto write_b = [&](const h16x8 (&w)[2], int stage) {
#pragma unroll
        for (int q = 0; q < 2; ++q) *reinterpret_cast<h16x8*>(&Bs[stage * B_STAGE + b_chunk[q]]) = w[q];
    };
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // fragment addresses (halves, inside a stage); a step's 32 k are four chunks, one per lane group of 16
    // (row offsets are multiples of 16: the same swizzle for all of a lane's rows)
    const int a_frag = (wm0 + (lane & 15)) * PK + (((lane >> 4) ^ pipe_swz(lane)) << 3);
    const int b_frag[2] = {((lane >> 4) * BN + wn0 + (lane & 15)) * 8, ((lane >> 4) * BN + wn0 + ((lane & 15) ^ 4)) * 8};
    auto load_frags = [&](int a_stage, int stage, h16x8 fa[TM], h16x8 fb[TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            fa[i] = *reinterpret_cast<const h16x8*>(&As[a_stage][a_frag + i * 16 * PK]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            fb[j] = *reinterpret_cast<const h16x8*>(&Bs[stage * B_STAGE + b_frag[j >> 1] + j * 128]);
    };
    auto mfma_step = [&](const h16x8 fa[TM], const h16x8 fb[TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    };

    // K steps kt0 .. last of the matrix belong to this workgroup (all of them unless SPLIT)
    const int ksteps = a.K / PK;
    // (whole pairs of steps; a share has at least four)
    const int kt0 = SPLIT ? ksteps / 2 * split / nsplit * 2 : 0;
    const int ktiles = (SPLIT ? ksteps / 2 * (split + 1) / nsplit * 2 : ksteps) - kt0;
    const int last = kt0 + ktiles - 1;

    // Cursors of the loads: weights run four K steps ahead of the MFMAs, states
    // A_AHEAD; both stop at the last step (the surplus loads re-read it, unused).
    Cursor cur = cursor_at(kt0);
    // (selects instead of branches: a branch here would split the scheduling
    // region of the step and invite the compiler to reuse the previous step's
    // scale / zero registers, which makes the step wait for its newest loads)
    // (plain integer arithmetic on purpose: conditions kept as booleans come out as
    // 64-bit lane-mask operations, several scalar instructions each)
    const int gu2 = a.group_units * 2;
    auto advance = [&]() {
        const int more = min(last - cur.kt, 1);                  // 1 until the last step is reached
        const int wrap = cur.left == 1 ? more : 0;
        cur.kt += more;
        cur.w += more * b_step;
        if constexpr (SPARSE) cur.m += more * m_step;
        cur.sz += wrap * g_step;
        cur.left += wrap * gu2 - more;
    };
    uint32_t a_cur = (uint32_t)kt0 * (PK * 2);
    int a_kt = kt0;
    auto advance_a = [&]() {
        const int more = min(last - a_kt, 1);
        a_kt += more;
        a_cur += more * (PK * 2);
    };
    Stage r[3];
    // the first steps' operands are requested before the look at the scales below, whose
    // round trip to memory they then share
    load_b(r[0], cur, true); advance();
    load_b(r[1], cur, false); advance();
#pragma unroll
    for (int i = 0; i < A_AHEAD; ++i) { dma_a(i, a_cur); advance_a(); }

    // Does any (group, column) of this tile use exponent quantisation (scale < 0
    // or NaN)?  One pass over the tile's scales (a few KB); the answer is
    // workgroup-uniform and selects between the pipelined loop, whose decode is
    // the linear one, and the one that also serves exponent groups.  (int2 and int3 have one decode for both.)
    bool tile_has_expo = false;
    if constexpr (BITS == 4) {
        int& any_expo = *reinterpret_cast<int*>(Bs);          // borrowed before the pipeline starts
        __syncthreads();
        if constexpr (SPARSE) {
            if (t < 256) {
                uint32_t e[8];
                sparse_lut_entry(t, e);
                *reinterpret_cast<u32x4*>(lut + t * 8) = u32x4{e[0], e[1], e[2], e[3]};
                *reinterpret_cast<u32x4*>(lut + t * 8 + 4) = u32x4{e[4], e[5], e[6], e[7]};
            }
        }
        if (t == 0) any_expo = 0;
        __syncthreads();
        {
            // the tile's scales are `groups` rows of BN / 2 aligned 32-bit words; the threads share them
            // out and fetch four words each per trip, all in flight together (one round trip to
            // memory instead of one per group)
            bool bad = false;
            const int groups = (ksteps + a.group_units * 2 - 1) / (a.group_units * 2);
            const int total = groups * (BN / 2);
            const uint32_t* tile_scales = reinterpret_cast<const uint32_t*>(a.scales + s0);
            const int64_t row_words = a.S / 2;
            const int last_word = (a.S - s0) / 2 - 1;
            for (int i0 = t; i0 < total; i0 += 4 * T) {
                uint32_t v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int i = min(i0 + k * T, total - 1);
                    v[k] = tile_scales[(int64_t)(i / (BN / 2)) * row_words + min(i % (BN / 2), last_word)];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const h16x2 h = as_h2(v[k]);
                    bad |= !(h.x >= (h16)0.0f) | !(h.y >= (h16)0.0f);
                }
            }
            if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) any_expo = 1;
        }
        __syncthreads();
        tile_has_expo = any_expo != 0;
        __syncthreads();
    }

    // Step kt, u = kt % 6, weights' stage b = kt % 3, states' stage u.  On entry states and decoded weights of
    // steps kt and kt + 1 are complete.  The step stores the decoded weights of step kt + 2 and asks for the packed ones of
    // kt + 4 and the states of kt + A_AHEAD.  Phase 0:
    // MFMAs, on fragments fetched in the step before, beside the decode of step kt + 2's weights; then stores, loads, the next
    // step's fragments.  Phase 1: the step's own fragments, stores of what the step before decoded, loads; then MFMAs
    // beside the decode of step kt + 3's weights.
    h16x8 fa[TM], fb[TN], dec[2];
    auto walk = [&](auto mode) {
        Coef<BITS, decltype(mode)::value> co[PAIR ? 2 : 1];
        auto body = [&](auto phase_tag, int u, Stage& r_new, const Stage& r_dec) {
            constexpr int phase = decltype(phase_tag)::value;
            const int b = u % P_STAGES, b1 = (u + 1) % P_STAGES, b2 = (u + 2) % P_STAGES;
            auto stores_and_loads = [&]() {
                write_b(dec, b2);
                __builtin_amdgcn_sched_barrier(0);
                dma_a((u + A_AHEAD) % A_STAGES, a_cur);
                load_b(r_new, cur, u % 2 == 0);
                advance_a();
                advance();
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (phase == 1) {
                load_frags(u, b, fa, fb);
                __builtin_amdgcn_sched_barrier(0);
                stores_and_loads();
            }
            if ((u + phase) % 2 == 0) take_sz(co);
            decode(r_dec, co, dec);
            mfma_step(fa, fb);
            // (the decode in the shadow of the MFMAs: one occupies the pipe for 16 cycles, and up to two other vector instructions per
            // MFMA go beside it.  Spread over the last two thirds, so that the packed words need not have arrived yet: 261 us where
            // three behind each of the first MFMAs take 288, 16 tiles at K = 16384; at full load 2 - 3 %)
            constexpr int MFMAS = TM * TN, LATE = MFMAS / 3, DECODE = (SPARSE ? 64 : BITS == 3 ? 52 : 40) + (decltype(mode)::value ? 26 : 0);
#pragma unroll
            for (int e = 0; e < MFMAS; ++e) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                const int n = e < LATE ? 0 : (e - LATE + 1) * DECODE / (MFMAS - LATE) - (e - LATE) * DECODE / (MFMAS - LATE);
                if (n == 1) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                else if (n == 2) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                else if (n == 3) __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                else if (n == 4) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                else if (n > 4) __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (phase == 0) stores_and_loads();
            // the step's stores are complete (lgkmcnt(0)) and, of the loads, all but the last two steps'
            __builtin_amdgcn_s_waitcnt(wait_counts(2 * (A_LOADS + W_LOADS) + 2, 0));
            if constexpr (phase == 0) {
                load_frags((u + 1) % A_STAGES, b1, fa, fb);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        take_sz(co);
        decode(r[0], co, dec);
        write_b(dec, 0);
        decode(r[1], co, dec);
        write_b(dec, 1);
        __builtin_amdgcn_s_waitcnt(wait_counts(0, 15));         // steps 0 ... A_AHEAD - 1 of the states
        load_b(r[2], cur, true); advance();             // step 2
        load_b(r[0], cur, false); advance();            // step 3
        __syncthreads();
        // weight stages and registers rotate with period 3, the states' stages with 6: six steps per trip, unrolled so that
        // all of them are compile-time names
        auto run = [&](auto phase_tag) {
            constexpr int ahead = 2 + decltype(phase_tag)::value;
            for (int kt = 0; kt < ktiles; kt += 6) {
#pragma unroll
                for (int u = 0; u < 6; ++u) {
                    if (u > 0 && kt + u >= ktiles) break;
                    body(phase_tag, u, r[(u + 1) % 3], r[(u + ahead) % 3]);
                }
            }
        };
        if (PING && wave < NW) {
            load_frags(0, 0, fa, fb);
            if constexpr (PING) run(std::integral_constant<int, 0>{});
        } else {
            take_sz(co);
            decode(r[2], co, dec);
            run(std::integral_constant<int, 1>{});
        }
    };
    if (BITS == 4 && tile_has_expo) walk(std::bool_constant<BITS == 4>{});
    else walk(std::false_type{});
    // (no load to LDS is in flight any more when the LDS is used otherwise or given back)
    __builtin_amdgcn_s_waitcnt(wait_counts(0, 15));
    if (SPLIT && nsplit > 1) {
        // Every workgroup of the tile stores its partial accumulators (16 bytes per lane and
        // store: register group g of thread t at (g * T + t) * 16 -- whole cache lines per wave)
        // and then counts itself in; whoever finds all the others counted adds the partials up
        // in split order (its own included, from memory: the sum has one order whoever is
        // last) and writes the tile.  Stores and loads go straight through to memory
        // (system-scope cache policy), the counter is a device-scope atomic: no cache-wide
        // fence, no waiting.  (Two workgroups per tile: the last one adds the other's partial to
        // its own registers -- a sum of two terms has one value in either order.)
        constexpr int SLOT_BYTES = BM * BN * 4, THROUGH = 17;      // sc0 | sc1
        char* const slots = reinterpret_cast<char*>(a.part) + (int64_t)tile * nsplit * SLOT_BYTES;
        const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc(
            slots + (int64_t)split * SLOT_BYTES, 0, SLOT_BYTES, RSRC_FLAGS);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                __builtin_amdgcn_raw_buffer_store_b128(bitcast<u32x4>(acc[i][j]), mine, ((i * TN + j) * T + t) * 16, 0, THROUGH);
        __builtin_amdgcn_s_waitcnt(0);                 // every store of this thread has been acknowledged
        int* const flag = reinterpret_cast<int*>(Bs);
        __syncthreads();
        if (t == 0) *flag = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*flag != nsplit - 1) return;
        if (t == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // clean for the next call
        if (nsplit > 2) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int sp = nsplit > 2 ? 0 : 1 - split; sp < (nsplit > 2 ? nsplit : 2 - split); ++sp) {
            const __amdgpu_buffer_rsrc_t theirs = __builtin_amdgcn_make_buffer_rsrc(
                slots + (int64_t)sp * SLOT_BYTES, 0, SLOT_BYTES, RSRC_FLAGS);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] += bitcast<f32x4>(__builtin_amdgcn_raw_buffer_load_b128(theirs, ((i * TN + j) * T + t) * 16, 0, THROUGH));
        }
    }
    if (s0 + wn0 >= a.S) return;                       // (a wave's 64 columns are inside or outside as one)
    // register r of tile (i, j) is row 16 i + 4 (lane / 16) + r, column 4 (lane % 16) + j of the wave's
    h16* const out = outs + (int64_t)(m0 + wm0 + 4 * (lane >> 4)) * a.S + s0 + wn0 + 4 * (lane & 15);
    const int rows = a.M - (m0 + wm0 + 4 * (lane >> 4));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (16 * i + r < rows)
                *reinterpret_cast<h16x4*>(out + (int64_t)(16 * i + r) * a.S) =
                    h16x4{(h16)acc[i][0][r], (h16)acc[i][1][r], (h16)acc[i][2][r], (h16)acc[i][3][r]};
}

template <int BITS, bool SPARSE, int NW, int TM, bool PING, bool SPLIT>
__global__ __launch_bounds__(NW * 128, NW == 2 ? 2 : 1) void matmul_kernel_pipe(MatmulArgs a) {
    constexpr int BM = TM * 32, BN = NW * 64;
    constexpr int A_ROWS = NW * 32;
    // (each stage of the states an array of its own: in one array every fragment read would wait for all loads in flight)
    constexpr int A_HALVES = (BM + A_ROWS - 1) / A_ROWS * A_ROWS * PK;
    __shared__ __attribute__((aligned(16))) h16 A0[A_HALVES], A1[A_HALVES], A2[A_HALVES], A3[A_HALVES], A4[A_HALVES], A5[A_HALVES];
    __shared__ __attribute__((aligned(16))) h16 Bs[P_STAGES * PK * BN];
    __shared__ __attribute__((aligned(16))) uint32_t Lut[SPARSE ? SPARSE_LUT_WORDS : 4];
    // (split-K: the workgroups of a tile are neighbours in the grid, so they run at about the same time;
    // the tiles before `split_from` are whole)
    const int total = a.tiles_m * a.tiles_n;
    int bid = blockIdx.x, split = 0, nsplit = 1, slot = 0;
    if constexpr (SPLIT) {
        const int v = (int)blockIdx.x - a.split_from;
        if (v >= 0) {
            bid = a.split_from + v / a.ksplit;
            split = v % a.ksplit;
            nsplit = a.ksplit;
            slot = (int)blockIdx.z * (total - a.split_from) + v / a.ksplit;       // counter and partial tiles
        }
    }
    int tile_m, tile_n;
    if (total % 8 == 0) {
        // XCD-aware numbering: workgroups are dealt round-robin to the 8 XCDs (each
        // with its own L2), so XCD x takes the contiguous range x * total / 8 ... of tiles
        const int per_xcd = total / 8, l = bid / 8;
        if (a.by_columns) {
            // ... walked one tile row at a time across the XCD's tile columns: the tiles in
            // flight on an XCD then share few rows of states, whose 64 bytes per row and K
            // step outweigh the packed weights' 16 bytes per column (measured: 1-5 % faster
            // than column by column)
            const int cols = per_xcd / a.tiles_m;
            tile_m = l / cols;
            tile_n = (bid % 8) * cols + l % cols;
        } else {
            bid = (bid % 8) * per_xcd + l;
            tile_m = bid % a.tiles_m, tile_n = bid / a.tiles_m;
        }
    } else {
        tile_m = bid % a.tiles_m, tile_n = bid / a.tiles_m;
    }
    const int64_t boff = blockIdx.z;
    h16* const As[A_STAGES] = {A0, A1, A2, A3, A4, A5};
    pipe_tile<BITS, SPARSE, TM, NW, PING, SPLIT>(a, tile_m * BM, tile_n * BN, a.x + boff * a.M * (int64_t)a.K,
                                          a.outs + boff * a.M * (int64_t)a.S, As, Bs, Lut, slot, split, nsplit);
}

template <int BITS, bool SPARSE, int NW, int TM = 8, bool PING = false>
static void launch_pipe(MatmulArgs a, int64_t B, hipStream_t st) {
    a.tiles_m = (a.M + TM * 32 - 1) / (TM * 32);
    a.tiles_n = (a.S + NW * 64 - 1) / (NW * 64);
    const int total = a.tiles_m * a.tiles_n;
    const dim3 grid(a.split_from + (total - a.split_from) * a.ksplit, 1, (unsigned)B), block(NW * 128);
    a.by_columns = a.tiles_n % 8 == 0;
    if (noting("matmul_kernel_pipe<bits=%d,%s,tile=%dx%d,%s> tiles=%d ksplit=%d split_from=%d workgroups=%u batch=%d", BITS,
               SPARSE ? "16:32" : "dense", TM * 32, NW * 64, PING ? "two-phase" : "plain", total, a.ksplit, a.split_from, grid.x, (int)B))
        return;
    if (a.ksplit > 1) hipLaunchKernelGGL((matmul_kernel_pipe<BITS, SPARSE, NW, TM, PING, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((matmul_kernel_pipe<BITS, SPARSE, NW, TM, PING, false>), grid, block, 0, st, a);
}

// The pipelined kernel takes any whole number of 64 columns; the last tile may be partly empty, up to half of the
// columns in all (128-column tiles: an eighth).  Before, such outputs went to the general tiles, which hide
// less of their loads and cannot split K (us, general / here: int4, K=9280, S=1600, 700 rows 135 / 54, S=14400, 1100 rows 422 /
// 351; int2 there 239 / 54 and 699 / 341; 16:32 280 / 73 and 846 / 385; int4, K=9280, S=9344 -- 256 x 128 tiles before --
// 1100 rows 280 / 214).
static bool tile_columns(int64_t S, int width, bool half) {
    return S % 64 == 0 && (S + width - 1) / width * width * 8 <= S * (half ? 12 : 9);
}

constexpr int64_t MM_SPLIT_MAX_TILES = 1024;             // counters: one int per tile in 4 KB
constexpr int64_t MM_SPLIT_MAX_BYTES = 192ll << 20;      // cap of the partial tiles

// ---- plan of the tiles.  Heights of 128 ... 256 rows in steps of 32, all 256 columns wide, one workgroup per CU, each K split
// `ksplit` ways or not, or only the tiles of a last, partly filled round (from `split_from` on): the candidate that a cost model
// finds cheapest, in us,
//     rounds of 256 workgroups, each  steps x step(height) x (1 + fill x share of the CUs^3) + fixed(height)      (*)
//     + (split: (way x ways + hand x share of the CUs) x height / 256)
// the last of several rounds with its share of the CUs raised towards 1 by `last`, full ones times `round`.  (*) is the power limit:
// a GPU filled to the last CU runs its K steps 40 % slower than an almost empty one.  Fitted per format to 870 ... 2050 timed
// launches (K = 1024 ... 28672, S = 1024 ... 28672, 257 ... 4096 rows); on these shapes its pick is 1.0 - 1.2 % off the best
// candidate on average, 9 - 16 % at worst.  Before, a tree of rules chose among 128, 192 and 256 rows and 256 x 128 tiles, of which
// the last are the best candidate on none of 210 shapes: above 512 rows this plan takes 10 % (int4), 15 % (int3), 14 % (int2) and
// 11 % (16:32) less time on average, at most 3 % more on a shape (us: int4, K=16128, S=3072, 1411 rows 217 / 151; K=9216, S=2304, 1151
// rows 98 / 70; int3, K=28096, S=2176, 880 rows 201 / 134; K=S=4096, 777 rows on S=11008 77 / 72).  Preferences on top of the model -- whole
// 256-row tiles, 16:32 split in 256 rows and never in 224 -- were made for single shapes and cost 2 % (90 random products of multiples
// of 256 rows; int4, K=20480, S=5120, 2048 rows 420 / 373) and 4 % (121 of 16:32; K=4096, S=8192, 896 rows 79.5 / 74.9).
struct TileCost { double step[5], fixed[5], fill, way, hand, round, last; };
static const TileCost tile_cost[4] = {                // int4, int3, int2, 16:32
    {{0.373, 0.434, 0.466, 0.521, 0.555}, {4.151, 4.233, 4.77, 4.391, 5.388}, 0.369, 2.82, 19.858, 1.065, 0.292},
    {{0.405, 0.462, 0.493, 0.536, 0.58}, {3.632, 4.086, 3.915, 4.283, 5.317}, 0.406, 2.965, 19.124, 1.027, 0.321},
    {{0.376, 0.423, 0.463, 0.515, 0.544}, {2.878, 3.789, 3.887, 3.45, 5.247}, 0.344, 2.974, 18.171, 1.042, 0.363},
    {{0.59, 0.659, 0.686, 0.759, 0.817}, {5.287, 5.577, 5.793, 5.759, 6.161}, 0.131, 3.381, 18.391, 1.061, 0.347}};
struct TilePlan { int tm; int ksplit; int64_t split_from, tiles; size_t part_bytes; double us; };
// `only`: this height alone (0: any); `scratch`: bytes for partial tiles, splits that need more are no candidates
static TilePlan plan_tiles(int bits, bool sparse, int64_t M, int64_t K, int64_t S, size_t scratch, int only) {
    TilePlan best{0, 1, 0, 0, 0, 1e30};
    const TileCost& c = tile_cost[sparse ? 3 : 4 - bits];
    const int64_t columns = (S + 255) / 256, steps = K / 32, forced = tuning(TUNE_MM_SPLIT), tail_knob = tuning(TUNE_MM_TAIL);
    const int64_t room = (int64_t)std::min<size_t>(scratch, MM_SPLIT_MAX_BYTES);
    for (int tm = 4; tm <= 8; ++tm) {
        if (only != 0 && tm != only) continue;
        const int64_t total = (M + 32 * tm - 1) / (32 * tm) * columns, tile_bytes = 32 * 256 * 4 * (int64_t)tm;
        const double share = tm / 8.0;
        auto one = [&](double n, double fill) { return n * c.step[tm - 4] * (1.0 + c.fill * fill * fill * fill) + c.fixed[tm - 4]; };
        auto take = [&](double us, int64_t ks, int64_t from) {
            if (us < best.us) best = TilePlan{tm, (int)ks, from, total, ks > 1 ? (size_t)((total - from) * ks * tile_bytes) : 0, us};
        };
        for (int64_t ks = 1; ks <= 8; ++ks) {
            if (ks > 1 && (steps / ks < 8 || total > MM_SPLIT_MAX_TILES || total * ks * tile_bytes > room || forced == 1)) break;
            const int64_t wgs = total * ks, rounds = (wgs + 255) / 256;
            const double n = (double)steps / ks, last = (wgs - (rounds - 1) * 256) / 256.0;
            double us = (rounds - 1) * c.round * one(n, 1.0) + one(n, rounds > 1 ? last + (1.0 - last) * c.last : last);
            if (ks > 1) us += (c.way * ks + c.hand * (rounds - 1 + last)) * share;
            take(forced >= 2 && ks == forced ? 0.0 : us, ks, 0);
        }
        // the tiles of the last round alone, over at most half of the GPU (two ways from 64 tiles on, where the second adds the first
        // one's partial tile to its registers and nothing else is read back) in shares of at least 32 steps (K=4096, S=8192, 2304 rows,
        // 32 tiles in the tail: eight ways 197 us, four ways 170)
        const int64_t tail = total % 256;
        if (tm != 8 || total <= 256 || tail == 0 || tail > 128 || tail_knob == 1 || (tail > 96 && K < 3072)) continue;
        const int64_t ks = std::min<int64_t>({std::max<int64_t>(2, 128 / tail), tail_knob >= 2 ? tail_knob : 8, steps / 32});
        if (ks < 2 || tail * ks * tile_bytes > room) continue;
        const double fill = tail * ks / 256.0;
        const double us = total / 256 * c.round * one(steps, 1.0) + one((double)steps / ks, fill + (1.0 - fill) * c.last) + (c.way * ks + c.hand * fill) * share;
        // (preferred within 5 %: the model has few of these to go by)
        take(us / 1.05, ks, total - tail);
    }
    best.us += 2.0;
    return best;
}

// ---- what earlier forms of the tile kernels split along K.  It decides still which workspaces the last chunk of a large batch is taken
// to have (last_chunk_as_others, a line of precision), and nothing else.  Shapes with at most 128 tiles of 256 x 256: 256 x 128 tiles
// (16:32: 256 x 256) with `ksplit` workgroups per tile, by a cost in K steps.
struct SplitPlan { int ksplit; int64_t tiles; int64_t tile_bytes; };
static SplitPlan plan_split(bool sparse, int64_t B, int64_t M, int64_t K, int64_t S) {
    const SplitPlan none{1, 0, 0};
    if (!tile_columns(S, sparse ? 256 : 128, sparse)) return none;
    const int64_t m_pad = (M + 255) / 256 * 256, tiles4 = m_pad / 256 * ((S + 255) / 256) * B;
    if (tiles4 > 128) return none;
    SplitPlan p{1, m_pad / 256 * ((S + (sparse ? 255 : 127)) / (sparse ? 256 : 128)) * B, sparse ? 256 * 256 * 4 : 256 * 128 * 4};
    if (p.tiles > MM_SPLIT_MAX_TILES) return none;
    const int64_t steps = K / 32, forced = tuning(TUNE_MM_SPLIT);
    auto cost = [&](int64_t ks) -> double {
        const int64_t wgs = p.tiles * ks, rounds = (wgs + 255) / 256;
        const double own = (double)(rounds * ((steps + ks - 1) / ks + 20));
        if (!sparse) return own + (ks > 1 ? 6.0 * ks : 0.0);
        const double fill = wgs >= 256 ? 1.0 : wgs / 256.0;
        return own * (1.0 + 0.39 * std::pow(fill, 3.2)) + (ks > 1 ? 5.0 * ks : 0.0);
    };
    int64_t best = 1;
    for (int64_t ks = 2; ks <= 8; ++ks) {
        if (steps / ks < 8 || p.tiles * ks * p.tile_bytes > MM_SPLIT_MAX_BYTES) break;
        if (forced == ks) { best = ks; break; }
        if (forced == 0 && cost(ks) < cost(best)) best = ks;
    }
    if (best < 2) return none;
    p.ksplit = (int)best;
    return p;
}

// and the tiles of a last round of 256 x 256 ones that fills at most half of the GPU
struct TailPlan { int ksplit; int64_t split_from, tiles; };
static TailPlan plan_tail(bool sparse, int64_t B, int64_t M, int64_t K, int64_t S) {
    const TailPlan none{1, 0, 0};
    if (B != 1 || !tile_columns(S, 256, sparse) || tuning(TUNE_MM_TAIL) == 1) return none;
    const int64_t total = (M + 255) / 256 * ((S + 255) / 256), tail = total % 256;
    if (total <= 256 || tail == 0 || tail > 128) return none;
    if (tail > 96 && K < 3072) return none;
    const int64_t cap = tuning(TUNE_MM_TAIL) >= 2 ? tuning(TUNE_MM_TAIL) : 8;
    const int64_t ks = std::min<int64_t>({std::max<int64_t>(2, 128 / tail), cap, K / 32 / 32});
    if (ks < 2 || tail * ks * (256 * 256 * 4) > MM_SPLIT_MAX_BYTES) return none;
    return TailPlan{(int)ks, total - tail, tail};
}

template <int BITS, bool SPARSE, int BM, int BN, int WM, int WN>
static void launch_tile(MatmulArgs a, int64_t B, hipStream_t st) {
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = (a.S + BN - 1) / BN;
    const dim3 grid(a.tiles_m * a.tiles_n, 1, (unsigned)B), block((BM / WM) * (BN / WN) * 64);
    if (noting("matmul_kernel<bits=%d,%s,tile=%dx%d> tiles=%u batch=%d", BITS, SPARSE ? "16:32" : "dense", BM, BN, grid.x, (int)B)) return;
    hipLaunchKernelGGL((matmul_kernel<BITS, SPARSE, BM, BN, WM, WN>), grid, block, 0, st, a);
}

// (the kernel addresses with 32-bit byte offsets into buffer resources: 256 rows of states,
// the whole packed matrix and the whole of scales / zeros have to stay below 2 GB each)
static bool pipe_shape(int bits, bool sparse, int64_t K, int64_t S, int64_t group_units) {
    const int64_t w_bytes = K / 32 * (sparse ? 2 : bits) * 4 * S, sz_bytes = (K / 64 + group_units - 1) / group_units * S * 2;
    return K <= (1 << 22) && S <= (1 << 27) && w_bytes < (1ll << 31) && sz_bytes < (1ll << 31);
}
// (a short K on a small dense grid: the pipelined kernel's prologue costs more than its faster steps return: 2048 rows,
// K=S=128 8.7 -> 5.3 us; 512 rows, K=512, S=1024 14.6 -> 10.7; from K = 1024 on there is nothing in it)
static bool takes_tiles(int bits, bool sparse, int64_t M, int64_t K, int64_t S, int64_t group_units) {
    return pipe_shape(bits, sparse, K, S, group_units) && tile_columns(S, 256, true) &&
           (sparse || K >= 1024 || (M + 255) / 256 * ((S + 255) / 256) > 128);
}

// ---- outputs of 128 columns, of which a tile of 256 would leave half empty: tiles of 128 x 128, two workgroups of four waves per CU, in the
// two phases as well.  On many rows the states' reads are the bound, 5.1 TB/s at 65536 rows.  K is split as many ways as fit 256 workgroups, in
// shares of 16 steps and more (int4, us: K=8192, 128 tiles 95 unsplit, two ways 69, three 73, four 75; 80 tiles three ways 38, four
// 44), or 512 where these are filled better (160 tiles, K=4096: one way 44, three 41; 96 tiles, K=16384: two ways 134, five 110) or the
// states are more than the 256 MB of the cache beside memory (110 tiles, K=28672: two ways 217, four 195).  Before, 256 x 128 tiles with
// the states through registers, whose decode spilled (int4, us, so / now: K=8192, 2048 rows 41.4 / 23.7, without room for a split 146 /
// 76, 65536 rows 249 / 211; K=4096, 600 rows 31.5 / 17.0; with 32x32x16 MFMAs and no spill 39.7, 126, 233, 30.4).
static bool takes_narrow_tiles(int bits, bool sparse, int64_t M, int64_t K, int64_t S, int64_t group_units) {
    const int64_t variant = tuning(TUNE_MM_VARIANT);
    return !sparse && M > 128 && pipe_shape(bits, sparse, K, S, group_units) && tile_columns(S, 128, false) &&
           (variant == 5 || (variant == 0 && K > 1024 && !tile_columns(S, 256, true)));
}
struct NarrowPlan { int ksplit; size_t part_bytes; };
static NarrowPlan plan_narrow(int64_t M, int64_t K, int64_t S, size_t scratch) {
    const int64_t tiles = (M + 127) / 128 * ((S + 127) / 128), steps = K / 32, forced = tuning(TUNE_MM_SPLIT), tile_bytes = 128 * 128 * 4;
    const int64_t room = (int64_t)std::min<size_t>(scratch, MM_SPLIT_MAX_BYTES);
    auto ways = [&](int64_t workgroups) { return std::max<int64_t>(1, std::min<int64_t>({8, workgroups / tiles, steps / 16})); };
    int64_t ks = forced >= 1 ? std::min(forced, steps / 8) : ways(256);
    if (forced < 1 && (ways(512) * 10 > ks * 22 || M * K * 2 > 256ll << 20)) ks = ways(512);
    if (tiles > MM_SPLIT_MAX_TILES) ks = 1;
    while (ks > 1 && tiles * ks * tile_bytes > room) --ks;
    return ks > 1 ? NarrowPlan{(int)ks, (size_t)(tiles * ks * tile_bytes)} : NarrowPlan{1, 0};
}

double tiles_us(int bits, bool sparse, int64_t M, int64_t K, int64_t S, int64_t group_units, size_t scratch) {
    return takes_tiles(bits, sparse, M, K, S, group_units) ? plan_tiles(bits, sparse, M, K, S, scratch, 0).us : 1e30;
}

// height of a forced variant's tiles, in 32 rows (0: none)
static int forced_height(int64_t variant) {
    static const int heights[12] = {0, 0, 0, 0, 0, 0, 8, 4, 6, 8, 5, 7};
    return variant >= 0 && variant < 12 ? heights[variant] : 0;
}

template <int BITS, bool SPARSE>
static void launch(MatmulArgs a, int64_t B, hipStream_t st, void* workspace, size_t workspace_bytes) {
    // variant 0 = automatic: the plan of the pipelined kernel's tiles; where that kernel does not take the shape its 128 x 128 tiles
    // or the general ones, 128 x 256, and 128 x 128 for narrow outputs or few rows
    const int variant = (int)tuning(TUNE_MM_VARIANT);
    const WorkspaceParts wsp = workspace_parts(workspace, workspace_bytes);
    // (a single row comes here where its matvec has a group longer than a launch covers: the size query asks nothing for it)
    const size_t scratch = wsp.counters != nullptr && B == 1 && (a.M > 1 || variant != 0) ? wsp.scratch_bytes : 0;
    a.counters = reinterpret_cast<int*>(wsp.counters);
    a.part = reinterpret_cast<float*>(wsp.scratch);
    const bool shape_ok = pipe_shape(BITS, SPARSE, a.K, a.S, a.group_units);
    const bool narrow = B == 1 && takes_narrow_tiles(BITS, SPARSE, a.M, a.K, a.S, a.group_units);
    const int only = forced_height(variant);
    const bool tiles = !narrow && (variant == 0 ? takes_tiles(BITS, SPARSE, a.M, a.K, a.S, a.group_units) : only != 0 && shape_ok && tile_columns(a.S, 256, true));
    if (narrow) {
        a.ksplit = plan_narrow(a.M, a.K, a.S, scratch).ksplit;
        if constexpr (!SPARSE) launch_pipe<BITS, false, 2, 4, true>(a, B, st);
    } else if (tiles) {
        const TilePlan p = plan_tiles(BITS, SPARSE, a.M, a.K, a.S, scratch, only);
        a.ksplit = p.ksplit;
        a.split_from = (int)p.split_from;
        // (variant 9 forces 256 x 256 without the two phases: 9 % slower, 16:32 4 %)
        if (variant == 9) launch_pipe<BITS, SPARSE, 4>(a, B, st);
        else if (p.tm == 4) launch_pipe<BITS, SPARSE, 4, 4, true>(a, B, st);
        else if (p.tm == 5) launch_pipe<BITS, SPARSE, 4, 5, true>(a, B, st);
        else if (p.tm == 6) launch_pipe<BITS, SPARSE, 4, 6, true>(a, B, st);
        else if (p.tm == 7) launch_pipe<BITS, SPARSE, 4, 7, true>(a, B, st);
        else launch_pipe<BITS, SPARSE, 4, 8, true>(a, B, st);
    } else if (variant == 3 || (variant != 1 && a.M > 512 && a.S >= 256 && !(!SPARSE && a.K <= 1024))) {
        launch_tile<BITS, SPARSE, 128, 256, 128, 64>(a, B, st);
    } else {
        launch_tile<BITS, SPARSE, 128, 128, 64, 64>(a, B, st);
    }
}

}  // namespace i4

using namespace i4;

extern "C" int int4mm_matmul(int bits, void* outs, const void* matrix, const void* multiplier,
                             const void* scales, const void* zeros, const void* sparse_mask,
                             const int4mm_shape* shape, void* workspace, size_t workspace_bytes,
                             void* stream) {
    int rc = validate_product(bits, outs, matrix, multiplier, scales, zeros, sparse_mask, shape, false);
    if (rc != INT4MM_OK) return rc;
    int64_t B = shape->batch, M = shape->seq_len;
    const int64_t K = shape->in_size, S = shape->out_size;
    if (B * M * S == 0) return INT4MM_OK;
    // Batches are contiguous ([B, M, K] states, [B, M, S] outputs) and every kernel's rows are independent: B
    // products of M rows are one product of B * M rows -- whole tiles instead of B padded ones (K=5120, S=20480: 32
    // batch elements of 20 rows 970 -> 152 us, 5 of 130 rows 258 -> 153).
    if (B > 1 && B * M <= ((int64_t)1 << 31) - 256) { M *= B; B = 1; }
    if (((M + 127) / 128) * ((S + 127) / 128) > 0x7FFFFFFF / 2) return INT4MM_ERR_SHAPE;
    const int64_t g = shape->group_size < 0 ? ONE_GROUP : shape->group_size;

    hipStream_t st = (hipStream_t)stream;
    // 2 .. 96 rows in all (batches are contiguous, so they flatten; on suitable shapes up to 512): the few-row
    // kernels, which read every packed word once for all rows -- unless a tile-kernel variant is forced
    if (B * M == 1 && !tuning(TUNE_NO_SKINNY) && !tuning(TUNE_MM_VARIANT) &&
        matvec_one_row(bits, (h16*)outs, (const uint32_t*)matrix, (const uint32_t*)sparse_mask, (const h16*)multiplier,
                       (const h16*)scales, (const h16*)zeros, K, S, g, st, workspace, workspace_bytes, &rc))
        return rc;
    if (B * M >= 2 && B * M <= 4 && !sparse_mask && !tuning(TUNE_NO_SKINNY) && !tuning(TUNE_MM_VARIANT) &&
        matvec_rows(bits, (h16*)outs, (const uint32_t*)matrix, (const h16*)multiplier, (const h16*)scales, (const h16*)zeros,
                    B * M, K, S, g, false, st, workspace, workspace_bytes))
        return check_launch("matmul");
    if (B * M >= 2 && B * M <= SK_WIDE_MAX_ROWS && !tuning(TUNE_NO_SKINNY) && !tuning(TUNE_MM_VARIANT) &&
        skinny_rows(bits, (h16*)outs, (const uint32_t*)matrix, (const h16*)multiplier, (const h16*)scales,
                    (const h16*)zeros, B * M, K, S, g, false, st, (const uint32_t*)sparse_mask, workspace, workspace_bytes, FOR_MATMUL))
        return check_launch("matmul");

    MatmulArgs a;
    a.outs = (h16*)outs;
    a.matrix = (const uint32_t*)matrix;
    a.mask = (const uint32_t*)sparse_mask;
    a.x = (const h16*)multiplier;
    a.scales = (const h16*)scales;
    a.zeros = (const h16*)zeros;
    a.M = (int)M;
    a.K = (int)K;
    a.S = (int)S;
    a.group_units = (int)(g / 64 > 0x7FFFFFF ? 0x7FFFFFF : g / 64);
    a.tiles_m = a.tiles_n = 0;
    a.by_columns = 0;
    a.ksplit = 1;
    a.split_from = 0;
    a.part = nullptr;
    a.counters = nullptr;

    if (sparse_mask) launch<4, true>(a, B, st, workspace, workspace_bytes);
    else if (bits == 4) launch<4, false>(a, B, st, workspace, workspace_bytes);
    else if (bits == 3) launch<3, false>(a, B, st, workspace, workspace_bytes);
    else launch<2, false>(a, B, st, workspace, workspace_bytes);
    return check_launch("matmul");
}

bool i4::last_chunk_as_others(bool sparse, int64_t B, int64_t n, int64_t K, int64_t S, int64_t group_units) {
    if (tuning(TUNE_NO_WIDE) >= 2) return true;
    const size_t others = rounded_room(sparse, SK_WIDE_MAX_ROWS, K, S, group_units, true), room = rounded_room(sparse, n, K, S, group_units, true);
    if (others == SIZE_MAX) return false;
    if (room <= others || room == SIZE_MAX) return true;                 // (never admitted: nothing to decide)
    const SplitPlan sp = plan_split(sparse, 1, B, K, S);
    const TailPlan tp = plan_tail(sparse, 1, B, K, S);
    size_t bytes = int4mm_workspace_bytes(S) + 2 * round_to_page(std::max(rounded_room(sparse, SK_WIDE_MAX_ROWS, K, S, 0, false),
                                                                          sp.ksplit > 1 ? (size_t)(sp.tiles * sp.ksplit * sp.tile_bytes) : 0));
    if (sp.ksplit == 1 && tp.ksplit > 1) bytes += 2 * round_to_page((size_t)(tp.tiles * tp.ksplit * (256 * 256 * 4)));
    return room <= bytes - ((bytes / 2) & ~size_t(4095));
}

// Workspace with which int4mm_matmul may split K for this shape: what the matvec needs, plus room for
// the partial tiles in the scratch half.  A smaller workspace is not an error: the product then runs unsplit.
extern "C" size_t int4mm_matmul_workspace_bytes(const int4mm_shape* shape, int sparse) {
    if (shape == nullptr) return 0;
    int64_t B = shape->batch, M = shape->seq_len;
    const int64_t K = shape->in_size, S = shape->out_size;
    size_t need = int4mm_workspace_bytes(S);
    // (below 128 columns two to four rows keep the launches that they have with the matvec's workspace)
    if (B <= 0 || M <= 0 || K < 64 || S < (B * M < 5 ? 128 : 64)) return need;
    if (B > 1 && B * M <= ((int64_t)1 << 31) - 256) { M *= B; B = 1; }           // (as int4mm_matmul does)
    // (a caller who asks with the sizes alone leaves matrix_rows or group_size 0)
    int bits = 0;
    for (const int b : {4, 3, 2})
        if (shape->matrix_rows * 32 == K * b) bits = b;
    const int64_t g = shape->group_size, group_units = g < 0 ? ONE_GROUP / 64 : g / 64;
    auto few = [&](int64_t rows, RowsCall call) { return skinny_workspace_bytes(bits, rows, K, S, sparse != 0, group_units, call); };
    size_t few_rows = B * M <= FEW_ROWS_MAX ? few(B * M, FOR_MATMUL) : 0;
    // (the matvec entry takes many batch elements of one row in chunks through the few-row kernels: as many as the kernel
    // for more rows takes, else even shares, which may be one fewer towards the end; its callers may ask with the flattened
    // shape too)
    if (B * M > FEW_ROWS_MAX && (shape->seq_len == 1 || B * M <= SK_WIDE_MAX_ROWS))
        for (const int64_t n : {std::min<int64_t>(B * M, SK_WIDE_MAX_ROWS), B * M > SK_WIDE_MAX_ROWS ? B * M % SK_WIDE_MAX_ROWS : 0}) {
            if (n < 2) continue;
            const bool as_others = B * M <= SK_WIDE_MAX_ROWS || n == SK_WIDE_MAX_ROWS || last_chunk_as_others(sparse != 0, B * M, n, K, S, group_units);
            if (as_others) few_rows = std::max(few_rows, few(n, FOR_MATVEC));
            for (const int64_t share : {exact_sums_at_once(n, S), exact_sums_at_once(B * M, S)})
                if ((n > FEW_ROWS_MAX || !as_others) && share >= 2)
                    few_rows = std::max({few_rows, few(share, EXACT_SUMS), few(std::max<int64_t>(2, share - 1), EXACT_SUMS)});
        }
    size_t part = few_rows;
    if (shape->seq_len == 1 && B * M > SK_WIDE_MAX_ROWS) {           // (chunks of the matvec entry: last_chunk_as_others)
        const SplitPlan sp = plan_split(sparse != 0, B, M, K, S);
        const TailPlan tp = plan_tail(sparse != 0, B, M, K, S);
        if (sp.ksplit > 1) part = std::max(part, (size_t)(sp.tiles * sp.ksplit * sp.tile_bytes));
        else if (tp.ksplit > 1) part = round_to_page(part) + (size_t)(tp.tiles * tp.ksplit * (256 * 256 * 4));
    }
    // (rows that the few-row kernels leave to the tiles are asked for as well: what a product is split into, and with it the order of its
    // sums, may not hang on what a workspace was made for)
    const int64_t variant = tuning(TUNE_MM_VARIANT);
    auto others_serve = [&](int b) {
        if (variant != 0 || tuning(TUNE_NO_SKINNY) || B != 1 || M > SK_WIDE_MAX_ROWS) return false;
        if (M <= FEW_ROWS_MAX) return M == 1 || few_rows_serve(b, sparse != 0, M, K, S, group_units);
        size_t bytes = 0;
        if (!wide_serves(b, sparse != 0, M, K, S, std::max<int64_t>(1, group_units), &bytes)) return false;
        part = std::max(part, bytes);
        return true;
    };
    for (const int b : {4, 3, 2}) {
        if (B != 1 || (sparse ? b != 4 : bits != 0 && b != bits) || others_serve(b)) continue;
        const int64_t gu = std::max<int64_t>(1, group_units);
        if (takes_narrow_tiles(b, sparse != 0, M, K, S, gu)) part = std::max(part, plan_narrow(M, K, S, SIZE_MAX).part_bytes);
        else if (variant != 0 || takes_tiles(b, sparse != 0, M, K, S, gu)) part = std::max(part, plan_tiles(b, sparse != 0, M, K, S, SIZE_MAX, forced_height(variant)).part_bytes);
    }
    return need + 2 * round_to_page(part);
}
