// Products of 17 ... 512 rows, every format, S a multiple of 256 (more than 96 rows: of 64): wide_rows_kernel, for the products of the
// matmul entry and, within a line of precision (rounded_line), for up to 96 rows and for the matvec entry's batches.  Every weight is dequantised once per
// block of up to 128 rows, with the reference's own two roundings fp16(fp16(q - z) s) (matmul.cuh:115-125) or, in exponent
// mode, its single-rounded fma (matmul.cuh:127-136), and multiplied on v_mfma_f32_32x32x16_f16 into accumulators that hold
// the product itself.
//
// A workgroup of eight waves owns a strip of 64 WN columns (WN = 4 or 2) and a range of K; wave (cg, kg) takes 64 of the
// columns and one of the WK = 8 / WN K groups into which the range is cut.  A step is one 64-row unit of every K group: its
// states (32 MT rows x WK x 128 bytes) are moved to LDS once per workgroup, two steps ahead (three buffers, one barrier per
// step), and a wave keeps two units of its packed weights in flight.  At the end the K groups' tiles are summed by halving
// through LDS and, where K is also split across workgroups (blockIdx.z), through the workspace: a workgroup stores its fp32
// tile write-through, counts itself in, and the last to arrive adds the others' up in split order, its own from registers.
//
// What bounds it is the issue of vector instructions, at the 2 GHz that the power limit leaves, and beside the loop the first
// loads and the hand-over (counters of a launch of 64 rows at K=5120, S=20480: VALU 36 % of the SIMDs' cycles, MFMA 26 %, no bank
// conflicts; 16:32, 45 rows at K=S=8192: 44 % and 16 %; int2, 200 rows at K=11008, S=4096: 49 % and 33 %).  Hence
//  * 32x32x16 MFMAs: half the instructions of 16x16x32 for the same product;
//  * 64 columns per wave: a fragment of states that is read from LDS serves two operands;
//  * int4 codes become halves through the 8-bit float conversion: the byte q < 16 is q 2^-9 in e4m3, so mask, shift, mask and
//    four v_cvt_scalef32_pk_f16_fp8 give eight exact codes (7 instructions; magic numbers and their removal: 9), in k order
//    0,2,4,6,1,3,5,7, in which the states are stored;
//  * int2: the group's four weights, dequantised once per column in either mode, are a v_perm table: 15 instructions for
//    eight weights; int3: the eight values' upper bytes are (their lower ones are 0), then add and fma: 23 -- one loop for
//    both modes; int4 and 16:32 have a second loop for waves whose scales hold a negative one, which forms +-2^e as 8-bit
//    floats as well;
//  * scales and zeros are fetched by each wave a group ahead (copying them to LDS first, behind a barrier, cost 2 us a launch);
//  * compact code: a launch runs cold, and a loop unrolled by four with its remainders apart was 1 - 2 us slower than two steps.
//
// Measured (us a launch, cold weights; before: 16x16x32 MFMAs, 32 columns per wave, a barrier per unit, eight waves on the same K):
// K=5120, S=20480, 64 rows int4 30.9 -> 25.0, int3 32.8 -> 27.3, int2 31.3 -> 23.3, one group in 40 in exponent mode 41.6 ->
// 28.1, 16:32 42.8 -> 32; 128 rows int4 46.6 -> 38.3, 16:32 59.9 -> 42.4; K=S=8192, 64 rows 26.4 -> 18.8, 16:32 45 rows 30.7 ->
// 22.3; int2, K=11008, S=4096, 200 rows with exponent mode 62.3 -> 32.3.
#include "rows.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace i4 {

constexpr int RSRC_FLAGS = 0x00020000;                // raw buffer, 32-bit data format
constexpr uint32_t BEYOND = 0x80000000u;              // ORed into a lane's offset: beyond every buffer here, the load returns 0

// packed rows of a 64-row unit, and words per column that a lane loads of it
template <int BITS, bool SPARSE> struct WideFmt;
template <> struct WideFmt<4, false> { static constexpr int ROWS = 8, WORDS = 4; };
template <> struct WideFmt<3, false> { static constexpr int ROWS = 6, WORDS = 6; };
template <> struct WideFmt<2, false> { static constexpr int ROWS = 4, WORDS = 4; };
template <> struct WideFmt<4, true> { static constexpr int ROWS = 4, WORDS = 6; };

struct WideArgs {
    h16* outs;
    const uint32_t* mask;
    float* part;
    int* counters;
    int accumulate;
};

template <int BITS, int MT, bool SPARSE, int WN>
__global__ __launch_bounds__(512, MT == 1 && !SPARSE && !(BITS == 4 && WN == 2) ? 4 : 2) void wide_rows_kernel(const uint32_t* matrix, const h16* x, const h16* scales, const h16* zeros,
                                                         int S, int K, int R_all, int group_units, uint32_t group_magic, int units_per_split,
                                                         WideArgs a) {
    using F = WideFmt<BITS, SPARSE>;
    constexpr int T = 512, WK = 8 / WN, STRIP = 64 * WN;
    constexpr int PITCH = WK * 128 + 16;              // bytes between the rows of a staged step (WK units)
    constexpr int ROWS = 32 * MT, XBUF = ROWS * PITCH, XCH = WK * 8, XPASS = T / XCH, XN = ROWS / XPASS;
    constexpr bool LEAN = MT > 2;                     // (tall blocks: registers for one step of states and one slice's fragments)
    constexpr int XD = LEAN ? 1 : 2;
    constexpr bool TABLE = BITS == 2, BYTES = BITS == 3, TWO_MODES = !TABLE && !BYTES;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ int arrived;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int j = lane & 31, h = lane >> 5;
    const int cg = wave % WN, kg = wave / WN;
    // (a last strip that is not full: the waves beyond the last column repeat the last 64 and write nothing)
    const int wcol = min((int)blockIdx.x * STRIP + cg * 64, S - 64);
    const int units = K / 64;
    const int z0 = blockIdx.z * units_per_split, share = min(units - z0, units_per_split);
    // K group kg takes units kg steps ... of the share; the last ones may get fewer
    const int steps = (share + WK - 1) / WK, u_base = kg * steps;
    const int row0 = blockIdx.y * ROWS, R = min(ROWS, R_all - row0);
    const uint32_t row2 = 2u * (uint32_t)S, row4 = 4u * (uint32_t)S;

    // ---- does any of the wave's groups use exponent mode (a negative or NaN scale)?  Its scales, a row of 64 columns per
    // half wave, are asked for before anything else, so that the answer waits for nothing else; groups beyond the last
    // read as 0.  (int2 and int3 look their weights up and have one loop for both modes.)
    const int u_first = z0 + min(u_base, share - 1), u_last = z0 + min(u_base + steps, share) - 1;       // (u_last < u_first: no unit)
    const int g_first = magic_div(u_first, group_units, group_magic);
    const int groups = magic_div(max(u_last, u_first), group_units, group_magic) + 1 - g_first;
    // (a wave without a unit has empty buffers: everything reads as 0)
    const int row_bytes = u_base < share ? (int)((uint32_t)(groups - 1) * row2 + 128) : 0;
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(scales) + (int64_t)g_first * S + wcol, 0, row_bytes, RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t z_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(zeros) + (int64_t)g_first * S + wcol, 0, row_bytes, RSRC_FLAGS);
    constexpr int BATCH = 4;                          // of two groups each
    uint32_t vs[BATCH], scan_off = (uint32_t)h * row2 + 4u * j;
    auto ask_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < BATCH; ++k, scan_off += 2 * row2) vs[k] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, scan_off, 0, 0);
    };
    if constexpr (TWO_MODES) ask_scales();
    // the current group's scales and zeros are asked for a group ahead: {s, s'} and {z, z'} of the lane's two columns
    uint32_t next_s, next_z, sz_off = 4u * j;
    auto ask_sz = [&]() __attribute__((always_inline)) {
        next_s = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, sz_off, 0, 0);
        next_z = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc, sz_off, 0, 0);
        sz_off += row2;
    };
    ask_sz();

    // ---- states: thread t moves chunk t % XCH (8 k) of rows t / XCH + XPASS q of every step
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<h16*>(x) + (int64_t)row0 * K + (int64_t)z0 * 64, 0, (int)(((uint32_t)(R - 1) * (uint32_t)K + share * 64u) * 2u), RSRC_FLAGS);
    const int xrow = t / XCH, xchunk = t % XCH, x_base = (xchunk >> 3) * steps;
    uint32_t x_off[XN];
#pragma unroll
    for (int q = 0; q < XN; ++q)
        x_off[q] = (uint32_t)min(xrow + XPASS * q, R - 1) * (2u * (uint32_t)K) + 128u * x_base + 16u * (xchunk & 7);
    struct XRegs { u32x4 v[XN]; };
    auto load_x = [&](XRegs& r, int s) __attribute__((always_inline)) {
        const uint32_t beyond = s < min(steps, share - x_base) ? 0u : BEYOND, soff = (uint32_t)min(s, steps - 1) * 128u;
#pragma unroll
        for (int q = 0; q < XN; ++q) r.v[q] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, x_off[q] | beyond, soff, 0);
    };
    char* const x_dst = lds + xrow * PITCH + xchunk * 16;
    auto stage_x = [&](const XRegs& r, uint32_t buf) __attribute__((always_inline)) {
        char* const dst = x_dst + buf;
#pragma unroll
        for (int q = 0; q < XN; ++q) {
            const u32x4 v = r.v[q];
            u32x4 o = v;
            if constexpr (BITS == 4 && !SPARSE)      // k order 0,2,4,6,1,3,5,7
                o = u32x4{__builtin_amdgcn_perm(v[1], v[0], 0x05040100u), __builtin_amdgcn_perm(v[3], v[2], 0x05040100u),
                          __builtin_amdgcn_perm(v[1], v[0], 0x07060302u), __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)};
            else if constexpr (!SPARSE)              // 0,4,1,5,2,6,3,7
                o = u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                          __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
            *reinterpret_cast<u32x4*>(dst + XPASS * q * PITCH) = o;
        }
    };

    // ---- weights: lane (j, h) loads columns 2 j and 2 j + 1 of the wave's 64; in step s the s-th unit of its K group
    const uint32_t unit_bytes = F::ROWS * row4;
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(matrix) + (int64_t)z0 * F::ROWS * S, 0, (int)((uint32_t)share * unit_bytes), RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t m_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(SPARSE ? a.mask + (int64_t)z0 * 2 * S : matrix), 0, (int)((uint32_t)share * 2u * row4), RSRC_FLAGS);
    const uint32_t m_off = (uint32_t)(wcol + 2 * j) * 4u;
    const uint32_t w_off = m_off + (BITS == 4 && !SPARSE ? (uint32_t)h * row4 : 0u);
    struct Packed { u32x2 w[F::WORDS]; };
    // (slice i of a unit: 16 k; the words of a dense format come slice by slice -- int3's and 16:32's, which serve two
    // slices, with the block's second -- as soon as the registers are free)
    struct Cursor { uint32_t off, base; };
    auto cursor = [&](int s) __attribute__((always_inline)) {
        const int u = u_base + s;
        return Cursor{w_off | (s < steps && u < share ? 0u : BEYOND), (uint32_t)min(u, share - 1) * unit_bytes};
    };
    auto load_w = [&](Packed& w, const Cursor& c, int i) __attribute__((always_inline)) {
        if constexpr (SPARSE) {
            if (i & 1) {
                const int blk = i >> 1;
                w.w[3 * blk] = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, c.off, c.base + (2 * blk) * row4, 2);
                w.w[3 * blk + 1] = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, c.off, c.base + (2 * blk + 1) * row4, 2);
                w.w[3 * blk + 2] = __builtin_amdgcn_raw_buffer_load_b64(m_rsrc, c.off, (c.base >> 1) + blk * row4, 2);
            }
        } else if constexpr (BITS == 3) {
            if (i & 1) {
#pragma unroll
                for (int r = 3 * (i >> 1); r < 3 * (i >> 1) + 3; ++r)
                    w.w[r] = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, c.off, c.base + r * row4, 2);
            }
        } else {
            w.w[i] = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, c.off, c.base + (BITS == 4 ? 2 : 1) * i * row4, 2);
        }
    };
    Packed w[2];
    XRegs xr[XD];
    {
        XRegs first[2];
        load_x(first[0], 0);
        load_x(first[1], 1);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const Cursor c = cursor(f);
#pragma unroll
            for (int i = 0; i < 4; ++i) load_w(w[f], c, i);
        }
#pragma unroll
        for (int f = 0; f < XD; ++f) load_x(xr[f], 2 + f);
        stage_x(first[0], 0);
        stage_x(first[1], XBUF);
    }

    // 16:32: for mask byte b the v_perm selectors of its rows' code bytes (even nibbles, then odd ones; 0x0C: none)
    __shared__ __attribute__((aligned(16))) u32x2 lut_table[SPARSE ? 256 : 1];
    const char* const lut = reinterpret_cast<const char*>(lut_table);
    if constexpr (SPARSE) {
        if (t < 256) {
            uint32_t sel[2] = {0, 0}, rank = 0;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const bool k = (t >> r) & 1;
                sel[r >> 2] |= (k ? (rank & 1) * 4 + (rank >> 1) : 0x0Cu) << (8 * (r & 3));
                rank += k;
            }
            lut_table[(t >> 3) | ((t & 7) << 5)] = u32x2{sel[0], sel[1]};        // (under bits 3 .. 10 of the byte's repetition)
        }
    }
    bool general = false;
    if constexpr (TWO_MODES) {
        bool bad = false;
        for (int done = 0;;) {
#pragma unroll
            for (int k = 0; k < BATCH; ++k) bad = bad || !(as_h2(vs[k]).x >= (h16)0.0f) || !(as_h2(vs[k]).y >= (h16)0.0f);
            done += 2 * BATCH;
            if (done >= groups) break;
            ask_scales();
        }
        general = __builtin_amdgcn_ballot_w64(bad) != 0;
    }
    __syncthreads();

    // ---- the lane's two columns: coefficients of the current group
    //   A = P + N, w = fma(A, B, C): P = q, (N, B, C) = (-z, s, -0) in linear mode, P = +-2^e, (-0, -s, z) in exponent mode
    h16x2 cN[2], cB[2], cC[2];
    uint32_t em[2];                     // all ones in exponent mode
    float fs[2];                        // scale of the 8-bit floats: 2^9 for q, 1 for +-2^e
    uint32_t T0[2], T1[2];              // int2: the group's four weights; int3: the eight values' upper bytes
    auto take_sz = [&](auto mode) __attribute__((always_inline)) {
        constexpr bool gen = decltype(mode)::value;
        const uint32_t s1 = next_s, z1 = next_z;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint32_t dup = c ? 0x03020302u : 0x01000100u;
            const h16x2 s = as_h2(__builtin_amdgcn_perm(s1, s1, dup)), z = as_h2(__builtin_amdgcn_perm(z1, z1, dup));
            if constexpr (!gen && TWO_MODES) {
                cB[c] = s;
                cN[c] = z;              // (subtracted)
            } else {
                const uint32_t m = s.x >= (h16)0.0f ? 0u : 0xFFFFFFFFu;
                auto pick = [&](uint32_t e, uint32_t l) { return (e & m) | (l & ~m); };
                em[c] = m;
                cN[c] = as_h2(pick(0x80008000u, as_u32(z) ^ 0x80008000u));
                cB[c] = as_h2(as_u32(s) ^ (m & 0x80008000u));
                cC[c] = as_h2(pick(as_u32(z), 0x80008000u));
                fs[c] = bitcast<float>(pick(0x3F800000u, 0x44000000u));
                if constexpr (TABLE) {
                    const h16x2 p0 = as_h2(pick(0x40003C00u, 0x3C000000u)), p1 = as_h2(pick(0xC000BC00u, 0x42004000u));
                    T0[c] = as_u32(__builtin_elementwise_fma(p0 + cN[c], cB[c], cC[c]));
                    T1[c] = as_u32(__builtin_elementwise_fma(p1 + cN[c], cB[c], cC[c]));
                }
                if constexpr (BYTES) {
                    T0[c] = pick(0x4844403Cu, 0x42403C00u);
                    T1[c] = pick(0xC8C4C0BCu, 0x47464544u);
                }
            }
        }
    };
    const uint32_t half_sel = h ? 0x0C030C02u : 0x0C010C00u;          // int2: half h of a word, its bytes in two halves
    const uint32_t below0 = h ? 0xFFu : 0u, below1 = h ? 0xFFFFFFu : 0xFFFFu, rep0 = 0x01010101u * h, rep1 = 0x01010101u * (2 + h);
    const uint32_t sh0 = h ? 24u : 0u, sh1 = h ? 8u : 16u;
    // operand of k slice i (16 k) of the unit and column c of the lane
    auto operand = [&](auto mode, const Packed& wu, int i, int c) __attribute__((always_inline)) -> h16x8 {
        constexpr bool gen = decltype(mode)::value;
        u32x4 r;
        if constexpr (BITS == 2) {
            const uint32_t word = wu.w[i][c];
            const uint32_t u = __builtin_amdgcn_perm(word, word, half_sel);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t q = (u >> (2 * e)) & 0x00030003u;
                r[e] = __builtin_amdgcn_perm(T1[c], T0[c], __umul24(q, 0x0202u) + 0x01000100u);
            }
        } else if constexpr (BITS == 3) {
            const int b = 3 * (i >> 1);
            const uint32_t w0 = wu.w[b][c], w1 = wu.w[b + 1][c], w2 = wu.w[b + 2][c];
            const uint32_t f = (i & 1) ? __builtin_amdgcn_alignbit(w2, h ? w2 : w1, sh1) : __builtin_amdgcn_alignbit(w1, w0, sh0);
            const uint32_t u = (f & 0xFFFu) | ((f << 4) & ~0xFFFu);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t sh = 3 * e < 8 ? u << (8 - 3 * e) : u >> (3 * e - 8);
                const h16x2 p = as_h2(__builtin_amdgcn_perm(T1[c], T0[c], (sh & 0x07000700u) | 0x000C000Cu));
                r[e] = as_u32(__builtin_elementwise_fma(p + cN[c], cB[c], cC[c]));
            }
        } else {
            uint32_t b0, b1;                      // the codes as bytes
            h16x2 kept[4];                        // 16:32: 1.0 in the kept rows' halves; in the loop for both modes all ones, to be ANDed
            if constexpr (SPARSE) {
                const int b = 3 * (i >> 1);
                const uint32_t w0 = wu.w[b][c], w1 = wu.w[b + 1][c], m = wu.w[b + 2][c];
                const uint64_t st = ((uint64_t)w1 << 32) | w0;
                const uint32_t skip = (uint32_t)__builtin_popcount(m & ((i & 1) ? below1 : below0)) << 2;
                const uint32_t v = (uint32_t)(st >> (skip & 63));
                const uint32_t mb4 = __builtin_amdgcn_perm(m, m, (i & 1) ? rep1 : rep0);
                const u32x2 sel = *reinterpret_cast<const u32x2*>(lut + (mb4 & 0x7F8u));
                const uint32_t even = (v & 0x0F0F0F0Fu) | 0x10101010u, odd_ = ((v >> 4) & 0x0F0F0F0Fu) | 0x10101010u;
                const uint32_t r0 = __builtin_amdgcn_perm(odd_, even, sel.x), r1 = __builtin_amdgcn_perm(odd_, even, sel.y);
                b0 = r0 & 0x0F0F0F0Fu; b1 = r1 & 0x0F0F0F0Fu;
                const uint32_t k0 = r0 & 0x10101010u, k1 = r1 & 0x10101010u;        // the byte 0x10 is 2^-5
                if constexpr (gen && MT < 4) {
                    // (a byte's flag becomes the sign of byte 1 or 3, which selectors 8 ... 11 spread over whole bytes: K=S=8192, 45 rows,
                    // one group in 40 in exponent mode 26.9 us with the form below, 25.9 so.  Blocks of 128 rows have no registers for
                    // it: K=5120, S=20480, 128 rows 50.4 / 49.0, but 43.9 / 45.3 without such groups)
                    auto mask = [](uint32_t r, uint32_t sel) { return as_h2(__builtin_amdgcn_perm(r << 3, r << 11, sel)); };
                    kept[0] = mask(r0, 0x0A0A0808u); kept[1] = mask(r0, 0x0B0B0909u);
                    kept[2] = mask(r1, 0x0A0A0808u); kept[3] = mask(r1, 0x0B0B0909u);
                } else if constexpr (gen) {
                    const uint32_t f0 = (k0 << 4) - (k0 >> 4), f1 = (k1 << 4) - (k1 >> 4);        // 0x10 -> 0xFF, byte by byte
                    kept[0] = as_h2(__builtin_amdgcn_perm(f0, f0, 0x01010000u)); kept[1] = as_h2(__builtin_amdgcn_perm(f0, f0, 0x03030202u));
                    kept[2] = as_h2(__builtin_amdgcn_perm(f1, f1, 0x01010000u)); kept[3] = as_h2(__builtin_amdgcn_perm(f1, f1, 0x03030202u));
                } else {
                    kept[0] = from_fp8<false>(k0, 32.f); kept[1] = from_fp8<true>(k0, 32.f);
                    kept[2] = from_fp8<false>(k1, 32.f); kept[3] = from_fp8<true>(k1, 32.f);
                }
            } else {
                const uint32_t word = wu.w[i][c];
                b0 = word & 0x0F0F0F0Fu; b1 = (word >> 4) & 0x0F0F0F0Fu;
            }
            float scale = 512.f;
            if constexpr (gen) {
                auto expo = [&](uint32_t b) {
                    const uint32_t e = ((b & 0x07070707u) << 3) + 0x38383838u;
                    const uint32_t x = ((b & 0x08080808u) << 4) | e;
                    return (x & em[c]) | (b & ~em[c]);
                };
                b0 = expo(b0); b1 = expo(b1);
                scale = fs[c];
            }
            const h16x2 q[4] = {from_fp8<false>(b0, scale), from_fp8<true>(b0, scale), from_fp8<false>(b1, scale), from_fp8<true>(b1, scale)};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h16x2 o;
                if constexpr (gen) {
                    o = __builtin_elementwise_fma(q[e] + cN[c], cB[c], cC[c]);
                    // (a dropped row is 0, not 0 times its code 0's weight, which may be infinite)
                    if constexpr (SPARSE) o = as_h2(as_u32(o) & as_u32(kept[e]));
                } else if constexpr (SPARSE) {
                    o = __builtin_elementwise_fma(-kept[e], cN[c], q[e]) * cB[c];
                } else {
                    o = (q[e] - cN[c]) * cB[c];
                }
                r[e] = as_u32(o);
            }
        }
        return bitcast<h16x8>(r);
    };

    f32x16 acc[2][MT];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[c][mt][r] = 0.f;

    // ---- the loop.  Step s multiplies the s-th unit of each K group from buffer s % 3, moves the states of step s + 2 to LDS, asks for those
    // of step s + 4 (tall blocks: s + 3) and, as each slice's registers fall free, for the weights of step s + 2; the fragments of a slice are
    // fetched during the one before it, across the barrier too: what a step reads was complete a barrier earlier.
    int group_end = g_first * group_units;             // first unit (of the matrix) beyond the current group
    const int own_end = z0 + min(u_base + steps, share);                // and beyond the wave's
    const char* const xa = lds + j * PITCH + kg * 128 + h * 16;
    h16x8 fa[LEAN ? 1 : 2][MT];
    auto fetch = [&](h16x8 (&f)[MT], const char* from, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) f[mt] = *reinterpret_cast<const h16x8*>(from + 32 * mt * PITCH + i * 32);
    };
    uint32_t buf0 = 0, buf1 = XBUF, buf2 = 2 * XBUF;
    auto step = [&](auto mode, int s, Packed& wu, XRegs& xn) __attribute__((always_inline)) {
        // (a step without a unit multiplies states and codes of 0; its scale and zero are those beyond the wave's last group, which
        // read as 0: a group's own may make an infinity of code 0)
        if (z0 + u_base + s >= min(group_end, own_end)) {
            group_end += group_units;
            take_sz(mode);
            ask_sz();
        }
        stage_x(xn, buf2);
        load_x(xn, s + 2 + XD);
        const Cursor next = cursor(s + 2);
        const char* const here = xa + buf0;
        const char* const there = xa + buf1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (LEAN) fetch(fa[0], here, i);
            else if (i < 3) fetch(fa[(i + 1) & 1], here, i + 1);
            else fetch(fa[0], there, 0);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const h16x8 fb = operand(mode, wu, i, c);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[c][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[LEAN ? 0 : i & 1][mt], fb, acc[c][mt], 0, 0, 0);
            }
            load_w(wu, next, i);
        }
        const uint32_t b = buf0;
        buf0 = buf1; buf1 = buf2; buf2 = b;
        __syncthreads();
    };
    if constexpr (!LEAN) fetch(fa[0], xa, 0);
    auto run = [&](auto mode) __attribute__((always_inline)) {
        int s = 0;
#pragma unroll 1
        for (; s + 2 <= steps; s += 2) {
            step(mode, s, w[0], xr[0]);
            step(mode, s + 1, w[1], xr[XD - 1]);
        }
        if (s < steps) step(mode, s, w[0], xr[0]);
    };
    if (general) run(std::true_type{});
    else run(std::false_type{});

    // ---- the K groups' tiles are summed by halving: in each round a wave gives half of its registers to the wave of the
    // other half of the K groups and adds what it gets; register r of a tile is row 8 (r / 4) + 4 h + r % 4, and the wave of
    // K group kg ends with registers kg 16 / WK ... of every tile (the loop's last barrier is behind every read of what this
    // overwrites)
    constexpr int OWN = 16 / WK, NV = OWN * MT * 2;            // values per lane: [register][row tile][column]
    float val[16 * MT * 2];
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int c = 0; c < 2; ++c) val[(r * MT + mt) * 2 + c] = acc[c][mt][r];
    auto halve = [&](auto level) __attribute__((always_inline)) {
        constexpr int bit = decltype(level)::value, n = 16 * MT * 2 / (WK / bit);        // values given away
        const bool upper = kg & bit;
        char* const out = lds + wave * (n * 256) + lane * 16;
        const char* const in = lds + (wave ^ (bit * WN)) * (n * 256) + lane * 16;
        if (bit != WK / 2) __syncthreads();
#pragma unroll
        for (int v = 0; v < n; v += 4) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = upper ? val[v + e] : val[n + v + e];
            *reinterpret_cast<f32x4*>(out + v * 256) = o;
        }
#pragma unroll
        for (int v = 0; v < n; ++v) val[v] = upper ? val[n + v] : val[v];
        __syncthreads();
#pragma unroll
        for (int v = 0; v < n; v += 4) {
            const f32x4 o = *reinterpret_cast<const f32x4*>(in + v * 256);
#pragma unroll
            for (int e = 0; e < 4; ++e) val[v + e] += o[e];
        }
    };
    if constexpr (WK >= 4) halve(std::integral_constant<int, 2>{});
    halve(std::integral_constant<int, 1>{});

    if (gridDim.z > 1) {
        constexpr int THROUGH = 17;                       // sc0 | sc1: straight to memory
        const int tile = blockIdx.y * gridDim.x + blockIdx.x, ks = gridDim.z;
        // (the slots of a strip: [split][wave][value / 4][lane][4])
        const __amdgpu_buffer_rsrc_t slots = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(a.part) + (int64_t)(tile * ks) * (8 * NV * 256), 0, ks * (8 * NV * 256), RSRC_FLAGS);
        const uint32_t at = (uint32_t)wave * (NV * 256) + lane * 16;
        const uint32_t mine = at + blockIdx.z * (8 * NV * 256);
#pragma unroll
        for (int v = 0; v < NV; v += 4)
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{bitcast<uint32_t>(val[v]), bitcast<uint32_t>(val[v + 1]), bitcast<uint32_t>(val[v + 2]), bitcast<uint32_t>(val[v + 3])},
                                                   slots, mine + v * 256, 0, THROUGH);
        __builtin_amdgcn_s_waitcnt(0);                 // every store of this thread has been acknowledged
        __syncthreads();
        if (t == 0) arrived = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (arrived != ks - 1) return;
        if (t == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        float sum[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) sum[v] = 0.f;
        uint32_t from = at;
#pragma unroll 1
        for (int sp = 0; sp < ks; ++sp, from += 8 * NV * 256) {
            if (sp == (int)blockIdx.z) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sum[v] += val[v];
                continue;
            }
            u32x4 o[NV / 4];
#pragma unroll
            for (int v = 0; v < NV; v += 4) o[v / 4] = __builtin_amdgcn_raw_buffer_load_b128(slots, from + v * 256, 0, THROUGH);
#pragma unroll
            for (int v = 0; v < NV; ++v) { const uint32_t b = o[v / 4][v & 3]; sum[v] += bitcast<float>(b); }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) val[v] = sum[v];
    }
    // ---- (rows beyond R lie beyond the buffer: their stores do nothing; a wave beyond the last column has an empty one)
    const __amdgpu_buffer_rsrc_t o_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.outs + (int64_t)row0 * S, 0, (int)(blockIdx.x * STRIP + cg * 64 < (unsigned)S ? (uint32_t)R * row2 : 0u), RSRC_FLAGS);
    const int m0 = WK == 2 ? 16 * kg : 8 * kg;         // first row of register kg OWN, in lane group 0
    const uint32_t o_off = (uint32_t)(m0 + 4 * h) * row2 + (uint32_t)(wcol + 2 * j) * 2u;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            const uint32_t off = o_off + (uint32_t)(32 * mt + 8 * (i >> 2) + (i & 3)) * row2;
            float v0 = val[(i * MT + mt) * 2], v1 = val[(i * MT + mt) * 2 + 1];
            if (a.accumulate) {
                const uint32_t prior = __builtin_amdgcn_raw_buffer_load_b32(o_rsrc, off, 0, 0);
                v0 += lo_f32(prior);
                v1 += hi_f32(prior);
            }
            __builtin_amdgcn_raw_buffer_store_b32(as_u32(h16x2{(h16)v0, (h16)v1}), o_rsrc, off, 0, 0);
        }
}

// LDS: three staged steps; the halving at the end keeps half of the workgroup's tile there
static constexpr size_t wide_lds_bytes(int mt, int wn) {
    const size_t staged = 3 * 32 * (size_t)mt * ((8 / wn) * 128 + 16), halved = 8 * 16 * (size_t)mt * 256;
    return staged > halved ? staged : halved;
}

// ---- which launch.  Blocks of 32 mt rows, strips of 64 wn columns, K split ksplit ways across workgroups: the candidate
// that a cost model finds cheapest, in us,
//     steps (step + filled x fill) + workgroup + (rounds - 1) (steps x more_step + more_workgroup) + last x fill of the last round
//     + (ksplit > 1: split + way x ksplit)
// with the steps of a workgroup (units of its share / K groups), fill = the share of the 256 CUs that get a workgroup and
// rounds of 256 workgroups (two of the smallest ones share a CU: their second round is cheaper).  Fitted per format and kernel
// to 930 ... 2440 timed launches each (K = 1024 ... 20480, S = 1024 ... 28672, 24 ... 512 rows, cold weights).  On 30 other random shapes
// of that range per format its pick was the best measured candidate on half of them and 1.1 / 1.8 / 1.0 / 0 % off it on
// average (int4, int3, int2, 16:32), 12 / 21 / 23 / 8 % at worst.
struct WidePlan { bool use; int mt, wn, row_blocks, ksplit, units_per_split; size_t part_bytes; double us; };
struct WideCost { int mt, wn; double step, filled, more_step, workgroup, more_workgroup, split, way, last; };
static const WideCost wide_cost[4][6] = {             // int4, int3, int2, 16:32
    {{1, 2, 0.736, 0.148, 0.824, 4.36, 2.51, 0.847, 0.445, 1.3},
     {2, 2, 0.858, 0.35, 1.09, 5.47, 3.79, 1.26, 0.492, 1.92},
     {1, 4, 0.653, 0.148, 0.62, 4.22, 0.644, 1.16, 0.484, 1.32},
     {2, 4, 0.866, 0.27, 0.989, 4.99, 4.32, 1.65, 0.655, 2.82},
     {3, 4, 1.14, 0.374, 1.29, 5.68, 5.53, 1.88, 0.922, 3.89},
     {4, 4, 1.24, 0.558, 1.53, 6.91, 6.48, 2.07, 1.24, 6.54}},
    {{1, 2, 1.04, 0.0999, 0.957, 4.42, 0, 0.864, 0.439, 0.838},
     {2, 2, 1.25, 0.203, 1.37, 5.51, 3.65, 1.26, 0.49, 1.74},
     {1, 4, 1.14, 0.069, 0.836, 3.95, 0.815, 0.882, 0.483, 1.07},
     {2, 4, 1.17, 0.196, 1.23, 4.88, 3.87, 1.61, 0.656, 2.43},
     {3, 4, 1.61, 0.19, 1.66, 5.69, 4.56, 1.58, 0.946, 3.28},
     {4, 4, 1.8, 0.323, 1.92, 6.76, 5.5, 1.66, 1.29, 5.09}},
    {{1, 2, 0.744, 0.0786, 0.657, 3.98, 0.211, 0.86, 0.449, 0.79},
     {2, 2, 0.944, 0.213, 1.07, 5.08, 3.51, 1.32, 0.496, 1.65},
     {1, 4, 0.805, 0.078, 0.517, 3.55, 1.25, 0.875, 0.481, 0.708},
     {2, 4, 0.873, 0.187, 0.957, 4.3, 3.86, 1.82, 0.661, 1.91},
     {3, 4, 1.28, 0.201, 1.37, 5.31, 4.57, 1.61, 0.956, 2.84},
     {4, 4, 1.45, 0.348, 1.63, 6.38, 5.58, 1.74, 1.29, 4.72}},
    {{1, 2, 1.3, 0.131, 1.33, 4.64, 2.59, 0.844, 0.442, 1.7},
     {2, 2, 1.44, 0.193, 1.46, 5.91, 4.3, 1.21, 0.491, 1.82},
     {1, 4, 1.26, 0.106, 1.23, 4.4, 2.54, 1.11, 0.487, 2.45},
     {2, 4, 1.4, 0.187, 1.36, 5.23, 4.64, 1.8, 0.663, 2.7},
     {3, 4, 1.71, 0.227, 1.65, 5.67, 5.77, 2.17, 0.946, 3.34},
     {4, 4, 1.76, 0.352, 1.84, 7.15, 6.6, 2.45, 1.26, 5.45}}};
constexpr int64_t WIDE_MAX_SPLIT_WGS = 512;              // workgroups of a launch that splits K (bounds its partial tiles)

// Which products of up to 96 rows, and which of the matvec entry, may take the kernel above.  Elsewhere they are sums of the
// exact codes, scale and zero applied in fp32; here each weight is rounded to fp16 twice (error against float64, 2-norm, 90
// rows at K=5120, S=2560: 2.07e-4 of the result there -- all of it the fp16 output's --, 3.23e-4 here).  Hence this is a line of precision and not of speed, and is not to be fitted to timings: it admits what an earlier form of
// the kernel took -- with its split of K, if its partial tiles have `room` in the workspace and a share's scales have room in the
// LDS, as that form kept them there -- so that no product that had the exact codes' sums loses them.
struct RoundedLine { bool admitted; size_t room; };
static RoundedLine rounded_line(bool sparse, int64_t R, int64_t K, int64_t S, int64_t group_units) {
    const RoundedLine none{false, 0};
    if (R < 17 || R > SK_WIDE_MAX_ROWS || S % 256 != 0) return none;
    // (32-bit: a query of the workspace comes here as well as a launch)
    const int rows = (int)R, units = (int)(K / 64), strips = (int)(S / 256), lds_limit = 150 * 1024 - (sparse ? 4096 : 0);
    const int gu = (int)std::min<int64_t>(group_units, units);
    int tiles = 0, blocks = 0, wgs = 0, ks = 1;             // row tiles of 16 in a block, blocks, unsplit workgroups, ways
    const int all_groups = (units + gu - 1) / gu;
    int64_t most_units = 0;                                 // of a share whose groups -- one more may be cut -- fit
    auto fits = [&](int share) { return share <= most_units; };
    auto shape = [&](int tallest) {
        blocks = (rows + tallest - 1) / tallest;
        tiles = ((rows + blocks - 1) / blocks + 15) / 16;
        if (tiles == 5 || tiles == 7) ++tiles;
        wgs = strips * blocks;
        const int most_groups = (lds_limit - 1040 - 16 * tiles * 288) / 1024;
        most_units = all_groups <= most_groups ? units : (int64_t)(most_groups - 1) * gu;
    };
    auto shape_and_split = [&](int tallest) {
        shape(tallest);
        ks = wgs > 128 && wgs < 256 ? 4 : 256 / wgs;
        ks = wgs > 1024 ? 1 : std::max(1, std::min(ks, units / 8));
        while (wgs * (ks + 1) <= 256 && ks < units / 8 && !fits((units + ks - 1) / ks)) ++ks;
    };
    shape_and_split(128);
    if (R <= 64 || ks > 6 || (ks > 1 && units / ks < 20)) shape_and_split(64);
    if (!sparse && R > 48 && R <= 64 && S <= 4096) shape_and_split(32);
    if (R > 64 && S >= (sparse ? 4096 : 1024) && S <= (sparse ? 8192 : 32768)) {
        struct Cost { double unit[9], workgroup, split, way, tile, last; };
        static const Cost costs[2] = {{{0, 0, 0, 0.617, 0.707, 0, 0.912, 0, 1.059}, 3.92, -4.164, 0.798, 1.915, 3.544},
                                      {{0, 0, 0, 1.12, 1.203, 0, 1.32, 0, 1.537}, 4.17, -3.744, 0.921, 1.701, 5.284}};
        const Cost& c = costs[sparse];
        double best = 1e30;
        int best_tallest = 0, best_ks = 1;
        for (const int tallest : {128, 96, 64, 48}) {
            shape(tallest);
            for (int k = 1; k <= 16 && (k == 1 || units >= 8 * k) && wgs * k <= 1024; ++k) {
                const int share = (units + k - 1) / k, rounds = (wgs * k + 255) >> 8, last = wgs * k - (rounds - 1) * 256;
                if (!fits(share)) continue;
                const double t = rounds * (c.unit[tiles] * share + c.workgroup) + (k > 1 ? c.split + c.way * k + c.tile * tiles : 0.0) +
                                 (rounds > 1 ? c.last * last / 256.0 : 0.0);
                if (t < best) { best = t; best_tallest = tallest; best_ks = k; }
            }
        }
        if (best_tallest != 0) { shape(best_tallest); ks = best_ks; }
        else shape_and_split(48);
    }
    const int share = (units + ks - 1) / ks;
    ks = (units + share - 1) / share;
    if (!fits(share)) return none;
    // one round of two row blocks of the few-row kernel, or that kernel's own split of K
    const bool one_round = [&] {
        if (S / 32 * 2 < 192) return true;
        for (const int c : {4, 2, 1}) {
            if (sparse && c == 4) continue;
            if (S / (16 * c) * 2 >= 128 && S / (16 * c) * 2 <= 256) return true;
        }
        return false;
    }();
    bool few_row;                                           // the few-row kernel or, beyond 96 rows, the matvec
    if (sparse) {
        few_row = R <= 32 ? K * S < (1ll << 26)
                : R <= 64 ? (one_round ? K <= 8192 || S < 3072 : K < 4096 && K * S < (1ll << 25))
                : R <= 96 ? false
                : R <= 128 ? S > 16384 && blocks > 1 : S > 8192 || (R > 256 && S > 4096);
    } else {
        few_row = R <= 32 ? wgs < (units >= 160 ? 24 : 32) || wgs > 96 || share < 16 || (S / 64 > 128 && S / 64 <= 256 && K <= 6144)
                : R <= 64 ? (one_round ? K <= 5120 || (K <= 8192 && S <= 4096) || S < 3072 : K * S < (1ll << 25))
                : R <= 128 ? false
                : S > 8192 && S > (R <= 192 || (R <= 256 && K <= 4096) ? 32768 : R <= 256 ? 10240 : 8192);
    }
    if (few_row) return none;
    return {true, ks > 1 ? (size_t)wgs * ks * tiles * 16384 : 0};
}

static bool needs_admission(int64_t R, RowsCall call) {
    return (R <= FEW_ROWS_MAX || call == FOR_MATVEC) && call != ROUNDED && tuning(TUNE_NO_WIDE) < 2;
}

// (groups of these units where the group is not known)
static constexpr int64_t SOME_GROUPS[] = {1, 2, 3, 4, 6, 8, 16, 0x7FFFFFF};

size_t rounded_room(bool sparse, int64_t R, int64_t K, int64_t S, int64_t group_units, bool least) {
    size_t room = least ? SIZE_MAX : 0;
    for (const int64_t units : SOME_GROUPS) {
        const RoundedLine line = rounded_line(sparse, R, K, S, group_units > 0 ? group_units : units);
        if (line.admitted) room = least ? std::min(room, line.room) : std::max(room, line.room);
        if (group_units > 0) break;
    }
    return room;
}

// Whole strips of 256 columns; beyond 96 rows, which the few-row kernel does not take, any number of whole 64 (the general
// tiles that served them cannot split K: int2, K=9280, S=1600, 220 rows 238 us there, 21 here).
static bool wide_columns(int64_t R, int64_t S) { return S % 256 == 0 || (R > FEW_ROWS_MAX && S % 64 == 0); }
static int64_t wide_strips(int64_t S, int wn) { return (S + 64 * wn - 1) / (64 * wn); }

// `scratch`: bytes for partial tiles; the splits that need more are no candidates
static WidePlan plan_wide(int bits, bool sparse, int64_t R, int64_t K, int64_t S, size_t scratch) {
    WidePlan p{false, 0, 0, 0, 1, 0, 0, 0.0};
    // (knob: 1 = never, n >= 2 = from n rows on whatever the shape)
    const int64_t knob = tuning(TUNE_NO_WIDE), min_rows = knob >= 2 ? knob : 17, forced = tuning(TUNE_MM_SPLIT);
    if (R < min_rows || R > SK_WIDE_MAX_ROWS || !wide_columns(R, S) || K % 64 != 0 || knob == 1) return p;
    const int64_t units = K / 64;
    // (32-bit byte offsets into buffer resources: a share of the packed matrix, its scales and the block's rows of states and
    // outputs stay below 2 GB)
    if (K * S >= (sparse ? 1ll << 33 : (1ll << 34) / bits) || K >= (1 << 22) || S >= (1 << 22)) return p;
    const int64_t few = (R + 127) / 128, tallest = ((R + few - 1) / few + 31) / 32;
    double best = 1e30;
    for (const WideCost& c : wide_cost[sparse ? 3 : 4 - bits]) {
        // (a block of rows that would hold no row more than the one below; 65 ... 256 rows up to K = 512 and 1024 columns keep the
        // fewest blocks, through which the tests of tall blocks go: K=S=512, 100 rows 12.0 us, 10.1 by the model's choice)
        if (32 * (c.mt - 1) >= R || (R > 64 && R <= 256 && units <= 8 && S <= 1024 && c.mt != tallest)) continue;
        // (49 ... 64 rows on 2048 ... 4096 columns and a long K: two blocks of 32 rows)
        if (!sparse && R > 48 && R <= 64 && S > 2048 && S <= 4096 && K > 8192 && forced < 1 && (c.mt != 1 || c.wn != 4)) continue;
        const int64_t blocks = (R + 32 * c.mt - 1) / (32 * c.mt), tiles = wide_strips(S, c.wn) * blocks;
        const auto too_large = [&](int64_t k) {
            const int64_t share = (units + k - 1) / k;
            return k > 1 && (size_t)((units + share - 1) / share * tiles * c.mt * c.wn) * 8192 > scratch;
        };
        // (below 1024 columns, where nothing was fitted: as many ways as leave shares of eight units)
        int64_t only = forced >= 1 ? std::min<int64_t>(forced, std::max<int64_t>(1, units / 4))
                     : S < 1024 ? std::max<int64_t>(1, std::min<int64_t>({256 / tiles, units / 8, 16})) : 0;
        while (only > 1 && too_large(only)) --only;
        for (int64_t k = only ? only : 1; k <= 16; ++k) {
            if (k > 1 && (units / k < 4 || tiles * k > WIDE_MAX_SPLIT_WGS || too_large(k))) break;
            const int64_t share = (units + k - 1) / k, steps = (share * c.wn + 7) / 8, wgs = tiles * k, rounds = (wgs + 255) / 256;
            const double t = steps * (c.step + c.filled * std::min(1.0, wgs / 256.0)) + c.workgroup + (k > 1 ? c.split + c.way * k : 0.0) +
                             (rounds > 1 ? (rounds - 1) * (c.more_step * steps + c.more_workgroup) + c.last * (wgs - (rounds - 1) * 256) / 256.0 : 0.0);
            if (t < best) { best = t; p.mt = c.mt; p.wn = c.wn; p.row_blocks = (int)blocks; p.units_per_split = (int)share; }
            if (only) break;
        }
    }
    if (p.mt == 0) return p;
    p.ksplit = (int)((units + p.units_per_split - 1) / p.units_per_split);
    // 257 rows and more on a wide output that is not split: the 256-row tiles, where the model's time is beyond what they
    // take (5 us and 0.75 PFLOP/s while the blocks fit one round of workgroups, 1.05 beyond: K=8192, S=28672, 512 rows 245 here,
    // 227 in tiles; int3, K=20480, S=11008 324 / 295; int4 K=8192, S=20480, 384 rows stays, 140 / 196; int3, K=512, S=17664, 442
    // rows 29 / 20; K=192, S=28416, 435 rows 22 / 14)
    if (knob < 2 && forced < 1 && R > 256 && S > 10240 && p.ksplit == 1) {
        const double flops = 2.0 * ((R + 255) / 256 * 256) * K * S;
        if (best > 5.0 + flops / (wide_strips(S, p.wn) * p.row_blocks > 256 ? 1.05e9 : 0.75e9)) return p;
    }
    p.part_bytes = p.ksplit > 1 ? (size_t)p.ksplit * p.row_blocks * p.mt * wide_strips(S, p.wn) * p.wn * 8192 : 0;
    p.us = best;
    p.use = true;
    return p;
}

// More than 256 rows through the matmul entry: the tile kernels where they are faster, by both models (us, here / there: int4, K=6656, S=14592,
// 306 rows 86 / 75; K=16000, S=14208, 432 rows 230 / 189; int3, K=2816, S=8448, 462 rows 47 / 39)
static bool tiles_instead(int bits, bool sparse, int64_t R, int64_t K, int64_t S, int64_t group_units, size_t scratch, const WidePlan& p) {
    return R > 256 && tuning(TUNE_NO_WIDE) < 2 && tuning(TUNE_MM_SPLIT) < 1 && tiles_us(bits, sparse, R, K, S, group_units, scratch) < 0.95 * p.us;
}

// Does the matmul entry leave a product of 97 ... 512 rows to this kernel, given room for any split?
bool wide_serves(int bits, bool sparse, int64_t R, int64_t K, int64_t S, int64_t group_units, size_t* part_bytes) {
    const WidePlan p = plan_wide(bits, sparse, R, K, S, SIZE_MAX);
    if (part_bytes) *part_bytes = p.part_bytes;
    return p.use && !tiles_instead(bits, sparse, R, K, S, group_units, SIZE_MAX, p);
}

// What the plan's partial tiles take with room for any split and, where a product has to be admitted, the room that it takes to be;
// bits = 0, group_units = 0: not known, the most of any
size_t wide_workspace_bytes(int bits, int64_t R, int64_t K, int64_t S, bool sparse, int64_t group_units, RowsCall call) {
    if (call == EXACT_SUMS || R < 2 || R > SK_WIDE_MAX_ROWS || !wide_columns(R, S) || K % 64 != 0) return 0;
    size_t need = 0;
    if (needs_admission(R, call)) {
        bool admitted = false;
        for (const int64_t units : SOME_GROUPS) {
            const RoundedLine line = rounded_line(sparse, R, K, S, group_units > 0 ? group_units : units);
            admitted = admitted || line.admitted;
            need = std::max(need, line.room);
            if (group_units > 0) break;
        }
        if (!admitted) return 0;
    }
    for (const int b : {4, 3, 2}) {
        if (sparse ? b != 4 : bits != 0 && b != bits) continue;
        const WidePlan p = plan_wide(b, sparse, R, K, S, SIZE_MAX);
        if (p.use) need = std::max(need, p.part_bytes);
    }
    return need;
}

template <int BITS, int MT, bool SPARSE, int WN>
static void launch_wide(const SkinnyArgs& s, const WidePlan& p, hipStream_t st) {
    constexpr size_t bytes = wide_lds_bytes(MT, WN);
    const dim3 grid((unsigned)wide_strips(s.S, WN), p.row_blocks, p.ksplit), block(512);
    auto kernel = wide_rows_kernel<BITS, MT, SPARSE, WN>;
    if constexpr (bytes > 64 * 1024) {                   // more than 64 KB of dynamic LDS has to be requested once per kernel and device
        static std::atomic<uint64_t> done;
        int dev = 0;
        (void)hipGetDevice(&dev);
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done.load(std::memory_order_relaxed) & bit)) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
            done.fetch_or(bit, std::memory_order_relaxed);
        }
    }
    const WideArgs a{s.outs, s.mask, s.part, s.counters, s.accumulate};
    hipLaunchKernelGGL(kernel, grid, block, bytes, st, s.matrix, s.x, s.scales, s.zeros, s.S, s.K, s.R, s.group_units,
                       div_magic((uint32_t)s.group_units), p.units_per_split, a);
}

template <int BITS, bool SPARSE>
static bool launch_wide(const SkinnyArgs& a, const WidePlan& p, hipStream_t st) {
    if (noting("wide_rows_kernel<bits=%d,%s,row_tiles=%d> strips=%d row_blocks=%d ksplit=%d columns=%d", BITS, SPARSE ? "16:32" : "dense",
               2 * p.mt, (int)wide_strips(a.S, p.wn), p.row_blocks, p.ksplit, 64 * p.wn))
        return true;
    if (p.wn == 2) {
        if (p.mt == 1) launch_wide<BITS, 1, SPARSE, 2>(a, p, st);
        else launch_wide<BITS, 2, SPARSE, 2>(a, p, st);
    } else if (p.mt == 1) launch_wide<BITS, 1, SPARSE, 4>(a, p, st);
    else if (p.mt == 2) launch_wide<BITS, 2, SPARSE, 4>(a, p, st);
    else if (p.mt == 3) launch_wide<BITS, 3, SPARSE, 4>(a, p, st);
    else launch_wide<BITS, 4, SPARSE, 4>(a, p, st);
    return true;
}

bool wide_rows(int bits, const SkinnyArgs& args, RowsCall call, void* workspace, size_t workspace_bytes, hipStream_t st) {
    const bool sparse = args.mask != nullptr;
    const WorkspaceParts ws = workspace_parts(workspace, workspace_bytes);
    if (call == EXACT_SUMS) return false;
    if (needs_admission(args.R, call)) {
        const RoundedLine line = rounded_line(sparse, args.R, args.K, args.S, args.group_units);
        if (!line.admitted || ws.scratch_bytes < line.room) return false;
    }
    const WidePlan p = plan_wide(bits, sparse, args.R, args.K, args.S, ws.scratch_bytes);
    if (!p.use) return false;
    if (call == FOR_MATMUL && tiles_instead(bits, sparse, args.R, args.K, args.S, args.group_units, ws.counters != nullptr ? ws.scratch_bytes : 0, p)) return false;
    SkinnyArgs a = args;
    a.counters = reinterpret_cast<int*>(ws.counters);
    a.part = reinterpret_cast<float*>(ws.scratch);
    if (sparse) return launch_wide<4, true>(a, p, st);
    return bits == 4 ? launch_wide<4, false>(a, p, st) : bits == 3 ? launch_wide<3, false>(a, p, st) : launch_wide<2, false>(a, p, st);
}

}  // namespace i4
