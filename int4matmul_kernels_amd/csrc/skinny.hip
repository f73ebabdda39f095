// Few-row products for gfx950: 2 .. 96 rows of states (32 per
// workgroup) against a dense int4 / int3 / int2 or 16:32 sparse int4 weight matrix, HBM-bound like the
// matvec (every packed word is read once and used for all rows).  17 .. 512 rows: wide_rows_kernel (csrc/wide.hip), which
// skinny_rows() at the end asks first.  The reference has no such path: it sends M >= 2 to its
// 64-row matmul tiles (int4matmul.cpp:27) and M == 1 with B > 1 to one matvec
// per batch element, re-reading the weights each time (matvec_kernel.cu:346).
//
// The rows are multiplied on the matrix core: v_mfma_f32_16x16x32_f16 takes 16
// rows of states as its 16 x 32 operand (rows >= R are zero; 17 .. 32 rows take
// two such tiles) and, as its 32 x 16 operand, 8 consecutive k of one column per
// lane -- which is exactly one packed int4 word; the four lane groups of a wave
// hold the four packed rows of a 32-row block.  A word becomes that operand
// without converting a single code: mask-and-OR of the word (and of the word
// shifted by 8) gives the half2 pairs {1024 + q0, 1024 + q4}, {64 + q1, 64 + q5},
// {1024 + q2, 1024 + q6}, {64 + q3, 64 + q7}; the states are stored to LDS in the
// same k order 0,4,1,5,2,6,3,7.  (int2 / int3: the chunk's 16 / 24 bits, pairs
// {1024 + q_even, 256 or 128 + q_odd} in natural order.)
// The offsets are removed once per quantisation group in fp32 together with
// scale and zero:
//     y[m, n] += s[n] * (acc[m, n] - sum_k off_k x[m, k] - z[n] * sum_k x[m, k])
// which is the exact value of sum_k x (q - z) s (the per-weight fp16 roundings of
// the reference's decode are not reproduced, as in the matvec).
//
// A workgroup owns a strip of 16 * CW columns (lane j of a wave holds the words
// of CW adjacent columns: CW * 64 contiguous bytes per packed row and wave) and
// its W waves split K; each wave stages the states of its own K range through
// a private LDS buffer, 64 k at a time, and the partial tiles are summed
// through LDS at the end; narrow matrices with a long K are also split along K across workgroups.
//
// 16:32 sparse int4 takes the same kernel.  Every lane group loads the block's
// mask word and both words of kept codes (the four groups of a wave ask for the
// same addresses); group h skips the codes of the rows before its eight with a
// population count of the lower mask bits, and expands its codes to their rows
// with the v_perm selectors of a 256-entry table in LDS (indexed by the mask
// byte), in the int4 k order.  No magic numbers here: the bytes 0x1q (bit 4: "this
// row is kept") become the halves 0x001q, i.e. the fp16 denormals (16 + q) 2^-24,
// which the matrix core multiplies exactly; a second MFMA on the same operand
// masked to 0x0010 gives 16 * 2^-24 * (sum of the kept rows' states), and
//     y[m, n] += s[n] * (2^24 (accA - accM) - z[n] * 2^20 accM).
#include "rows.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace i4 {

constexpr int SK_PITCH = 144;                   // bytes between rows of a staged unit (128 + 16: conflict-free)
constexpr int SK_XBUF = 32 * SK_PITCH;          // one staged unit: 32 rows x 64 k
constexpr int SK_WAVE_LDS = 2 * SK_XBUF + 256;  // two unit buffers + the group sums of 32 rows

constexpr int SK_BAL_WAVES = 8;

// Balanced launch: workgroup i of 256 takes the range [i q + i r / 256, (i + 1) q + (i + 1) r / 256) of
// strips x units (strip-major; q, r = quotient and remainder of the total by 256).  The range is at least one
// strip and less than two strips long, so it touches at most three strips: three segments, segment k on strip
// strip0 + k.  The workgroup's waves are dealt to the segments in proportion to their units (at least one each).
// For one wave: its segment (`mine`), the segment's units [lo, hi) within its strip, the segment's first wave
// and number of waves; of all segments: the first unit of the first one and the units of each.
struct BalancedShare { int strip0, mine, lo, hi, wave0, waves, first, n0, n1, n2; };
// (The quotients stand between a wave's start and its first loads, in code that every launch fetches anew: they are taken with
// magic numbers, which the host passes -- magic_div, csrc/common.h -- or through the float reciprocal.)
// a / b for 0 <= a < 2^22 through the float reciprocal, for a divisor without a magic number at hand
__device__ __forceinline__ int small_div(int a, int b, float inv_b) {
    int q = (int)((float)a * inv_b);
    int r = a - q * b;
    if (r < 0) { --q; r += b; }
    if (r >= b) ++q;
    return q;
}
__device__ __forceinline__ BalancedShare balanced_share(int q, int r, uint32_t units_magic, int i, int units, int wave) {
    BalancedShare b{};
    const int lo = i * q + ((i * r) >> 8), hi = (i + 1) * q + (((i + 1) * r) >> 8);           // (/ 256 workgroups)
    const int share = hi - lo;
    const float per_unit = (float)SK_BAL_WAVES * __builtin_amdgcn_rcpf((float)share);
    b.strip0 = magic_div(lo, units, units_magic);
    b.first = lo - b.strip0 * units;
    b.n0 = min(share, units - b.first);
    b.n1 = min(share - b.n0, units);
    b.n2 = share - b.n0 - b.n1;
    // waves in proportion, at least one each: the outer segments' are rounded, the middle one, a whole strip and more than half
    // of the range where there are three, has the rest (any deal is right; a rounding that differs moves a wave)
    const int w2 = b.n2 > 0 ? max(1, (int)((float)b.n2 * per_unit + 0.5f)) : 0;
    const int w0 = b.n1 > 0 ? min(max(1, (int)((float)b.n0 * per_unit + 0.5f)), SK_BAL_WAVES - 1 - w2) : SK_BAL_WAVES;
    const int w1 = SK_BAL_WAVES - w0 - w2;
    b.mine = wave < w0 ? 0 : wave < w0 + w1 ? 1 : 2;
    b.wave0 = b.mine == 0 ? 0 : b.mine == 1 ? w0 : w0 + w1;
    b.waves = b.mine == 0 ? w0 : b.mine == 1 ? w1 : w2;
    b.lo = b.mine == 0 ? b.first : 0;
    b.hi = b.mine == 0 ? b.first + b.n0 : b.mine == 1 ? b.n1 : b.n2;
    // (the same in every lane, which the compiler cannot see behind the float arithmetic)
    b.mine = __builtin_amdgcn_readfirstlane(b.mine);
    b.wave0 = __builtin_amdgcn_readfirstlane(b.wave0);
    b.waves = __builtin_amdgcn_readfirstlane(b.waves);
    b.lo = __builtin_amdgcn_readfirstlane(b.lo);
    b.hi = __builtin_amdgcn_readfirstlane(b.hi);
    return b;
}

// CW: columns per lane; RT: row groups of 8 that can hold real rows (R <= 8 RT);
// MT: 16-row MFMA tiles; PF: units of packed weights in flight per wave
// BAL: the workgroups share the work evenly instead of taking a strip each (more strips than CUs): a workgroup's
// range of (strip, unit) touches two or three strips, its waves are dealt to them in proportion, every wave works
// on one strip, and a strip that two workgroups share is summed through the hand-over below.
// XC = 1: a fifth column per lane (CW = 4 only, dense formats): the workgroup's columns are four or five slivers of
// 16, the lane's four adjacent columns in the first four and column j of the fifth (a.wide_wgs workgroups have one)
// PLAIN: the operand is the codes themselves or, in exponent mode, their powers of two -- no offsets to be removed from the sums, no
// weight that is rounded in a strip with a negative scale.  For the shares of a batch that would otherwise run one matvec per
// element (17 rows and more, a batch that the kernel with rounded weights does not take) and lose nothing to it.  2-norm of the error
// against float64 (1e-4), one matvec per element / shares with offsets and rounded weights / PLAIN, 110 ... 180 elements, S=1088: int3, K=4096, one
// group 2.07 / 2.13 / 2.06; int2, K=8192, g=128 2.11 / 2.16 / 2.08; one (group, column) in 40 in exponent mode, K=4096: int4, g=128 2.07 / 3.25 /
// 2.07 (1615 / 32 / 29 us), 16:32 2.06 / 3.24 / 2.06 (1102 / 45 / 32)
template <int BITS, int CW, int RT, bool SPARSE, bool BAL = false, int XC = 0, bool PLAIN = false>
__global__ __launch_bounds__(512) void skinny_kernel(const uint32_t* pre_matrix, const h16* pre_x, const h16* pre_scales, const h16* pre_zeros,
                                                   int pre_S, int pre_K, int pre_group_units, int pre_units, uint32_t pre_rows,
                                                   uint32_t pre_more, SkinnyArgs a) {
    // (what the first loads depend on, once more in front of the record: the first dwords of a kernel's arguments
    // reach a wave in registers at its start, a record's fields are fetched by the wave itself; with the rows, the ranges and the
    // waves among them nothing waits for the record before the loads: int4, K=5120, S=20480, 8 rows 18.2 -> 17.8 us a layer,
    // int3, K=4864, S=2304 10.1 -> 9.9)
    a.matrix = pre_matrix; a.x = pre_x; a.scales = pre_scales; a.zeros = pre_zeros; a.S = pre_S; a.K = pre_K;
    a.group_units = pre_group_units;
    // (pre_units, pre_rows, pre_more -- BAL: q, rows and r, the magic number of the units; XC: units per wave, rows and waves,
    // workgroups with a fifth sliver; else units per wave, rows and waves, units per split)
    a.R = (int)(pre_rows & 0xFFFF);
    if constexpr (BAL) { a.bal_q = pre_units; a.bal_r = (int)(pre_rows >> 16); a.bal_magics.units = pre_more; }
    else { a.units_per_wave = pre_units; if constexpr (XC != 0) a.wide_wgs = (int)pre_more; else a.units_per_split = (int)pre_more; }
    using F = SkFmt<BITS, SPARSE>;
    constexpr int NL = F::LOADS;
    constexpr int PF = (BITS == 3 && CW == 4) || (SPARSE && CW == 4) ? 2 : 4, MT = RT == 4 ? 2 : 1;
    constexpr int PFX = RT == 4 ? 2 : 4;            // units of states in flight per wave
    constexpr int CT = CW + XC;                     // columns per lane in all
    constexpr int STRIP = 16 * CT;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    typedef typename Words<CW>::type words_t;
    const int t = threadIdx.x, lane = t & 63, nwaves = BAL ? SK_BAL_WAVES : (int)(pre_rows >> 16);
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);   // scalar: the unit loop runs on SGPRs
    const int j = lane & 15, h = lane >> 4;
    const int units = a.K / 64;
    // the wave's strip, the part of the strip's units that its workgroup (BAL: its segment of the workgroup's
    // range) covers, and the wave's own units in it
    int strip = blockIdx.x, split_lo, split_hi, u0, u1;
    int seg_wave0 = 0, seg_waves = nwaves;                      // the waves that work on the same strip
    BalancedShare bs{};
    if constexpr (BAL) {
        bs = balanced_share(a.bal_q, a.bal_r, a.bal_magics.units, blockIdx.x, units, wave);
        strip = bs.strip0 + bs.mine;
        split_lo = bs.lo;
        split_hi = bs.hi;
        seg_wave0 = bs.wave0;
        seg_waves = bs.waves;
        const int upw = small_div(split_hi - split_lo + seg_waves - 1, seg_waves, 1.f / (float)seg_waves);
        u0 = min(split_hi, split_lo + (wave - seg_wave0) * upw);
        u1 = min(split_hi, u0 + upw);
    } else {
        split_lo = XC != 0 ? 0 : blockIdx.z * a.units_per_split;
        split_hi = XC != 0 ? units : min(units, split_lo + a.units_per_split);
        u0 = min(split_hi, split_lo + wave * a.units_per_wave);
        u1 = min(split_hi, u0 + a.units_per_wave);
    }
    // first column of the workgroup, of the lane's CW adjacent columns, and the lane's column in the fifth sliver
    // (a workgroup without one re-reads its first sliver there and does not write the result)
    const bool has_extra = XC != 0 && (int)blockIdx.x < a.wide_wgs;
    const int colbase = XC != 0 ? (has_extra ? 80 * (int)blockIdx.x : 80 * a.wide_wgs + 64 * ((int)blockIdx.x - a.wide_wgs))
                                : strip * STRIP;
    const int col0 = colbase + CW * j;
    const int colx = has_extra ? colbase + 16 * CW + j : colbase + j;
    // more than 32 rows: blockIdx.y takes rows 32 y .. 32 y + 31 (each block reads the strip's weights again)
    const int row0 = blockIdx.y * 32;
    const int R = min(32, a.R - row0);

    // The strip's scales and zeros ([groups][STRIP] halves each) are copied to LDS
    // once: the loop then never waits on a global load other than its prefetched
    // weights and states.  Exponent-mode scales (negative or NaN) anywhere in the
    // strip switch the whole workgroup to the exact per-weight decode.  (The copy
    // runs after the first loads have been issued, under their latency.)
    // (of the groups that the workgroup's share of K touches)
    // (BAL: the copies of the workgroup's segments one after the other; this wave's group gi is at sz_goff + gi)
    int sz_groups = 0, sz_goff = 0;
    // (16:32: the selector table is allocated statically: its LDS address is a compile-time constant)
    __shared__ __attribute__((aligned(16))) u32x4 lut_table[SPARSE ? 256 : 1];
    const char* lut = reinterpret_cast<const char*>(lut_table);
    if constexpr (SPARSE) {
        // for mask byte b, pair e = (row e, row e + 4): byte 0 picks the code byte of row e out of
        // {even nibbles, odd nibbles} by its rank among the kept rows, byte 2 that of row e + 4;
        // 0x0C yields 0.  Stored under the nibble-swapped byte (see the lookup).
        for (int b = t; b < 256; b += blockDim.x) {
            uint32_t selb[8];
            int rank = 0;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const bool k = (b >> r) & 1;
                selb[r] = k ? (uint32_t)((rank & 1) * 4 + (rank >> 1)) : 0x0Cu;
                rank += k;
            }
            u32x4 e;
#pragma unroll
            for (int q = 0; q < 4; ++q) e[q] = selb[q] | (0x0Cu << 8) | (selb[q + 4] << 16) | (0x0Cu << 24);
            lut_table[((b & 15) << 4) | (b >> 4)] = e;
        }
    }
    uint32_t* sz = reinterpret_cast<uint32_t*>(lds + nwaves * SK_WAVE_LDS + 16);      // scales, then zeros
    auto scan_scales = [&]() __attribute__((always_inline)) -> bool {
        int* flag = reinterpret_cast<int*>(lds + nwaves * SK_WAVE_LDS);
        if (t == 0) *flag = 0;
        // (BAL: the first group of the first segment -- the others start with their strip -- and where each segment's copy starts)
        int glo0 = 0, goff1 = 0, goff2 = 0;
        if constexpr (BAL) {
            const uint32_t magic = a.bal_magics.group_units;
            const int gu = a.group_units;
            glo0 = magic_div(bs.first, gu, magic);
            goff1 = magic_div(bs.first + bs.n0 - 1, gu, magic) + 1 - glo0;
            goff2 = goff1 + (bs.n1 > 0 ? magic_div(bs.n1 - 1, gu, magic) + 1 : 0);
            sz_groups = goff2 + (bs.n2 > 0 ? magic_div(bs.n2 - 1, gu, magic) + 1 : 0);
            sz_goff = bs.mine == 0 ? -glo0 : bs.mine == 1 ? goff1 : goff2;
        } else {
            glo0 = split_lo / a.group_units;
            sz_groups = (split_hi + a.group_units - 1) / a.group_units - glo0;
            sz_goff = -glo0;
        }
        __syncthreads();
        bool bad = false;
        const int n = sz_groups * (STRIP / 2);
        for (int i = t; i < n; i += blockDim.x) {
            const int g = i / (STRIP / 2), c = i % (STRIP / 2);
            int64_t at;
            if constexpr (BAL) {
                // (sums rather than selections among the three segments' values: the compiler turns a selection
                // among fields into an indexed load, which puts the whole record into scratch memory)
                const int k1 = g >= goff1 ? 1 : 0, k2 = g >= goff2 ? 1 : 0;
                const int first = glo0 - k1 * glo0;
                const int off = k1 * goff1 + k2 * (goff2 - goff1);
                at = (int64_t)(first + g - off) * a.S + (bs.strip0 + k1 + k2) * STRIP + 2 * c;
            } else {
                at = (int64_t)(glo0 + g) * a.S + colbase + ((XC != 0 && !has_extra && c >= 8 * CW) ? 2 * c - 16 * CW : 2 * c);
            }
            const uint32_t two = *reinterpret_cast<const uint32_t*>(a.scales + at);
            bad |= !(as_h2(two).x >= (h16)0.0f) || !(as_h2(two).y >= (h16)0.0f);
            sz[i] = two;
            sz[n + i] = *reinterpret_cast<const uint32_t*>(a.zeros + at);
        }
        if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) *flag = 1;
        __syncthreads();
        return *flag != 0;
    };
    bool general = false;

    char* my = lds + wave * SK_WAVE_LDS;
    float* sums = reinterpret_cast<float*>(my + 2 * SK_XBUF);   // [0..31] sum x, [32..63] sum off x

    // accumulators: acc = raw products of the current group, y = finished groups
    // (register e of tile mt is row 16 mt + 4 h + e, column j)
    // (16:32: accm = the same for the "kept" flags)
    f32x4 acc[CT][MT], accm[SPARSE ? CW : 1][MT], y[CT][MT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            acc[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            y[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (SPARSE || c == 0) accm[SPARSE ? c : 0][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    if (u0 >= u1) general = scan_scales();          // idle waves still take part in its barriers
    if (u0 < u1) {
        // ---- loaders
        // weights of unit u, CW words per load.  Lane group h needs chunk h (8 codes) of
        // each of the unit's two 32-row blocks:
        //   int4: packed row 4 blk + h;  int2: row 2 blk + h / 2, its low or high half;
        //   int3: bits 24 h .. 24 h + 23 of the block's 96-bit stream = rows {0,0,1,1}[h] and the
        //         next one, shifted right by {0, 24, 16, 40}[h]
        const int wrow = BITS == 4 ? h : (BITS == 2 ? (h >> 1) : (h >> 1));
        const int wshift = BITS == 4 ? 0 : (BITS == 2 ? 16 * (h & 1) : (h == 0 ? 0 : h == 1 ? 24 : h == 2 ? 16 : 40));
        //   16:32: every lane group loads both words of kept codes and the mask word of the block
        //          (w[3 blk], w[3 blk + 1], w[3 blk + 2])
        const uint32_t* wbase = a.matrix + (int64_t)(SPARSE ? 0 : wrow) * a.S + col0;
        const uint32_t* mbase = SPARSE ? a.mask + col0 : nullptr;
        const uint32_t* xbase = a.matrix + (int64_t)wrow * a.S + colx;
        auto load_w = [&](words_t w[NL], uint32_t wx[NL], int u) {
            const uint32_t* p = wbase + (int64_t)u * (2 * F::ROWS) * a.S;
            if constexpr (SPARSE) {
                const uint32_t* pm = mbase + (int64_t)u * 2 * a.S;
#pragma unroll
                for (int blk = 0; blk < 2; ++blk) {
                    w[3 * blk] = __builtin_nontemporal_load(reinterpret_cast<const words_t*>(p + (int64_t)(2 * blk) * a.S));
                    w[3 * blk + 1] = __builtin_nontemporal_load(reinterpret_cast<const words_t*>(p + (int64_t)(2 * blk + 1) * a.S));
                    w[3 * blk + 2] = __builtin_nontemporal_load(reinterpret_cast<const words_t*>(pm + (int64_t)blk * a.S));
                }
            } else {
#pragma unroll
                for (int i = 0; i < NL; ++i) {
                    const int row = BITS == 3 ? 3 * (i >> 1) + (i & 1) : F::ROWS * i;       // relative to the lane's first row
                    w[i] = __builtin_nontemporal_load(reinterpret_cast<const words_t*>(p + (int64_t)row * a.S));
                    if constexpr (XC != 0)
                        wx[i] = __builtin_nontemporal_load(xbase + ((int64_t)u * (2 * F::ROWS) + row) * a.S);
                }
            }
        };
        // 16:32: mask bits of the rows before the lane group's eight; selector that replicates mask byte h
        const uint32_t below = SPARSE ? (1u << (8 * h)) - 1u : 0u, rep_h = 0x01010101u * h;
        // the 8 codes of chunk h of block blk, column c
        auto chunk_bits = [&](const words_t w[NL], const uint32_t wx[NL], int blk, int c) -> uint32_t {
            auto word = [&](int idx) -> uint32_t { return c < CW ? word_of<CW>(w[idx], c < CW ? c : 0) : wx[idx]; };
            if constexpr (BITS == 3)
                return (uint32_t)((((uint64_t)word(2 * blk + 1) << 32) | word(2 * blk)) >> wshift);
            else
                return word(blk) >> wshift;
        };
        // states of unit u (8 RT rows x 128 bytes): 8 / RT lanes per row, RT 16-byte chunks
        // each; the rows of the LDS buffers beyond 8 RT stay zero
        constexpr int LPR = 8 / RT;                                   // lanes per row
        const int xm = lane / LPR, xpart = lane % LPR;
        const bool xreal = xm < R;
        const h16* xsrc = a.x + (int64_t)(row0 + min(xm, R - 1)) * a.K + xpart * (8 * RT);
        auto load_x = [&](u32x4 xr[RT], int u) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
                xr[i] = xreal ? *reinterpret_cast<const u32x4*>(xsrc + u * 64 + i * 8) : u32x4{0, 0, 0, 0};
        };
        // store a loaded unit to LDS buffer p and return its per-row sums (all lanes of a row get them)
        auto stage_x = [&](const u32x4 xr[RT], int p, float& sx, float& so) {
            const uint32_t ONES = 0x3C003C00u;
            sx = 0.f; so = 0.f;
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const u32x4 v = xr[i];
                // the k order inside the chunk that the operand decode produces (int4: 0,4,1,5,2,6,3,7)
                u32x4 q = v;
                if constexpr (BITS == 4)
                    q = u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                              __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
                if constexpr (!SPARSE) {                 // (16:32 has no offsets to remove)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sx = dot2(q[e], ONES, sx);
                        if constexpr (!PLAIN) so = dot2(q[e], F::offs(e), so);
                    }
                }
                *reinterpret_cast<u32x4*>(my + p * SK_XBUF + xm * SK_PITCH + (xpart * RT + i) * 16) = q;
            }
            if constexpr (!SPARSE) {
                // the other lanes of the row: lane ^ 1, lane ^ 2, lane ^ 4 as far as the row extends
                sx += dpp_f32<0xB1>(sx);
                so += dpp_f32<0xB1>(so);
                if constexpr (LPR >= 4) { sx += dpp_f32<0x4E>(sx); so += dpp_f32<0x4E>(so); }
                if constexpr (LPR >= 8) { sx += dpp_f32<0x141>(sx); so += dpp_f32<0x141>(so); }
            }
        };
        // rows that never receive states must read as zero
        for (int i = lane; i < 2 * SK_XBUF / 16; i += 64) *reinterpret_cast<u32x4*>(my + i * 16) = u32x4{0, 0, 0, 0};

        words_t w[PF][NL];
        uint32_t wx[PF][NL];                // (XC: the fifth column's words)
        u32x4 xr[PFX][RT];
        const uint32_t m0 = in_vgpr(BITS == 4 ? 0x000F000Fu : BITS == 2 ? 0x000C0003u : 0x00380007u);
        const uint32_t g0 = in_vgpr(BITS == 4 ? 0x64006400u : BITS == 2 ? 0x5C006400u : 0x58006400u);
        const uint32_t m1 = BITS == 4 ? in_vgpr(0x00F000F0u) : 0u, g1 = BITS == 4 ? in_vgpr(0x54005400u) : 0u;
        const uint32_t sp_nib = SPARSE ? in_vgpr(0x0F0F0F0Fu) : 0u, sp_flag = SPARSE ? in_vgpr(0x10101010u) : 0u;
        const uint32_t sp_kept = SPARSE ? in_vgpr(0x00100010u) : 0u, sp_idx = SPARSE ? in_vgpr(0x00000FF0u) : 0u;
        float gS = 0.f, gO = 0.f;           // sums of the current group so far (row lane / 2)
        float nS, nO;                       // sums of the unit staged last (the next to be multiplied)
        // scale / zero of the lane's CW columns for group gi, from the LDS copy
        h16 sc[CT], ze[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) { sc[c] = (h16)0.f; ze[c] = (h16)0.f; }
        auto load_sz = [&](int gi) {
            const h16* ps = reinterpret_cast<const h16*>(sz) + (sz_goff + gi) * STRIP + CW * j;
            const h16* pz = ps + sz_groups * STRIP;
            if constexpr (CW == 4) {
                const u32x2 s2 = *reinterpret_cast<const u32x2*>(ps), z2 = *reinterpret_cast<const u32x2*>(pz);
                sc[0] = as_h2(s2.x).x; sc[1] = as_h2(s2.x).y; sc[2] = as_h2(s2.y).x; sc[3] = as_h2(s2.y).y;
                ze[0] = as_h2(z2.x).x; ze[1] = as_h2(z2.x).y; ze[2] = as_h2(z2.y).x; ze[3] = as_h2(z2.y).y;
            } else if constexpr (CW == 2) {
                const uint32_t s1 = *reinterpret_cast<const uint32_t*>(ps), z1 = *reinterpret_cast<const uint32_t*>(pz);
                sc[0] = as_h2(s1).x; sc[1] = as_h2(s1).y; ze[0] = as_h2(z1).x; ze[1] = as_h2(z1).y;
            } else {
                sc[0] = ps[0]; ze[0] = pz[0];
            }
            if constexpr (XC != 0) { sc[CW] = ps[16 * CW + j - CW * j]; ze[CW] = pz[16 * CW + j - CW * j]; }
        };

#pragma unroll
        for (int f = 0; f < PF; ++f) load_w(w[f], wx[f], min(u0 + f, u1 - 1));
        load_x(xr[0], u0);
        general = scan_scales();
        stage_x(xr[0], 0, nS, nO);
        // set f holds unit u0 + f (f >= 1) and, for f = 0, unit u0 + PFX
#pragma unroll
        for (int f = 1; f <= PFX; ++f) load_x(xr[f % PFX], min(u0 + f, u1 - 1));

        // p: parity of the LDS buffer that holds unit u; xn: the register set with the states of unit u + 1.
        // The decode mode is a compile-time tag: one loop body per mode, no branches inside.
        auto step = [&](auto mode, int u, int p, words_t w[NL], uint32_t wx[NL], u32x4 xn[RT]) {
            constexpr bool general = decltype(mode)::value;
            if constexpr (general) {
                if (u == u0 || u % a.group_units == 0) load_sz(u / a.group_units);
            }
            gS += nS; gO += nO;
            // 2 blocks of 32 k: lane group h multiplies chunk h (8 k) of the block
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                h16x8 xa[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    xa[mt] = *reinterpret_cast<const h16x8*>(my + p * SK_XBUF + (j + 16 * mt) * SK_PITCH + (i * 4 + h) * 16);
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    if constexpr (SPARSE) {
                        const uint32_t m = word_of<CW>(w[3 * i + 2], c);
                        const uint64_t st = ((uint64_t)word_of<CW>(w[3 * i + 1], c) << 32) | word_of<CW>(w[3 * i], c);
                        // the codes of the rows before this chunk are skipped, 4 bits each (a full
                        // skip of 64 bits only happens when no row of the chunk is kept)
                        const uint32_t v = (uint32_t)(st >> ((uint32_t)__builtin_popcount(m & below) << 2));
                        const uint32_t mb4 = __builtin_amdgcn_perm(m, m, rep_h);           // mask byte h, four times
                        if constexpr (general && !PLAIN) {
                            const h16x8 wb = exact_operand_sparse(v, mb4 & 0xFFu, sc[c], ze[c]);
#pragma unroll
                            for (int mt = 0; mt < MT; ++mt)
                                acc[c][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[mt], wb, acc[c][mt], 0, 0, 0);
                        } else {
                            // (table entries sit under the nibble-swapped byte = bits 4 .. 11 of mb4)
                            const u32x4 sel = *reinterpret_cast<const u32x4*>(lut + (mb4 & sp_idx));
                            u32x4 b = sparse_operand(v, sel, sp_nib, sp_flag);
                            const u32x4 bm = u32x4{b.x & sp_kept, b.y & sp_kept, b.z & sp_kept, b.w & sp_kept};
                            if constexpr (general) {        // q 2^-24, or +-2^e, of the kept rows
                                const bool expo = !(sc[c] >= (h16)0.0f);
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const uint32_t power = ((b[e] & 0x00080008u) << 12) | (((b[e] & 0x00070007u) << 10) + 0x3C003C00u);
                                    b[e] = expo ? power & ((bm[e] << 12) - (bm[e] >> 4)) : b[e] & 0x000F000Fu;
                                }
                            }
#pragma unroll
                            for (int mt = 0; mt < MT; ++mt) {
                                acc[c][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[mt], bitcast<h16x8>(b), acc[c][mt], 0, 0, 0);
                                accm[c][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[mt], bitcast<h16x8>(bm), accm[c][mt], 0, 0, 0);
                            }
                        }
                    } else {
                        const uint32_t f = chunk_bits(w, wx, i, c);
                        h16x8 wb;
                        if constexpr (PLAIN) wb = plain_operand<BITS, general>(f, m0, m1, g0, g1, sc[c]);
                        else if constexpr (general) wb = exact_operand<BITS>(f, m0, m1, g0, g1, sc[c], ze[c]);
                        else wb = magic_operand<BITS>(f, m0, m1, g0, g1);
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            acc[c][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[mt], wb, acc[c][mt], 0, 0, 0);
                    }
                }
            }
            // refill this register set PF units ahead; move the next unit's states to LDS
            load_w(w, wx, min(u + PF, u1 - 1));
            stage_x(xn, p ^ 1, nS, nO);
            load_x(xn, min(u + 1 + PFX, u1 - 1));
            // group complete (or this wave's range ends): fold it into y
            if ((u + 1) % a.group_units == 0 || u + 1 == u1) {
                if constexpr (SPARSE && (PLAIN || !general)) {
                    if constexpr (!general) load_sz(u / a.group_units);
#pragma unroll
                    for (int c = 0; c < CW; ++c) {
                        // y += s (A - z M) with A = 2^24 (acc - accm), M = 2^20 accm
                        float ka = (float)sc[c] * 16777216.f;
                        float km = -(ka + (float)sc[c] * (float)ze[c] * 1048576.f);
                        if constexpr (general) {            // A = 2^24 acc, or z M - s acc
                            const bool expo = !(sc[c] >= (h16)0.0f);
                            km = (expo ? 1048576.f : (float)sc[c] * -1048576.f) * (float)ze[c];
                            ka = expo ? -(float)sc[c] : ka;
                        }
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                y[c][mt][e] = __builtin_fmaf(ka, acc[c][mt][e], __builtin_fmaf(km, accm[c][mt][e], y[c][mt][e]));
                            acc[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                            accm[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
                    }
                } else {
                if (xpart == 0) { sums[xm] = gS; sums[32 + xm] = gO; }
                if constexpr (!general) load_sz(u / a.group_units);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const f32x4 s4 = *reinterpret_cast<const f32x4*>(&sums[16 * mt + 4 * h]);
                    const f32x4 o4 = *reinterpret_cast<const f32x4*>(&sums[32 + 16 * mt + 4 * h]);
#pragma unroll
                    for (int c = 0; c < CT; ++c) {
                        if constexpr (general && PLAIN) {   // y += s (acc - z X), or z X - s acc
                            const bool expo = !(sc[c] >= (h16)0.0f);
                            const float ka = expo ? -(float)sc[c] : (float)sc[c], kx = (expo ? 1.f : -(float)sc[c]) * (float)ze[c];
#pragma unroll
                            for (int e = 0; e < 4; ++e) y[c][mt][e] = __builtin_fmaf(ka, acc[c][mt][e], __builtin_fmaf(kx, s4[e], y[c][mt][e]));
                        } else {
                            const float sf = general ? 1.f : (float)sc[c];
                            const float z = general ? 0.f : (float)ze[c];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float off = general ? 0.f : PLAIN ? z * s4[e] : o4[e] + z * s4[e];
                                y[c][mt][e] += sf * (acc[c][mt][e] - off);
                            }
                        }
                        acc[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                }
                }
                gS = 0.f; gO = 0.f;
            }
        };
        auto run = [&](auto mode) {
            constexpr int UN = PF > PFX ? PF : PFX;      // register sets rotate with periods PF and PFX
            for (int u = u0; u < u1; u += UN) {
#pragma unroll
                for (int f = 0; f < UN; ++f) {
                    if (f > 0 && u + f >= u1) break;
                    step(mode, u + f, f & 1, w[f % PF], wx[f % PF], xr[(f + 1) % PFX]);
                }
            }
        };
        if (general) run(std::integral_constant<bool, true>{});
        else run(std::integral_constant<bool, false>{});
    }

    // ---- sum the waves' partial tiles through LDS (tile: [16 MT rows][16 CW columns] fp32)
    __syncthreads();
    constexpr int TILE = MT * 16 * STRIP;
    float* red = reinterpret_cast<float*>(lds);
    auto tile_at = [&](float* base, int mt, int e) { return base + ((mt * 16 + 4 * h + e) * 16 + j) * CT; };
    if constexpr (BAL) {
        // every wave leaves its tile; the first wave of each segment adds up its segment's, in wave order
        float* dst = red + wave * TILE;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < CT; ++c) tile_at(dst, mt, e)[c] = y[c][mt][e];
        __syncthreads();
        if (wave != seg_wave0) return;
        for (int w = seg_wave0 + 1; w < seg_wave0 + seg_waves; ++w) {
            float* src = red + w * TILE;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < CT; ++c) y[c][mt][e] += tile_at(src, mt, e)[c];
        }
    }
    for (int s = BAL ? 0 : (nwaves >> 1); s >= 1; s >>= 1) {
        if (wave >= s && wave < 2 * s) {
            float* dst = red + (wave - s) * TILE;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < CT; ++c) tile_at(dst, mt, e)[c] = y[c][mt][e];
        }
        __syncthreads();
        if (wave < s) {
            float* src = red + wave * TILE;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < CT; ++c) y[c][mt][e] += tile_at(src, mt, e)[c];
        }
        __syncthreads();
    }
    if (BAL || wave == 0) {
        // (BAL: a strip shared by two workgroups -- never more: a workgroup's range is at least a strip long)
        const bool shared = BAL ? (split_lo > 0 || split_hi < units) : gridDim.z > 1;
        if (shared) {
            // hand-over between the workgroups of a strip: write-through stores of the partial tile
            // (value v of lane l at (v * 64 + l) * 4), a device-scope counter, and whoever finds all
            // the others counted reads every partial back in split order -- one summation order
            // whoever is last -- and goes on to write the strip.  One wave: no barrier involved.
            constexpr int NV = CW * MT * 4, THROUGH = 17;                 // sc0 | sc1: straight to memory
            const int tile = BAL ? strip : blockIdx.y * gridDim.x + blockIdx.x, ks = BAL ? 2 : gridDim.z;
            const int my_split = BAL ? (split_lo > 0 ? 1 : 0) : blockIdx.z;
            char* const slots = reinterpret_cast<char*>(a.part) + (int64_t)tile * ks * (NV * 256);
            const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc(
                slots + (int64_t)my_split * (NV * 256), 0, NV * 256, 0x00020000);
#pragma unroll
            for (int c = 0; c < CW; ++c)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = y[c][mt][e];       // (a bit_cast straight from the vector element reads element 0)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), mine,
                                                              (((c * MT + mt) * 4 + e) * 64 + lane) * 4, 0, THROUGH);
                    }
            // (the fences keep the compiler from moving the counter update ahead of the stores, or the
            // loads below ahead of it; the hardware side is the wait for the stores' acknowledgement)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_s_waitcnt(0);
            int arrived = 0;
            if (lane == 0) arrived = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            arrived = __builtin_amdgcn_readfirstlane(arrived);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (arrived != ks - 1) return;
            if (lane == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int c = 0; c < CW; ++c)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) y[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int sp = 0; sp < ks; ++sp) {
                const __amdgpu_buffer_rsrc_t theirs = __builtin_amdgcn_make_buffer_rsrc(
                    slots + (int64_t)sp * (NV * 256), 0, NV * 256, 0x00020000);
#pragma unroll
                for (int c = 0; c < CW; ++c)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            y[c][mt][e] += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                theirs, (((c * MT + mt) * 4 + e) * 64 + lane) * 4, 0, THROUGH));
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = mt * 16 + 4 * h + e;
                if (m < R) {
                    h16* o = a.outs + (int64_t)(row0 + m) * a.S + col0;
#pragma unroll
                    for (int c = 0; c < CW; ++c) {
                        float v = y[c][mt][e];
                        if (a.accumulate) v += (float)o[c];
                        o[c] = (h16)v;
                    }
                    if (XC != 0 && has_extra) {
                        h16* ox = a.outs + (int64_t)(row0 + m) * a.S + colx;
                        float v = y[CT - 1][mt][e];
                        if (a.accumulate) v += (float)ox[0];
                        ox[0] = (h16)v;
                    }
                }
            }
    }
}

// LDS of the unsplit kernel: per wave its units, then the scales and zeros of all of the strip's groups
static size_t skinny_lds_bytes(int cw, int waves, int groups) { return (size_t)waves * SK_WAVE_LDS + 16 + (size_t)groups * 16 * cw * 4; }
static constexpr size_t skinny_lds_limit(bool sparse) { return 150 * 1024 - (sparse ? 4096 : 0); }      // (16:32: 4 KB of static LDS for the selector table)

template <int BITS, int CW, bool SPARSE>
static bool launch_skinny(const SkinnyArgs& a, int waves, int ksplit, bool plain, hipStream_t st) {
    const int strips = a.S / (16 * CW);
    const int rt = ((a.R > 32 ? 32 : a.R) + 7) / 8;
    int groups = (a.K / 64 + a.group_units - 1) / a.group_units;
    if (ksplit > 1) groups = std::min(groups, (a.units_per_split + a.group_units - 1) / a.group_units + 1);
    size_t lds = skinny_lds_bytes(CW, waves, groups);
    const size_t red = (size_t)(waves / 2) * (rt <= 2 ? 1 : 2) * 16 * 16 * CW * 4;
    if (red > lds) lds = red;
    if (lds > skinny_lds_limit(SPARSE)) return false;
    const dim3 grid(strips, (a.R + 31) / 32, ksplit), block(waves * 64);
    plain = plain && rt > 2;
    if (noting("skinny_kernel<bits=%d,%s,columns_per_lane=%d,row_tiles=%d%s> strips=%d row_blocks=%u ksplit=%d waves=%d", BITS,
               SPARSE ? "16:32" : "dense", CW, rt <= 1 ? 1 : (rt <= 2 ? 2 : 4), plain ? ",plain" : "", strips, grid.y, ksplit, waves))
        return true;
    auto go = [&](auto kernel, int slot) {
        // more than 64 KB of dynamic LDS has to be requested once per kernel and device
        static std::atomic<uint64_t> done[4];
        int dev = 0;
        hipGetDevice(&dev);
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done[slot].load(std::memory_order_relaxed) & bit)) {
            hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                150 * 1024);
            done[slot].fetch_or(bit, std::memory_order_relaxed);
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, st, a.matrix, a.x, a.scales, a.zeros, a.S, a.K, a.group_units, a.units_per_wave, (uint32_t)a.R | (uint32_t)waves << 16,
                           (uint32_t)a.units_per_split, a);
    };
    if constexpr (!(SPARSE && CW == 4)) {                           // (which up to 16 rows have alone)
        if (plain) { go(skinny_kernel<BITS, CW, 4, SPARSE, false, 0, true>, 3); return true; }
    }
    if (rt <= 1) go(skinny_kernel<BITS, CW, 1, SPARSE>, 0);
    else if (rt <= 2) go(skinny_kernel<BITS, CW, 2, SPARSE>, 1);
    else go(skinny_kernel<BITS, CW, 4, SPARSE>, 2);
    return true;
}

// The balanced launch: 64-column strips, eight waves, `wgs` workgroups that share strips x units evenly.
// Partial tiles of the strips that two workgroups share: two slots per strip in `part`, one counter per strip.
constexpr int SK_BAL_WGS = 256;
static_assert(SK_BAL_WGS == 1 << 8, "balanced_share divides by it with a shift");
static size_t skinny_balanced_part_bytes(int64_t S) { return (size_t)(S / 64) * 2 * (4 * 2 * 4 * 256); }
// Where it pays (8 and 16 rows, K = 3072 ... 14336, us, a workgroup per strip / shared): int4 K=5120, S=20480 19.1 / 16.6,
// K=8192, S=18432 27.4 / 21.0, K=3072, S=20480 13.8 / 12.9; 16:32 K=5120, S=20480 29.5 / 24.5, K=8192, S=18432 43.5 / 31.0;
// beyond a quarter more strips than CUs only on a long K, where a workgroup per strip means eight waves each and two
// rounds (K=12288, S=28672 48.5 / 39.8, K=10240, S=24576 39.0 / 30.9; K=8192, S=22016 28.7 / 29.3 and K=4096, S=28672
// 17.2 / 18.0 do not gain).  17 ... 32 rows, whose accumulators fill the register file, lose (K=2048, S=20480 14.8 / 15.9).
static bool balanced_shape(int64_t R, int64_t K, int64_t S) {
    const int64_t strips = S / 64, units = K / 64;
    if (R < 2 || R > 16 || S % 64 != 0 || strips <= SK_BAL_WGS || strips >= 2 * SK_BAL_WGS || strips * units >= (1ll << 22)) return false;
    return units >= (strips <= SK_BAL_WGS * 5 / 4 ? 48 : 160);
}
template <int BITS, bool SPARSE>
static bool launch_skinny_balanced(SkinnyArgs a, hipStream_t st) {
    constexpr int CW = 4, WAVES = SK_BAL_WAVES;
    const int strips = a.S / 64, units = a.K / 64;
    const int rt = (a.R + 7) / 8;
    const int64_t total = (int64_t)strips * units;
    a.bal_q = (int)(total / SK_BAL_WGS);
    a.bal_r = (int)(total % SK_BAL_WGS);
    a.bal_magics = {div_magic((uint32_t)units), div_magic((uint32_t)a.group_units)};
    // scales in LDS: a workgroup's range is less than two strips long and touches at most three
    const int groups = 2 * ((units + a.group_units - 1) / a.group_units) + 3;
    size_t lds = (size_t)WAVES * SK_WAVE_LDS + 16 + (size_t)groups * 16 * CW * 4;
    const size_t red = (size_t)WAVES * 16 * 16 * CW * 4;
    if (red > lds) lds = red;
    if (lds > 150 * 1024 - (SPARSE ? 4096 : 0)) return false;
    const dim3 grid(SK_BAL_WGS, 1, 1), block(WAVES * 64);
    if (noting("skinny_kernel<bits=%d,%s,columns_per_lane=%d,row_tiles=%d,balanced> strips=%d row_blocks=1 workgroups=%d waves=%d",
               BITS, SPARSE ? "16:32" : "dense", CW, rt <= 1 ? 1 : 2, strips, SK_BAL_WGS, WAVES))
        return true;
    auto go = [&](auto kernel) {
        static std::atomic<uint64_t> done;
        int dev = 0;
        hipGetDevice(&dev);
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done.load(std::memory_order_relaxed) & bit)) {
            hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                150 * 1024);
            done.fetch_or(bit, std::memory_order_relaxed);
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, st, a.matrix, a.x, a.scales, a.zeros, a.S, a.K, a.group_units, a.bal_q, (uint32_t)a.R | (uint32_t)a.bal_r << 16,
                           a.bal_magics.units, a);
    };
    if (rt <= 1) go(skinny_kernel<BITS, CW, 1, SPARSE, true>);
    else go(skinny_kernel<BITS, CW, 2, SPARSE, true>);            // (up to 16 rows: balanced_shape)
    return true;
}

// Between 256 and 320 strips of 64 columns: 256 workgroups of four or five slivers of 16 columns each, so that
// every CU has one workgroup and none a second (dense formats, up to 16 rows).
// int3 and int2 (8 and 16 rows, us, a workgroup per strip / shared strips / slivers): K=5120, S=20480 int3 22.5 / 19.3 / 17.8,
// int2 21.2 / 18.2 / 16.6; K=8192, S=18432 int3 32.4 / 24.1 / 24.2; K=14336, S=19200 int3 56.2 / 44.8 / 38.8, int2 53.0 / 41.3 /
// 34.6.  int4, whose words carry a third more bytes per unit, does better with shared strips (K=5120, S=20480 18.5 with
// slivers), and so does 16:32, which has no registers for a fifth column.
static bool sliver_shape(int bits, int64_t R, int64_t K, int64_t S, bool sparse) {
    const int64_t slivers = S / 16;
    return !sparse && bits != 4 && R >= 2 && R <= 16 && S % 64 == 0 && slivers > 4 * SK_BAL_WGS && slivers <= 5 * SK_BAL_WGS &&
           K / 64 >= 48;
}
template <int BITS>
static bool launch_skinny_slivers(SkinnyArgs a, hipStream_t st) {
    constexpr int CW = 4, CT = 5, WAVES = 8;
    const int rt = (a.R + 7) / 8;
    a.wide_wgs = a.S / 16 - 4 * SK_BAL_WGS;
    a.units_per_split = a.K / 64;
    a.units_per_wave = (a.units_per_split + WAVES - 1) / WAVES;
    const int groups = (a.K / 64 + a.group_units - 1) / a.group_units;
    size_t lds = (size_t)WAVES * SK_WAVE_LDS + 16 + (size_t)groups * 16 * CT * 4;
    const size_t red = (size_t)(WAVES / 2) * 16 * 16 * CT * 4;
    if (red > lds) lds = red;
    if (lds > 150 * 1024) return false;
    const dim3 grid(SK_BAL_WGS, 1, 1), block(WAVES * 64);
    if (noting("skinny_kernel<bits=%d,dense,columns_per_lane=4+1,row_tiles=%d> strips=%d (%d of 80 columns, the others of 64) "
               "row_blocks=1 ksplit=1 waves=%d", BITS, rt <= 1 ? 1 : 2, SK_BAL_WGS, a.wide_wgs, WAVES))
        return true;
    auto go = [&](auto kernel) {
        static std::atomic<uint64_t> done;
        int dev = 0;
        hipGetDevice(&dev);
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done.load(std::memory_order_relaxed) & bit)) {
            hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                150 * 1024);
            done.fetch_or(bit, std::memory_order_relaxed);
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, st, a.matrix, a.x, a.scales, a.zeros, a.S, a.K, a.group_units, a.units_per_wave, (uint32_t)a.R | (uint32_t)WAVES << 16,
                           (uint32_t)a.wide_wgs, a);
    };
    if (rt <= 1) go(skinny_kernel<BITS, CW, 1, false, false, 1>);
    else go(skinny_kernel<BITS, CW, 2, false, false, 1>);
    return true;
}

template <int BITS, bool SPARSE = false>
static bool launch_skinny_cw(const SkinnyArgs& a, int cw, int waves, int ksplit, bool plain, hipStream_t st) {
    if (cw == 4) return launch_skinny<BITS, 4, SPARSE>(a, waves, ksplit, plain, st);
    if (cw == 2) return launch_skinny<BITS, 2, SPARSE>(a, waves, ksplit, plain, st);
    return launch_skinny<BITS, 1, SPARSE>(a, waves, ksplit, plain, st);
}

// Columns per lane of the unsplit kernel: the widest strips (64, 32 or 16 columns) that still give at
// least 256 workgroups, else at least 128 (narrow strips use half a cache line per packed row).
static int unsplit_cw(int64_t R, int64_t S, bool sparse) {
    int cw = 1;
    // (more than 32 rows run as two or three row blocks per strip, each a workgroup: the widest strips -- within what
    // the format's registers allow -- that give one round of 128 ... 256 workgroups, where there are such: K=2048,
    // S=8192, 40 rows in 256 workgroups of 64 columns instead of 512 of 32)
    if (R > 32) {
        const int64_t blocks = (R + 31) / 32;
        int64_t best = 0;
        for (const int c : {4, 2, 1}) {
            if (sparse && c == 4) continue;
            const int64_t wgs = S / (16 * c) * blocks;
            if (S % (16 * c) == 0 && wgs >= 128 && wgs <= 256 && wgs > best) { best = wgs; cw = c; }
        }
        if (best != 0) return cw;
    }
    // (64-column strips as soon as they give more than half a round of workgroups: 129 ... 255 of them finish in one
    // round where twice as many 32-column strips need two -- up to 16 rows, us: K=8192, S=12288 21.5 -> 17.4; K=14336,
    // S=14336 38.3 -> 25.5; K=4096, S=10240 12.9 -> 11.9; 16:32, K=8192, S=12288 32.8 -> 26.0)
    const int prefer[4][2] = {{4, 129}, {2, 256}, {4, 128}, {2, 128}};       // {columns per lane, workgroups}
    for (const auto& c : prefer)
        if (S % (16 * c[0]) == 0 && S / (16 * c[0]) >= c[1]) { cw = c[0]; break; }
    // (16:32 with more than 16 rows: four columns per lane would not fit the register file)
    if (sparse && R > 16 && cw == 4) cw = 2;
    return cw;
}

// Split-K plan of the few-row kernel: when even 32-column strips would give fewer than 192 workgroups,
// 64-column strips with as many workgroups per strip as come closest to one per CU, each with at least
// six units per wave -- if that makes at least as many workgroups as the unsplit choice of narrower
// strips (with more than 16 rows, where wide strips matter more: half as many).  `part_bytes`: room for
// the partial tiles (0: no split).
struct SkinnySplit { int cw, ksplit; size_t tiles, part_bytes; };
static SkinnySplit plan_skinny_split(int64_t R, int64_t K, int64_t S, bool sparse) {
    SkinnySplit p{0, 1, 0, 0};
    if (S % 64 != 0 || R < 2 || R > 96) return p;
    const int64_t row_blocks = (R + 31) / 32, units = K / 64;
    if (S / 32 * row_blocks >= 192) return p;
    const int cw = sparse && R > 16 ? 2 : 4;
    const int64_t wgs = S / (16 * cw) * row_blocks;
    int64_t ks = std::min<int64_t>(256 / wgs, units / (8 * 6));
    if ((R > 16 ? 2 : 1) * wgs * ks < S / (16 * unsplit_cw(R, S, sparse)) * row_blocks) ks = 1;
    const int64_t forced = tuning(TUNE_MM_SPLIT);
    if (forced >= 1) ks = std::min<int64_t>(forced, std::max<int64_t>(1, units / 16));
    if (ks < 2 || wgs > 1024) return p;
    p.cw = cw;
    p.ksplit = (int)ks;
    p.tiles = (size_t)wgs;
    p.part_bytes = (size_t)wgs * ks * (cw * 2 * 4 * 256);       // up to 32 rows x 16 cw columns of fp32 per partial
    return p;
}

// Waves of the unsplit kernel.  Four split K when there are more workgroups than CUs (three of them fit a CU) and K
// is short (each wave should walk a dozen units or more), eight otherwise -- also at exactly one
// workgroup per CU, where eight waves keep twice the bytes in flight (K=5120, S=16384, 8 rows:
// 14.6 -> 12.0 us; K=S=8192: 16.5 -> 12.3 us; 320 and 448 strips: 17.7 against 22.2, 27 against 32)
static int unsplit_waves(int64_t S, int cw, int64_t units) { return S / (16 * cw) > 256 && units < 160 ? 4 : 8; }

// Do the scales of a strip's groups, or of those of a share of K, leave the LDS room for the waves' units?  (a group that is not known: the
// smallest)
static bool few_row_groups_fit(int64_t R, int64_t K, int64_t S, bool sparse, int64_t group_units) {
    const int64_t units = K / 64, gu = std::max<int64_t>(1, std::min(group_units, units)), groups = (units + gu - 1) / gu;
    auto fits = [&](int cw, int waves, int64_t n) { return skinny_lds_bytes(cw, waves, (int)n) <= skinny_lds_limit(sparse); };
    const SkinnySplit p = plan_skinny_split(R, K, S, sparse);
    if (p.ksplit > 1) {
        const int64_t share = (units + p.ksplit - 1) / p.ksplit;
        if (fits(p.cw, 8, std::min(groups, (share + gu - 1) / gu + 1))) return true;
    }
    const int cw = unsplit_cw(R, S, sparse);
    return fits(cw, unsplit_waves(S, cw, units), groups);
}

bool few_rows_serve(int bits, bool sparse, int64_t R, int64_t K, int64_t S, int64_t group_units) {
    if (!sparse && matvec_takes_rows(R, K, S)) return true;
    if (few_row_groups_fit(R, K, S, sparse, group_units)) return true;
    for (const int b : {4, 3, 2})
        if ((sparse ? b == 4 : bits == 0 || b == bits) && (R < 17 || !wide_serves(b, sparse, R, K, S, std::max<int64_t>(1, group_units)))) return false;
    return true;
}

size_t skinny_workspace_bytes(int bits, int64_t R, int64_t K, int64_t S, bool sparse, int64_t group_units, RowsCall call) {
    const SkinnySplit p = plan_skinny_split(R, K, S, sparse);
    size_t wide = wide_workspace_bytes(bits, R, K, S, sparse, group_units, call);
    // (a product that falls through skinny_rows)
    if (call == FOR_MATMUL && wide == 0 && R >= 17 && R <= FEW_ROWS_MAX && !few_row_groups_fit(R, K, S, sparse, group_units))
        wide = wide_workspace_bytes(bits, R, K, S, sparse, group_units, ROUNDED);
    const size_t balanced = balanced_shape(R, K, S) ? skinny_balanced_part_bytes(S) : 0;
    return std::max(std::max<size_t>(p.ksplit > 1 ? p.part_bytes : 0, wide), balanced);
}

// Product of 2 <= R <= 96 rows with a dense or (sparse_mask != nullptr) 16:32 sparse int4 matrix; beyond that
// the tile kernels are faster.  Returns false when the shape is not one this kernel takes (the caller then
// uses the general kernels).
bool skinny_rows(int bits, h16* outs, const uint32_t* matrix, const h16* x, const h16* scales, const h16* zeros,
                 int64_t R, int64_t K, int64_t S, int64_t group_size, bool accumulate, hipStream_t st,
                 const uint32_t* sparse_mask, void* workspace, size_t workspace_bytes, RowsCall call) {
    if (R < 2 || R > SK_WIDE_MAX_ROWS || S % 16 != 0 || K % 64 != 0 || K > (1 << 30) || S > (1 << 28)) return false;
    if (sparse_mask && bits != 4) return false;
    SkinnyArgs a;
    a.outs = outs; a.matrix = matrix; a.mask = sparse_mask; a.x = x; a.scales = scales; a.zeros = zeros;
    a.R = (int)R; a.K = (int)K; a.S = (int)S;
    const int64_t gu = group_size / 64;
    a.group_units = (int)(gu > 0x7FFFFFF ? 0x7FFFFFF : gu);
    a.accumulate = accumulate ? 1 : 0;
    a.part = nullptr;
    a.counters = nullptr;
    a.bal_q = 0; a.bal_r = 0;
    a.wide_wgs = 0;
    // 17 rows and more: the kernel whose waves share the staged states, where its plan says so
    if (wide_rows(bits, a, call, workspace, workspace_bytes, st)) return true;
    if (R > FEW_ROWS_MAX) return false;
    int cw = unsplit_cw(R, S, sparse_mask != nullptr);
    {   // (tuning: columns per lane of the few-row kernel where the shape allows them)
        const int64_t forced_cw = tuning(TUNE_MV_LK);
        if ((forced_cw == 1 || forced_cw == 2 || (forced_cw == 4 && !(sparse_mask && R > 16))) && S % (16 * forced_cw) == 0)
            cw = (int)forced_cw;
    }
    const int units = (int)(K / 64);
    int waves = (int)tuning(TUNE_MV_WAVES);
    if (waves != 2 && waves != 4 && waves != 8) waves = unsplit_waves(S, cw, units);
    while (waves > 1 && units < 2 * waves) waves >>= 1;
    auto launch = [&](int cw_, int waves_, int ksplit_) {
        a.units_per_wave = (a.units_per_split + waves_ - 1) / waves_;
        if (sparse_mask) return launch_skinny_cw<4, true>(a, cw_, waves_, ksplit_, call == EXACT_SUMS, st);
        if (bits == 4) return launch_skinny_cw<4>(a, cw_, waves_, ksplit_, call == EXACT_SUMS, st);
        if (bits == 3) return launch_skinny_cw<3>(a, cw_, waves_, ksplit_, call == EXACT_SUMS, st);
        return launch_skinny_cw<2>(a, cw_, waves_, ksplit_, call == EXACT_SUMS, st);
    };
    // split-K across workgroups where the plan asks for it and the scratch half of the workspace has room
    // for the partial tiles (per-strip counters: last page of the half that is kept zero)
    a.part = nullptr;
    a.counters = nullptr;
    const SkinnySplit sp = plan_skinny_split(R, K, S, sparse_mask != nullptr);
    const WorkspaceParts ws = workspace_parts(workspace, workspace_bytes);
    if (sp.ksplit > 1 && ws.counters != nullptr && ws.scratch_bytes >= sp.part_bytes) {
        a.units_per_split = (units + sp.ksplit - 1) / sp.ksplit;
        a.counters = reinterpret_cast<int*>(ws.counters);
        a.part = reinterpret_cast<float*>(ws.scratch);
        const int ksplit = (units + a.units_per_split - 1) / a.units_per_split;          // no empty split
        if (launch(sp.cw, 8, ksplit)) return true;
    }
    a.units_per_split = units;
    // a quarter more 64-column strips than CUs at most: a workgroup per CU, of 64 or 80 columns
    if (tuning(TUNE_NO_BALANCE) == 0 && tuning(TUNE_MV_LK) == 0 && sliver_shape(bits, R, K, S, sparse_mask != nullptr)) {
        const bool ok = bits == 3 ? launch_skinny_slivers<3>(a, st) : launch_skinny_slivers<2>(a, st);
        if (ok) return true;
    }
    // more 64-column strips than CUs, fewer than twice as many: one workgroup per CU, the strips' units shared evenly
    // (16:32 with more than 16 rows has no 64-column strips)
    if (cw == 4 && tuning(TUNE_NO_BALANCE) == 0 && balanced_shape(R, K, S) && ws.counters != nullptr &&
        ws.scratch_bytes >= skinny_balanced_part_bytes(S)) {
        a.counters = reinterpret_cast<int*>(ws.counters);
        a.part = reinterpret_cast<float*>(ws.scratch);
        a.units_per_wave = 0;
        const bool ok = sparse_mask ? launch_skinny_balanced<4, true>(a, st)
                      : bits == 4 ? launch_skinny_balanced<4, false>(a, st)
                      : bits == 3 ? launch_skinny_balanced<3, false>(a, st) : launch_skinny_balanced<2, false>(a, st);
        if (ok) return true;
        a.counters = nullptr;
        a.part = nullptr;
    }
    // (so many groups that their scales do not fit the LDS beside the waves' units: narrower strips, where the matvec entry would run an
    // element at a time else -- us, so / now: int4, g=64, K=25344, S=27648, 48 elements 2945 / 378, K=22784, S=18688, 368 elements
    // 16601 / 1435; four waves on strips of 64 columns take 402 and 1447)
    for (; cw >= 1; cw >>= 1) {
        if (launch(cw, waves, 1)) return true;
        if (call != EXACT_SUMS || R < 17) break;
    }
    // a long K with small groups, whose scales do not fit the LDS: the matmul entry's tile kernels round the weights too
    return call == FOR_MATMUL && wide_rows(bits, a, ROUNDED, workspace, workspace_bytes, st);
}

}  // namespace i4
