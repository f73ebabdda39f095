// Pack / unpack / dequantise helpers for the packed weight formats.  These are
// integer kernels bound by HBM traffic: one thread owns one (32-row block,
// column) cell, lanes run along the column index so every global access of the
// [rows, S] matrices is coalesced.
#include "common.h"

#include <algorithm>
#include <mutex>

namespace i4 {

// 32 codes of one column, blocks of 32 rows: the shared decode step.
template <int BITS, bool SPARSE>
__device__ __forceinline__ void decode_block32(const uint32_t* __restrict__ matrix,
                                               const uint32_t* __restrict__ mask, int64_t S,
                                               int64_t blk, int64_t s, uint32_t codes[32],
                                               uint32_t& keep) {
    keep = 0xFFFFFFFFu;
    if constexpr (SPARSE) {
        const uint32_t lo = matrix[(2 * blk) * S + s], hi = matrix[(2 * blk + 1) * S + s];
        uint64_t v = (uint64_t)lo | ((uint64_t)hi << 32);
        keep = mask[blk * S + s];
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const bool k = (keep >> t) & 1u;
            codes[t] = k ? (uint32_t)(v & 0xF) : 0u;
            v >>= k ? 4 : 0;
        }
    } else if constexpr (BITS == 3) {
        const uint32_t w0 = matrix[(3 * blk) * S + s], w1 = matrix[(3 * blk + 1) * S + s],
                       w2 = matrix[(3 * blk + 2) * S + s];
        const uint64_t lo = (uint64_t)w0 | ((uint64_t)w1 << 32);   // stream bits 0..63
        const uint64_t hi = (uint64_t)w1 | ((uint64_t)w2 << 32);   // stream bits 32..95
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const int pos = 3 * t;
            codes[t] = pos + 3 <= 64 ? (uint32_t)(lo >> pos) & 7u : (uint32_t)(hi >> (pos - 32)) & 7u;
        }
    } else {
        constexpr int PER = 32 / BITS;
#pragma unroll
        for (int i = 0; i < BITS; ++i) {
            uint32_t v = matrix[(BITS * blk + i) * S + s];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                codes[i * PER + j] = v & ((1u << BITS) - 1u);
                v >>= BITS;
            }
        }
    }
}

template <int BITS, bool SPARSE>
__global__ __launch_bounds__(256) void unpack_kernel(uint8_t* __restrict__ codes_out,
                                                     uint8_t* __restrict__ keep_out,
                                                     const uint32_t* __restrict__ matrix,
                                                     const uint32_t* __restrict__ mask, int64_t K,
                                                     int64_t S) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, blk = blockIdx.y;
    if (s >= S) return;
    uint32_t codes[32], keep;
    decode_block32<BITS, SPARSE>(matrix, mask, S, blk, s, codes, keep);
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        codes_out[(blk * 32 + t) * S + s] = (uint8_t)codes[t];
        if (keep_out) keep_out[(blk * 32 + t) * S + s] = (uint8_t)((keep >> t) & 1u);
    }
}

// The same for four adjacent columns per thread (S a multiple of 4): a row's four codes leave as one 32-bit
// store, a wave's store is 256 contiguous bytes of a row instead of 64 (K = S = 16384, int4: 87 -> 76 us).
template <int BITS, bool SPARSE>
__global__ __launch_bounds__(256) void unpack4_kernel(uint8_t* __restrict__ codes_out,
                                                      uint8_t* __restrict__ keep_out,
                                                      const uint32_t* __restrict__ matrix,
                                                      const uint32_t* __restrict__ mask, int64_t K,
                                                      int64_t S) {
    const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4, blk = blockIdx.y;
    if (s >= S) return;
    uint32_t out[32], kept[32];
#pragma unroll
    for (int t = 0; t < 32; ++t) { out[t] = 0u; kept[t] = 0u; }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        uint32_t codes[32], keep;
        decode_block32<BITS, SPARSE>(matrix, mask, S, blk, s + c, codes, keep);
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            out[t] |= (codes[t] & 0xFFu) << (8 * c);
            kept[t] |= ((keep >> t) & 1u) << (8 * c);
        }
    }
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        *reinterpret_cast<uint32_t*>(codes_out + (blk * 32 + t) * S + s) = out[t];
        if (keep_out) *reinterpret_cast<uint32_t*>(keep_out + (blk * 32 + t) * S + s) = kept[t];
    }
}

template <int BITS, bool SPARSE>
__global__ __launch_bounds__(256) void dequantize_kernel(h16* __restrict__ w_out,
                                                         const uint32_t* __restrict__ matrix,
                                                         const uint32_t* __restrict__ mask,
                                                         const h16* __restrict__ scales,
                                                         const h16* __restrict__ zeros, int64_t K,
                                                         int64_t S, int64_t group_size) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, blk = blockIdx.y;
    if (s >= S) return;
    uint32_t codes[32], keep;
    decode_block32<BITS, SPARSE>(matrix, mask, S, blk, s, codes, keep);
    const int64_t gi = (blk * 32) / group_size;      // group_size is a multiple of 64
    const h16 sc = scales[gi * S + s], ze = zeros[gi * S + s];
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        h16 w = dequant_code<BITS>(codes[t], sc, ze);
        if (SPARSE && !((keep >> t) & 1u)) w = (h16)0.0f;
        w_out[(blk * 32 + t) * S + s] = w;
    }
}

// codes uint8 [K, S] -> packed words, LSB-first bitstream of 32 codes per block
template <int BITS>
__global__ __launch_bounds__(256) void dense_pack_kernel(uint32_t* __restrict__ matrix_out,
                                                         const uint8_t* __restrict__ codes_in,
                                                         int64_t K, int64_t S) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, blk = blockIdx.y;
    if (s >= S) return;
    uint64_t lo = 0, hi = 0;                          // stream bits 0..63 and 64..127
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        const uint64_t c = codes_in[(blk * 32 + t) * S + s] & ((1u << BITS) - 1u);
        const int pos = BITS * t;
        if (pos < 64) {
            lo |= c << pos;
            if (pos + BITS > 64) hi |= c >> (64 - pos);
        } else {
            hi |= c << (pos - 64);
        }
    }
    const uint32_t w[4] = {(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
#pragma unroll
    for (int i = 0; i < BITS; ++i) matrix_out[(BITS * blk + i) * S + s] = w[i];
}

// 16:32 packer.  Inputs are in the [S, K] orientation (row = output column), outputs have lanes along the column
// index, so the job is a transposition.  It is done on the outputs, which are 3 / 16 of the inputs' bytes: a workgroup
// takes a tile of 16 LANES input rows x COLS columns, LANES threads along K and PASSES loads of each input per thread (a
// load: half a 32-row cell, 16 bytes), a wave's load is whole runs of consecutive bytes of a column, and the packed words
// go through LDS, from where they are stored along the columns.  Kept codes are compacted eight rows at a time: keep flags
// gathered by a multiply, code bytes moved to the front by v_perm with selectors from a 256-entry table, squeezed to
// nibbles; the two lanes of a cell exchange rank, mask and one word each.  Consecutive workgroups walk along K, so that the
// runs in flight are consecutive in memory.
// Bound by memory traffic.  A kernel with one 128-byte line of each input per thread, lanes K bytes apart, and this one,
// whose loads are non-temporal (every byte is read once), us a launch:
//   K x S                    16384 x 16384   15968 x 16385   8192 x 8192   11008 x 4096   1024 x 1024
//   a line per thread          146 ... 164             184            49             36           5.8
//   this kernel (5.5 TB/s)             116             127            28             20           3.9
// The tile follows K: the fewest lanes that span it, at most 32, so that a tile is more than half full whatever K is.
// A line per thread / 32 lanes and eight loads at any K / the fewest lanes:
//   S = 2^20, K = 32: 15 / 80 / 14; K = 64: 32 / 82 / 27; S = 2^18, K = 128: 21 / 26 / 15; S = 4096, K = 64: 3.4 / 4.6 / 3.3 us.
// Two loads of each input in flight per thread, four at 32 lanes, so that a tile has at least 32 columns and a store
// fills whole lines.  Eight leave a small matrix to too few workgroups (1024 x 1024 5.2 us, 8192 x 63 5.2 against 3.8) and
// gain nothing on a large one; two at 32 lanes (16 columns) take 105 instead of 116 us at 16384 x 16384, but 16.4 instead of
// 15.3 at K = 512, S = 65536 and 24.9 instead of 22.5 at K = 544.
constexpr int SPARSE_PACK_MAX_LANES = 32;
constexpr int64_t SPARSE_PACK_TILES_LAUNCH = 1 << 20;               // tiles of a launch: a grid has no more than 2^32 threads
constexpr int sparse_pack_passes(int lanes) { return lanes == 32 ? 4 : 2; }
constexpr int sparse_pack_cols(int lanes) { return 256 / lanes * sparse_pack_passes(lanes); }
template <int LANES>
__global__ __launch_bounds__(256) void sparse_pack_kernel(uint32_t* __restrict__ wt_outs,
                                                          uint32_t* __restrict__ msk_outs,
                                                          const uint8_t* __restrict__ wt_in,
                                                          const uint8_t* __restrict__ msk_in,
                                                          int64_t S, int64_t K, int64_t s_first, uint32_t k_tiles,
                                                          int* __restrict__ bad_blocks, int* bad_flag) {
    constexpr int PASSES = sparse_pack_passes(LANES), CELLS = LANES / 2, COLS_PASS = 256 / LANES, COLS = sparse_pack_cols(LANES);
    // compaction table: for a byte of eight keep flags, the v_perm selectors that move the kept rows' code bytes to
    // the front in row order (0 ... 7: that row of the eight; 0x0C: a zero byte)
    __shared__ u32x2 front[256];
    __shared__ uint32_t tile[3][CELLS][COLS + 1];                   // low words, high words, masks
    const int64_t k0 = (int64_t)(blockIdx.x % k_tiles) * (16 * LANES);
    const int64_t s0 = s_first + (int64_t)(blockIdx.x / k_tiles) * COLS;
    const int lane = threadIdx.x % LANES, col0 = threadIdx.x / LANES;
    const bool in_k = k0 + 16 * lane < K;                           // (K is a multiple of 32: both lanes of a cell or neither)
    u32x4 wq[PASSES], mq[PASSES];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int64_t s = s0 + col0 + i * COLS_PASS;
        wq[i] = mq[i] = u32x4{0, 0, 0, 0};
        if (in_k && s < S) {
            wq[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wt_in + s * K + k0 + 16 * lane));
            mq[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(msk_in + s * K + k0 + 16 * lane));
        }
    }
    {
        uint32_t sel[2] = {0x0C0C0C0Cu, 0x0C0C0C0Cu};
        int p = 0;
        for (int r = 0; r < 8; ++r)
            if ((threadIdx.x >> r) & 1u) {
                sel[p >> 2] = (sel[p >> 2] & ~(0xFFu << (8 * (p & 3)))) | ((uint32_t)r << (8 * (p & 3)));
                ++p;
            }
        front[threadIdx.x] = u32x2{sel[0], sel[1]};
    }
    __syncthreads();
    // keep flags of four rows (bytes > 0) as four bits: the top bit of every non-zero byte, gathered by a multiply
    auto flags4 = [](uint32_t m) {
        const uint32_t nz = ((((m & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | m) & 0x80808080u) >> 7;
        return ((nz * 0x00204081u) >> 21) & 0xFu;
    };
    // four code bytes (each at most 15) to four nibbles
    auto nibbles4 = [](uint32_t o) {
        const uint32_t n = (o | (o >> 4)) & 0x00FF00FFu;
        return (n | (n >> 8)) & 0xFFFFu;
    };
    auto other_lane = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true); };  // lane ^ 1
    const bool odd = lane & 1;
    int bad = 0;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        uint32_t keep = 0;
        uint64_t v = 0;
        int rank = 0;
#pragma unroll
        for (int g8 = 0; g8 < 2; ++g8) {                            // eight rows at a time
            const uint32_t m8 = flags4(mq[i][2 * g8]) | (flags4(mq[i][2 * g8 + 1]) << 4);
            const u32x2 sel = front[m8];
            const uint32_t clo = wq[i][2 * g8] & 0x0F0F0F0Fu, chi = wq[i][2 * g8 + 1] & 0x0F0F0F0Fu;
            const uint32_t kept = nibbles4(__builtin_amdgcn_perm(chi, clo, sel.x)) |
                                  (nibbles4(__builtin_amdgcn_perm(chi, clo, sel.y)) << 16);
            keep |= m8 << (8 * g8);
            v |= (uint64_t)kept << (4 * rank);
            rank += __builtin_popcount(m8);
        }
        // the odd lane's codes follow the even lane's (those beyond the sixteenth fall off the top)
        const int rank_other = (int)other_lane((uint32_t)rank);
        if (odd) v = rank_other < 16 ? v << (4 * rank_other) : 0;
        const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
        const uint32_t word = (odd ? hi : lo) | other_lane(odd ? lo : hi);
        const uint32_t keep_other = other_lane(keep);
        const int col = col0 + i * COLS_PASS;
        tile[odd][lane / 2][col] = word;
        if (!odd) {
            tile[2][lane / 2][col] = keep | (keep_other << 16);
            bad += in_k && s0 + col < S && rank + rank_other != 16;
        }
    }
    __syncthreads();
    const int cells = (int)min((int64_t)CELLS, (K - k0) / 32);
#pragma unroll
    for (int i = 0; i < CELLS * COLS / 256; ++i) {
        const int at = i * 256 + (int)threadIdx.x, c = at / COLS, col = at % COLS;
        const int64_t s = s0 + col, blk = k0 / 32 + c;
        if (c >= cells || s >= S) continue;
        wt_outs[(2 * blk) * S + s] = tile[0][c][col];
        wt_outs[(2 * blk + 1) * S + s] = tile[1][c][col];
        msk_outs[blk * S + s] = tile[2][c][col];
    }
    if (bad && bad_blocks) {
        atomicAdd(bad_blocks, bad);
        // (pinned host memory: a plain store, which every bus carries)
        if (bad_flag) __hip_atomic_store(bad_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

static dim3 cell_grid(int64_t S, int64_t K) { return dim3((unsigned)((S + 255) / 256), (unsigned)(K / 32)); }

// What a checked packing reports through: a device counter that is 0 between calls, and a word of pinned host memory that the kernel
// sets when it counts.  A call takes one for itself and gives it back; MOST are kept.
struct PackReport { int device; int* count; int* flag; };
constexpr int MOST_REPORTS = 16;
static std::mutex g_reports_mutex;
static PackReport g_reports[MOST_REPORTS];
static int g_n_reports = 0;

// (on the caller's stream: a copy on the null stream would wait for, or under a capture elsewhere be refused because of, other streams)
static bool clear_count(const PackReport& r, hipStream_t stream) {
    static const int zero = 0;
    return hipMemcpyAsync(r.count, &zero, sizeof(int), hipMemcpyHostToDevice, stream) == hipSuccess;
}
static void free_report(const PackReport& r) {
    if (r.count) (void)hipFree(r.count);
    if (r.flag) (void)hipHostFree(r.flag);
}

static bool take_report(PackReport& r, hipStream_t stream) {
    r = PackReport{0, nullptr, nullptr};
    if (hipGetDevice(&r.device) != hipSuccess) return false;
    {
        std::lock_guard<std::mutex> lock(g_reports_mutex);
        for (int i = 0; i < g_n_reports; ++i)
            if (g_reports[i].device == r.device) {
                r = g_reports[i];
                g_reports[i] = g_reports[--g_n_reports];
                return true;
            }
    }
    // (another thread may be capturing a graph, which allocations must not end)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const bool ok = hipMalloc(&r.count, sizeof(int)) == hipSuccess && hipHostMalloc(&r.flag, sizeof(int), hipHostMallocDefault) == hipSuccess &&
                    clear_count(r, stream);
    if (ok) *r.flag = 0;
    else free_report(r);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return ok;
}

static void give_back(const PackReport& r) {
    {
        std::lock_guard<std::mutex> lock(g_reports_mutex);
        if (g_n_reports < MOST_REPORTS) {
            g_reports[g_n_reports++] = r;
            return;
        }
    }
    free_report(r);
}

static int validate_pack(const void* wt_outs, const void* msk_outs, const void* wt_in, const void* msk_in, int64_t out_size, int64_t in_size) {
    if (out_size < 0 || in_size < 0 || in_size % 32 != 0) return INT4MM_ERR_SHAPE;
    if (in_size / 32 > 65535) return INT4MM_ERR_SHAPE;
    if (out_size == 0 || in_size == 0) return INT4MM_OK;
    if (!wt_outs || !msk_outs || !wt_in || !msk_in) return INT4MM_ERR_NULL;
    if (((uintptr_t)wt_in | (uintptr_t)msk_in) & 15u) return INT4MM_ERR_ALIGN;
    return INT4MM_OK;
}

static int sparse_pack(void* wt_outs, void* msk_outs, const void* wt_in, const void* msk_in,
                       int64_t out_size, int64_t in_size, int* bad_blocks, int* bad_flag, void* stream) {
    const int wrong = validate_pack(wt_outs, msk_outs, wt_in, msk_in, out_size, in_size);
    if (wrong != INT4MM_OK || out_size == 0 || in_size == 0) return wrong;
    int lanes = 2;
    while (lanes < SPARSE_PACK_MAX_LANES && 16 * lanes < in_size) lanes *= 2;
    const int64_t k_tiles = (in_size + 16 * lanes - 1) / (16 * lanes);
    const int64_t cols = sparse_pack_cols(lanes), cols_launch = SPARSE_PACK_TILES_LAUNCH / k_tiles * cols;   // (k_tiles <= 4096)
    for (int64_t s_first = 0; s_first < out_size; s_first += cols_launch) {
        const int64_t tiles = k_tiles * ((std::min(cols_launch, out_size - s_first) + cols - 1) / cols);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(256), 0,
                               (hipStream_t)stream, (uint32_t*)wt_outs, (uint32_t*)msk_outs,
                               (const uint8_t*)wt_in, (const uint8_t*)msk_in, out_size, in_size, s_first,
                               (uint32_t)k_tiles, bad_blocks, bad_flag);
        };
        switch (lanes) {
            case 2: launch(sparse_pack_kernel<2>); break;
            case 4: launch(sparse_pack_kernel<4>); break;
            case 8: launch(sparse_pack_kernel<8>); break;
            case 16: launch(sparse_pack_kernel<16>); break;
            default: launch(sparse_pack_kernel<32>); break;
        }
    }
    return check_launch("sparse_pack");
}

}  // namespace i4

using namespace i4;

extern "C" {

int int4mm_sparse_pack(void* wt_outs, void* msk_outs, const void* wt_in, const void* msk_in,
                       int64_t out_size, int64_t in_size, void* bad_blocks, void* stream) {
    return sparse_pack(wt_outs, msk_outs, wt_in, msk_in, out_size, in_size, (int*)bad_blocks, nullptr, stream);
}

// Nothing runs before the kernel and nothing but the wait after it: a fill that clears a counter and a copy that reads it back
// make a call at 16384 x 16384 134 us instead of 129.
int int4mm_sparse_pack_checked(void* wt_outs, void* msk_outs, const void* wt_in, const void* msk_in,
                               int64_t out_size, int64_t in_size, int* bad_blocks, void* stream) {
    if (bad_blocks == nullptr) return INT4MM_ERR_NULL;
    *bad_blocks = 0;
    const int wrong = validate_pack(wt_outs, msk_outs, wt_in, msk_in, out_size, in_size);
    if (wrong != INT4MM_OK || out_size == 0 || in_size == 0) return wrong;
    // (refused before anything is enqueued: a recorded kernel would go on reporting into what the next call takes)
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)stream, &capture) != hipSuccess) return launch_error();
    if (capture != hipStreamCaptureStatusNone) return launch_error(hipErrorStreamCaptureUnsupported);
    PackReport r;
    if (!take_report(r, (hipStream_t)stream)) return launch_error();
    const int rc = sparse_pack(wt_outs, msk_outs, wt_in, msk_in, out_size, in_size, r.count, r.flag, stream);
    if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) {          // (the kernel may still write: the report is not used again)
        const int failed = launch_error();
        return rc != INT4MM_OK ? rc : failed;
    }
    bool clean = true;
    if (*(volatile int*)r.flag != 0) {
        clean = hipMemcpyAsync(bad_blocks, r.count, sizeof(int), hipMemcpyDeviceToHost, (hipStream_t)stream) == hipSuccess &&
                clear_count(r, (hipStream_t)stream) && hipStreamSynchronize((hipStream_t)stream) == hipSuccess;
        *r.flag = 0;
    }
    if (!clean) {
        free_report(r);
        return launch_error();
    }
    give_back(r);
    return rc;
}

int int4mm_dense_pack(int bits, void* matrix_out, const void* codes_in, int64_t in_size,
                      int64_t out_size, void* stream) {
    if (bits != 4 && bits != 3 && bits != 2) return INT4MM_ERR_BITS;
    if (out_size < 0 || in_size < 0 || in_size % 32 != 0 || in_size / 32 > 65535)
        return INT4MM_ERR_SHAPE;
    if (out_size == 0 || in_size == 0) return INT4MM_OK;
    if (!matrix_out || !codes_in) return INT4MM_ERR_NULL;
    const dim3 grid = cell_grid(out_size, in_size), block(256);
    hipStream_t st = (hipStream_t)stream;
    uint32_t* o = (uint32_t*)matrix_out;
    const uint8_t* c = (const uint8_t*)codes_in;
    if (bits == 4) hipLaunchKernelGGL(dense_pack_kernel<4>, grid, block, 0, st, o, c, in_size, out_size);
    if (bits == 3) hipLaunchKernelGGL(dense_pack_kernel<3>, grid, block, 0, st, o, c, in_size, out_size);
    if (bits == 2) hipLaunchKernelGGL(dense_pack_kernel<2>, grid, block, 0, st, o, c, in_size, out_size);
    return check_launch("dense_pack");
}

int int4mm_unpack(int bits, void* codes_out, void* keep_out, const void* matrix,
                  const void* sparse_mask, int64_t in_size, int64_t out_size, void* stream) {
    if (bits != 4 && bits != 3 && bits != 2) return INT4MM_ERR_BITS;
    if (sparse_mask && bits != 4) return INT4MM_ERR_SPARSE_BITS;
    if (out_size < 0 || in_size < 0 || in_size % 32 != 0 || in_size / 32 > 65535)
        return INT4MM_ERR_SHAPE;
    if (out_size == 0 || in_size == 0) return INT4MM_OK;
    if (!codes_out || !matrix) return INT4MM_ERR_NULL;
    const dim3 grid = cell_grid(out_size, in_size), block(256);
    hipStream_t st = (hipStream_t)stream;
    uint8_t* o = (uint8_t*)codes_out;
    uint8_t* k = (uint8_t*)keep_out;
    const uint32_t* m = (const uint32_t*)matrix;
    const uint32_t* msk = (const uint32_t*)sparse_mask;
    if (out_size % 4 == 0 && (((uintptr_t)codes_out | (uintptr_t)keep_out) & 3u) == 0) {
        const dim3 grid4((unsigned)((out_size / 4 + 255) / 256), grid.y);
        if (msk) hipLaunchKernelGGL((unpack4_kernel<4, true>), grid4, block, 0, st, o, k, m, msk, in_size, out_size);
        else if (bits == 4) hipLaunchKernelGGL((unpack4_kernel<4, false>), grid4, block, 0, st, o, k, m, msk, in_size, out_size);
        else if (bits == 3) hipLaunchKernelGGL((unpack4_kernel<3, false>), grid4, block, 0, st, o, k, m, msk, in_size, out_size);
        else hipLaunchKernelGGL((unpack4_kernel<2, false>), grid4, block, 0, st, o, k, m, msk, in_size, out_size);
        return check_launch("unpack");
    }
    if (msk) hipLaunchKernelGGL((unpack_kernel<4, true>), grid, block, 0, st, o, k, m, msk, in_size, out_size);
    else if (bits == 4) hipLaunchKernelGGL((unpack_kernel<4, false>), grid, block, 0, st, o, k, m, msk, in_size, out_size);
    else if (bits == 3) hipLaunchKernelGGL((unpack_kernel<3, false>), grid, block, 0, st, o, k, m, msk, in_size, out_size);
    else hipLaunchKernelGGL((unpack_kernel<2, false>), grid, block, 0, st, o, k, m, msk, in_size, out_size);
    return check_launch("unpack");
}

int int4mm_dequantize(int bits, void* w_out, const void* matrix, const void* scales,
                      const void* zeros, const void* sparse_mask, int64_t in_size,
                      int64_t out_size, int64_t n_groups, int64_t group_size, void* stream) {
    if (bits != 4 && bits != 3 && bits != 2) return INT4MM_ERR_BITS;
    if (sparse_mask && bits != 4) return INT4MM_ERR_SPARSE_BITS;
    if (out_size < 0 || in_size < 0 || in_size % 64 != 0 || in_size / 32 > 65535 || n_groups <= 0)
        return INT4MM_ERR_SHAPE;
    if (group_size == 0 || (group_size > 0 && group_size % 64 != 0)) return INT4MM_ERR_GROUP;
    const int64_t g = group_size < 0 ? ONE_GROUP : group_size;
    if (n_groups > ((int64_t)1 << 40) || g * n_groups < in_size) return INT4MM_ERR_SHAPE;
    if (out_size == 0 || in_size == 0) return INT4MM_OK;
    if (!w_out || !matrix || !scales || !zeros) return INT4MM_ERR_NULL;
    const dim3 grid = cell_grid(out_size, in_size), block(256);
    hipStream_t st = (hipStream_t)stream;
    h16* o = (h16*)w_out;
    const uint32_t* m = (const uint32_t*)matrix;
    const uint32_t* msk = (const uint32_t*)sparse_mask;
    const h16* sc = (const h16*)scales;
    const h16* ze = (const h16*)zeros;
    if (msk) hipLaunchKernelGGL((dequantize_kernel<4, true>), grid, block, 0, st, o, m, msk, sc, ze, in_size, out_size, g);
    else if (bits == 4) hipLaunchKernelGGL((dequantize_kernel<4, false>), grid, block, 0, st, o, m, msk, sc, ze, in_size, out_size, g);
    else if (bits == 3) hipLaunchKernelGGL((dequantize_kernel<3, false>), grid, block, 0, st, o, m, msk, sc, ze, in_size, out_size, g);
    else hipLaunchKernelGGL((dequantize_kernel<2, false>), grid, block, 0, st, o, m, msk, sc, ze, in_size, out_size, g);
    return check_launch("dequantize");
}

}  // extern "C"
