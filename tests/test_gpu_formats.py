"""GPU parity, integer side: pack / unpack / dequantise kernels against the CPU
oracle, bit for bit, through the C ABI."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(4, False), (3, False), (2, False), (4, True)]


@pytest.fixture(scope="module")
def H():
    from tests import helpers
    return helpers


@pytest.mark.parametrize("bits,sparse", CASES)
@pytest.mark.parametrize("K,S,g", [(64, 64, 64), (256, 320, 128), (1024, 1024, 64), (384, 64, -1)])
def test_dequantize_bit_exact(H, bits, sparse, K, S, g):
    p = O.make_problem(K=K, S=S, bits=bits, group_size=g, sparse=sparse, seed=K + S + bits)
    # mix in exponent-mode (negative scale) columns and groups
    p["scales"][:, ::3] *= np.float16(-1)
    d = H.dev_problem(p)
    out = torch.empty((K, S), dtype=torch.float16, device=H.DEV)
    H.capi.dequantize(bits, out, d["matrix"], d["scales"], d["zeros"], g, d["mask"])
    want = O.dequantize_matrix(bits, p["matrix"], p["scales"], p["zeros"], g, p["sparse_mask"])
    got = out.cpu().numpy()
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


def test_dequantize_exhaustive_codes_and_zeros(H):
    """every int4 code x every fp16 zero in [0, 15] x 64 scales, both modes"""
    zbits = np.arange(0, int(np.float16(15).view(np.uint16)) + 1, dtype=np.uint16)
    n = (len(zbits) + 63) // 64 * 64
    zeros = np.zeros(n, np.float16)
    zeros[:len(zbits)] = zbits.view(np.float16)
    rng = np.random.default_rng(2)
    for sign in (1.0, -1.0):
        for srow in range(4):
            scales = (sign * rng.uniform(0.001, 1.01, n)).astype(np.float16)
            codes = np.tile(np.arange(16, dtype=np.uint8)[:, None], (4, n))      # K = 64
            matrix = O.pack_dense(4, codes)
            out = torch.empty((64, n), dtype=torch.float16, device=H.DEV)
            H.capi.dequantize(4, out, H.t(matrix), H.t(scales[None]), H.t(zeros[None]), 64, None)
            want = O.dequantize_matrix(4, matrix, scales[None], zeros[None], 64)
            assert np.array_equal(out.cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("bits,sparse", CASES)
def test_unpack_bit_exact(H, bits, sparse):
    K, S = 512, 192
    p = O.make_problem(K=K, S=S, bits=bits, sparse=sparse, seed=11 + bits)
    d = H.dev_problem(p)
    codes = torch.empty((K, S), dtype=torch.uint8, device=H.DEV)
    keep = torch.empty((K, S), dtype=torch.uint8, device=H.DEV)
    H.capi.unpack(bits, codes, keep, d["matrix"], d["mask"])
    assert np.array_equal(codes.cpu().numpy(), p["codes"])
    want_keep = p["keep"] if sparse else np.ones((K, S), bool)
    assert np.array_equal(keep.cpu().numpy().astype(bool), want_keep)


@pytest.mark.parametrize("bits", [4, 3, 2])
def test_dense_pack_bit_exact_and_round_trip(H, bits):
    K, S = 640, 448
    rng = np.random.default_rng(bits)
    codes = rng.integers(0, 1 << bits, (K, S), dtype=np.uint8)
    out = torch.empty((K * bits // 32, S), dtype=torch.int32, device=H.DEV)
    H.capi.dense_pack(bits, out, H.t(codes))
    assert np.array_equal(out.cpu().numpy(), O.pack_dense(bits, codes))
    back = torch.empty((K, S), dtype=torch.uint8, device=H.DEV)
    H.capi.unpack(bits, back, None, out, None)
    assert np.array_equal(back.cpu().numpy(), codes)


def test_sparse_pack_bit_exact_capi_and_extension(H):
    S, K = 192, 1024
    p = O.make_problem(K=K, S=S, bits=4, sparse=True, seed=5)
    rng = np.random.default_rng(6)
    codes_sk = rng.integers(0, 16, (S, K), dtype=np.uint8)      # dropped rows carry junk codes
    keep_sk = np.ascontiguousarray(p["keep"].T).astype(np.uint8) * 3   # any value > 0 keeps
    want_w, want_m = O.sparse_pack(codes_sk, keep_sk)
    for via in ("capi", "ext"):
        w = torch.full((K // 16, S), -1, dtype=torch.int32, device=H.DEV)
        m = torch.full((K // 32, S), -1, dtype=torch.int32, device=H.DEV)
        if via == "capi":
            bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
            H.capi.sparse_pack(w, m, H.t(codes_sk), H.t(keep_sk), bad)
            assert int(bad.item()) == 0
        else:
            H.pkg.load_extension().weight_matrix_packing(w, m, H.t(codes_sk), H.t(keep_sk))
        assert np.array_equal(w.cpu().numpy(), want_w)
        assert np.array_equal(m.cpu().numpy(), want_m)


@pytest.mark.parametrize("S,K", [(1, 32), (300, 96), (4096, 1024)])
def test_weight_matrix_packing_counts_bad_blocks_anew_each_time(H, S, K):
    """the report of a bad packing does not reach the next one, on whichever stream or thread that runs"""
    from concurrent.futures import ThreadPoolExecutor
    ext = H.pkg.load_extension()
    codes = torch.full((S, K), 5, dtype=torch.uint8, device=H.DEV)
    good = (torch.arange(K, device=H.DEV) % 2).to(torch.uint8).repeat(S, 1).contiguous()
    torch.cuda.synchronize()

    def pack(bad):
        with torch.cuda.stream(torch.cuda.Stream()):
            keep = good.clone()
            if bad > 0:
                keep.view(-1, 32)[:bad, 0] = 1                # 17 rows of 32
            w = torch.empty((K // 16, S), dtype=torch.int32, device=H.DEV)
            m = torch.empty((K // 32, S), dtype=torch.int32, device=H.DEV)
            if bad == 0:
                ext.weight_matrix_packing(w, m, codes, keep)
                assert int((m != -0x55555556).sum()) == 0
            else:
                with pytest.raises(RuntimeError, match=f" {bad} 32-row blocks"):
                    ext.weight_matrix_packing(w, m, codes, keep)

    def pack_through_the_c_api(bad):
        # (ctypes lets go of the interpreter's lock: several reports are out at once)
        with torch.cuda.stream(torch.cuda.Stream()):
            keep = good.clone()
            keep.view(-1, 32)[:bad, 0] = 1
            w = torch.empty((K // 16, S), dtype=torch.int32, device=H.DEV)
            m = torch.empty((K // 32, S), dtype=torch.int32, device=H.DEV)
            for _ in range(4):
                assert H.capi.sparse_pack_checked(w, m, codes, keep) == bad

    most = S * K // 32
    counts = [0, 1, most, 0, min(2, most), 0]
    for n in counts:
        pack(n)
    with ThreadPoolExecutor(4) as pool:
        list(pool.map(pack_through_the_c_api, counts * 4))


def test_checked_packing_is_refused_on_a_stream_that_is_being_captured(H):
    """with nothing recorded: the capture goes on, and the packing after it counts as ever"""
    codes = torch.full((64, 64), 5, dtype=torch.uint8, device=H.DEV)
    keep = (torch.arange(64, device=H.DEV) % 2).to(torch.uint8).repeat(64, 1).contiguous()
    keep[0, 0] = 1
    w = torch.full((4, 64), 3, dtype=torch.int32, device=H.DEV)
    m = torch.empty((2, 64), dtype=torch.int32, device=H.DEV)
    x = torch.zeros(4, device=H.DEV)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        with pytest.raises(H.capi.Int4mmError) as e:
            H.capi.sparse_pack_checked(w, m, codes, keep)
        assert e.value.code == 7
    for n in range(1, 4):
        graph.replay()
        torch.cuda.synchronize()
        assert x.tolist() == [float(n)] * 4 and bool((w == 3).all())
    assert H.capi.sparse_pack_checked(w, m, codes, keep) == 1


@pytest.mark.parametrize("S,K", [(64, 64), (63, 96), (65, 512), (1, 544), (128, 1056), (200, 480), (320, 1600)])
def test_sparse_pack_tile_edges(H, S, K):
    """edges of the packer's tiles; cells that keep more or fewer than 16 rows are counted once each"""
    rng = np.random.default_rng(S * 10007 + K)
    codes_sk = rng.integers(0, 256, (S, K), dtype=np.uint8)
    keep_sk = (rng.random((S, K // 32, 32)).argsort(axis=2) < 16).astype(np.uint8)
    want_w, want_m = O.sparse_pack(codes_sk & 15, keep_sk.reshape(S, K))
    spoilt = rng.random((S, K // 32)) < 0.1
    for extra in (False, True):
        if extra:                                   # the last row of a cell flips: 15 or 17 kept, checked by count alone
            keep_sk[..., 31][spoilt] ^= 1
        w = torch.full((K // 16, S), -1, dtype=torch.int32, device=H.DEV)
        m = torch.full((K // 32, S), -1, dtype=torch.int32, device=H.DEV)
        bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
        H.capi.sparse_pack(w, m, H.t(codes_sk), H.t(keep_sk.reshape(S, K)), bad)
        assert int(bad.item()) == (int(spoilt.sum()) if extra else 0)
        if not extra:
            assert np.array_equal(w.cpu().numpy(), want_w)
            assert np.array_equal(m.cpu().numpy(), want_m)


@pytest.mark.parametrize("S,K", [(1, 32), (255, 32), (257, 32), (600, 32), (127, 64), (129, 64), (63, 128), (65, 128), (33, 160),
                                 (31, 256), (33, 256), (31, 288), (33, 992)])
def test_sparse_pack_tile_follows_narrow_k(H, S, K):
    """a tile has the fewest lanes that span K, and as many more columns: edges of each of the five tiles"""
    rng = np.random.default_rng(S * 10007 + K)
    codes = rng.integers(0, 256, (S, K), dtype=np.uint8)
    keep = (rng.random((S, K // 32, 32)).argsort(axis=2) < 16).astype(np.uint8).reshape(S, K)
    want_w, want_m = O.sparse_pack(codes & 15, keep)
    # a row of guard words before and behind each output
    w = torch.full((K // 16 + 2, S), -1, dtype=torch.int32, device=H.DEV)
    m = torch.full((K // 32 + 2, S), -1, dtype=torch.int32, device=H.DEV)
    keep[S // 2, 0] ^= 1                                # one cell keeps 15 or 17 rows: counted once, its words are not compared
    bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
    H.capi.sparse_pack(w[1:-1], m[1:-1], H.t(codes), H.t(keep), bad)
    assert int(bad.item()) == 1
    w, m = w.cpu().numpy(), m.cpu().numpy()
    assert (w[[0, -1]] == -1).all() and (m[[0, -1]] == -1).all()
    spoilt = np.zeros(S, bool)
    spoilt[S // 2] = True
    assert np.array_equal(w[1:-1][:, ~spoilt], want_w[:, ~spoilt]) and np.array_equal(w[3:-1], want_w[2:])
    assert np.array_equal(m[1:-1][:, ~spoilt], want_m[:, ~spoilt]) and np.array_equal(m[2:-1], want_m[1:])


@pytest.mark.parametrize("K", [32, 64])
def test_sparse_pack_narrow_k_is_as_fast_as_a_square(H, K):
    """the same bytes in 2^20 columns of one or two cells and in columns of 2048 rows: within a factor of two (they take
    equal time; a tile that is 512 rows deep whatever K is took five and three times as long)"""
    def best_us(k, s):
        codes = torch.randint(0, 16, (s, k), dtype=torch.uint8, device=H.DEV)
        keep = torch.zeros((s, k // 32, 32), dtype=torch.uint8, device=H.DEV)
        keep[..., ::2] = 1
        w = torch.empty((k // 16, s), dtype=torch.int32, device=H.DEV)
        m = torch.empty((k // 32, s), dtype=torch.int32, device=H.DEV)
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                H.capi.sparse_pack(w, m, codes, keep.reshape(s, k))
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end) * 50)
        return min(times)

    narrow, square = best_us(K, 1 << 20), best_us(2048, (1 << 20) * K // 2048)
    assert narrow < 2 * square + 5, (narrow, square)


@pytest.mark.parametrize("K,S", [(544, (1 << 25) + 336), (32, (1 << 30) + 4304)])
def test_sparse_pack_more_columns_than_a_launch_takes(H, K, S):
    """two launches and more; the second is 2^30 columns of one cell, more than 2^32 input bytes each"""
    need = 2 * S * K + 3 * S * K // 8
    if torch.cuda.mem_get_info()[0] < need + (16 << 30):
        pytest.skip(f"needs {need >> 30} GB")
    P = 16 * 13                                         # the columns repeat with a period that no tile's width divides
    assert S % P == 0
    rng = np.random.default_rng(K)
    codes = rng.integers(0, 16, (P, K), dtype=np.uint8)
    keep = (rng.random((P, K // 32, 32)).argsort(axis=2) < 16).astype(np.uint8).reshape(P, K)
    want_w, want_m = O.sparse_pack(codes, keep)
    codes_all = torch.empty((S // P, P, K), dtype=torch.uint8, device=H.DEV)
    keep_all = torch.empty_like(codes_all)
    codes_all.copy_(H.t(codes)[None])
    keep_all.copy_(H.t(keep)[None])
    w = torch.full((K // 16, S), -1, dtype=torch.int32, device=H.DEV)
    m = torch.full((K // 32, S), -1, dtype=torch.int32, device=H.DEV)
    bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
    try:
        H.capi.sparse_pack(w, m, codes_all.reshape(S, K), keep_all.reshape(S, K), bad)
        assert int(bad.item()) == 0
        for got, want in ((w, want_w), (m, want_m)):
            for row, want_row in zip(got, H.t(want)):
                assert bool((row.reshape(-1, P) == want_row).all())
    finally:
        del codes_all, keep_all, w, m
        torch.cuda.empty_cache()


def test_sparse_pack_flags_wrong_popcount(H):
    S, K = 64, 64
    keep = np.zeros((S, K), np.uint8)
    keep[:, :16] = 1
    keep[:, 32:48] = 1
    keep[5, 40] = 0                       # one block keeps 15
    codes = np.zeros((S, K), np.uint8)
    w = torch.empty((K // 16, S), dtype=torch.int32, device=H.DEV)
    m = torch.empty((K // 32, S), dtype=torch.int32, device=H.DEV)
    bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
    H.capi.sparse_pack(w, m, H.t(codes), H.t(keep), bad)
    assert int(bad.item()) == 1
    with pytest.raises(RuntimeError):
        H.pkg.load_extension().weight_matrix_packing(w, m, H.t(codes), H.t(keep))


def test_sparse_pack_any_popcount_any_flag_value_high_code_bits(H):
    """the packer is rank based (utils_kernel.cu:29-63): a row is kept when its mask byte is > 0 (any value), only the
    low nibble of a code byte counts, the code of rank p < 16 lands at bits 4p and later ones are dropped -- checked
    cell by cell against that closed form for blocks keeping 0 ... 32 rows; S and K / 32 not multiples of the tile"""
    rng = np.random.default_rng(23)
    S, K = 70, 32 * 9
    codes = rng.integers(0, 256, (S, K), dtype=np.uint8)                       # high nibbles are noise
    prob = rng.random((S, K // 32, 1))
    keep = (rng.random((S, K // 32, 32)) < prob).astype(np.uint8) * rng.integers(1, 256, (S, K // 32, 32), dtype=np.uint8)
    keep[0, 0, :] = 0
    keep[1, 0, :] = 7
    keep = keep.reshape(S, K)
    w = torch.zeros((K // 16, S), dtype=torch.int32, device=H.DEV)
    m = torch.zeros((K // 32, S), dtype=torch.int32, device=H.DEV)
    bad = torch.zeros(1, dtype=torch.int32, device=H.DEV)
    H.capi.sparse_pack(w, m, H.t(codes), H.t(keep), bad)
    torch.cuda.synchronize()
    got_w = w.cpu().numpy().view(np.uint32)
    got_m = m.cpu().numpy().view(np.uint32)
    wrong = 0
    for s in range(S):
        for b in range(K // 32):
            bits, v, rank = 0, 0, 0
            for t in range(32):
                if keep[s, 32 * b + t] > 0:
                    bits |= 1 << t
                    if rank < 16:
                        v |= int(codes[s, 32 * b + t] & 0xF) << (4 * rank)
                    rank += 1
            wrong += rank != 16
            assert got_m[b, s] == bits, (s, b)
            assert got_w[2 * b, s] == (v & 0xFFFFFFFF) and got_w[2 * b + 1, s] == (v >> 32), (s, b)
    assert int(bad.item()) == wrong
