"""Host-only: which kernel, tile shape and split the launchers choose.
``int4mm_describe_launch`` runs the launchers' own decision code with the launches
switched off.  The benchmark configurations are pinned exactly -- an edit of a shape
rule that silently reroutes one of them fails here, without a GPU; every other shape
is held to properties: a kernel that exists, launched within its limits."""
import pytest

from int4matmul_kernels_amd import capi

K, S = 5120, 20480


def d(*a, **kw):
    return capi.describe_launch(*a, **kw)


def test_matvec_configurations():
    # C1: K = S = 1024, g = 64
    assert d("vec", 4, 1, 1, 1024, 1024, 64).startswith(
        "matvec_kernel<bits=4,dense,lane_groups=4,prefetch=0> strips=16 splits=4 waves=2 units_per_workgroup=5")
    # C2: 640 workgroups of four waves; the three writing splits take 23 units each, the summing one 11.
    # Its transposed shape has 8 splits, which share K equally
    assert d("vec", 4, 1, 1, K, S, 128).startswith(
        "matvec_kernel<bits=4,dense,lane_groups=2,prefetch=0> strips=160 splits=4 waves=4 units_per_workgroup=23")
    assert d("vec", 4, 1, 1, S, K, 128).startswith(
        "matvec_kernel<bits=4,dense,lane_groups=4,prefetch=0> strips=80 splits=8 waves=4 units_per_workgroup=40")
    # C4: 16:32 at K = S = 16384, g = 64
    assert d("vec", 4, 1, 1, 16384, 16384, 64, sparse=True).startswith(
        "matvec_kernel<bits=4,16:32,lane_groups=4,prefetch=1> strips=256 splits=3 waves=4 units_per_workgroup=103")
    # C5: int3 / int2 take the shape of C2
    for bits in (3, 2):
        assert d("vec", bits, 1, 1, K, S, 128).startswith(
            f"matvec_kernel<bits={bits},dense,lane_groups=2,prefetch=0> strips=160 splits=4 waves=4 units_per_workgroup=23")


@pytest.mark.parametrize("bits", [4, 3, 2])
def test_dense_matmul_m2048(bits):
    # 640 tiles of 256 x 256 in the two-phase order; the 128 tiles of the third round split in two along K
    want = (f"matmul_kernel_pipe<bits={bits},dense,tile=256x256,two-phase> tiles=640 ksplit=2 split_from=512 "
            "workgroups=768")
    assert d("mtx", bits, 1, 2048, K, S, 128).startswith(want)
    # without room for the partial tiles the last round stays whole
    assert "ksplit=1 split_from=0 workgroups=640" in d("mtx", bits, 1, 2048, K, S, 128, workspace_bytes=0)


def test_other_matmul_configurations():
    # eleven rows of 192-row tiles, the last a third empty, fill the GPU better than eight rows of whole 256-row ones
    assert d("mtx", 4, 1, 2048, S, K, 128).startswith("matmul_kernel_pipe<bits=4,dense,tile=192x256,two-phase> tiles=220")
    # C3 small: one group, 16 tiles of the general kernel (the pipelined kernel's prologue would dominate)
    assert d("mtx", 4, 1, 2048, 128, 128, 128).startswith("matmul_kernel<bits=4,dense,tile=128x128> tiles=16")
    # C4: the 16:32 format, in the two phases as well
    assert d("mtx", 4, 1, 2048, K, S, 64, sparse=True).startswith(
        "matmul_kernel_pipe<bits=4,16:32,tile=256x256,two-phase> tiles=640 ksplit=2 split_from=512 workgroups=768")
    # every height and format runs the two phases; tuning key 3 = 9 forces 256 x 256 tiles without them
    for variant, order in ((5, "two-phase"), (6, "two-phase"), (7, "two-phase"), (8, "two-phase"), (9, "plain"), (10, "two-phase"), (11, "two-phase")):
        capi.tune(3, variant)
        try:
            for bits, sparse in ((4, False), (3, False), (2, False), (4, True)):
                if variant != 5 or not sparse:
                    assert f",{order}> " in d("mtx", bits, 1, 2048, K, S, 128, sparse), (variant, bits, sparse)
        finally:
            capi.tune(3, 0)


def test_baseline_shape_with_few_rows():
    # the few-row legs that bench.py reports at the benchmark shape (K=5120, S=20480): 2 rows through the matvec kernel (a row per
    # MFMA result register), 8 rows through the few-row kernel, 64 rows through the kernel with shared staging
    assert d("mtx", 4, 1, 2, K, S, 128).startswith("matvec_kernel<bits=4,dense,lane_groups=2,prefetch=0,rows=2> strips=160 splits=4")
    # (320 strips of 64 columns on 256 CUs: 256 workgroups share the strips' units evenly)
    shared = "skinny_kernel<bits=4,dense,columns_per_lane=4,row_tiles=1,balanced> strips=320 row_blocks=1 workgroups=256 waves=8"
    assert d("mtx", 4, 1, 8, K, S, 128).startswith(shared)
    assert d("vec", 4, 8, 1, K, S, 128).startswith(shared)
    assert d("mtx", 4, 1, 64, K, S, 128).startswith("wide_rows_kernel<bits=4,dense,row_tiles=4> strips=80 row_blocks=1 ksplit=3")
    # a single row through the matmul entry: the matvec kernel (all formats), the same launch as the matvec entry's
    for bits, sparse, g in ((4, False, 128), (3, False, 128), (2, False, 128), (4, True, 64)):
        assert d("mtx", bits, 1, 1, K, S, g, sparse) == d("vec", bits, 1, 1, K, S, g, sparse)
        assert d("mtx", bits, 1, 1, K, S, g, sparse).startswith("matvec_kernel<bits=%d," % bits)


# ---- every other shape: properties of the choice, not the choice itself (the shape rules are tuned on
# measurements and may move; what must hold is that a kernel that exists is launched within its limits)
KERNELS = ("matvec_kernel", "skinny_kernel", "wide_rows_kernel", "matmul_kernel_pipe", "matmul_kernel")
SHAPES = [(k, s) for k in (64, 512, 2048, 4096, 5120, 8192, 14336, 28672) for s in (64, 512, 2048, 4096, 5120, 11008, 20480, 32768)]
ROWS = (1, 2, 3, 4, 5, 8, 16, 17, 32, 33, 64, 65, 96, 128, 129, 192, 256, 257, 384, 512, 513, 1024, 1280, 2048, 4097)


def fields(line):
    """'name<template args> key=value key=value ...; ' -> (name, {key: int})"""
    import re
    head = line.split(";")[0]
    name = head.split("<")[0]
    return name, {k: int(v) for k, v in re.findall(r"(\w+)=(\d+)(?![x\d])", head)}, head


@pytest.mark.parametrize("fmt", [(4, False, 128), (3, False, 128), (2, False, -1), (4, True, 64)])
def test_every_shape_gets_a_kernel_within_its_limits(fmt):
    bits, sparse, g = fmt
    for k, s in SHAPES:
        for rows in ROWS:
            line = d("mtx", bits, 1, rows, k, s, g, sparse)
            name, f, head = fields(line)
            assert name in KERNELS, line
            assert f"bits={bits}," in head and ("16:32" in head) == sparse, line
            if name == "matvec_kernel":
                cols = 256 // f["lane_groups"]
                assert f["strips"] * cols >= s and (f["strips"] - 1) * cols < s, line
                nr = int(head.split(",rows=")[1][0]) if ",rows=" in head else 1
                assert 1 <= f["splits"] * nr <= 32 and 1 <= f["waves"] <= 8, line
                assert f["splits"] * f["units_per_workgroup"] >= k // 64 and f["units_per_workgroup"] * nr <= 224, line
                assert rows <= 4
            elif name in ("skinny_kernel", "wide_rows_kernel"):
                assert 2 <= rows <= 512 and f["strips"] >= 1, line
                assert f.get("ksplit", 1) >= 1 and f.get("row_blocks", 1) * 16 * f["row_tiles"] >= rows, line
            else:
                tm, tn = (int(v) for v in head.split("tile=")[1].split(",")[0].split(">")[0].split("x"))
                assert f["tiles"] >= -(-rows // tm) * -(-s // tn) // 1 and f["tiles"] >= 1, line
                assert 1 <= f.get("ksplit", 1) <= 8, line
            # without a workspace nothing may split K across workgroups
            bare = d("mtx", bits, 1, rows, k, s, g, sparse, workspace_bytes=0)
            n2, f2, _ = fields(bare)
            assert n2 in KERNELS and f2.get("ksplit", 1) == 1 and f2.get("splits", 1) == 1, bare


# ---- the kernels that sum exact codes keep the products that they had: a workspace too small for the split of K that the kernel with
# rounded weights was admitted with, and a long K with small groups
@pytest.mark.parametrize("product", ["mtx", "vec"])
@pytest.mark.parametrize("bits,sparse,rows,k,s,g,ws", [(4, False, 64, 8192, 8192, 128, "matvec"), (3, False, 40, 20480, 4096, 64, "matvec"),
                                                       (2, False, 96, 8192, 4096, -1, "matvec"), (4, True, 90, 8192, 8192, 64, "matvec"),
                                                       (4, True, 72, 14016, 768, 64, 3 << 20), (4, False, 52, 16896, 23296, 64, None),
                                                       (4, True, 18, 17920, 23808, 64, None)])
def test_few_rows_keep_the_sums_of_exact_codes(product, bits, sparse, rows, k, s, g, ws):
    nbytes = capi.lib().int4mm_workspace_bytes(s) if ws == "matvec" else ws
    line = d(product, bits, *((rows, 1) if product == "vec" else (1, rows)), k, s, g, sparse, nbytes)
    assert line.startswith("skinny_kernel"), line
    if ws is not None:                                     # (with the workspace that the size query asks for they are rounded, as before)
        assert d("mtx", bits, 1, rows, k, s, g, sparse).startswith("wide_rows_kernel")


# ---- a long K with so many groups that the few-row kernel has no room for their scales: the matmul entry, whose tile kernels round the
# weights as well, has the kernel with shared staging for it, with or without a workspace
@pytest.mark.parametrize("bits,rows,k,s,g", [(4, 34, 23296, 25600, 64), (4, 17, 28672, 28672, 64), (3, 34, 28672, 14336, 64),
                                             (2, 61, 28672, 16384, 64), (4, 50, 46656, 8192, 128), (4, 96, 20480, 25600, 64)])
def test_few_rows_on_many_groups_are_not_left_to_the_tiles(bits, rows, k, s, g):
    for ws in (None, 0, 1 << 34):
        assert d("mtx", bits, 1, rows, k, s, g, workspace_bytes=ws).startswith("wide_rows_kernel")
    nbytes = capi.matmul_workspace_bytes(1, rows, k, s)
    assert d("mtx", bits, 1, rows, k, s, g) == d("mtx", bits, 1, rows, k, s, g, False, 1 << 34) == d("mtx", bits, 1, rows, k, s, g, False, nbytes)


# ---- the matvec entry with more batch elements than the few-row kernel takes at once: the kernel with rounded weights where it is
# admitted, else shares of at most 96 elements with sums of exact codes; never a launch per element
@pytest.mark.parametrize("bits,sparse,batch,k,s", [(4, False, 256, 5120, 20480), (4, False, 256, 8192, 28672), (4, False, 300, 4096, 11008),
                                                   (4, False, 512, 4096, 14336), (4, True, 133, 4096, 11008), (4, True, 100, 2048, 20480),
                                                   (4, False, 385, 5120, 20480), (4, False, 1000, 5120, 20480), (3, False, 481, 4096, 11008),
                                                   (4, True, 257, 8192, 28672), (2, False, 330, 4096, 11008), (3, False, 97, 4096, 576)])
def test_many_batch_elements_keep_the_sums_of_exact_codes(bits, sparse, batch, k, s):
    line = d("vec", bits, batch, 1, k, s, 64 if sparse else 128, sparse)
    assert line.startswith("skinny_kernel") and "row_tiles=4,plain>" in line and "wide_rows" not in line, line


@pytest.mark.parametrize("bits,batch,k,s,g", [(4, 619, 1344, 5888, 128), (2, 877, 19200, 3584, -1), (4, 1740, 1536, 8192, -1), (3, 625, 1024, 7424, 128)])
def test_the_last_chunk_of_many_batch_elements_keeps_the_sums_of_exact_codes(bits, batch, k, s, g):
    # it asks for a split of K that the chunks of 512 do not: whatever the workspace has room for
    for ws in (None, 1 << 34):
        lines = d("vec", bits, batch, 1, k, s, g, False, ws).split("; ")[:-1]
        assert all(line.startswith("wide_rows_kernel") for line in lines[:batch // 512]), lines
        assert lines[batch // 512:] and all(line.startswith("skinny_kernel") for line in lines[batch // 512:]), lines
    # (no room is asked for a chunk that follows none of 512: 180 MB here)
    assert capi.matmul_workspace_bytes(657, 1, 18176, 16896) < 10 << 20
    # a last chunk that asks no more than those before it goes with them
    assert d("vec", 4, 1000, 1, 4096, 4096, 128).count("wide_rows_kernel") == 2


@pytest.mark.parametrize("bits,sparse", [(4, False), (3, False), (2, False), (4, True)])
def test_many_batch_elements_never_run_one_by_one(bits, sparse):
    for k, s in ((512, 256), (4096, 512), (2048, 1600), (4096, 11008), (5120, 20480), (8192, 28672), (2048, 40960)):
        for batch in (5, 17, 96, 97, 128, 193, 320, 384, 385, 481, 512, 513, 777, 1000):
            for ws in (None, capi.lib().int4mm_workspace_bytes(s)):
                line = d("vec", bits, batch, 1, k, s, 64 if sparse else 128, sparse, ws)
                assert line.startswith(("skinny_kernel", "wide_rows_kernel")), (batch, k, s, line)
    # (so many groups that the strips have to be narrower for their scales)
    for batch, k, s in ((368, 22784, 18688), (501, 19968, 15104), (48, 25344, 27648), (17, 28672, 28672), (90, 22400, 2752), (130, 57344, 17728)):
        for ws in (None, capi.lib().int4mm_workspace_bytes(s)):
            line = d("vec", bits, batch, 1, k, s, 64, sparse, ws)
            assert line.startswith(("skinny_kernel", "wide_rows_kernel")) and "matvec" not in line, (batch, k, s, line)


def test_many_rows_on_a_short_k_are_not_left_to_few_workgroups():
    # outputs wide enough for the tile kernels go to them from 257 rows on; narrower ones get more than the fewest blocks of rows
    for bits, rows, k, s in ((3, 442, 512, 17664), (4, 435, 192, 28416), (4, 494, 192, 12288), (4, 476, 64, 14848)):
        assert d("mtx", bits, 1, rows, k, s, 128).startswith("matmul_kernel"), (rows, k, s)
    for bits, rows, k, s in ((4, 469, 448, 1920), (4, 363, 448, 1536), (4, 117, 448, 2560), (2, 441, 320, 1536)):
        name, f, line = fields(d("mtx", bits, 1, rows, k, s, 128))
        assert name == "wide_rows_kernel" and f["strips"] * f["row_blocks"] >= 40, line


def evenly_shared(line):
    return "balanced" in line or "columns_per_lane=4+1" in line


def test_more_strips_than_cus_are_shared_out_evenly_within_limits():
    assert evenly_shared(d("mtx", 4, 1, 8, 12288, 28672, 128)) and evenly_shared(d("mtx", 4, 1, 16, 3072, 16448, 64, True))
    assert not evenly_shared(d("mtx", 4, 1, 17, 3072, 17408, 128))          # more than 16 rows
    assert not evenly_shared(d("mtx", 4, 1, 8, 2048, 20480, 128))           # a short K
    assert not evenly_shared(d("mtx", 4, 1, 8, 8192, 22016, 128))           # many more strips than CUs, K not long
    assert not evenly_shared(d("mtx", 4, 1, 8, 5120, 16384, 128))           # a strip per CU
    # without a workspace there is nowhere to sum a shared strip: a workgroup per strip; slivers need none
    assert not evenly_shared(d("mtx", 4, 1, 8, 5120, 20480, 128, False, 0))
    assert "columns_per_lane=4+1" in d("mtx", 3, 1, 8, 5120, 20480, 128, False, 0)
    # tuning key 9 = 1 switches both off
    capi.tune(9, 1)
    try:
        assert not evenly_shared(d("mtx", 4, 1, 8, K, S, 128)) and not evenly_shared(d("mtx", 3, 1, 8, K, S, 128))
    finally:
        capi.tune(9, 0)
    # the shared launch's partial tiles fit the workspace that the size query asks for
    for bits, sparse in ((4, False), (4, True)):
        for k, s in ((3072, 16448), (5120, 20480), (12288, 32704)):
            assert capi.matmul_workspace_bytes(1, 16, k, s, sparse) >= 2 * ((s // 64) * 2 * 8192), (k, s)


def test_workspace_sizes_are_consistent():
    lib = capi.lib()
    prev = 0
    for s in (64, 256, 1024, 4096, 20480, 32768, 131072):
        n = lib.int4mm_workspace_bytes(s)
        assert n >= prev and n >= 2 * (32 * 8 * s)              # 32 splits of {fp32, flag} per column, kept twice
        prev = n
        for k in (64, 4096, 28672):
            for rows in (1, 8, 64, 300, 2048):
                for sparse in (False, True):
                    assert capi.matmul_workspace_bytes(1, rows, k, s, sparse) >= n


@pytest.mark.parametrize("s", [64, 192, 512, 1600, 4096, 8192, 11008, 14400, 28672])
def test_the_workspace_asked_for_is_all_that_a_product_uses(s):
    # the launch with it is the launch with any amount more, whether the query knew the format and the group or only the sizes; and
    # an unsplit product does not ask for partial tiles
    for k in (512, 1088, 4096, 8192, 12352):
        for rows in (2, 8, 17, 33, 60, 72, 96, 97, 128, 200, 256, 300, 384, 512, 600, 1000):
            for bits, sparse, g in ((4, False, 128), (3, False, -1), (2, False, 64), (4, True, 64)):
                for product, shape in (("mtx", (1, rows)), ("vec", (rows, 1))):
                    plenty = d(product, bits, *shape, k, s, g, sparse, 1 << 34)
                    assert d(product, bits, *shape, k, s, g, sparse) == plenty, (rows, k, s)
                    nbytes = capi.matmul_workspace_bytes(*((1, rows) if rows <= 512 else shape), k, s, sparse)
                    assert d(product, bits, *shape, k, s, g, sparse, nbytes) == plenty, (rows, k, s)
    if s == 64:                                            # (one strip: K is all that there is to share out)
        assert "ksplit=16" in d("mtx", 4, 1, 300, 18048, 64, 128) and "ksplit=5" in d("mtx", 4, 1, 44, 17728, 64, 128)
    # (K = 8192, S = 28672: 200 and 512 rows asked for 134 MB and used nothing of it)
    if s == 28672:
        for rows in (200, 512):
            assert "ksplit=1" in d("mtx", 4, 1, rows, 8192, s, 128)
            assert capi.matmul_workspace_bytes(1, rows, 8192, s) == capi.lib().int4mm_workspace_bytes(s)


@pytest.mark.parametrize("bits,sparse,rows,k,s,g", [(4, False, 75, 20864, 17856, 64), (4, True, 14, 23232, 10944, 64), (4, False, 16, 28672, 9216, 64),
                                                    (2, False, 72, 43776, 10048, 64), (3, False, 2, 40960, 9216, 64), (4, True, 27, 49472, 4736, 64),
                                                    (4, True, 2, 46720, 27264, 128), (2, False, 5, 21376, 34560, 64), (3, False, 96, 20480, 12352, 64),
                                                    (4, False, 1, 917504, 1024, 524288)])
def test_few_rows_that_are_left_to_the_tiles_are_split_alike_on_any_workspace(bits, sparse, rows, k, s, g):
    # so many groups that their scales do not fit the few-row kernel's LDS (and a single row with a group longer than a launch of the
    # matvec covers): the launch with the workspace that the query asks for, knowing the group or not, is the launch with any amount
    # more, which other products on the stream may have left there
    plenty = d("mtx", bits, 1, rows, k, s, g, sparse, 1 << 34)
    assert d("mtx", bits, 1, rows, k, s, g, sparse) == plenty
    nbytes = capi.matmul_workspace_bytes(1, rows, k, s, sparse)
    assert d("mtx", bits, 1, rows, k, s, g, sparse, nbytes) == plenty
    name, f, line = fields(plenty)
    assert name == "matmul_kernel_pipe" and (f["ksplit"] > 1) == (rows > 1), line


@pytest.mark.parametrize("bits,sparse", [(4, False), (3, False), (2, False), (4, True)])
def test_a_row_more_or_fewer_takes_the_same_tiles(bits, sparse):
    # 640 and 1152 rows on a long K, multiples of 256 rows, and 224-row tiles of 16:32 are no rules of their own: the tiles that a row
    # fewer takes (which is padded to the same height)
    for rows, k, s in ((640, 28672, 3840), (1152, 14336, 4096), (1152, 20480, 4096), (1152, 28672, 2048), (2048, 20480, 5120), (1024, 8192, 9216),
                       (1536, 4096, 6400), (896, 4096, 8192), (672, 14336, 6144)):
        line = d("mtx", bits, 1, rows, k, s, 64, sparse)
        assert "x256," in line and line == d("mtx", bits, 1, rows - 1, k, s, 64, sparse), line
    if sparse:
        assert "tile=224x256," in d("mtx", 4, 1, 896, 4096, 8192, 64, True) and "ksplit=2 " in d("mtx", 4, 1, 896, 4096, 8192, 64, True)


@pytest.mark.parametrize("bits,rows,k,s,g", [(3, 546, 30272, 8832, 128), (4, 703, 31104, 9088, -1), (2, 2643, 31872, 2432, -1), (3, 293, 23936, 13568, -1),
                                             (4, 289, 24320, 13440, 128), (4, 2048, 8192, 128, 128), (2, 600, 4096, 128, 64), (4, 1152, 14336, 4096, 128)])
def test_the_workspace_asked_for_is_the_partial_tiles_of_the_launch(bits, rows, k, s, g):
    # not what a kernel that the product does not go to would split into (int3, K=23936, S=13568, 293 rows asked for 340 MB and used 35)
    name, f, line = fields(d("mtx", bits, 1, rows, k, s, g))
    tm, tn = (int(v) for v in line.split("tile=")[1].split(",")[0].split("x"))
    assert name == "matmul_kernel_pipe" and f["ksplit"] > 1, line
    used = (f["tiles"] - f["split_from"]) * f["ksplit"] * tm * tn * 4
    sh = capi.Shape(1, rows, k, s, k * bits // 32, 1 if g < 0 else -(-k // g), g)
    assert capi.lib().int4mm_matmul_workspace_bytes(sh, 0) - capi.lib().int4mm_workspace_bytes(s) == 2 * (-(-used // 4096) * 4096)


@pytest.mark.parametrize("bits", [4, 3, 2])
def test_outputs_of_128_columns_take_tiles_of_128(bits):
    for rows, k, want in ((513, 1088, 2), (600, 4096, 8), (4096, 2048, 4), (10240, 8192, 3), (16384, 8192, 2), (20480, 4096, 3), (24576, 4096, 1),
                          (12288, 16384, 5), (32768, 16384, 2), (65536, 8192, 1)):
        line = d("mtx", bits, 1, rows, k, 128, 128)
        assert line.startswith("matmul_kernel_pipe") and "tile=128x128," in line and f"tiles={-(-rows // 128)} ksplit={want} " in line, line
        assert "ksplit=1 " in d("mtx", bits, 1, rows, k, 128, 128, workspace_bytes=0)
    # up to 512 rows the kernel with shared staging, on a short K the general tiles
    assert d("mtx", bits, 1, 512, 8192, 128, 128).startswith("wide_rows_kernel")
    assert d("mtx", bits, 1, 2048, 1024, 128, 128).startswith("matmul_kernel<")


def test_matvec_of_a_k_beyond_one_launch():
    # 32 x 224 units of 64 rows is what one launch covers: a longer K runs as several launches (one line each)
    line = d("vec", 4, 1, 1, 1 << 20, 256, 128)
    assert line.count("matvec_kernel<") == 3, line
    assert d("vec", 4, 1, 1, 458752, 256, 128).count("matvec_kernel<") == 1
    with pytest.raises(capi.Int4mmError):                     # a single group longer than a launch covers, on a longer K
        d("vec", 4, 1, 1, 1 << 20, 256, 1 << 19)
    assert d("vec", 4, 1, 1, 1 << 20, 256, -1).count("matvec_kernel<") == 3       # one group: any cut will do


@pytest.mark.parametrize("k,s", [(28736, 32768), (32192, 16896), (46656, 26624), (60544, 11008), (430144, 1344), (14400, 109312), (458752, 32768)])
def test_matvec_of_a_long_k_on_a_wide_output(k, s):
    # K is split more ways than the output's width asks for, so that a workgroup's units fit its staged states
    for bits, sparse in ((4, False), (3, False), (2, False), (4, True)):
        line = d("vec", bits, 1, 1, k, s, 128, sparse)
        name, f, _ = fields(line)
        assert name == "matvec_kernel" and line.count("matvec_kernel<") == 1 and f["units_per_workgroup"] <= 224 and f["splits"] <= 32, line
        assert f["splits"] * f["units_per_workgroup"] >= k // 64 > (f["splits"] - 1) * f["units_per_workgroup"], line


def test_matvec_needs_its_workspace_whatever_the_shape():
    # K = 64: a single unit, nothing to hand over -- the documented rule holds all the same
    with pytest.raises(capi.Int4mmError) as e:
        d("vec", 4, 1, 1, 64, 64, 64, workspace_bytes=0)
    assert e.value.code == 6
    assert d("vec", 4, 1, 1, 64, 64, 64, workspace_bytes=capi.lib().int4mm_workspace_bytes(64)).startswith("matvec_kernel")


def test_tuning_is_per_thread_and_describe_leaves_no_trace():
    import threading
    capi.tune(3, 1)
    try:
        seen = {}
        t = threading.Thread(target=lambda: seen.setdefault("other", d("mtx", 4, 1, 2048, K, S, 128)))
        t.start()
        t.join()
        assert seen["other"].startswith("matmul_kernel_pipe")            # the other thread keeps the defaults
        assert d("mtx", 4, 1, 2048, K, S, 128).startswith("matmul_kernel<bits=4,dense,tile=128x128>")
    finally:
        capi.tune(3, 0)
    assert d("mtx", 4, 1, 2048, K, S, 128).startswith("matmul_kernel_pipe")
