"""QuantLinear: the caller-side holder of the packed formats (quantise / pack on
the device, forward through the `int4matmul` extension)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,sparse,tol", [(4, False, 0.08), (3, False, 0.17), (2, False, 0.4), (4, True, 0.08)])
@pytest.mark.parametrize("shape", [(1, 1), (2, 5), (1, 300)])
def test_quantise_pack_forward(bits, sparse, tol, shape):
    from int4matmul_kernels_amd.quant_linear import QuantLinear

    torch.manual_seed(bits)
    K, S = 512, 384
    w = (torch.randn((K, S), device="cuda") * 0.05).half()
    keep = None
    if sparse:
        keys = torch.rand((S, K // 32, 32), device="cuda")
        keep = torch.zeros((S, K // 32, 32), dtype=torch.bool, device="cuda")
        keep.scatter_(2, keys.argsort(dim=2)[:, :, :16], True)
        keep = keep.reshape(S, K).t().contiguous()
    bias = torch.randn((S,), device="cuda").half()
    layer = QuantLinear.from_float(w, bits=bits, group_size=64, keep=keep, bias=bias)
    wq = layer.dequantized_weight()
    target = w if keep is None else w * keep
    # quantisation error of round-to-nearest: at most half a step of the group's range
    step = (w.float().reshape(K // 64, 64, S).amax(1) - w.float().reshape(K // 64, 64, S).amin(1)) / ((1 << bits) - 1)
    err = (wq.float() - target.float()).abs().reshape(K // 64, 64, S).amax(1)
    assert torch.all(err <= 0.51 * step + 2e-3)
    if keep is not None:
        assert torch.all(wq[~keep] == 0)
    x = torch.randn((*shape, K), device="cuda").half()
    y = layer(x)
    ref = x.float() @ wq.float() + bias.float()
    assert y.shape == (*shape, S) and y.dtype == torch.float16
    rms = ref.pow(2).mean().sqrt()
    assert ((y.float() - ref).abs().max() / rms).item() < 1e-2
    # and close to the unquantised layer within the format's resolution
    full = x.float() @ target.float() + bias.float()
    assert ((y.float() - full).pow(2).mean().sqrt() / full.pow(2).mean().sqrt()).item() < tol


def test_from_packed_round_trip_and_state_dict():
    from int4matmul_kernels_amd.quant_linear import QuantLinear

    w = (torch.randn((256, 128), device="cuda") * 0.1).half()
    a = QuantLinear.from_float(w, bits=4, group_size=-1)
    b = QuantLinear.from_packed(4, a.matrix, a.scales, a.zeros, -1)
    c = QuantLinear(4, 256, 128, group_size=-1)
    c.load_state_dict(a.state_dict())
    x = torch.randn((3, 1, 256), device="cuda").half()
    assert torch.equal(a(x), b(x)) and torch.equal(a(x), c(x))
    with pytest.raises(ValueError):
        QuantLinear(3, 256, 128, sparse=True)


@pytest.mark.parametrize("bits,sparse", [(4, False), (3, False), (2, False), (4, True)])
@pytest.mark.parametrize("shape", [(1, 1), (3, 1), (8, 1), (70, 1), (130, 1), (515, 1), (1, 2), (2, 5), (1, 45), (1, 300), (0, 1), (2, 0)])
def test_forward_overwrites_as_quant_matmul_on_zeros(bits, sparse, shape):
    """a layer's output is allocated without a fill: whatever the memory held, every element is written, with the bits that
    quant_matmul gives on a zeroed tensor"""
    import int4matmul_kernels_amd as pkg
    from int4matmul_kernels_amd.quant_linear import QuantLinear

    gen = torch.Generator(device="cuda").manual_seed(bits)
    K, S = 8192, 320                                 # few columns, long K: K is split, partial sums are handed over
    matrix = torch.randint(-2 ** 31, 2 ** 31, (K // 16 if sparse else K * bits // 32, S), dtype=torch.int32, generator=gen, device="cuda")
    scales = (torch.rand((K // 64, S), generator=gen, device="cuda") * 0.02 + 0.001).half()
    zeros = (torch.rand((K // 64, S), generator=gen, device="cuda") * 3).half()
    mask = torch.full((K // 32, S), 0x0FF00FF0, dtype=torch.int32, device="cuda") if sparse else None
    layer = QuantLinear.from_packed(bits, matrix, scales, zeros, 64, mask)
    x = torch.randn((*shape, K), generator=gen, device="cuda").half()
    want = torch.zeros((*shape, S), dtype=torch.float16, device="cuda")
    pkg.load_extension().quant_matmul(bits, want, matrix, x, scales, zeros, 64, mask)
    stale = torch.full((*shape, S), float("nan"), dtype=torch.float16, device="cuda")
    at = stale.data_ptr()
    del stale
    got = layer(x)
    assert got.numel() == 0 or got.data_ptr() == at  # the allocator has handed the block of NaN to the layer's output
    assert torch.equal(got, want)
    assert torch.equal(layer(x.float()), want)       # converted on the way in
    # strided states: every second of 2 K columns; the first two dimensions in the other order
    apart = torch.stack((x, x + 1), dim=-1).flatten(-2)[..., ::2]
    assert x.numel() == 0 or not apart.is_contiguous()
    assert torch.equal(layer(apart), want)
    if min(shape) > 1:
        turned = x.transpose(0, 1).contiguous().transpose(0, 1)
        assert not turned.is_contiguous()
        assert torch.equal(layer(turned), want)


ROUTES = [  # bits, sparse, batch, K, S, the launches in order
    (4, False, 1, 4096, 512, [("matvec_kernel<bits=4,dense", "batch=1")]),
    (4, True, 1, 4096, 512, [("matvec_kernel<bits=4,16:32", "batch=1")]),
    (4, False, 1, 460800, 64, [("matvec_kernel", "batch=1"), ("matvec_kernel", "batch=1")]),          # two ranges of K
    (4, False, 3, 460800, 64, [("matvec_kernel", "batch=3"), ("matvec_kernel", "batch=3")]),
    (4, False, 2, 5120, 20480, [("matvec_kernel", "rows=2>")]),
    (3, False, 3, 5120, 20480, [("matvec_kernel", "rows=4>")]),
    (2, False, 4, 5120, 20480, [("matvec_kernel", "rows=4>")]),
    (4, False, 8, 5120, 20480, [("skinny_kernel", "balanced")]),
    (4, True, 8, 5120, 20480, [("skinny_kernel<bits=4,16:32", "balanced")]),
    (3, False, 8, 8192, 16448, [("skinny_kernel", "columns_per_lane=4+1")]),
    (4, False, 2, 4096, 512, [("skinny_kernel", "ksplit=1")]),
    (2, False, 70, 8192, 320, [("skinny_kernel", "ksplit=2")]),
    (4, False, 70, 4096, 512, [("wide_rows_kernel", "ksplit=8")]),
    (4, True, 130, 4096, 512, [("wide_rows_kernel<bits=4,16:32", "ksplit=8")]),
    (4, False, 130, 4096, 4096, [("wide_rows_kernel", "ksplit")]),
    # the 512-row chunks: a remainder for the wide kernel, for the few-row kernel, a single row, and none that fits at all
    (4, False, 600, 4096, 512, [("wide_rows_kernel", "ksplit"), ("wide_rows_kernel", "ksplit")]),
    (4, False, 515, 4096, 512, [("wide_rows_kernel", "ksplit"), ("skinny_kernel", "ksplit")]),
    (3, False, 513, 4096, 512, [("wide_rows_kernel", "ksplit"), ("matvec_kernel", "batch=1")]),
    (4, False, 130, 8192, 320, [("matvec_kernel", "batch=130")]),
]


@pytest.mark.parametrize("bits,sparse,batch,K,S,launches", ROUTES)
def test_matvec_overwrite_writes_every_element_on_every_route(bits, sparse, batch, K, S, launches):
    """int4mm_matvec_overwrite on NaN, between guard rows: the bits of int4mm_matvec on zeros, and nothing beyond"""
    from int4matmul_kernels_amd import capi

    line = capi.describe_launch("vec", bits, batch, 1, K, S, 64, sparse).split("; ")[:-1]
    assert len(line) == len(launches), line
    for got, (kernel, form) in zip(line, launches):
        assert got.startswith(kernel) and form in got, line
    gen = torch.Generator(device="cuda").manual_seed(batch)
    matrix = torch.randint(-2 ** 31, 2 ** 31, (K // 16 if sparse else K * bits // 32, S), dtype=torch.int32, generator=gen, device="cuda")
    scales = (torch.rand((K // 64, S), generator=gen, device="cuda") * 0.02 + 0.001).half()
    zeros = (torch.rand((K // 64, S), generator=gen, device="cuda") * 3).half()
    mask = torch.full((K // 32, S), 0x0FF00FF0, dtype=torch.int32, device="cuda") if sparse else None
    x = torch.randn((batch, 1, K), generator=gen, device="cuda").half() / 8
    ws = capi.new_matmul_workspace(batch, 1, K, S, sparse)
    want = torch.zeros((batch, 1, S), dtype=torch.float16, device="cuda")
    capi.matvec(bits, want, matrix, x, scales, zeros, 64, mask, ws)
    assert bool(torch.isfinite(want).all()) and bool((want != 0).any())
    outs = torch.full((batch + 2, 1, S), float("nan"), dtype=torch.float16, device="cuda")
    guard = outs[0].clone()
    capi.matvec_overwrite(bits, outs[1:-1], matrix, x, scales, zeros, 64, mask, ws)
    assert torch.equal(outs[1:-1].view(torch.int16), want.view(torch.int16))
    assert torch.equal(outs[0].view(torch.int16), guard.view(torch.int16))
    assert torch.equal(outs[-1].view(torch.int16), guard.view(torch.int16))
