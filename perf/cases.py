"""The workloads whose speed is watched: passes through the public entry points, from one token against a
small matrix to a batch of long prompts, in every weight format.

A case is a dict:

  path    "linear"  a ``QuantLinear`` layer (or several, one after another) applied to its input
          "matmul"  ``int4matmul.quant_matmul`` on tensors that the caller keeps, as the reference's callers use it
          "pack"    ``int4matmul.weight_matrix_packing``: codes and mask of a 16:32 matrix to its packed layout
  bits, sparse, group   the weight format: 4, 3 or 2 bits; 16:32 rows kept; rows per scale (-1: one group)
  expo    share of the (group, column) pairs in exponent mode (negative scale)
  k, s    input and output features
  batch, rows   the input is [batch, rows, k]; rows = 1 is one generated token per sequence
  layers  weight matrices of this shape that a pass goes through, each used once: while tokens are generated
          every pass walks through all layers of a model, so a layer's weights come from memory and not from a cache

Sizes are those of the test-suite, of ``bench.py`` and of the tables of measurements kept with this code.
"""
import math

import torch

import int4matmul_kernels_amd as pkg
from int4matmul_kernels_amd.quant_linear import QuantLinear

DEV = "cuda"


def _product(name, path, k, s, batch, rows, layers=1, bits=4, group=128, sparse=False, expo=0.0):
    case = dict(path=path, bits=bits, sparse=sparse, group=group, expo=expo, k=k, s=s, batch=batch, rows=rows, layers=layers)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # a small model generating one sequence: every call is a launch and little else
        _product("token_1k", "linear", 1024, 1024, 1, 1, layers=16, group=64),
        # one token through the up- and the down-projections of a feed-forward stack
        _product("token_up", "linear", 5120, 20480, 1, 1, layers=4),
        _product("token_down", "matmul", 20480, 5120, 1, 1, layers=4),
        # the same with a 16:32 matrix
        _product("token_sparse", "matmul", 16384, 16384, 1, 1, layers=2, group=64, sparse=True),
        # eight, and sixty-four, sequences that generate a token each
        _product("tokens_8", "linear", 5120, 20480, 8, 1, layers=4),
        _product("tokens_64", "linear", 5120, 20480, 64, 1, layers=4),
        # a short prompt of odd length through a square 16:32 projection; one through a 2-bit matrix whose groups
        # are partly in exponent mode
        _product("prompt_45_sparse", "matmul", 8192, 8192, 1, 45, layers=2, group=64, sparse=True),
        _product("prompt_200_int2", "linear", 11008, 4096, 1, 200, bits=2, expo=0.025),
        # a prompt of ragged length, three bits with one group; the benchmark's prompt; a batch of two long ones
        _product("prompt_777_int3", "linear", 4096, 11008, 1, 777, bits=3, group=-1),
        _product("prompt_2048", "linear", 5120, 20480, 1, 2048),
        _product("prompts_2x2048", "matmul", 8192, 28672, 2, 2048),
        # a matrix on its way in: 16:32 codes and mask, one byte each, to the packed layout
        dict(name="pack_sparse", path="pack", k=16384, s=16384),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    bits, sparse = rng.choice([(4, False), (4, False), (4, False), (3, False), (2, False), (4, True)])
    group = rng.choice([64, 128, 128, -1] if not sparse else [64, 128])
    expo = rng.choice([0.0, 0.0, 0.0, 0.0, 0.025])
    path = rng.choice(["linear", "linear", "matmul"])
    # features: multiples of 64, most of them of 256 as layers have, odd multiples too
    step = rng.choice([64, 256, 256, 256])
    while True:
        k, s = (max(1024, int(_log(rng, 1024, 28672)) // step * step) for _ in range(2))
        if k * s <= 16384 * 16384:
            break
    kind = rng.choice(["token", "token", "tokens", "tokens", "prompt", "prompt", "pack"])
    if kind == "pack":
        return dict(path="pack", k=k, s=s)
    if kind == "token":
        batch, rows = 1, 1
    elif kind == "tokens":
        batch, rows = int(_log(rng, 2, 129)), 1
    else:
        batch, rows = rng.choice([1, 1, 1, 2, 4]), int(_log(rng, 2, 4096))
        batch = max(1, min(batch, 4096 // rows))
    # no more than the largest listed case
    while batch * rows * k * s > 4096 * 8192 * 28672:
        rows = max(1, rows // 2)
    layers = 1 if batch * rows > 256 else max(1, min(16, int(4.2e8 / (k * s))))
    return _product(None, path, k, s, batch, rows, layers, bits, group, sparse, expo)


def _kept_rows(gen):
    """uint8 [65536, 32]: uniformly random choices of 16 rows of 32"""
    return (torch.rand((65536, 32), generator=gen, device=DEV).argsort(dim=1) < 16).to(torch.uint8)


def _masks(n, s, gen):
    """int32 [n, s]: words with exactly 16 bits set"""
    words = (_kept_rows(gen).to(torch.int64) << torch.arange(32, device=DEV)).sum(dim=1).to(torch.int32)
    return words[torch.randint(0, 65536, (n, s), generator=gen, device=DEV)]


def _weights(case, gen):
    """packed matrix, scales, zeros, mask: uniform codes are uniform words in every dense format"""
    bits, k, s, group = case["bits"], case["k"], case["s"], case["group"]
    rows = k // 16 if case["sparse"] else k * bits // 32
    groups = 1 if group < 0 else (k + group - 1) // group
    matrix = torch.randint(-2 ** 31, 2 ** 31, (rows, s), dtype=torch.int32, generator=gen, device=DEV)
    lo, hi = (0.001, 0.02) if bits == 4 else (0.004, 0.08)
    scales = torch.empty((groups, s), device=DEV).uniform_(lo, hi, generator=gen)
    if bits == 4:
        zeros = torch.empty((groups, s), device=DEV).uniform_(0.0, 15.0, generator=gen).half()
    else:
        zeros = torch.full((groups, s), (2 ** bits - 1) / 2, device=DEV).half()
    if case["expo"] > 0:
        chosen = torch.rand((groups, s), generator=gen, device=DEV) < case["expo"]
        # (an exponent-mode weight is z -+ s 2^e: a zero next to 0 and a scale that keeps 2^7 within the linear range)
        scales = torch.where(chosen, -scales / 2 ** (2 ** (bits - 1) - bits + 1), scales)
        zeros = torch.where(chosen, torch.zeros_like(zeros), zeros)
    mask = _masks(k // 32, s, gen) if case["sparse"] else None
    return matrix, scales.half(), zeros, mask


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    state = dict(case=case, ext=pkg.load_extension())
    if case["path"] == "pack":
        k, s = case["k"], case["s"]
        state["codes"] = torch.randint(0, 16, (s, k), dtype=torch.uint8, generator=gen, device=DEV)
        chosen = torch.randint(0, 65536, (s * k // 32,), generator=gen, device=DEV)
        state["kept"] = _kept_rows(gen)[chosen].reshape(s, k)
        return state
    state["x"] = torch.randn((case["batch"], case["rows"], case["k"]), generator=gen, device=DEV).half()
    layers = []
    for _ in range(case["layers"]):
        matrix, scales, zeros, mask = _weights(case, gen)
        if case["path"] == "linear":
            layers.append(QuantLinear.from_packed(case["bits"], matrix, scales, zeros, case["group"], mask))
        else:
            layers.append((matrix, scales, zeros, mask))
    state["layers"] = layers
    return state


def run(state):
    case = state["case"]
    if case["path"] == "pack":
        k, s = case["k"], case["s"]
        matrix = torch.empty((k // 16, s), dtype=torch.int32, device=DEV)
        mask = torch.empty((k // 32, s), dtype=torch.int32, device=DEV)
        state["ext"].weight_matrix_packing(matrix, mask, state["codes"], state["kept"])
        return matrix, mask
    x, outs = state["x"], []
    for layer in state["layers"]:
        if case["path"] == "linear":
            outs.append(layer(x))
        else:
            # a product of one row per sequence adds onto `out`, one of several overwrites it
            matrix, scales, zeros, mask = layer
            new = torch.zeros if case["rows"] == 1 else torch.empty
            out = new((case["batch"], case["rows"], case["s"]), dtype=torch.float16, device=x.device)
            state["ext"].quant_matmul(case["bits"], out, matrix, x, scales, zeros, case["group"], mask)
            outs.append(out)
    return outs


def work(case):
    k, s = case["k"], case["s"]
    if case["path"] == "pack":
        return {"bytes": 2 * k * s + 3 * k * s // 8, "flops": 0}
    n = case["batch"] * case["rows"]
    groups = 1 if case["group"] < 0 else (k + case["group"] - 1) // case["group"]
    packed = k * s * (3 if case["sparse"] else case["bits"]) // 8
    one = packed + 2 * groups * s * 2 + n * s * 2
    return {"bytes": case["layers"] * one + n * k * 2, "flops": case["layers"] * 2 * n * k * s}


def tolerance(case):
    if case["path"] == "pack":
        return "exact"
    # against float64 on unrounded weights the kernels that apply scale and zero in fp32 are at rel 2.1e-4, max 6e-4 (the
    # fp16 output's rounding); those that round each weight to fp16 twice, as the reference's decode does, at 3.3e-4, 1.9e-3
    return {"rel": 1.3e-3, "max": 8e-3}


def _codes(bits, matrix, mask):
    """uint8 [k, s] of a packed matrix; with a mask bool [k, s] of the rows kept, else None"""
    words = matrix.to(torch.int64) & 0xFFFFFFFF
    s = words.shape[1]
    if mask is None and bits != 3:
        shifts = torch.arange(0, 32, bits, device=words.device)[None, :, None]
        return ((words[:, None] >> shifts) & (2 ** bits - 1)).to(torch.uint8).reshape(-1, s), None
    if mask is None:
        # 32 codes of a column are a stream of 96 bits in three words
        words = words.reshape(-1, 3, s)
        codes = torch.empty((words.shape[0], 32, s), dtype=torch.uint8, device=words.device)
        for i in range(32):
            word, bit = divmod(3 * i, 32)
            value = words[:, word] >> bit
            if bit > 29:
                value = value | (words[:, word + 1] << (32 - bit))
            codes[:, i] = (value & 7).to(torch.uint8)
        return codes.reshape(-1, s), None
    # sixteen codes of 32 rows, in the order of the mask's set bits
    kept = ((mask[:, None].to(torch.int64) >> torch.arange(32, device=mask.device)[None, :, None]) & 1).to(torch.uint8)
    rank = kept.cumsum(dim=1, dtype=torch.int16) - kept
    stored = ((words[:, None] >> torch.arange(0, 32, 4, device=words.device)[None, :, None]) & 15).to(torch.uint8)
    stored = stored.reshape(-1, 16, s)
    codes = stored.gather(1, rank.clamp(max=15).to(torch.int64))
    return codes.reshape(-1, s), kept.reshape(-1, s).bool()


def exact(case, seed):
    """The products in float64, of weights that are not rounded on the way; packing gives whole numbers and has none."""
    if case["path"] == "pack":
        return None
    state, outs = prepare(case, seed), []
    x = state["x"].double()
    for layer in state["layers"]:
        if case["path"] == "linear":
            layer = layer.matrix, layer.scales.reshape(-1, case["s"]), layer.zeros.reshape(-1, case["s"]), layer.sparse_mask
        matrix, scales, zeros, mask = layer
        codes, kept = _codes(case["bits"], matrix, mask)
        out = torch.zeros((case["batch"] * case["rows"], case["s"]), dtype=torch.float64, device=DEV)
        step = case["k"] if case["group"] < 0 else case["group"]
        for group, first in enumerate(range(0, case["k"], step)):
            code = codes[first:first + step].double()
            scale, zero = scales[group].double(), zeros[group].double()
            half = 2 ** (case["bits"] - 1)
            power = torch.where(code >= half, -1.0, 1.0) * 2.0 ** (code % half)
            weight = torch.where(scale >= 0, (code - zero) * scale, zero - scale * power)
            if kept is not None:
                weight = weight * kept[first:first + step]
            out += x.reshape(-1, case["k"])[:, first:first + step] @ weight
        outs.append(out.reshape(case["batch"], case["rows"], case["s"]))
    return outs
