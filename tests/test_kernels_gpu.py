"""Each HIP kernel alone against a plain float32 reference of the same
operation, at sizes other than the engine's (odd widths, tails of tiles)."""
import math

import numpy as np
import pytest
import torch

import plain_impl
from litinfer_amd.engine.batch import AttentionMeta

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def tol(dtype, f32=1e-5, bf16=2e-2):
    return f32 if dtype is torch.float32 else bf16


def rel(got, ref):
    got = got.double().cpu().numpy() if isinstance(got, torch.Tensor) else got
    return float(np.abs(got - ref).max() / max(np.abs(ref).max(), 1e-30))


@pytest.fixture(scope="module")
def ops():
    from litinfer_amd.kernels import ops
    ops.require_gpu(DEV)
    return ops


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 2, 3), (50, 301, 120), (7, 1000, 4096)])
def test_embedding(ops, dtype, shape):
    t, v, h = shape
    g = torch.Generator().manual_seed(0)
    table = torch.randn(v, h, generator=g).to(dtype)
    ids = torch.randint(0, v, (t,), generator=g, dtype=torch.int32)
    out = torch.empty(t, h, device=DEV)
    ops.embedding(ids.to(DEV), table.to(DEV), out)
    ref = plain_impl.embedding(ids.numpy(), table.double().numpy())
    assert np.array_equal(out.double().cpu().numpy(), ref)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,eps", [((1, 4), 1e-5), ((33, 120), 1e-6), ((512, 4096), 1e-5), ((3, 3584), 1e-6),
                                        ((300, 1002), 1e-6), ((257, 8196), 1e-5), ((256, 20), 0.1)])      # many rows: of any length, too long for registers, short
def test_rmsnorm(ops, dtype, shape, eps):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(*shape, generator=g) * 3
    w = 1 + 0.1 * torch.randn(shape[1], generator=g)
    out = torch.empty(*shape, dtype=dtype, device=DEV)
    ops.rmsnorm(x.to(DEV), w.to(DEV), eps, out)
    ref = plain_impl.rms_norm(x.double().numpy(), w.double().numpy(), eps)
    assert rel(out, ref) < tol(dtype, 2e-6, 8e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(2, 70), (255, 1024), (255, 1025), (3, 9001), (256, 1025), (1100, 300)])      # few rows of one column a thread and more, many rows
def test_rmsnorm_of_bfloat16_rows(ops, dtype, shape):
    g = torch.Generator().manual_seed(84)
    x = (torch.randn(*shape, generator=g) * 3).to(torch.bfloat16)
    w = 1 + 0.1 * torch.randn(shape[1], generator=g)
    out = torch.full(shape, float("nan"), dtype=dtype, device=DEV)
    ops.rmsnorm(x.to(DEV), w.to(DEV), 1e-6, out)
    assert rel(out, plain_impl.rms_norm(x.double().numpy(), w.double().numpy(), 1e-6)) < tol(dtype, 2e-6, 8e-3)


def test_rmsnorm_zero_row_is_zero_not_nan(ops):
    x = torch.zeros(2, 64, device=DEV)
    out = torch.empty(2, 64, device=DEV)
    ops.rmsnorm(x, torch.ones(64, device=DEV), 1e-6, out)
    assert torch.equal(out, torch.zeros_like(out))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mnk,bias,acc", [
    ((2, 3, 4), True, False), ((1, 8, 16), False, False), ((5, 301, 120), True, False),
    ((70, 200, 96), False, True), ((130, 129, 264), True, True), ((512, 512, 1024), True, False),
    ((64, 3584, 3584), False, False), ((3, 37, 90), True, False), ((257, 64, 36), False, False),
    ((17, 37, 264), True, True), ((33, 130, 1160), False, False), ((48, 16, 8), True, False),
    ((8, 4608, 3584), True, False), ((65, 50, 128), False, True),
    ((1, 1000, 3584), True, False), ((16, 70, 260), True, True), ((40, 19, 100), False, True),      # few rows in 32-bit
    ((9, 18, 4), True, False),
    ((300, 200, 130), True, True), ((256, 128, 64), False, False), ((1000, 333, 1027), True, False),     # the large 32-bit tile
    ((2048, 3584, 128), True, True), ((2000, 4600, 64), True, False),           # large tiles, ragged
    ((1100, 4600, 128), True, True), ((1167, 6627, 128), False, False),         # a last row of tiles with few rows
    ((585, 3979, 128), True, False), ((779, 6296, 128), False, True)])          # columns that few tiles divide
def test_linear(ops, dtype, mnk, bias, acc):
    m, n, k = mnk
    g = torch.Generator().manual_seed(2)
    x = torch.randn(m, k, generator=g).to(dtype)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(dtype)
    b = torch.randn(n, generator=g) if bias else None
    ref = plain_impl.linear(x.double().numpy(), w.double().numpy(), None if b is None else b.double().numpy())
    if acc:
        base = torch.randn(m, n, generator=g)
        out = base.to(DEV)
        ref = ref + base.double().numpy()
    else:
        out = torch.empty(m, n, dtype=dtype, device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, accumulate=acc)
    # operands are exact in both dtypes; what differs is the float32 accumulation over K terms
    # (a random-walk error of about sqrt(K) half-ulps) and, for a bfloat16 out, its rounding
    assert rel(out, ref) < (4 * math.sqrt(k) * 2.0 ** -24 if out.dtype is torch.float32 else 5e-3)


# Tiles of many rows: rows and columns past the last, widths that no 16-byte piece divides, and one, an odd number and an even number of
# steps of 64 k-values (which tile each takes, and every tile in its steady state: test_every_tile_of_a_product).
@pytest.mark.parametrize("m,n,k,form", [
    (129, 32771, 64, "residual"), (129, 32776, 192, "bf16"), (769, 20488, 256, "relu2"),
    (641, 14344, 64, "residual"), (385, 20491, 320, "residual"), (705, 14341, 64, "bf16"), (385, 20488, 192, "relu2"),
    (385, 24584, 192, "residual"), (193, 32776, 320, "bf16"), (385, 24589, 128, "residual"),
    (769, 14344, 192, "residual"), (1537, 8200, 448, "residual"),
    (129, 8203, 64, "gated"), (130, 8200, 192, "gelu_gate"),
    (129, 16388, 320, "gated"), (257, 16388, 64, "clamped"), (300, 16385, 128, "gated"),
    (385, 10244, 192, "gated"), (385, 10241, 64, "gelu_gate"),
    (513, 8200, 320, "gated"), (577, 8200, 64, "gated"), (577, 8203, 192, "clamped"),
    (641, 10244, 64, "gelu_gate"), (577, 10241, 192, "gated"), (600, 10244, 448, "clamped")])
def test_linear_in_large_tiles(ops, m, n, k, form):
    _product_is_right(ops, m, n, k, form)


# Every tile of more than 64 rows that `tiling_of` and `gated_tiling_of` know, with each of its epilogues: more steps of 64 k-values than
# stages, an odd and an even number of them (so that stages are filled again while the loop runs, and the step of zeros behind an odd number
# takes the place of one that was in use), ragged both ways.  "pieces": stages handed back in pieces (gemm_bf16_tile_kernel).
@pytest.mark.parametrize("bm,bn,how,m,n,k,form", [
    (128, 128, "whole", 129, 8067, 448, "bf16"),
    (192, 128, "whole", 129, 16387, 320, "residual"), (192, 128, "whole", 129, 16392, 448, "relu2"),
    (256, 128, "whole", 385, 14339, 320, "residual"), (256, 128, "whole", 193, 16387, 512, "bf16"),
    (128, 224, "whole", 193, 16387, 320, "residual"), (128, 224, "whole", 257, 16387, 512, "bf16"), (128, 224, "whole", 257, 16392, 448, "relu2"),
    (256, 256, "whole", 641, 16387, 320, "residual"), (256, 256, "whole", 577, 16387, 384, "bf16"), (256, 256, "whole", 577, 16392, 448, "relu2"),
    (192, 224, "pieces", 385, 16387, 320, "residual"), (192, 224, "pieces", 257, 19075, 384, "bf16"), (192, 224, "pieces", 385, 16392, 448, "relu2"),
    (192, 256, "pieces", 385, 19075, 384, "residual"), (192, 256, "pieces", 577, 14339, 320, "bf16"), (192, 256, "pieces", 385, 19080, 448, "relu2"),
    (256, 224, "pieces", 641, 16387, 384, "residual"), (256, 224, "pieces", 385, 21763, 832, "residual"),
    (256, 224, "pieces", 577, 16387, 768, "bf16"), (256, 224, "pieces", 385, 21768, 1216, "relu2"),
    (256, 256, "pieces", 577, 19075, 1536, "residual"), (256, 256, "pieces", 577, 19075, 3520, "bf16"), (256, 256, "pieces", 577, 19080, 1536, "relu2"),
    (128, 128, "gated", 300, 1003, 448, "clamped"),
    (128, 192, "gated", 129, 8195, 320, "gated"), (128, 192, "gated", 130, 8195, 384, "gelu_gate"), (128, 192, "gated", 129, 8200, 448, "clamped"),
    (128, 256, "gated", 257, 8195, 320, "gated"), (128, 256, "gated", 257, 8195, 384, "gelu_gate"), (128, 256, "gated", 257, 8200, 448, "clamped"),
    (256, 128, "gated", 641, 5379, 320, "gated"), (256, 128, "gated", 641, 5379, 512, "gelu_gate"), (256, 128, "gated", 641, 5384, 448, "clamped"),
    (256, 256, "gated", 641, 8195, 320, "gated"), (256, 256, "gated", 385, 9283, 64, "gelu_gate"), (256, 256, "gated", 641, 8200, 448, "clamped"),
    (128, 320, "gated pieces", 385, 8195, 320, "gated"), (128, 320, "gated pieces", 385, 8195, 384, "gelu_gate"), (128, 320, "gated pieces", 385, 8200, 448, "clamped"),
    (192, 256, "gated pieces", 513, 8195, 320, "gated"), (192, 256, "gated pieces", 513, 8195, 384, "gelu_gate"), (192, 256, "gated pieces", 513, 8200, 448, "clamped"),
    (192, 320, "gated pieces", 769, 6531, 384, "gated"), (192, 320, "gated pieces", 1025, 6531, 320, "gelu_gate"), (192, 320, "gated pieces", 1025, 6536, 448, "clamped"),
    (256, 192, "gated pieces", 385, 10883, 320, "gated"), (256, 192, "gated pieces", 385, 10883, 384, "gelu_gate"), (256, 192, "gated pieces", 385, 10888, 448, "clamped"),
    (256, 256, "gated pieces", 577, 8195, 384, "gated"), (256, 256, "gated pieces", 1537, 4483, 1600, "gelu_gate"), (256, 256, "gated pieces", 577, 8200, 512, "clamped")])
def test_every_tile_of_a_product(ops, bm, bn, how, m, n, k, form):
    import ctypes
    gated = how.startswith("gated")
    tile = ops._lib_fn("gemm", "li_linear_tile", [ctypes.c_int] * 5, ctypes.c_int)
    units = torch.cuda.get_device_properties(0).multi_processor_count
    if units == 256:                                          # (the sizes are for that many)
        assert tile(int(gated), m, 2 * n if gated else n, k, 8 if form == "residual" else 2) == (-1 if "pieces" in how else 1) * (bm * 65536 + bn)
    _product_is_right(ops, m, n, k, form)


def _product_is_right(ops, m, n, k, form):
    g = torch.Generator(device=DEV).manual_seed(91)
    gated = form in ("gated", "gelu_gate", "clamped")
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn((2 if gated else 1) * n, k, generator=g, device=DEV) * 2 / math.sqrt(k)).bfloat16()
    y = x.double() @ w.double().t()
    # the float32 sums of K products (a random walk of half-ulps of terms of size y), carried on by slopes of 3 at most
    slack = 12 * math.sqrt(k) * 2.0 ** -24 * (1 + y.abs())
    if gated:
        gate, up = y[:, :n], y[:, n:]
        slack = (slack[:, :n] + slack[:, n:]) * (1 + gate.abs() + up.abs())
        limit = {"gated": 0.0, "gelu_gate": ops.GELU_TANH_GATE, "clamped": 1.5}[form]
        if form == "gated":
            want = up * gate * torch.sigmoid(gate)
        elif form == "gelu_gate":
            want = up * torch.nn.functional.gelu(gate, approximate="tanh")
        else:
            gc, uc = gate.clamp(max=1.5), up.clamp(-1.5, 1.5)
            want = gc * torch.sigmoid(1.702 * gc) * (uc + 1)
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.linear_swiglu(x, w, out, limit=limit)
    else:
        b = torch.randn(n, generator=g, device=DEV)
        y = y + b.double()
        if form == "residual":
            out = torch.randn(m, n, generator=g, device=DEV)
            want = out.double() + 0.5 * y
            ops.linear(x, w, b, out, accumulate=True, factor=0.5)
        elif form == "bf16":
            out, want = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV), y
            ops.linear(x, w, b, out)
        else:
            out, want = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV), y.clamp(min=0) ** 2
            slack = slack * (1 + y.abs())
            assert ops.linear_act(x, w, b, out, "relu2", (0.0, 0.0), None)
    if out.dtype is torch.bfloat16:
        slack = slack + want.abs() * 2.0 ** -8
    assert bool(((out.double() - want).abs() <= slack).all())


@pytest.mark.parametrize("m,n,k,swiglu,out_dtype,bias,acc", [
    (1, 16, 8, False, torch.bfloat16, False, False),
    (8, 4608, 3584, False, torch.bfloat16, True, False),        # decode: qkv + bias
    (8, 18944, 3584, True, torch.bfloat16, False, False),       # decode: gate/up + swiglu
    (8, 3584, 18944, False, torch.float32, False, True),        # decode: down + residual
    (5, 301, 120, False, torch.float32, False, False),          # odd sizes: head
    (17, 200, 96, True, torch.bfloat16, False, False),
    (32, 37, 264, False, torch.bfloat16, True, False),
    (33, 130, 1160, True, torch.bfloat16, False, False),
    (64, 50, 128, False, torch.float32, True, True),
    (7, 2049, 72, False, torch.float32, True, True),            # few columns: 9 a block, the last block ragged
    (16, 4100, 40, False, torch.bfloat16, True, False),         # 17 a block: two tiles, the second nearly empty
    (12, 8191, 32, False, torch.bfloat16, False, False),        # 32 a block
    (24, 4100, 72, False, torch.float32, True, True),           # the same shares with 17 to 32 rows
    (30, 2500, 40, False, torch.bfloat16, False, False),
    (3, 9000, 64, False, torch.bfloat16, True, False),          # wide output: two tiles a wave
    (16, 8200, 1160, False, torch.float32, True, True),         # wide outputs at other sizes
    (7, 40000, 264, False, torch.float32, False, False),
    (11, 8300, 520, True, torch.bfloat16, False, False),
    (1, 152064, 64, False, torch.float32, False, False),
    (20, 9000, 520, False, torch.bfloat16, False, False),
    (4, 8960, 64, True, torch.bfloat16, False, False),          # gate/up in equal shares of the columns: 12 a block,
    (25, 4101, 40, True, torch.bfloat16, False, False),         # 9 a block with a ragged last one,
    (40, 4864, 72, True, torch.bfloat16, False, False),         # 10 a block
])
def test_linear_skinny_with_fused_swiglu(ops, m, n, k, swiglu, out_dtype, bias, acc):
    g = torch.Generator().manual_seed(12)
    x = (torch.randn(m, k, generator=g) * 2).to(torch.bfloat16)
    w = (torch.randn(2 * n if swiglu else n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) if bias else None
    y = x.double().numpy() @ w.double().numpy().T
    if swiglu:
        y = plain_impl.swiglu(y[:, :n], y[:, n:])
    if b is not None:
        y = y + b.double().numpy()
    if acc:
        base = torch.randn(m, n, generator=g)
        out = base.to(DEV)
        y = y + base.double().numpy()
    else:
        out = torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)     # a column left out shows
    assert ops.skinny_takes(m, k, w.dtype)
    ops.linear_skinny(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, acc, swiglu=swiglu)
    assert rel(out, y) < (4 * math.sqrt(k) * 2.0 ** -24 if out_dtype is torch.float32 else 5e-3)


class _Lender:
    """Stands in for the engine's workspace."""
    made = 0

    def buffer(self, name, shape, dtype, zero=False):
        self.made += 1
        return (torch.zeros if zero else torch.empty)(*shape, dtype=dtype, device=DEV)


@pytest.mark.parametrize("m,n,k,out_dtype,bias,acc", [
    (33, 200, 1024, torch.float32, True, True),          # K in parts: few tiles
    (64, 3584, 3584, torch.float32, False, True),
    (48, 300, 18944, torch.bfloat16, True, False),
    (64, 136, 512, torch.bfloat16, False, False),        # too short a K for parts
    (40, 20000, 128, torch.float32, True, False),        # many tiles of 128 columns
    (64, 37000, 64, torch.bfloat16, False, False),       # many tiles of 256 columns
    (128, 3584, 18944, torch.float32, False, True),      # more rows, but few tiles over a long K: parts again
    (200, 300, 4096, torch.bfloat16, True, False),
    (500, 1000, 1024, torch.float32, True, False),       # 32 tiles, two parts
    (13, 3584, 18944, torch.float32, True, True),        # the fewest rows that take the tiles with K in parts (a large matrix)
    (16, 3584, 3584, torch.float32, True, True),         # a small one at 16 rows: the few-row kernel
    (50, 4608, 3584, torch.bfloat16, True, False),       # 36 tiles in 7 parts: not whole eighths, the XCDs share one sequence
    (384, 3584, 2048, torch.float32, False, True),       # 84 tiles in 3 parts, three rows of tiles
    (130, 2048, 1536, torch.float32, True, True),        # 32 tiles in 3 parts: an eighth of the tiles each, part by part
    (64, 1100, 1984, torch.bfloat16, False, False),      # 9 tiles in 3 parts of 11, 10 and 10 steps
])
def test_linear_with_k_in_parts(ops, m, n, k, out_dtype, bias, acc):
    g = torch.Generator().manual_seed(15)
    x = (torch.randn(m, k, generator=g) * 2).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) if bias else None
    y = x.double().numpy() @ w.double().numpy().T
    if b is not None:
        y = y + b.double().numpy()
    if acc:
        base = torch.randn(m, n, generator=g)
        y = y + base.double().numpy()
    outs = []
    for ws in (_Lender(), None):                         # with and without memory for partial sums
        out = base.to(DEV) if acc else torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)
        ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, acc, ws=ws)
        assert rel(out, y) < (4 * math.sqrt(k) * 2.0 ** -24 if out_dtype is torch.float32 else 5e-3)
        outs.append(out)
    again = base.to(DEV) if acc else torch.empty(m, n, dtype=out_dtype, device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), again, acc, ws=_Lender())
    assert torch.equal(again, outs[0])                   # the parts are added in a fixed order


@pytest.mark.parametrize("m,n,k,bias,factor", [
    (65, 100, 204, False, 1.0),              # one row more than the few-row kernel takes; parts of 7 and 6 steps, the last step of 12 k-values
    (129, 1536, 8960, True, 1.0),            # the most parts
    (300, 1537, 1540, True, 0.5),            # a column and a piece of a step over
    (810, 1536, 1536, False, 1.0),
    (257, 260, 4096, True, 0.0),             # not accumulating
    (2048, 300, 92, True, 1.0),              # too short a K for parts
    (65, 4, 4, False, 1.0),                  # a quarter of a step
    (70, 130, 20, True, 1.0),                # one whole step and a quarter
    (129, 257, 36, False, 0.5),              # two and a quarter, tiles of one row and one column
    (200, 96, 52, True, 1.0),                # three and a quarter: the loop's first whole round
])
def test_float32_linear_with_k_in_parts(ops, m, n, k, bias, factor):
    from litinfer_amd.kernels.ops import _work_bytes
    g = torch.Generator().manual_seed(62)
    x = torch.randn(m, k, generator=g)
    w = torch.randn(n, k, generator=g) / math.sqrt(k)
    b = torch.randn(n, generator=g) if bias else None
    base = torch.randn(m, n, generator=g)
    assert (_work_bytes(m, n, k, 0) > 0) == (k > 100)          # the case is what it says
    y = x.double().numpy() @ w.double().numpy().T + (0 if b is None else b.double().numpy())
    y = base.double().numpy() + factor * y if factor else y
    outs = []
    for ws in (_Lender(), None, _Lender()):
        out = base.to(DEV) if factor else torch.full((m, n), float("nan"), device=DEV)
        ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, bool(factor), ws=ws, factor=factor or 1.0)
        assert rel(out, y) < 4 * math.sqrt(k) * 2.0 ** -24     # (as for the product in one piece)
        outs.append(out)
    assert torch.equal(outs[0], outs[2])                       # the parts are added in a fixed order


@pytest.mark.parametrize("m,n,k,bias,factor", [
    (8, 1536, 8960, False, 1.0),             # six columns a block, the most trips
    (3, 2048, 1536, True, 0.0),              # eight columns a block
    (8, 2049, 1540, True, 0.5),              # nine: both halves of a piece one after the other; one piece of a row over
    (9, 1536, 1536, False, 0.0),             # a row more than both halves of a piece take
    (1, 5, 4, True, 1.0),                    # one column a block, a single 16-byte piece a row
    (7, 300, 20, False, 0.0),                # the second half of the only piece is cut
    (8, 257, 8212, True, 1.0),               # the last piece ends inside its second half
    (4, 300, 2052, False, 1.0),              # four pieces a trip: one trip and a piece of its own half over
    (5, 300, 2052, False, 0.0),              # ... a row more: one piece a trip
    (2, 100, 4096, True, 0.5),
])
def test_float32_linear_of_few_rows_and_columns(ops, m, n, k, bias, factor):
    g = torch.Generator().manual_seed(63)
    x = torch.randn(m, k, generator=g)
    w = torch.randn(n, k, generator=g) / math.sqrt(k)
    b = torch.randn(n, generator=g) if bias else None
    base = torch.randn(m, n, generator=g)
    y = x.double().numpy() @ w.double().numpy().T + (0 if b is None else b.double().numpy())
    y = base.double().numpy() + factor * y if factor else y
    out = base.to(DEV) if factor else torch.full((m, n), float("nan"), device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, bool(factor), factor=factor or 1.0)
    assert rel(out, y) < 4 * math.sqrt(k) * 2.0 ** -24         # (sums of k float32 products)


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [
    (5, 64), (200, 448),                 # fewer units of 64 than waves: some waves have none
    (897, 512), (1536, 2048),            # up to four units a wave, a ragged last block; the longest rows of a wide matrix
    (5000, 1088), (9000, 192),           # more columns than a round of blocks
    (300, 2112), (70, 5120),             # five to ten units a wave at once
    (33, 5184), (300, 8960),             # ... and in rounds of four: a last round of one unit, of two
])
def test_products_of_one_to_four_rows(ops, m, n, k):
    g = torch.Generator().manual_seed(81)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b, base = torch.randn(n, generator=g), torch.randn(m, n, generator=g)
    y = x.double().numpy() @ w.double().numpy().T + b.double().numpy()
    bound = 4 * math.sqrt(k) * 2.0 ** -24                       # sums of k float32 products
    plain = torch.full((m, n), float("nan"), device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), plain)
    assert rel(plain, y) < bound
    added = base.to(DEV)
    ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), added, True, factor=0.5)
    assert rel(added, base.double().numpy() + 0.5 * y) < bound
    short = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), short)
    assert rel(short, y) < 2.0 ** -8
    if n % 8 == 0:
        assert ops.linear_act(x.to(DEV), w.to(DEV), b.to(DEV), short, "relu2")
        assert rel(short, np.maximum(y, 0) ** 2) < 2.0 ** -8
    # a value that is not finite stays with its row
    x[m - 1, k - 1] = float("inf")
    ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), plain)
    assert rel(plain[:m - 1], y[:m - 1]) < bound if m > 1 else True
    assert not torch.isfinite(plain[m - 1]).any()


@pytest.mark.parametrize("m", [33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(64, 512), (1536, 1536), (1100, 1032), (4096, 1024), (2048, 2048)])      # the last one up to 48 rows only
def test_products_of_33_to_64_rows_against_small_matrices(ops, m, n, k):
    assert ops.four_tiles_preferred(m, n, k) == (m <= 48 or k <= 1536)
    g = torch.Generator().manual_seed(82)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b, base = torch.randn(n, generator=g), torch.randn(m, n, generator=g) * torch.logspace(-2, 2, m)[:, None]
    gamma, beta, eps = torch.rand(n, generator=g) + 0.5, torch.randn(n, generator=g), 1e-5
    y = base.double().numpy() + x.double().numpy() @ w.double().numpy().T + b.double().numpy()
    bound = 4 * math.sqrt(k) * 2.0 ** -24
    alone, xn = base.to(DEV), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), alone, True, ws=_Lender())
    for i in range(m):
        assert rel(alone[i], y[i]) < bound, i
    # with a norm behind it: wherever K has whole steps (the last product above 48 rows in parts), and where not, nothing is touched;
    # K whole takes no lent memory
    out, lent = base.to(DEV), _Lender()
    if k % 64:
        assert not ops.linear_then_norm(x.to(DEV), w.to(DEV), b.to(DEV), out, gamma.to(DEV), eps, xn, lent)
        assert not ops.linear_tanh_norm(x.to(DEV), w.to(DEV), b.to(DEV), out, 0.7, gamma.to(DEV), beta.to(DEV), xn, lent)
        assert torch.equal(out.cpu(), base) and torch.isnan(xn.float()).all()
    else:
        assert ops.linear_then_norm(x.to(DEV), w.to(DEV), b.to(DEV), out, gamma.to(DEV), eps, xn, lent)
        assert torch.equal(out, alone)
        ref = plain_impl.rms_norm(y, gamma.double().numpy(), eps)
        for i in range(m):
            assert rel(xn[i], ref[i]) < 8e-3, i
        out, xn = base.to(DEV), torch.full_like(xn, float("nan"))
        assert ops.linear_tanh_norm(x.to(DEV), w.to(DEV), b.to(DEV), out, 0.7, gamma.to(DEV), beta.to(DEV), xn, lent)
        assert rel(out, y) < bound and rel(xn, np.tanh(0.7 * y) * gamma.double().numpy() + beta.double().numpy()) < 8e-3
        short = torch.empty_like(xn)
        assert ops.linear_act(x.to(DEV), w.to(DEV), b.to(DEV), short, "relu2", ws=lent)
        assert bool(lent.made) == (not ops.four_tiles_preferred(m, n, k))
    # the packed projection with rotary encoding and page write, in one launch
    if n % 64 == 0 and n >= 256:
        nkv, dh, page = 1, 64, 16
        nh = n // dh - 2
        pos = torch.randint(0, 3000, (m,), generator=g, dtype=torch.int32)
        slots = torch.randperm(5 * page, generator=g)[:m].to(torch.int32)
        cos, sin = torch.empty(m, dh // 2, device=DEV), torch.empty(m, dh // 2, device=DEV)
        ops.rope_table(pos.to(DEV), 1e6, dh, cos, sin)
        kc = torch.zeros((5, nkv, page, dh), dtype=torch.bfloat16, device=DEV)
        vc, q = torch.zeros_like(kc), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert ops.linear_rope_store_parts(x.to(DEV), w.to(DEV), b.to(DEV), q, nh, nkv, dh, cos, sin, slots.to(DEV), kc, vc, page, _Lender())
        yq = (y - base.double().numpy()).reshape(m, nh + 2 * nkv, dh)
        ref = np.concatenate([plain_impl.rope_neox(yq[:, :nh + nkv], pos.numpy(), 1e6), yq[:, nh + nkv:]], axis=1)
        assert rel(q, ref.reshape(m, n)) < 5e-3
        qv = q.cpu().view(m, nh + 2 * nkv, dh)
        for i in range(m):
            sl = int(slots[i])
            assert torch.equal(kc[sl // page, :, sl % page].cpu(), qv[i, nh:nh + nkv]) and torch.equal(vc[sl // page, :, sl % page].cpu(), qv[i, nh + nkv:])


@pytest.mark.parametrize("m,n,k", [(48, 1536, 1536), (64, 4096, 1024), (64, 3584, 3584)])      # K whole, twice, and in parts
def test_norm_behind_a_product_that_counts_for_nothing(ops, m, n, k):
    g = torch.Generator().manual_seed(83)
    x, w = torch.randn(m, k, generator=g).to(torch.bfloat16), torch.randn(n, k, generator=g).to(torch.bfloat16)
    base, gamma = torch.randn(m, n, generator=g), torch.rand(n, generator=g) + 0.5
    out, xn = base.to(DEV), torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV)
    assert ops.linear_then_norm(x.to(DEV), w.to(DEV), None, out, gamma.to(DEV), 1e-5, xn, _Lender(), factor=0.0)
    assert torch.equal(out.cpu(), base)
    assert rel(xn, plain_impl.rms_norm(base.double().numpy(), gamma.double().numpy(), 1e-5)) < 4 * math.sqrt(n) * 2.0 ** -24


@pytest.mark.parametrize("m,n,k,bias,taken", [
    (64, 3584, 18944, False, True),      # a decoding batch of 64 at the 7B sizes
    (40, 200, 1024, True, True),
    (200, 300, 4096, True, True),        # more than 64 rows, few tiles
    (64, 37000, 64, False, False),       # no cut along K: nothing is done
    (8, 200, 1024, False, False),        # few rows: another kernel's business
    (12, 3584, 18944, False, False),     # the most rows of that kernel's whatever the matrix
    (13, 3584, 3584, True, False),       # 13 to 16 rows against a small matrix: still the few-row kernel
    (13, 3584, 18944, True, True),       # against a large one (136 MB): tiles with K in parts
])
def test_linear_into_the_residual_sum_with_its_norm(ops, m, n, k, bias, taken):
    g = torch.Generator().manual_seed(19)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) * 0.1 if bias else None
    base = torch.randn(m, n, generator=g) * torch.logspace(-2, 2, m)[:, None]       # rows of very different size
    gamma, eps = torch.rand(n, generator=g) + 0.5, 1e-5
    out = base.to(DEV)
    xn = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    did = ops.linear_then_norm(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, gamma.to(DEV), eps, xn, _Lender())
    assert did == taken
    if not taken:
        assert torch.equal(out.cpu(), base) and torch.isnan(xn.float()).all()        # nothing was touched
        return
    y = base.double().numpy() + x.double().numpy() @ w.double().numpy().T + (0 if b is None else b.double().numpy())
    ref = plain_impl.rms_norm(y, gamma.double().numpy(), eps)
    for i in range(m):
        assert rel(out[i], y[i]) < 4 * math.sqrt(k) * 2.0 ** -24, i
        assert rel(xn[i], ref[i]) < 8e-3, i
    # the sum is the one that the product alone leaves, bit for bit
    alone = base.to(DEV)
    ops.linear(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), alone, True, ws=_Lender())
    assert torch.equal(alone, out)
    # and the norm is the one that the norm's own kernel makes of that sum, up to the order of its additions
    own = torch.empty_like(xn)
    ops.rmsnorm(out, gamma.to(DEV), eps, own)
    assert (own.float() - xn.float()).abs().max().item() <= 2.0 ** -7 * own.float().abs().max().item()


@pytest.mark.parametrize("m,n,k,bias", [(255, 1536, 1536, True), (256, 1536, 1536, True), (1027, 1536, 1024, False), (300, 512, 8192, True), (700, 896, 1088, False),
                                        (257, 2052, 2048, True), (256, 4096, 1024, False), (300, 5124, 1024, True), (256, 8192, 1024, False), (300, 1538, 4096, True),
                                        (257, 4096, 1024, True), (258, 8192, 1024, False), (280, 2048, 4864, True), (599, 1536, 8960, True), (600, 1536, 8960, True)])
def test_parts_of_many_rows_with_their_norm(ops, m, n, k, bias):
    """From 256 rows on four columns a load: two, three, four and eight parts; one to eight pieces a thread; rows of no multiple of four."""
    test_linear_into_the_residual_sum_with_its_norm(ops, m, n, k, bias, ops._work_bytes(m, n, k, ops._DT[torch.bfloat16]) > 0)


@pytest.mark.parametrize("m,n,k", [
    (8, 200, 96),                # few rows: the decode kernel
    (13, 9500, 128),             # 13 to 64 rows: tiles of 64 rows
    (40, 20000, 128),
    (64, 9500, 192),
    (50, 18944, 128),            # tiles of 64 x 192: the gates in one wave, the ups in the wave beside it
    (33, 12300, 192),            # the same with a ragged last tile
    (65, 32, 64),                # one tile, one step of K
    (100, 200, 128),             # an output width that is no multiple of 32
    (300, 1000, 192),            # several tiles both ways, ragged edges
    (700, 4700, 256),            # (which tiles the larger ones take, and every tile there is: test_every_tile_of_a_product)
    (2048, 18944, 128),          # enough tiles for the largest tiling
    (97, 7419, 128),             # few rows against many columns
    (300, 9001, 128),
    (1101, 2500, 192),           # several rows of tiles: the last XCD's share of the tiles is short
    (1024, 4800, 192),
    (2000, 4793, 192),           # ragged edges both ways
])
def test_linear_with_swiglu_epilogue(ops, m, n, k):
    g = torch.Generator().manual_seed(14)
    x = (torch.randn(m, k, generator=g) * 2).to(torch.bfloat16)
    w = (torch.randn(2 * n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    y = x.double().numpy() @ w.double().numpy().T
    y = plain_impl.swiglu(y[:, :n], y[:, n:])
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.swiglu_takes(m, k, w.dtype)
    ops.linear_swiglu(x.to(DEV), w.to(DEV), out)
    assert rel(out, y) < 5e-3
    # a gate far from zero either way and single outputs that stand out
    w2 = torch.zeros(2 * n, k)
    w2[3, 0] = 30.0; w2[n + 3, 0] = 1.0          # silu(+large) * up
    w2[5, 0] = -30.0; w2[n + 5, 0] = 1.0         # silu(-large) -> 0
    w2[n - 1, 1] = 1.0; w2[2 * n - 1, 1] = 2.0   # the last output
    x2 = torch.zeros(m, k); x2[:, 0] = 1.0; x2[m - 1, 1] = 3.0
    ops.linear_swiglu(x2.to(torch.bfloat16).to(DEV), w2.to(torch.bfloat16).to(DEV), out)
    o = out.float().cpu()
    assert abs(o[0, 3].item() - 30.0) < 0.2 and abs(o[0, 5].item()) < 1e-9
    want_last = 2.0 * 3.0 * (3.0 / (1 + math.exp(-3.0)))
    assert abs(o[m - 1, n - 1].item() - want_last) < 0.1 and o[0, n - 1].item() == 0.0
    assert torch.count_nonzero(o).item() <= 2 * m + 1


@pytest.mark.parametrize("m,inter,k", [(1, 300, 264), (8, 2000, 3584), (16, 37, 100), (17, 4200, 512), (33, 200, 96),
                                       (64, 500, 128), (5, 9000, 1160), (40, 16500, 64)])
def test_float32_few_row_product_with_swiglu_epilogue(ops, m, inter, k):
    """The 32-bit path's gate/up product of a decoding step: on the float32 matrix cores, the activation in
    the epilogue; one, two and four row tiles, one to four column tiles, short and long K."""
    g = torch.Generator().manual_seed(12)
    x = torch.randn(m, k, generator=g)
    w = torch.randn(2 * inter, k, generator=g) / math.sqrt(k)
    y = x.double().numpy() @ w.double().numpy().T
    ref = plain_impl.swiglu(y[:, :inter], y[:, inter:])
    out = torch.full((m, inter), float("nan"), device=DEV)
    assert ops.swiglu_takes(m, k, torch.float32) == (m <= 16)         # (the parts ask; the kernel takes up to 64 rows)
    ops.linear_swiglu(x.to(DEV), w.to(DEV), out)
    assert rel(out, ref) < 8 * math.sqrt(k) * 2.0 ** -24


@pytest.mark.parametrize("m,n,kprev,inter,eps", [
    (8, 3584, 512, 1024, 1e-6),      # a decoding step at the 7B width
    (8, 5120, 256, 27648, 1e-6),     # the 32B's gate/up matrix (566 MB): tiles of 64 x 256 scale the rows
    (3, 3584, 512, 18944, 1e-6),     # the 7B's (272 MB): tiles of 64 x 192
    (16, 5120, 128, 20480, 1e-5),    # 419 MB: tiles of 64 x 192, gates and ups in two waves
    (1, 40, 8, 24, 1e-5),
    (16, 8200, 64, 48, 1e-5),        # a width from which the product before takes 32 columns a block; ragged
    (5, 200, 136, 301, 0.1),         # a ragged last block of 16 columns; an eps that counts
    (9, 264, 72, 8210, 1e-5),        # many outputs, ragged; fewer chunks of K than waves
    (4, 1096, 40, 9000, 1e-6),
    (17, 3584, 512, 1024, 1e-6),     # two tiles of rows a block: the same three ways out, 32 places a block for the shares
    (32, 1536, 8960, 8960, 1e-6),    # the 1.5B's sizes at 32 rows: few-row kernels on both sides
    (24, 3584, 512, 18944, 1e-6),    # the 7B's gate/up at 24 rows: tiles of 64 x 192 scale 24 rows
    (29, 5120, 128, 20480, 1e-5),    # gates and ups in two waves
    (19, 8200, 64, 48, 1e-5),
    (32, 200, 136, 301, 0.1),
    (21, 264, 72, 8210, 1e-5),
])
def test_rms_norm_shared_between_the_products_on_its_two_sides(ops, m, n, kprev, inter, eps):
    """x += h Wo^T leaves gamma * x and the shares of the rows' sums of squares; the gate/up product
    with SwiGLU (and the packed projection with rotary encoding and page write) scales its rows."""
    g = torch.Generator().manual_seed(18)
    h = torch.randn(m, kprev, generator=g).to(torch.bfloat16)
    wo = (torch.randn(n, kprev, generator=g) / math.sqrt(kprev)).to(torch.bfloat16)
    bias = torch.randn(n, generator=g) * 0.1
    base = torch.randn(m, n, generator=g) * torch.logspace(-2, 2, m)[:, None]       # rows of very different size
    gamma = torch.rand(n, generator=g) + 0.5
    x = base.double().numpy() + h.double().numpy() @ wo.double().numpy().T + bias.double().numpy()
    assert ops.residual_norm_takes(m, n, kprev, wo.dtype)
    out = base.to(DEV)
    xg = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    places = ops.row_scale_rows(m)                       # 16 up to 16 rows, 32 above
    parts = torch.full((ops.RESIDUAL_NORM_MAX_PARTS * places,), float("nan"), device=DEV)
    nparts = ops.linear_residual_norm(h.to(DEV), wo.to(DEV), bias.to(DEV), out, gamma.to(DEV), xg, parts)
    assert nparts == ops.residual_norm_parts(n) <= ops.RESIDUAL_NORM_MAX_PARTS
    for i in range(m):
        assert rel(out[i], x[i]) < 1e-5, i
        assert rel(xg[i], gamma.double().numpy() * x[i]) < 2.0 ** -8, i
    sq = parts[:nparts * places].view(nparts, places)[:, :m].double().sum(dim=0).cpu().numpy()
    assert np.allclose(sq, (x * x).sum(axis=1), rtol=1e-5)
    # the same sum as the product alone leaves it
    alone = base.to(DEV)
    ops.linear(h.to(DEV), wo.to(DEV), bias.to(DEV), alone, True)
    assert torch.equal(alone, out)
    scale = ops.RowScale(parts, nparts, eps)
    xn = plain_impl.rms_norm(x, gamma.double().numpy(), eps)
    xb = xg.double().cpu().numpy()                       # what the product after the norm multiplies
    inv = 1.0 / np.sqrt((x * x).mean(axis=1, keepdims=True) + eps)
    # -- gate/up with SwiGLU
    w = (torch.randn(2 * inter, n, generator=g) / math.sqrt(n)).to(torch.bfloat16)
    y = xn @ w.double().numpy().T
    ref = plain_impl.swiglu(y[:, :inter], y[:, inter:])
    got = torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear_swiglu(xg, w.to(DEV), got, row_scale=scale)
    yb = (xb @ w.double().numpy().T) * inv
    refb = plain_impl.swiglu(yb[:, :inter], yb[:, inter:])
    for i in range(m):                                   # the kernel's own arithmetic, row by row
        assert rel(got[i], refb[i]) < 5e-3, i
    # against the plain norm and product, element by element within what rounding the rows to
    # bfloat16 (each term by at most 2^-9 of itself) and the output can do:
    # |d out| <= |silu(g)| |d u| + |u| |silu'(g)| |d g| + 2^-9 |out|, |silu'| <= 1.1
    ya = np.abs(xn) @ np.abs(w.double().numpy()).T
    g_, u_ = y[:, :inter], y[:, inter:]
    bound = 2.0 ** -9 * (np.abs(g_ / (1 + np.exp(-g_))) * ya[:, inter:] + 1.1 * np.abs(u_) * ya[:, :inter] + np.abs(ref))
    err = np.abs(got.double().cpu().numpy() - ref)
    assert (err <= 1.01 * bound + 1e-30).all(), float((err / (bound + 1e-30)).max())
    # -- the packed projection with rotary encoding and page write
    nh, nkv, dh, page, pages = 3, 1, 32, 8, 5
    nq = (nh + 2 * nkv) * dh
    wq = (torch.randn(nq, n, generator=g) / math.sqrt(n)).to(torch.bfloat16)
    bq = torch.randn(nq, generator=g)
    pos = torch.randint(0, 3000, (m,), generator=g, dtype=torch.int32)
    slots = torch.randperm(pages * page, generator=g)[:m].to(torch.int32)
    cos = torch.empty(m, dh // 2, device=DEV)
    sin = torch.empty(m, dh // 2, device=DEV)
    ops.rope_table(pos.to(DEV), 1e6, dh, cos, sin)
    kc = torch.zeros((pages, nkv, page, dh), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    q = torch.full((m, nq), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear_rope_store(xg, wq.to(DEV), bq.to(DEV), q, nh, nkv, dh, cos, sin, slots.to(DEV), kc, vc, page,
                          row_scale=scale)
    yq = ((xb @ wq.double().numpy().T) * inv + bq.double().numpy()).reshape(m, nh + 2 * nkv, dh)
    refq = np.concatenate([plain_impl.rope_neox(yq[:, :nh + nkv], pos.numpy(), 1e6), yq[:, nh + nkv:]], axis=1)
    assert rel(q, refq.reshape(m, nq)) < 5e-3
    qv = q.cpu().view(m, nh + 2 * nkv, dh)
    for i in range(m):
        sl = int(slots[i])
        assert torch.equal(kc[sl // page, :, sl % page].cpu(), qv[i, nh:nh + nkv])
        assert torch.equal(vc[sl // page, :, sl % page].cpu(), qv[i, nh + nkv:])
    with pytest.raises(ValueError):                      # more rows than the kernels scale
        ops.linear_swiglu(torch.zeros(33, n, dtype=torch.bfloat16, device=DEV), w.to(DEV),
                          torch.empty(33, inter, dtype=torch.bfloat16, device=DEV), row_scale=scale)


@pytest.mark.parametrize("dtype", DTYPES)
def test_linear_rows_do_not_depend_on_the_batch(ops, dtype):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(200, 264, generator=g).to(dtype).to(DEV)
    w = torch.randn(150, 264, generator=g).to(dtype).to(DEV)
    full = torch.empty(200, 150, dtype=torch.float32, device=DEV)
    ops.linear(x, w, None, full)
    for rows in (slice(0, 1), slice(17, 19), slice(100, 200)):
        part = torch.empty(rows.stop - rows.start, 150, dtype=torch.float32, device=DEV)
        ops.linear(x[rows].contiguous(), w, None, part)
        # kernels for few and for many rows may add the K terms in another order: rounding only
        assert rel(part, full[rows].double().cpu().numpy()) < 4 * math.sqrt(264) * 2.0 ** -24


def test_the_rule_for_few_rows_is_the_same_in_the_library_and_in_the_host_stand_in(ops):
    # parts ask the kernel library which kernels few rows should take; the stand-in that the host-side tests
    # run the parts with answers the same
    import torch_ops
    for m in (1, 8, 12, 13, 16, 17, 24, 32, 33, 64, 65):
        for n, k in ((1536, 1536), (3584, 18944), (18944, 3584), (4608, 3584), (5120, 27648), (10240, 8192), (14000, 3745),
                     (17920, 1536), (1536, 8960), (2048, 11008), (5120, 5120), (7168, 5120), (22016, 2048), (300, 100)):
            assert ops.few_rows_preferred(m, n, k) == torch_ops.few_rows_preferred(m, n, k), (m, n, k)
    assert ops.few_rows_preferred(12, 3584, 18944) and not ops.few_rows_preferred(13, 3584, 18944)
    assert ops.few_rows_preferred(16, 3584, 3584) and ops.few_rows_preferred(32, 3584, 3584) and not ops.few_rows_preferred(33, 3584, 3584)
    assert not ops.few_rows_preferred(17, 3584, 18944) and not ops.few_rows_preferred(17, 5120, 5120)
    assert ops.few_rows_preferred(32, 1536, 8960) and not ops.few_rows_preferred(17, 2048, 11008)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(2, 3), (33, 200), (512, 4096)])
def test_swiglu(ops, dtype, shape):
    t, i = shape
    g = torch.Generator().manual_seed(4)
    gu = (torch.randn(t, 2 * i, generator=g) * 3).to(dtype)
    out = torch.empty(t, i, dtype=dtype, device=DEV)
    ops.swiglu(gu.to(DEV), out)
    gd = gu.double().numpy()
    ref = plain_impl.swiglu(gd[:, :i], gd[:, i:])
    assert rel(out, ref) < tol(dtype, 1e-6, 8e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("t,heads,dh,theta,start", [(3, 1, 4, 1e4, 0), (40, 5, 48, 5e4, 7), (64, 4, 128, 1e6, 500)])
def test_rope(ops, dtype, t, heads, dh, theta, start):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(t, heads * dh, generator=g).to(dtype)
    pos = torch.arange(start, start + t, dtype=torch.int32)
    cos = torch.empty(t, dh // 2, device=DEV)
    sin = torch.empty(t, dh // 2, device=DEV)
    ops.rope_table(pos.to(DEV), theta, dh, cos, sin)
    xd = x.to(DEV).clone()
    ops.rope_apply(xd, heads, dh, dh, cos, sin)
    ref = plain_impl.rope_neox(x.double().numpy().reshape(t, heads, dh), pos.numpy(), theta).reshape(t, -1)
    # float32 angles: an angle near `start + t` carries an absolute error of about its ulp
    assert rel(xd, ref) < tol(dtype, 2e-4 if start else 2e-6, 8e-3)


def _paged_case(ops, dtype, seg_specs, nh, nkv, dh, page, window, seed, scale_one=None, row=None, ws=None,
                pad_pow2=False):
    """seg_specs: list of (ctx_len, q_len).  Builds random K/V for every
    segment, scatters them into shuffled pages, and compares the kernel with
    the plain attention on the logical sequences.  `scale_one` is the index of a
    key that is made to stand out for query `row` of its segment (the last one
    when `row` is None).  `pad_pow2`: the block table is widened to the next power
    of two and the decode kernel is told the table's width as its longest context,
    as a recorded decode step sees its batch."""
    g = torch.Generator().manual_seed(seed)
    nseg = len(seg_specs)
    blocks = [-(-c // page) for c, _ in seg_specs]
    num_pages = sum(blocks) + 3
    perm = torch.randperm(num_pages, generator=g).tolist()
    kc = torch.randn(num_pages, nkv, page, dh, generator=g).to(dtype)      # garbage everywhere first
    vc = torch.randn(num_pages, nkv, page, dh, generator=g).to(dtype)
    width = max(blocks) if not pad_pow2 else max(16, 1 << (max(blocks) - 1).bit_length())
    tab = np.full((nseg, width), -1, dtype=np.int32)
    T = sum(q for _, q in seg_specs)
    q = (torch.randn(T, nh * dh, generator=g)).to(dtype)
    ks, vs = [], []
    o = 0
    for s, (c, ql) in enumerate(seg_specs):
        k = torch.randn(c, nkv, dh, generator=g).to(dtype)
        v = torch.randn(c, nkv, dh, generator=g).to(dtype)
        if scale_one is not None:             # make one far key stand out for the last query
            far = scale_one
            big = math.sqrt(12.0 * math.sqrt(dh))      # its score is 12 after scaling: e^12 against some hundred keys near 1
            k[far] = 0
            k[far, :, 0] = big
            r = ql - 1 if row is None else row
            q[o + r].view(nh, dh)[:, :] = 0
            q[o + r].view(nh, dh)[:, 0] = big
        for b in range(blocks[s]):
            tab[s, b] = perm.pop()
            n = min(page, c - b * page)
            kc[tab[s, b], :, :n] = k[b * page:b * page + n].transpose(0, 1)
            vc[tab[s, b], :, :n] = v[b * page:b * page + n].transpose(0, 1)
        ks.append(k)
        vs.append(v)
        o += ql
    q_len = np.array([ql for _, ql in seg_specs], dtype=np.int32)
    ctx_len = np.array([c for c, _ in seg_specs], dtype=np.int32)
    q_start = np.concatenate([[0], np.cumsum(q_len)[:-1]]).astype(np.int32)
    seg_of = np.repeat(np.arange(nseg, dtype=np.int32), q_len)
    dev = lambda a: torch.from_numpy(a).to(DEV)
    single = np.nonzero(q_len[seg_of] == 1)[0].astype(np.int32)
    multi = np.nonzero(q_len[seg_of] != 1)[0].astype(np.int32)
    meta = AttentionMeta(block_table=dev(tab), max_blocks=tab.shape[1], seg_of_token=dev(seg_of),
                         q_start=dev(q_start), q_len=dev(q_len), ctx_len=dev(ctx_len), num_segments=nseg,
                         num_tokens=T, max_q_len=int(q_len.max()), max_ctx_len=int(ctx_len.max()),
                         host_q_start=q_start, host_q_len=q_len, host_ctx_len=ctx_len,
                         single_tokens=dev(single) if len(multi) else None, num_single=len(single),
                         multi_tokens=dev(multi) if len(single) else None, num_multi=len(multi),
                         tiles=dev(np.asarray([(i, int(q_start[i]) + a, min(32, int(q_len[i]) - a), 0)
                                               for i in range(nseg) if q_len[i] > 1
                                               for a in range(0, int(q_len[i]), 32)], dtype=np.int32).reshape(-1, 4)),
                         num_tiles=sum(-(-int(n) // 32) for n in q_len if n > 1), tile_rows=32,
                         max_single_ctx=(width * page if pad_pow2 else int(ctx_len[q_len == 1].max())) if len(single) else 0)
    out = torch.empty(T, nh * dh, dtype=dtype, device=DEV)
    scale = 1.0 / math.sqrt(dh)
    ops.paged_attention(q.to(DEV), out, kc.to(DEV), vc.to(DEV), meta, nh, nkv, dh, page, window, scale, ws=ws)
    refs = []
    o = 0
    for s, (c, ql) in enumerate(seg_specs):
        qq = q[o:o + ql].double().numpy().reshape(ql, nh, dh)
        refs.append(plain_impl.attention(qq, ks[s].double().numpy(), vs[s].double().numpy(),
                                         np.arange(c - ql, c), np.arange(c), scale, window).reshape(ql, -1))
        o += ql
    return out, np.concatenate(refs)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("segs,nh,nkv,dh,page,window", [
    ([(2, 2)], 1, 1, 4, 16, 0),                       # the reference's smallest case
    ([(11, 5)], 4, 2, 8, 16, 0),                      # a 5-token portion after 6 cached tokens
    ([(20, 20), (20, 1)], 4, 2, 8, 16, 0),            # shuffled table, last page partly filled
    ([(20, 1), (28, 1)], 4, 2, 8, 16, 0),             # two decoding requests with interleaved pages
    ([(100, 37), (1, 1), (300, 1), (64, 64)], 6, 2, 48, 8, 0),
    ([(100, 37), (33, 2), (300, 1), (70, 70)], 5, 5, 32, 16, 20),    # window crosses pages
    ([(130, 130), (257, 3)], 28, 4, 128, 16, 0),      # the 7B layer's head layout
    ([(200, 8)], 3, 1, 112, 16, 64),
    ([(4096, 1), (37, 1), (1, 1), (700, 1)], 28, 4, 128, 16, 0),    # decoding: keys split over blocks
    ([(900, 1), (64, 1), (2000, 1)], 12, 1, 64, 16, 300),           # 12 heads in one group, window
    ([(1000, 1), (50, 3), (513, 1)], 4, 2, 16, 8, 0),               # decoding beside a portion
    ([(300, 1), (77, 1)], 6, 3, 80, 16, 0),                         # a head size the split kernel does not take
    ([(300, 1), (1025, 1), (31, 1)], 40, 2, 64, 16, 0),             # 20 heads in a group: two blocks of MFMA rows
    ([(33, 1), (32, 1), (1, 1)], 7, 7, 128, 8, 0),                  # one head per group, keys around a block's edge
    ([(700, 700), (40, 3), (513, 1), (300, 17)], 28, 4, 128, 16, 0),    # portions on the matrix cores
    ([(257, 100), (90, 90), (64, 33)], 20, 2, 64, 8, 50),           # 10 heads a group (two turns of waves), window
    ([(2, 2), (17, 16), (33, 2)], 3, 3, 128, 16, 0),
    ([(500, 300), (70, 70), (45, 2)], 8, 2, 128, 12, 0),            # page sizes that do not divide a block of 32 keys
    ([(400, 150), (130, 130)], 6, 3, 128, 64, 90),                  # pages longer than a block of keys, window
    ([(333, 200), (64, 5)], 10, 2, 64, 5, 0),
    ([(300, 300), (100, 9)], 4, 1, 64, 24, 40),
    ([(1, 1), (3000, 700)], 14, 2, 128, 1, 0),                      # one key a page: a long table
    ([(1200, 1200), (40, 3)], 28, 4, 128, 16, 0),                   # more blocks than compute units: the tile's keys in one go
    ([(1300, 1300)], 32, 8, 64, 8, 200),
    ([(5000, 300)], 4, 2, 128, 1, 0),                               # a table too long for the kernel that keeps the pages' offsets in LDS
    ([(1500, 400), (9, 9)], 7, 1, 128, 1, 0),                       # one key a page, within its table
    ([(1100, 1100), (40, 3)], 40, 8, 128, 16, 0),                   # groups of 5 heads
    ([(1100, 1100)], 48, 8, 64, 12, 0),                             # groups of 6, pages that do not divide a block of keys
    ([(2100, 2100)], 18, 2, 64, 8, 700),                            # groups of 9
])
def test_paged_attention(ops, dtype, segs, nh, nkv, dh, page, window):
    out, ref = _paged_case(ops, dtype, segs, nh, nkv, dh, page, window, seed=6)
    assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2)


@pytest.mark.parametrize("m,n,k,parts", [(33, 200, 4096, 8), (64, 136, 5888, 8), (64, 136, 6144, 12), (40, 300, 7744, 15), (64, 264, 9024, 16), (65, 264, 9024, 8)])
def test_products_of_many_parts_and_what_follows_them(ops, m, n, k, parts):
    """K in up to sixteen parts (eight above 64 rows): every kernel that adds them up adds all of them."""
    assert ops._work_bytes(m, n, k, ops._DT[torch.bfloat16]) == 4 * m * n * parts
    g = torch.Generator().manual_seed(83)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b, base = torch.randn(n, generator=g), torch.randn(m, n, generator=g)
    gamma, beta, eps = torch.rand(n, generator=g) + 0.5, torch.randn(n, generator=g), 1e-5
    y = x.double().numpy() @ w.double().numpy().T + b.double().numpy()
    total, bound = base.double().numpy() + y, 4 * math.sqrt(k) * 2.0 ** -24
    dev = [v.to(DEV) for v in (x, w, b)]
    alone, short = base.to(DEV), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear(*dev, alone, True, ws=_Lender())
    ops.linear(*dev, short, ws=_Lender())
    assert rel(alone, total) < bound and rel(short, y) < 2.0 ** -8
    for dtype, near in ((torch.bfloat16, 2.0 ** -8), (torch.float32, 2 * bound)):
        xn, out = torch.full((m, n), float("nan"), dtype=dtype, device=DEV), base.to(DEV)
        assert ops.linear_then_norm(*dev, out, gamma.to(DEV), eps, xn, _Lender())
        assert torch.equal(out, alone) and rel(xn, plain_impl.rms_norm(total, gamma.double().numpy(), eps)) < near
        xn, out = torch.full((m, n), float("nan"), dtype=dtype, device=DEV), base.to(DEV)
        assert ops.linear_tanh_norm(*dev, out, 0.7, gamma.to(DEV), beta.to(DEV), xn, _Lender())
        assert torch.equal(out, alone) and rel(xn, np.tanh(0.7 * total) * gamma.double().numpy() + beta.double().numpy()) < near
    act = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.linear_act(*dev, act, "relu2", ws=_Lender())
    assert rel(act, np.maximum(y, 0) ** 2) < 2.0 ** -8


@pytest.mark.parametrize("T,nh,nkv,dk,dv,rot,split,norm,store", [
    (1, 1, 1, 2, 1, 2, False, True, True), (3, 16, 2, 64, 48, 64, True, True, True),          # a unit; two units a thread, all pairs
    (2, 12, 2, 128, 128, 64, True, True, True), (2, 17, 3, 128, 128, 4, False, True, True),       # 1,024 threads, their units; one head too many for them
    (5, 8, 8, 32, 32, 0, False, True, True), (2, 3, 1, 40, 257, 8, True, False, True), (4, 24, 1, 64, 64, 32, True, True, False)])
def test_query_and_key_norms_of_short_and_long_rows(ops, T, nh, nkv, dk, dv, rot, split, norm, store):
    """At and around the units a thread holds; float32 in the page cache, against float64 (a sum of n squares and a few roundings)."""
    g = torch.Generator().manual_seed(dk * 7 + nh)
    nq, nk, page = nh * dk, nkv * dk, 4
    rows = torch.randn(T, nq + nk + nkv * dv + 3, generator=g)
    wq, wk = 1 + torch.randn(nq, generator=g) / 8, 1 + torch.randn(nk, generator=g) / 8
    ang = torch.rand(T, max(rot // 2, 1), generator=g) * 6
    cos, sin = ang.cos(), ang.sin()
    slots = torch.randperm(3 * page, generator=g)[:T].to(torch.int32)
    gpu = lambda x: x.to(DEV)
    d = gpu(rows)
    kc, vc = torch.full((3, nkv, page, dk), 7.0, device=DEV), torch.full((3, nkv, page, dv), 7.0, device=DEV)
    ops.qk_norm_pairs_store(d, nh, nkv, dk, dv, rot, gpu(wq) if norm else None, gpu(wk) if norm else None, 1e-5, gpu(cos[:, :rot // 2].contiguous()),
                            gpu(sin[:, :rot // 2].contiguous()), gpu(slots) if store else None, kc if store else None, vc if store else None, page, half_split=split)

    def ref(x, w, heads):
        x = x.double()
        y = x / (x.square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double() if norm else x
        y, half = y.view(T, heads, dk).clone(), rot // 2
        i = torch.arange(half)
        a, b = (i, i + half) if split else (2 * i, 2 * i + 1)
        c, s_ = cos[:, None, :half].double(), sin[:, None, :half].double()
        u, v = y[..., a], y[..., b]
        y[..., a], y[..., b] = u * c - v * s_, u * s_ + v * c
        return y
    bound = (nq + 16) * 2 ** -24 * 6
    assert (d.cpu()[:, :nq].double() - ref(rows[:, :nq], wq, nh).reshape(T, nq)).abs().max() < bound
    assert torch.equal(d.cpu()[:, nq:], rows[:, nq:])
    k, v = kc.cpu().transpose(1, 2).reshape(-1, nkv, dk), vc.cpu().transpose(1, 2).reshape(-1, nkv, dv)
    other = torch.ones(3 * page, dtype=torch.bool)
    if store:
        other[slots.long()] = False
        assert (k[slots.long()].double() - ref(rows[:, nq:nq + nk], wk, nkv)).abs().max() < bound
        assert torch.equal(v[slots.long()], rows[:, nq + nk:nq + nk + nkv * dv].reshape(T, nkv, dv))
    assert (k[other] == 7.0).all() and (v[other] == 7.0).all()


@pytest.mark.parametrize("taps,C,slots,bias", [(2, 5, [2], True), (3, 256, [0, 3], False), (4, 300, [4, 1, 0], True), (5, 257, [1, 2], True)])
def test_convolution_of_one_token_a_request(ops, taps, C, slots, bias):
    """A decoding step's outputs and moved tails (bit for bit), also of 5 taps, which the general kernel takes; other slots' tails stay."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(taps * 100 + C)
    T = len(slots)
    wide, w, b, tail = torch.randn(T, C + 8, generator=g), torch.randn(C, taps, generator=g), torch.randn(C, generator=g), torch.randn(6, taps - 1, C, generator=g)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(num_tokens=T, num_segments=T, max_q_len=1, seg_of_token=i32(list(range(T))), q_start=i32(list(range(T))), q_len=i32([1] * T),
                          state_slots=i32(slots), host_state_slots=np.array(slots, np.int32), host_q_len=np.ones(T, np.int32), host_q_start=np.arange(T, dtype=np.int32))
    dev_tail, out = tail.to(DEV), torch.empty(T, C, device=DEV)
    ops.causal_conv_silu(wide.to(DEV)[:, 4:4 + C], w.to(DEV), b.to(DEV) if bias else None, dev_tail, ctx, out)
    seen = torch.cat([tail[slots], wide[:, None, 4:4 + C]], dim=1)
    z = (seen.double() * w.t().double()).sum(1) + (b.double() if bias else 0.0)
    assert (out.cpu().double() - z * torch.sigmoid(z)).abs().max() < 16 * taps * 2 ** -24 * (seen.abs() * w.t().abs()).sum(1).max()
    moved = tail.clone()
    moved[slots] = seen[:, 1:]
    assert torch.equal(dev_tail.cpu(), moved)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ctx,nh,nkv,dh,page,pad", [
    ([1, 7, 8, 31, 32, 33, 95, 96], 14, 2, 64, 16, False), ([97, 128, 129], 6, 1, 64, 8, False), ([144] * 2, 12, 2, 128, 12, False),      # four runs a block, one
    ([449, 450], 12, 2, 128, 16, False), ([513, 640, 700], 7, 1, 128, 16, False), ([700] * 3, 12, 2, 128, 8, False),       # runs of 64 keys and more
    ([61, 300, 15], 12, 2, 128, 24, False), ([200, 9], 20, 1, 64, 16, False),                     # runs of 32 (float32); 20 heads: two passes
    ([257, 130, 8], 5, 1, 128, 1, True), ([260 * 16 - 3, 4], 4, 1, 64, 16, False)])               # tables beyond the pages that are asked for ahead
def test_single_tokens_of_few_keys(ops, dtype, ctx, nh, nkv, dh, page, pad):
    """A request a token, in order, at the edges of the cuts of short contexts; a portion among them (then the tokens come by a
    list) must not change what a token gets, and neither the requests' number passed or left out."""
    from litinfer_amd.engine.workspace import Workspace
    segs = [(c, 1) for c in ctx]
    ws = Workspace(DEV)
    out, ref = _paged_case(ops, dtype, segs, nh, nkv, dh, page, 0, seed=8, ws=ws, pad_pow2=pad)
    assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2)
    told, was = [], ops._seg_of_token
    try:
        ops._seg_of_token = lambda meta, takes=True: told.append(was(meta, takes)) or meta.seg_of_token.data_ptr()
        by_list, _ = _paged_case(ops, dtype, segs, nh, nkv, dh, page, 0, seed=8, ws=ws, pad_pow2=pad)
    finally:
        ops._seg_of_token = was
    assert told == [0] and torch.equal(out, by_list)
    out, ref = _paged_case(ops, dtype, segs[:1] + [(40, 5)] + segs[1:], nh, nkv, dh, page, 0, seed=9, ws=ws, pad_pow2=pad)
    assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("far", [3, 1000, 1999])
def test_a_far_key_stands_out_in_a_decode_batch_of_unequal_contexts(ops, far, dtype):
    # contexts of 2,000 to 5,000 keys: the batch gets one run length and a list of its runs; one key of every
    # request (in its first run or a later one) takes nearly all of the weight
    rng = np.random.default_rng(9)
    segs = [(int(c), 1) for c in rng.integers(2000, 5000, 24)] + [(5000, 1), (2000, 1)]
    from litinfer_amd.kernels.ops import _ragged_splits, decode_splits
    class _M: pass
    m = _M()
    m.host_q_len = np.ones(len(segs), dtype=np.int32)
    m.host_ctx_len = np.array([c for c, _ in segs], dtype=np.int32)
    planned = decode_splits(len(segs) * 2, 5000, 1024)
    assert _ragged_splits(planned, m, 0) > planned                 # the case is what it says
    got, ref = _paged_case(ops, dtype, segs, 12, 2, 128, 16, 0, seed=43, scale_one=far, ws=_Lender())
    assert rel(got, ref) < tol(dtype, 1e-5, 8e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("runs", [2, 16, 17, 32, 33, 64])
def test_any_number_of_runs_is_joined(ops, monkeypatch, runs, dtype):
    # sixteen runs a group of the joining kernel's threads, one group, two or four; contexts that are equal, and that leave some of
    # the runs without keys
    monkeypatch.setattr(ops, "_decode_cut", lambda *a: (runs, 1, runs))
    out, ref = _paged_case(ops, dtype, [(64 * 32, 1), (64 * 32, 1)], 6, 2, 64, 16, 0, seed=61, scale_one=777, ws=_Lender())
    assert rel(out, ref) < tol(dtype, 1e-5, 8e-3)
    monkeypatch.setattr(ops, "_decode_cut", lambda *a: (runs, 1, 1))
    out, ref = _paged_case(ops, dtype, [(64 * 32, 1), (70, 1), (1, 1), (1033, 1)], 6, 2, 128, 16, 0, seed=62, ws=_Lender())
    assert rel(out, ref) < tol(dtype, 1e-5, 8e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("requests,runs", [(160, 64), (161, 64), (171, 17), (172, 33), (560, 64)])
def test_runs_of_many_tokens_with_a_long_one_among_them_are_joined(ops, monkeypatch, requests, runs, dtype):
    # from 171 x 6 (token, head)s on one group of the joining kernel's threads takes a token's runs sixteen at a time; from 161 x 64 x 2
    # blocks on the listed runs go head by head
    monkeypatch.setattr(ops, "_decode_cut", lambda *a: (runs, 1, 1))
    segs = [(1 + (7 * i) % 45, 1) for i in range(requests)]
    segs[requests // 2], segs[3] = (32 * runs - 5, 1), (16 * 32, 1)
    out, ref = _paged_case(ops, dtype, segs, 6, 2, 64, 16, 0, seed=64, ws=_Lender())
    assert rel(out, ref) < tol(dtype, 1e-5, 8e-3)


@pytest.mark.parametrize("dh,ctx", [(256, 16 * 256), (256, 17 * 256), (128 + 64, 33 * 256), (16, 20 * 256)])
def test_runs_of_the_vector_kernel_are_joined(ops, dh, ctx):
    for dtype in DTYPES:
        out, ref = _paged_case(ops, dtype, [(ctx, 1)], 2, 1, dh, 16, 0, seed=63, ws=_Lender())
        assert rel(out, ref) < tol(dtype, 1e-5, 8e-3)


@pytest.mark.parametrize("window", [0, 900])
def test_decode_run_length_of_a_batch_with_unequal_contexts(ops, window):
    # the run length chosen on the device against the same search written out, for contexts from 3 to 5,000
    # keys; then the attention of that batch
    rng = np.random.default_rng(5)
    ctx = rng.integers(3, 5000, 37).astype(np.int32)
    ctx[11] = 5000
    nseg, page, nkv, nsplit, simds = len(ctx), 16, 2, 9, 128
    ones = np.ones(nseg, dtype=np.int32)
    dev = lambda a: torch.from_numpy(a).to(DEV)
    max_blocks = 512
    meta = AttentionMeta(block_table=torch.zeros(nseg, max_blocks, dtype=torch.int32, device=DEV), max_blocks=max_blocks,
                         seg_of_token=dev(np.arange(nseg, dtype=np.int32)), q_start=dev(np.arange(nseg, dtype=np.int32)),
                         q_len=dev(ones), ctx_len=dev(ctx), num_segments=nseg, num_tokens=nseg, max_q_len=1,
                         max_ctx_len=int(ctx.max()), host_q_start=np.arange(nseg, dtype=np.int32), host_q_len=ones,
                         host_ctx_len=ctx, num_single=nseg)
    out = torch.full((2 + nseg + nseg * nsplit,), -1, dtype=torch.int32, device=DEV)
    ops.decode_run_keys(meta, None, nseg, page, window, nkv, nsplit, simds, out)
    keys = np.minimum(ctx, window) if window else ctx
    widest = min(max_blocks * page, window) if window else max_blocks * page
    lower, cap = (-(-int(keys.max()) // nsplit) + 31) & ~31, (-(-widest // nsplit) + 31) & ~31
    cost = {c: -(-int(nkv * np.sum(-(-keys // c))) // simds) * (c + 24) for c in range(lower, max(cap, lower) + 1, 32)}
    want = min(cost, key=lambda c: (cost[c], c))
    got = out.cpu().numpy()
    assert int(got[0]) == want
    runs = -(-keys // want)
    assert int(got[1]) == int(runs.sum()) and np.array_equal(got[2:2 + nseg], runs)
    items = got[2 + nseg:2 + nseg + int(runs.sum())]
    assert [(int(i) & 0xffff, int(i) >> 16) for i in items] == [(t, r) for t in range(nseg) for r in range(int(runs[t]))]
    assert want == (832 if not window else 128)      # (without a window the shortest run, 576, is not the cheapest)
    segs = [(int(c), 1) for c in ctx]
    got, ref = _paged_case(ops, torch.bfloat16, segs, 12, 2, 128, 16, window, seed=41, ws=_Lender())
    assert rel(got, ref) < 8e-3


@pytest.mark.parametrize("segs,nh,nkv,dh,page,window", [
    ([(3000, 64)], 28, 4, 128, 16, 0),                              # two tiles behind 2,936 cached tokens: their keys in five runs
    ([(3000, 64), (500, 1), (1200, 40), (40, 40)], 28, 4, 128, 16, 0),   # beside a decoding token; a short tile leaves runs without keys
    ([(6000, 96)], 12, 2, 64, 8, 3000),                             # a window, six heads a group
    ([(2500, 33), (2600, 2)], 8, 8, 128, 12, 0),                    # pages that do not divide a block of keys; a tile of one row
])
def test_prompt_portions_behind_long_contexts_with_their_keys_in_runs(ops, segs, nh, nkv, dh, page, window):
    from litinfer_amd.kernels.ops import _prefill_runs
    ql, cl = np.array([q for _, q in segs], dtype=np.int32), np.array([c for c, _ in segs], dtype=np.int32)
    blocks = max(-(-c // page) for c, _ in segs)
    assert _prefill_runs(ql, cl, nh, nkv, dh, blocks, window, int(ql.sum())) > 1       # the case is what it says
    out, ref = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, page, window, seed=31, ws=_Lender())
    assert rel(out, ref) < 1.5e-2
    # and one far key among thousands, in a run of its own
    for far in (5, 1000, 2900):
        out, ref = _paged_case(ops, torch.bfloat16, [(3000, 64)], 28, 4, 128, 16, 0, seed=32, scale_one=far, row=40, ws=_Lender())
        assert rel(out, ref) < 1.5e-2


@pytest.mark.parametrize("heads", [1, 2])
@pytest.mark.parametrize("segs,nh,nkv,dh,page,window", [
    ([(300, 300), (40, 3), (1, 1), (257, 129), (64, 33)], 5, 1, 128, 16, 0),      # segments that end in any of a block's tiles
    ([(500, 300), (70, 70), (45, 2)], 6, 2, 128, 12, 0),                          # pages that do not divide a block of keys
    ([(700, 500), (90, 90), (200, 161)], 3, 3, 64, 8, 50),                        # a window shorter than a block's tiles
    ([(260, 129)], 14, 2, 64, 64, 100),                                           # one row in a block's second tile or first of the next
])
def test_prompt_attention_with_several_tiles_a_block(ops, monkeypatch, segs, nh, nkv, dh, page, window, heads):
    monkeypatch.setattr(ops, "_prefill_heads", lambda *a: heads)
    out, ref = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, page, window, seed=33)
    assert rel(out, ref) < 1.5e-2
    # one far key among the keys that only a later tile of the block sees
    out, ref = _paged_case(ops, torch.bfloat16, [(1000, 300)], nh, nkv, dh, page, 0, seed=34, scale_one=770, row=90)
    assert rel(out, ref) < 1.5e-2


@pytest.mark.parametrize("dh,page,window", [(128, 16, 0), (128, 4, 0), (128, 2, 40), (64, 8, 0), (64, 4, 33), (128, 32, 70)])
@pytest.mark.parametrize("heads", [1, 2])
def test_prompt_attention_over_few_blocks_of_keys(ops, monkeypatch, dh, page, window, heads):
    # one to seven blocks of 32 keys: the turns before the stages of LDS are all in use and the last ones; pages down to less than a load
    monkeypatch.setattr(ops, "_prefill_heads", lambda *a: heads)
    segs = [(2, 2), (32, 32), (33, 33), (64, 2), (65, 64), (97, 33), (128, 128), (130, 5), (161, 161), (224, 31)]
    out, ref = _paged_case(ops, torch.bfloat16, segs, 6, 2, dh, page, window, seed=37)
    assert rel(out, ref) < 1.5e-2


@pytest.mark.parametrize("heads,tiles,runs", [(4, 1, 2), (4, 7, 5), (2, 2, 3), (2, 10, 16), (1, 4, 4), (1, 12, 2)])
def test_prompt_attention_with_the_keys_of_its_first_tiles_in_runs(ops, monkeypatch, heads, tiles, runs):
    segs = [(700, 300), (1, 1), (90, 70), (400, 40), (257, 129)]                # 10 + 3 + 2 + 5 tiles, a decoding token among them
    blocks = 128 // heads                                                        # tokens of a block; one goes by its first tile
    of = [(s, a, min(blocks, q - a)) for s, a, q in [(s, a, q) for s, (_, q) in enumerate(segs) if q > 1 for a in range(0, q, 32)][:tiles] if a % blocks == 0]
    starts = np.concatenate([[0], np.cumsum([q for _, q in segs])])
    monkeypatch.setattr(ops, "_prefill_runs", lambda *a: 1)
    monkeypatch.setattr(ops, "_prefill_heads", lambda *a: heads)
    monkeypatch.setattr(ops, "_prefill_tail", lambda *a: (runs, tiles, sum(r for _, _, r in of), int(starts[of[-1][0]] + of[-1][1] + of[-1][2])))
    for nh, nkv, dh, window in ((5, 1, 128, 0), (6, 2, 64, 90)):
        out, ref = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, 16, window, seed=35, ws=_Lender())
        assert rel(out, ref) < 1.5e-2


@pytest.mark.parametrize("segs,nh,nkv,dh,page,window", [
    # one head, four groups: as few as one block of keys, so that groups have none; a window that begins inside a block of keys
    ([(2, 2), (32, 32), (33, 33), (64, 5), (65, 2), (1, 1)], 6, 2, 128, 16, 0), ([(700, 500), (90, 90), (200, 161)], 3, 3, 128, 8, 50),
    ([(500, 300), (70, 70), (97, 2)], 5, 1, 64, 12, 0),
    # two heads, two groups: whole pairs of heads and a wave without one
    ([(400, 400), (33, 33)], 28, 4, 128, 16, 0), ([(990, 990), (300, 40)], 12, 2, 64, 8, 100),
    # four heads, two groups, with idle waves; and one group
    ([(960, 960), (31, 2)], 28, 4, 64, 16, 0), ([(1056, 1056)], 32, 16, 64, 16, 0), ([(990, 990), (300, 40)], 24, 12, 128, 16, 100),
])
def test_prompt_attention_in_32_bits_with_its_keys_over_groups_of_waves(ops, segs, nh, nkv, dh, page, window):
    out, ref = _paged_case(ops, torch.float32, segs, nh, nkv, dh, page, window, seed=36)
    assert rel(out, ref) < 5e-6                     # float32 sums of up to some thousand terms: 2^-24 times the square root of their number


def test_which_tiles_of_prompt_attention_have_their_keys_in_runs(ops):
    from litinfer_amd.kernels.ops import _prefill_tail
    tail = lambda new, cached, nh, nkv, heads: _prefill_tail(np.array(new, dtype=np.int32), np.array(cached, dtype=np.int32) + np.array(new, dtype=np.int32), nh, nkv, 128, 2000, 0, heads)
    assert tail([1999], [16000], 40, 8, 1) == (3, 16, 512, 512)                   # 640 blocks: 512 and the first four rows of tiles
    assert tail([1, 1999], [50, 16000], 40, 8, 1) == (3, 16, 512, 513)
    assert tail([1999], [16000], 40, 8, 4)[0] == 1 and tail([990], [16000], 40, 8, 4)[0] == 1      # a last round that is nearly full; less than one round
    assert tail([1999], [100], 40, 8, 1)[0] == 1                                  # too few keys


def test_how_many_heads_a_block_of_prompt_attention_takes(ops):
    from litinfer_amd.kernels.ops import _prefill_heads
    heads = lambda new, cached, nh, nkv, window=0, pages=2000: _prefill_heads(np.array(new, dtype=np.int32), np.array(cached, dtype=np.int32) + np.array(new, dtype=np.int32), nh, nkv, pages, window)
    assert heads([1999], [16000], 40, 8) == 1 and heads([2048], [0], 32, 32) < 4 and heads([2000], [4000], 32, 16) == 2
    assert heads([1999], [16000], 64, 8) == 4 and heads([1999], [16000], 28, 4) == 4      # whole groups; a chip that is not filled
    assert heads([990], [517], 40, 8) == 4 and heads([1] * 9, [700] * 9, 32, 32) == 4     # one round; no portion at all
    assert heads([1999], [16000], 40, 8, pages=5000) == 4                                 # a table for the form without


@pytest.mark.parametrize("segs,nh,nkv,dh", [
    ([(1056, 1056)], 32, 16, 128),                 # more blocks than compute units: the form with four waves a block
    ([(700, 700), (300, 40)], 24, 12, 64),
    ([(500, 500)], 16, 4, 128),                    # fewer: the keys in two halves
    ([(3000, 64)], 28, 4, 128),                    # the keys in runs that are joined
])
def test_prompt_attention_gives_the_same_bits_again(ops, segs, nh, nkv, dh):
    """The scores' maxima are taken of finished sums: a maximum of unfinished ones is only the reference of the
    exponentials, so the output stays close, but its last bits then depend on how the waves happened to run."""
    first, ref = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, 16, 0, seed=61, ws=_Lender())
    assert rel(first, ref) < 1.5e-2
    for _ in range(4):
        again, _ = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, 16, 0, seed=61, ws=_Lender())
        assert torch.equal(first, again)


# ---- the context lengths of the long workloads (8 x 30,000-token prompts in portions of 2,048, then decoding):
# block tables of 1,875 to 2,048 pages, a portion behind 28,000 cached keys, splits of many pages
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("pad_pow2", [False, True])
@pytest.mark.parametrize("far", [3, 15000, 29940])
def test_decoding_over_thirty_thousand_keys_finds_one_far_key(ops, far, pad_pow2, dtype):
    """Eight requests of 30,000 keys each, pages of 16, 40 heads on 8 kv heads of size 128: one key of every
    request, near the start, in the middle or near the end, carries nearly all the weight.  Also with the
    block table widened to 2,048 pages, as a recorded step sees it."""
    segs = [(30000 - 7 * i, 1) for i in range(8)]
    out, ref = _paged_case(ops, dtype, segs, 40, 8, 128, 16, 0, seed=51, scale_one=far, ws=_Lender(),
                           pad_pow2=pad_pow2)
    assert rel(out, ref) < tol(dtype, 1e-5, 8e-3)


@pytest.mark.parametrize("page,ctx,window", [(1, 5000, 0), (2, 8400, 0), (1, 6000, 4500)])
def test_decode_splits_that_would_hold_more_pages_than_the_kernel_keeps_get_more_runs(ops, page, ctx, window):
    """Many requests with small pages: the number of runs that fills the SIMDs once would give every run
    more than the 1,024 pages the matrix-core decode kernel keeps in LDS, so the host raises the number
    of runs until a run fits; a far key in the first, a middle and the last run."""
    from litinfer_amd.kernels import ops as O
    n, nkv = 64, 4
    segs = [(ctx - 3 * i, 1) for i in range(n)]
    blocks = -(-ctx // page)
    keys = min(ctx, window) if window else ctx
    planned = O.decode_splits(n * nkv, keys, O._simd_count(torch.device(DEV)))
    assert O.decode_split_blocks(blocks, page, window, planned) > O.DECODE_TABLE_CAP      # the case is what it says
    for far in (ctx - 3 * n - 5, ctx // 2, max(ctx - window, 0) + 7 if window else 2):
        out, ref = _paged_case(ops, torch.bfloat16, segs, 8, nkv, 64, page, window, seed=52, scale_one=far, ws=_Lender())
        assert rel(out, ref) < 8e-3
    out, ref = _paged_case(ops, torch.float32, segs, 8, nkv, 64, page, window, seed=52, scale_one=ctx // 2, ws=_Lender())
    assert rel(out, ref) < 1e-5


@pytest.mark.parametrize("far", [5, 14000, 29000])
def test_a_portion_of_2048_behind_28000_cached_keys_finds_one_far_key(ops, far):
    """A prompt portion of 2,048 queries behind 28,000 cached keys (pages of 16: a block table of 1,878
    pages), its tiles' keys cut into runs that are joined afterwards: one key in the first, a middle or
    the last run stands out for one row; all rows against the plain attention."""
    from litinfer_amd.kernels.ops import _prefill_runs
    segs, nh, nkv, dh, page = [(30048, 2048)], 8, 2, 128, 16
    ql, cl = np.array([2048], dtype=np.int32), np.array([30048], dtype=np.int32)
    assert _prefill_runs(ql, cl, nh, nkv, dh, -(-30048 // page), 0, 2048) > 1             # the case is what it says
    out, ref = _paged_case(ops, torch.bfloat16, segs, nh, nkv, dh, page, 0, seed=53, scale_one=far, row=1500, ws=_Lender())
    assert rel(out, ref) < 1.5e-2


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh", [32, 64, 128])          # 64 and 128 take the matrix-core kernels
def test_paged_attention_finds_one_far_key(ops, dtype, dh):
    # one key among hundreds carries almost all the weight: a kernel that skips
    # or misplaces a page gives a visibly different output
    for far in (0, 15, 16, 333, 511):
        out, ref = _paged_case(ops, dtype, [(512, 1)], 4, 2, dh, 16, 0, seed=7, scale_one=far)
        assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("ctx,ql", [(512, 70), (300, 33)])
def test_portions_find_one_far_key_for_any_row_of_a_tile(ops, dtype, dh, ctx, ql):
    # portions: the standout key for the first row of a 32-row tile, its last row, the first
    # row of the next tile and the portion's last row; at the start of the sequence, in the
    # middle, just before the portion and at the row's own position
    for row in (0, 31, 32, ql - 1):
        p = ctx - ql + row
        for far in (0, 97, ctx - ql - 1, p):
            out, ref = _paged_case(ops, dtype, [(ctx, ql)], 6, 2, dh, 16, 0, seed=7, scale_one=far, row=row)
            assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2), (row, far)
        if p + 1 < ctx:                                # the key after the row's own is not seen
            out, ref = _paged_case(ops, dtype, [(ctx, ql)], 6, 2, dh, 16, 0, seed=7, scale_one=p + 1, row=row)
            assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2), (row, "next")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh", [32, 64, 128])
def test_window_edge(ops, dtype, dh):
    # the key just outside the window must not count, the one just inside must
    for window, far, visible in ((32, 512 - 32, True), (32, 512 - 33, False)):
        out, ref = _paged_case(ops, dtype, [(512, 1)], 2, 1, dh, 8, window, seed=8, scale_one=far)
        assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("ctx,ql,window", [(512, 70, 48), (300, 33, 100), (512, 70, 37)])
def test_window_edge_for_any_row_of_a_tile(ops, dtype, dh, ctx, ql, window):
    # the first and last row of a 32-row tile, the first row of the next tile, a row whose
    # window begins on a block of 32 keys, and the last row: the key at the window's first
    # position counts, the one before it does not
    rows = {0, 31, 32, ql - 1}
    rows.add(next(r for r in range(ql) if (ctx - ql + r - window + 1) % 32 == 0))
    for row in sorted(rows):
        first = ctx - ql + row - window + 1            # the first key that the row sees
        for far in (first, first - 1):
            assert far >= 0
            out, ref = _paged_case(ops, dtype, [(ctx, ql)], 4, 2, dh, 16, window, seed=8, scale_one=far, row=row)
            assert rel(out, ref) < tol(dtype, 3e-6, 1.5e-2), (row, far - first)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh,pad", [(48, 5), (48, 16), (128, 0), (20, 0)])      # rows that do and do not start on 16 bytes
def test_rope_kv_store_and_plain_store(ops, dtype, dh, pad):
    g = torch.Generator().manual_seed(9)
    t, nh, nkv, page, pages = 37, 3, 2, 8, 11
    qkv = torch.randn(t, (nh + 2 * nkv) * dh + pad, generator=g).to(dtype)[:, :(nh + 2 * nkv) * dh]
    pos = torch.randint(0, 200, (t,), generator=g, dtype=torch.int32)
    slots = torch.randperm(pages * page, generator=g)[:t].to(torch.int32)
    cos = torch.empty(t, dh // 2, device=DEV)
    sin = torch.empty(t, dh // 2, device=DEV)
    ops.rope_table(pos.to(DEV), 1e4, dh, cos, sin)
    outs = []
    for fused in (True, False):
        d = qkv.to(DEV)
        d = d.clone() if d.is_contiguous() else d      # keep the row stride with its pad
        kc = torch.zeros(pages, nkv, page, dh, dtype=dtype, device=DEV)
        vc = torch.zeros_like(kc)
        if fused:
            ops.rope_kv_store(d, nh, nkv, dh, dh, cos, sin, slots.to(DEV), kc, vc, page)
        else:
            ops.rope_apply(d, nh + nkv, dh, dh, cos, sin)
            ops.kv_store(d, nh, nkv, dh, slots.to(DEV), kc, vc, page)
        outs.append((d[:, :nh * dh].clone(), kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    x = qkv.double().numpy()
    kref = plain_impl.rope_neox(x[:, nh * dh:(nh + nkv) * dh].reshape(t, nkv, dh), pos.numpy(), 1e4)
    got = outs[0][1].double().cpu().numpy()
    for i in range(t):
        s = int(slots[i])
        assert np.abs(got[s // page, :, s % page] - kref[i]).max() < tol(dtype, 1e-4, 3e-2)
        assert torch.equal(outs[0][2][s // page, :, s % page].cpu(),
                           qkv[i, (nh + nkv) * dh:].reshape(nkv, dh))


@pytest.mark.parametrize("t,nh,nkv,dh,k,bias", [
    (64, 28, 4, 128, 3584, True),       # a decoding batch of 64 at the 7B layer sizes
    (33, 12, 2, 128, 1536, True),
    (13, 64, 8, 128, 8192, True),       # the fewest rows that are cut along K, against a large matrix (168 MB)
    (40, 6, 2, 64, 1280, False),
    (100, 28, 4, 128, 3584, True),      # more than 64 rows: tiles of 128 rows, K still cut
    (200, 12, 2, 128, 1536, False),
])
def test_projection_cut_along_k_with_rotary_encoding_and_page_write_in_the_adding_up(ops, t, nh, nkv, dh, k, bias):
    g = torch.Generator().manual_seed(31)
    n, page, pages = (nh + 2 * nkv) * dh, 16, max(8, t // 16 + 3)
    x = torch.randn(t, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) if bias else None
    pos = torch.randint(0, 5000, (t,), generator=g, dtype=torch.int32)
    slots = torch.randperm(pages * page, generator=g)[:t].to(torch.int32)
    cos = torch.empty(t, dh // 2, device=DEV)
    sin = torch.empty(t, dh // 2, device=DEV)
    ops.rope_table(pos.to(DEV), 1e6, dh, cos, sin)
    kc = torch.full((pages, nkv, page, dh), 7.0, dtype=torch.bfloat16, device=DEV)
    vc = torch.full_like(kc, 7.0)
    out = torch.full((t, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    took = ops.linear_rope_store_parts(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, nh, nkv, dh, cos, sin,
                                       slots.to(DEV), kc, vc, page, _Lender())
    assert took
    y = x.double().numpy() @ w.double().numpy().T + (0 if b is None else b.double().numpy())
    y = y.reshape(t, nh + 2 * nkv, dh)
    ref = np.concatenate([plain_impl.rope_neox(y[:, :nh + nkv], pos.numpy(), 1e6), y[:, nh + nkv:]], axis=1).reshape(t, n)
    assert rel(out, ref) < 5e-3
    ov = out.cpu().view(t, nh + 2 * nkv, dh)
    touched = torch.zeros(pages, page, dtype=torch.bool)
    for i in range(t):
        sl = int(slots[i])
        touched[sl // page, sl % page] = True
        assert torch.equal(kc[sl // page, :, sl % page].cpu(), ov[i, nh:nh + nkv])
        assert torch.equal(vc[sl // page, :, sl % page].cpu(), ov[i, nh + nkv:])
    untouched = ~touched[:, None, :, None].expand(pages, nkv, page, dh)
    assert (kc.cpu()[untouched] == 7.0).all() and (vc.cpu()[untouched] == 7.0).all()
    # few rows, or no workspace: not taken
    assert not ops.linear_rope_store_parts(x[:8].to(DEV), w.to(DEV), None, out[:8], nh, nkv, dh, cos[:8], sin[:8],
                                           slots[:8].to(DEV), kc, vc, page, _Lender())


@pytest.mark.parametrize("t,nh,nkv,dh,k,bias", [
    (8, 28, 4, 128, 3584, True),        # a decoding step at the 7B layer sizes
    (1, 3, 1, 32, 96, True),
    (16, 5, 5, 48, 120, False),         # a head size that is no power of two
    (3, 6, 2, 64, 136, True),
    (5, 35, 1, 80, 72, True),           # 1480 rotation pairs: 6 a block, blocks that straddle heads, a ragged last one
    (16, 40, 8, 128, 64, False),        # 3584 pairs: 14 a block, two tiles
    (2, 70, 1, 128, 40, True),          # more pairs than two tiles a compute unit hold: whole tiles again
    (17, 28, 4, 128, 3584, True),       # two tiles of rows a block
    (32, 12, 2, 128, 1536, True),
    (25, 5, 5, 48, 120, False),
    (31, 35, 1, 80, 72, True),
    (20, 70, 1, 128, 40, False),
])
def test_projection_with_rotary_encoding_and_page_write_as_its_epilogue(ops, t, nh, nkv, dh, k, bias):
    g = torch.Generator().manual_seed(16)
    n, page, pages = (nh + 2 * nkv) * dh, 8, 9
    assert t <= page * pages
    x = (torch.randn(t, k, generator=g) * 2).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) if bias else None
    pos = torch.randint(0, 3000, (t,), generator=g, dtype=torch.int32)
    slots = torch.randperm(pages * page, generator=g)[:t].to(torch.int32)
    cos = torch.empty(t, dh // 2, device=DEV)
    sin = torch.empty(t, dh // 2, device=DEV)
    ops.rope_table(pos.to(DEV), 1e6, dh, cos, sin)
    kc = torch.full((pages, nkv, page, dh), 7.0, dtype=torch.bfloat16, device=DEV)
    vc = torch.full_like(kc, 7.0)
    out = torch.full((t, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.rope_store_takes(t, k, w.dtype, dh, dh)
    ops.linear_rope_store(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, nh, nkv, dh, cos, sin,
                          slots.to(DEV), kc, vc, page)
    y = x.double().numpy() @ w.double().numpy().T
    if b is not None:
        y = y + b.double().numpy()
    y = y.reshape(t, nh + 2 * nkv, dh)
    ref = np.concatenate([plain_impl.rope_neox(y[:, :nh + nkv], pos.numpy(), 1e6), y[:, nh + nkv:]], axis=1)
    assert rel(out, ref.reshape(t, n)) < 5e-3
    o = out.cpu().view(t, nh + 2 * nkv, dh)
    touched = torch.zeros(pages, page, dtype=torch.bool)
    for i in range(t):                                   # the pages hold exactly what out holds
        s = int(slots[i])
        touched[s // page, s % page] = True
        assert torch.equal(kc[s // page, :, s % page].cpu(), o[i, nh:nh + nkv])
        assert torch.equal(vc[s // page, :, s % page].cpu(), o[i, nh + nkv:])
    untouched = ~touched[:, None, :, None].expand(pages, nkv, page, dh)
    assert (kc.cpu()[untouched] == 7.0).all() and (vc.cpu()[untouched] == 7.0).all()


@pytest.mark.parametrize("shape", [(1, 4), (3, 4096), (5, 152064), (2, 301)])
def test_argmax_rows_lowest_index_wins(ops, shape):
    g = torch.Generator().manual_seed(10)
    x = torch.randn(*shape, generator=g)
    x[0, shape[1] // 2] = 50.0
    x[0, shape[1] - 1] = 50.0          # an equal maximum later in the row
    out = torch.empty(shape[0], dtype=torch.int32, device=DEV)
    ops.argmax_rows(x.to(DEV), out)
    assert out.cpu().tolist() == [plain_impl.argmax_first(r) for r in x.numpy()]
    assert out[0].item() == shape[1] // 2


def test_gather_and_cast(ops):
    x = torch.randn(10, 37)
    rows = torch.tensor([9, 0, 0, 4], dtype=torch.int32)
    out = torch.empty(4, 37, device=DEV)
    ops.gather_rows(x.to(DEV), rows.to(DEV), out)
    assert torch.equal(out.cpu(), x[rows.long()])
    b = torch.empty(10, 37, dtype=torch.bfloat16, device=DEV)
    ops.cast(x.to(DEV), b)
    assert torch.equal(b.cpu(), x.to(torch.bfloat16))       # round to nearest even, as torch does
    f = torch.empty(10, 37, device=DEV)
    ops.cast(b, f)
    assert torch.equal(f.cpu(), x.to(torch.bfloat16).float())


def _sample(ops, logits, temperature, top_k, top_p, u):
    n = logits.shape[0]
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    f = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
    ops.sample_rows(logits.to(DEV), f(temperature, torch.float32), f(top_k, torch.int32),
                    f(top_p, torch.float32), f(u, torch.float32), out)
    return out.cpu().tolist()


def _pick_is_right(row, temperature, top_k, top_p, u, pick, slack=2e-5):
    """The kernel sums in float32 in another order than the plain sampler: the
    pick is right if the uniform number lies within its interval of the CDF,
    give or take the rounding of the sums."""
    ids, p = plain_impl.sampling_candidates(row, temperature, top_k, top_p)
    assert pick in ids.tolist(), f"token {pick} is not among the candidates"
    cum = np.cumsum(p)
    i = ids.tolist().index(pick)
    lo = cum[i - 1] if i else 0.0
    return lo - slack <= u <= cum[i] + slack


@pytest.mark.parametrize("vocab", [8, 301, 4096, 152064])
def test_sample_rows_against_the_plain_sampler(ops, vocab):
    g = torch.Generator().manual_seed(13)
    n = 12
    logits = torch.randn(n, vocab, generator=g) * 3
    logits[1, : min(5, vocab)] = 7.0                       # equal maxima: ties go by index
    temperature = [0.0, 0.7, 1.0, 1.3, 0.8, 1.0, 0.5, 2.0, 1.0, 1.0, 0.9, 1.0]
    top_k = [0, 3, 0, 0, 50, 1, 0, 7, vocab, 0, 5, 2]
    top_p = [1.0, 1.0, 0.9, 0.5, 0.8, 0.3, 1.0, 0.95, 1.0, 0.01, 0.99, 1.0]
    u = torch.rand(n, generator=g).tolist()
    picks = _sample(ops, logits, temperature, top_k, top_p, u)
    rows = logits.double().numpy()
    assert picks[0] == plain_impl.argmax_first(rows[0])                    # temperature 0: greedy
    assert picks[5] == plain_impl.argmax_first(rows[5])                    # top_k 1
    assert picks[9] == plain_impl.argmax_first(rows[9])                    # a tiny top_p keeps the maximum only
    for r in range(1, n):
        assert _pick_is_right(rows[r], temperature[r], top_k[r], top_p[r], u[r], picks[r]), r
    # exact agreement wherever the uniform number is not at an interval's edge
    same = sum(picks[r] == plain_impl.sample_with_uniform(rows[r], temperature[r], top_k[r], top_p[r], u[r])
               for r in range(n))
    assert same >= n - 1


@pytest.mark.parametrize("vocab", [8, 301, 8192, 8193, 152064])
def test_sample_rows_with_temperature_alone(ops, vocab):
    # no top-k and no top-p: the kernel's short way; uniform numbers at both ends among them
    g = torch.Generator().manual_seed(15)
    n = 24
    logits = torch.randn(n, vocab, generator=g) * 4
    temperature = [0.3 + 0.1 * i for i in range(n)]
    u = torch.rand(n, generator=g).tolist()
    u[0], u[1], u[2] = 0.0, 0.99999994, 0.5
    picks = _sample(ops, logits, temperature, [0] * n, [1.0] * n, u)
    rows = logits.double().numpy()
    for r in range(n):
        assert 0 <= picks[r] < vocab
        assert _pick_is_right(rows[r], temperature[r], 0, 1.0, u[r], picks[r]), r
    # and mostly the very id of the float64 sampler (among 152,064 ids a float32 sum's rounding moves an
    # interval's edge past the uniform number now and then; each such pick was checked above)
    same = sum(picks[r] == plain_impl.sample_with_uniform(rows[r], temperature[r], 0, 1.0, u[r]) for r in range(n))
    assert same >= n - 4


def test_sample_rows_with_tiles_of_the_vocabulary_masked_out(ops):
    # the rows' ids are summed in tiles of 8,192 first: a tile of -inf alone, a tile so far below the
    # maximum that it has no mass in float32, and the last tile cut short must not disturb the pick
    g = torch.Generator().manual_seed(16)
    vocab, n = 3 * 8192 + 5, 16
    logits = torch.randn(n, vocab, generator=g) * 2
    logits[:8, 8192:16384] = float("-inf")
    logits[8:12, :8192] -= 200.0
    logits[12:, 16384:] = float("-inf")                      # the last two tiles, the short one among them
    temperature = [0.0, 1.0, 0.7, 1.5] * 4
    u = torch.rand(n, generator=g).tolist()
    u[1], u[2], u[5], u[13] = 0.99999994, 0.0, 0.99999994, 0.99999994
    picks = _sample(ops, logits, temperature, [0] * n, [1.0] * n, u)
    rows = logits.double().numpy()
    for r in range(n):
        assert np.isfinite(rows[r][picks[r]]), r
        if temperature[r] == 0.0:
            assert picks[r] == plain_impl.argmax_first(rows[r])
        else:
            assert _pick_is_right(rows[r], temperature[r], 0, 1.0, u[r], picks[r]), r
    assert all(p < 8192 or p >= 16384 for p in picks[:8]) and all(p >= 8192 for p in picks[9:12]) and all(p < 16384 for p in picks[12:])


@pytest.mark.parametrize("vocab", [1000, 20000, 152064])
def test_sample_rows_with_many_equal_logits_at_the_thresholds(ops, vocab):
    # logits on a coarse grid: hundreds of ids share the k-th largest value and the value at which top-p
    # cuts, spread over the threads and tiles of the kernel; which of them survive goes by ascending id
    g = torch.Generator().manual_seed(17)
    n = 16
    logits = torch.round(torch.randn(n, vocab, generator=g) * 2) / 2
    temperature = [1.0, 0.5, 2.0, 0.8] * 4
    top_k = [50, 0, 300, 7, 1000, 0, 2, 64, 999, 0, 50, 50, 0, 5000, 20, 1][:n]
    top_k = [min(k, vocab - 1) for k in top_k]
    top_p = [1.0, 0.6, 0.9, 0.5, 0.95, 0.99, 1.0, 0.3, 1.0, 0.05, 0.8, 0.999, 0.9, 0.7, 1.0, 1.0]
    u = torch.rand(n, generator=g).tolist()
    u[0], u[1], u[2] = 0.99999994, 0.0, 0.99999994
    picks = _sample(ops, logits, temperature, top_k, top_p, u)
    rows = logits.double().numpy()
    for r in range(n):
        assert _pick_is_right(rows[r], temperature[r], top_k[r], top_p[r], u[r], picks[r]), r
    same = sum(picks[r] == plain_impl.sample_with_uniform(rows[r], temperature[r], top_k[r], top_p[r], u[r]) for r in range(n))
    assert same >= n - 2


@pytest.mark.parametrize("order", ["mixed", "rounded", "ascending", "few", "one_value"])
def test_sample_rows_with_the_candidates_found_by_a_bound(ops, order):
    # ids above a bound are held against each other (mixed: some more than the wanted ones lie above it); where one wave
    # holds all large ids (ascending), most ids are -inf (few) or all are equal, too many lie above it and the search goes
    # through the digits; of bfloat16's values (rounded) several ids share one, at the threshold of top-p too
    g = torch.Generator().manual_seed(66)
    vocab, top_k = 8192 + 4097, [1, 15, 16, 17, 50, 128, 255, 256]
    n = len(top_k)
    logits = torch.randn(n, vocab, generator=g) * 3
    if order == "rounded":
        logits = logits.bfloat16().float()
    elif order == "ascending":
        logits = logits.sort(dim=1).values
    elif order == "few":
        logits[:, torch.randperm(vocab, generator=g)[:vocab - 40]] = float("-inf")
    elif order == "one_value":
        logits[:] = 1.5
        logits[:, 9000:9003] = torch.tensor([2.0, 1.75, 2.0])
    rows = logits.double().numpy()
    for top_p in (1.0, 0.9):
        for temperature in (0.7, 1.0):
            u = torch.rand(n, generator=g).tolist()
            picks = _sample(ops, logits, [temperature] * n, top_k, [top_p] * n, u)
            for r in range(n):
                assert np.isfinite(rows[r][picks[r]]), (r, top_k[r])
                assert _pick_is_right(rows[r], temperature, top_k[r], top_p, u[r], picks[r]), (r, top_k[r])


@pytest.mark.parametrize("vocab", [32 * 8192, 32 * 8192 + 1, 5 * 8192 + 3])
def test_sample_rows_with_tiles_that_hand_over_different_numbers_of_candidates(ops, vocab):
    # up to 32 tiles hand over all ids above their own bound, more tiles exactly k of them; here one tile's large ids lie in one wave
    # (so many above its bound that it hands over k), one has a single value, one next to nothing, the last one is cut short
    g = torch.Generator().manual_seed(68)
    top_k = [1, 17, 50, 200, 256, 50]
    n = len(top_k)
    logits = torch.randn(n, vocab, generator=g) * 3
    logits[:, 8192:16384] = logits[:, 8192:16384].sort(dim=1).values
    logits[:, 16384:24576] = 9.0
    logits[5, 16384:24576] = 2.0
    logits[:, 24576:32768 - 20] = float("-inf")
    rows = logits.double().numpy()
    for top_p in (1.0, 0.9, 0.05):
        u = torch.rand(n, generator=g).tolist()
        u[1] = 0.99999994
        picks = _sample(ops, logits, [0.8] * n, top_k, [top_p] * n, u)
        for r in range(n):
            assert _pick_is_right(rows[r], 0.8, top_k[r], top_p, u[r], picks[r]), (r, top_k[r], top_p)


@pytest.mark.parametrize("vocab", [6 * 8192 + 1, 6 * 8192 + 2049, 7 * 8192 - 1, 7 * 8192])
def test_sample_rows_takes_the_same_ids_where_the_tiles_are_many(ops, vocab):
    # 768 tiles and more are taken by other blocks (four stretches of ids a wave): the same sums in the same order, so the same ids, as
    # when a few rows are sampled alone; the largest are found among the logits (neighbours of one quotient included), quotients come from
    # a reciprocal where all sizes allow it
    g = torch.Generator().manual_seed(18)
    n = 110
    logits = torch.randn(n, vocab, generator=g) * 3
    logits[10:20] = torch.round(logits[10:20] * 2) / 2                  # ids of one value, zeros of both signs among them
    logits[20:25] = logits[20:25].to(torch.bfloat16).float()
    logits[25:30, ::3] = float("-inf")
    logits[30:33] = -logits[30:33].abs() - 100.0
    logits[33:36] *= 1e-13                                              # (too small for the reciprocal)
    logits[36:39] *= 1e12
    logits[39, : vocab - 40] = float("-inf")
    big = torch.full((vocab,), 8388608.0) + torch.randint(0, 40, (vocab,), generator=g)
    logits[40:44] = big                                                 # neighbouring float32 numbers, two of which share a quotient now and then
    temperature = [(0.0, 0.7, 3.0, 0.8, 1.3)[i % 5] for i in range(n)]
    for r in range(33, 36):
        temperature[r] = 1e-13
    for r in (*range(36, 39), *range(40, 44)):
        temperature[r] = (3e12, 3.0, 5.0, 3.0, 7.0, 1e12, 1.7)[r % 7]
    top_k = [(0, 50, 3, 256, 0, 200, 1)[i % 7] for i in range(n)]
    top_p = [(1.0, 0.9, 0.5)[i % 3] if top_k[i] else 1.0 for i in range(n)]
    u = torch.rand(n, generator=g).tolist()
    picks = _sample(ops, logits, temperature, top_k, top_p, u)
    for r in range(n):
        one = _sample(ops, logits[r:r + 1], temperature[r:r + 1], top_k[r:r + 1], top_p[r:r + 1], u[r:r + 1])[0]
        assert picks[r] == one, r
        if r < 45:
            row = logits[r].double().numpy()
            if temperature[r] == 0.0:
                assert picks[r] == plain_impl.argmax_first(row), r
            elif r < 40:                                                # (beyond: the float64 quotients differ where the float32 ones are one)
                assert _pick_is_right(row, temperature[r], top_k[r], top_p[r], u[r], picks[r], 1e-4), r


@pytest.mark.parametrize("mask", ["half", "lowest", "behind", "few", "zeros", "tiny"])
def test_masked_logits_where_the_tiles_are_many_and_few(ops, mask):
    # ids that may not come (-inf, the lowest number), scattered, behind a place within a tile (its stretches without a mask give the
    # bound), or all but a few (fewer than are wanted above a tile's lowest); zeros and values too small for the reciprocal; top-p alone too
    g = torch.Generator().manual_seed(72)
    vocab, n = 6 * 8192 + 2049, 112                                     # 784 tiles of seven a row; six rows are 42
    logits = torch.randn(n, vocab, generator=g) * 3
    hit = torch.rand(n, vocab, generator=g)
    if mask == "behind":
        logits[:, 3 * 8192 + 2100:] = float("-inf")
        logits[1::2, :8192 + 4090] = float("-inf")
    elif mask in ("zeros", "tiny"):
        logits[hit < 0.02] = 0.0 if mask == "zeros" else 1e-20
    else:
        logits[hit < (0.9995 if mask == "few" else 0.5)] = torch.finfo(torch.float32).min if mask == "lowest" else float("-inf")
    temperature = [(0.7, 1.3, 0.0, 0.9, 2.0)[i % 5] for i in range(n)]
    top_k = [(0, 50, 200, 0, 3, 0, 256)[i % 7] for i in range(n)]
    top_p = [(1.0, 0.9, 0.5, 0.7, 1.0, 1.0, 0.95)[i % 7] for i in range(n)]
    u = torch.rand(n, generator=g).tolist()
    many = _sample(ops, logits, temperature, top_k, top_p, u)
    few = sum((_sample(ops, logits[r:r + 6], temperature[r:r + 6], top_k[r:r + 6], top_p[r:r + 6], u[r:r + 6]) for r in range(0, 42, 6)), [])
    assert many[:42] == few
    for r in range(42):
        row = logits[r].double().numpy()
        assert row[many[r]] > -1e30, r
        if temperature[r] == 0.0:
            assert many[r] == plain_impl.argmax_first(row), r
        else:
            assert _pick_is_right(row, temperature[r], top_k[r], top_p[r], u[r], many[r], 1e-4), r


@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 128, 129])
def test_options_in_the_arguments_choose_what_options_in_arrays_choose(ops, n):
    # sample_async hands options that are packed to the launch itself, up to 128 rows; objects that hold the same numbers unpacked go
    # the arrays' way.  Several results at a time, one of them never asked for
    from types import SimpleNamespace

    from litinfer_amd.sampling import Sampler, SamplingParams, sampler
    sm, g = Sampler(DEV), torch.Generator().manual_seed(19)
    logits = (torch.randn(n, 5000, generator=g) * 3).to(DEV)
    params = [SamplingParams(temperature=(0.7, 0.0, 1.2, float("nan"), -1.0)[i % 5], top_k=(0, 5, 50, -3, 6000)[i % 5], top_p=(1.0, 0.9, 2.0)[i % 3],
                             seed=(i, -i, 2 ** 64 - 1 - i, 2 ** 70 + i)[i % 4]) for i in range(n)]
    plain = [SimpleNamespace(temperature=p.temperature, top_k=p.top_k, top_p=p.top_p, seed=p.seed, greedy=p.greedy) for p in params]
    counters = [3 * i for i in range(n)]
    ids, other = torch.empty(n, dtype=torch.int32, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
    first = sm.sample_async(logits, params, counters, out=ids)
    sm.sample_async(logits, params, counters)                            # (let go at once)
    second = sm.sample_async(logits, plain, counters, out=other)
    third = sm.sample_async(logits * 0.5, params, counters)
    want = second.result()
    assert first.result() == want == ids.tolist() == other.tolist()
    assert third.result() == sm.sample_async(logits * 0.5, plain, counters).result()
    torch.cuda.synchronize()
    sm.sample(logits, params, counters)                                  # (a call lets go of what has been written by now)
    assert not sampler._unread


def test_sample_rows_frequencies_and_ties(ops):
    lg = torch.tensor([[2.0, 1.0, 3.0, 3.0, -1.0, 0.5, 2.5, 0.0]])
    n = 4000
    g = torch.Generator().manual_seed(14)
    u = torch.rand(n, generator=g).tolist()
    picks = _sample(ops, lg.repeat(n, 1), [1.0] * n, [0] * n, [1.0] * n, u)
    freq = np.bincount(picks, minlength=8) / n
    want = np.exp(lg[0].double().numpy())
    assert np.abs(freq - want / want.sum()).max() < 0.03
    # top_k = 1 with two equal maxima: the lower index; top_k = 3: ids 2, 3 and 6 only
    assert set(_sample(ops, lg.repeat(50, 1), [1.0] * 50, [1] * 50, [1.0] * 50, u[:50])) == {2}
    assert set(_sample(ops, lg.repeat(500, 1), [1.0] * 500, [3] * 500, [1.0] * 500, u[:500])) == {2, 3, 6}
    # top_p = 0.5: the shortest prefix reaching half the mass is {2, 3}
    assert set(_sample(ops, lg.repeat(500, 1), [1.0] * 500, [0] * 500, [0.5] * 500, u[:500])) == {2, 3}


def test_sampling_table_rows_become_the_arrays_of_a_step_with_uniform_numbers_drawn_on_the_device(ops):
    """li_sample_prepare against the host's stream: the same uniform numbers bit for bit for any seed and
    count, a count that goes up for sampling rows only, greedy flags, slots outside the table."""
    from litinfer_amd.sampling import Sampler, SamplingParams, uniform
    smp = Sampler(DEV, slots=6)
    opts = [SamplingParams(temperature=0.8, top_k=7, top_p=0.9, seed=0), SamplingParams(temperature=1.5, seed=2 ** 64 - 1),
            SamplingParams(), SamplingParams(temperature=0.3, top_p=0.5, seed=-12345678901234),
            SamplingParams(temperature=1.0, seed=0x9E3779B97F4A7C15)]
    draws = [0, 5, 0, 2 ** 31 - 3, 1000000]
    for slot, (sp, c) in enumerate(zip(opts, draws)):
        smp.bind(slot, sp, c)
    rows = torch.tensor([4, 0, 3 | ops.SAMPLE_ROW_GREEDY, 2, 1, 5, 77], dtype=torch.int32, device=DEV)
    n = rows.numel()
    t, p, u = (torch.full((n,), -1.0, device=DEV) for _ in range(3))
    k = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    for step in range(3):
        ops.sample_prepare(rows, smp.table, t, k, p, u)
        for i, slot in enumerate((4, 0, None, 2, 1, None, None)):      # None: greedy by flag, an unbound row, outside the table
            if slot is None or opts[slot].greedy:
                assert float(t[i]) == 0.0 and float(u[i]) == 0.0
                continue
            sp = opts[slot]
            assert float(t[i]) == np.float32(sp.temperature) and int(k[i]) == sp.top_k and float(p[i]) == np.float32(sp.top_p)
            assert float(u[i]) == uniform(sp.seed, draws[slot] + step), (slot, step)
    counts = smp.table[:, 5].cpu().tolist()
    assert counts == [3, 8, 0, draws[3], 1000003, 0]               # slot 3 was greedy by flag: its count stayed


def test_decode_attention_refuses_block_tables_beyond_the_keys_its_page_quotient_is_exact_for(ops):
    """The matrix-core decode kernel finds a key's page by a float32 product that is exact below 2^22; the host
    refuses a table that could hold more than 2^21 keys instead of reading a wrong page."""
    nh, nkv, dh, page = 4, 2, 128, 16
    width = (1 << 21) // page + 1
    tab = torch.zeros(1, width, dtype=torch.int32, device=DEV)
    one = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)
    ql, cl, qs = np.array([1], np.int32), np.array([40], np.int32), np.array([0], np.int32)
    meta = AttentionMeta(block_table=tab, max_blocks=width, seg_of_token=one(0), q_start=one(0), q_len=one(1),
                         ctx_len=one(40), num_segments=1, num_tokens=1, max_q_len=1, max_ctx_len=40, host_q_start=qs,
                         host_q_len=ql, host_ctx_len=cl, single_tokens=None, num_single=1, multi_tokens=None,
                         num_multi=0, max_single_ctx=40)
    kc = torch.zeros(4, nkv, page, dh, dtype=torch.bfloat16, device=DEV)
    q = torch.zeros(1, nh * dh, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="beyond the decode kernel"):
        ops.paged_attention(q, torch.empty_like(q), kc, kc.clone(), meta, nh, nkv, dh, page, 0, 0.1)


@pytest.mark.parametrize("counts,n_out,k,act,weigh,gather,out_dtype", [
    ([1, 16, 0, 17, 32, 3], 36, 1000, 0, False, True, torch.float32),      # one row, whole and broken halves of a tile; a last chunk of 104 k-values, a last column tile of 4
    ([5, 2], 4, 8, 0, False, False, torch.bfloat16),                       # less than a chunk
    ([3, 0, 2], 64, 1280, 2, False, True, torch.bfloat16),                 # pairs of gate and up
    ([2, 9, 40], 100, 520, 3, False, True, torch.float32),                 # the clamped pairs; an expert of two tiles
    ([7, 6, 1], 20, 136, 4, True, True, torch.bfloat16),                   # weights on the input, gelu
    ([30, 1, 28], 132, 1160, 1, False, False, torch.bfloat16),
    ([9, 11, 10], 34, 264, 0, False, True, torch.float32),                 # 34 outputs: not a multiple of 4, another kernel
])
def test_routed_product_of_a_decoding_batch(ops, counts, n_out, k, act, weigh, gather, out_dtype):
    """Rows of every expert against its matrix; a float32 result within the random walk of K products' sums, a bfloat16
    one within its rounding (2^-9 of a value, taken twice)."""
    g = torch.Generator().manual_seed(63)
    rows, E = sum(counts), len(counts)
    tokens = rows if not gather else rows + 3
    a = torch.randn(tokens, k + 8, generator=g).to(torch.bfloat16)[:, :k]             # rows with a stride of their own
    w = (torch.randn(E, n_out, k, generator=g) / math.sqrt(k) * 2).to(torch.bfloat16)
    src = torch.randperm(tokens, generator=g)[:rows] if gather else torch.arange(rows)
    row_wt = torch.rand(rows, generator=g) + 0.5 if weigh else None
    tiles, r, ref = [], 0, []
    for e, n in enumerate(counts):
        tiles += [(e, r + o, min(32, n - o), 0) for o in range(0, n, 32)]
        y = a[src[r:r + n]].double() @ w[e].double().t()
        ref.append(y * row_wt[r:r + n, None].double() if weigh else y)
        r += n
    y = torch.cat(ref)
    if act == 1:
        y = y.clamp(min=0) ** 2
    elif act == 2:
        y = torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
    elif act == 3:
        gate, up = y[:, 0::2].clamp(max=1.5), y[:, 1::2].clamp(-1.5, 1.5)
        y = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
    elif act == 4:
        y = torch.nn.functional.gelu(y)
    plan = torch.tensor([len(tiles), rows, 0, 0] + [v for t in tiles for v in t], dtype=torch.int32)
    plan = torch.cat([plan, torch.full((16,), -1, dtype=torch.int32)])                 # four tiles that the plan does not have
    out = torch.full((rows, y.shape[1]), float("nan"), dtype=out_dtype, device=DEV)
    wide = torch.zeros(tokens, k + 8, dtype=torch.bfloat16, device=DEV)
    wide[:, :k] = a.to(DEV)
    ops.moe_linear(wide[:, :k], src.to(torch.int32).to(DEV) if gather else None, w.to(DEV), plan.to(DEV), len(tiles) + 4, out, rows,
                   act=act, limit=1.5 if act == 3 else 0.0, row_wt=None if row_wt is None else row_wt.to(DEV))
    assert rel(out, y.numpy()) < (8 * math.sqrt(k) * 2.0 ** -24 if out_dtype is torch.float32 else 8e-3)


@pytest.mark.parametrize("counts,n_out,k,act,out_dtype", [([1, 0, 2], 20, 2560, 0, torch.float32), ([1, 0, 3], 22, 2568, 2, torch.bfloat16),
                                                           ([1], 37, 4096, 0, torch.float32)])      # pieces held by a wave, and one piece more
def test_routed_product_of_few_long_rows(ops, counts, n_out, k, act, out_dtype):
    test_routed_product_of_a_decoding_batch(ops, counts, n_out, k, act, False, True, out_dtype)


@pytest.mark.parametrize("counts,tile,n_out,k,act,weigh,gather,out_dtype", [
    ([1, 64, 0, 65, 63], 64, 32, 64, 0, False, True, torch.float32),           # one step of k; a quarter of a block's outputs
    ([130, 5, 200], 64, 160, 192, 2, False, True, torch.bfloat16),             # three steps, pairs of gate and up
    ([1, 128, 0, 129, 127], 128, 96, 128, 4, True, True, torch.bfloat16),      # two steps, weights on the input
    ([300, 3], 128, 288, 320, 3, False, False, torch.float32),
    ([70, 200, 1], 128, 224, 96, 1, False, True, torch.float32),               # k no multiple of 64: the kernel that stages through registers
    ([400, 390, 410, 401, 399, 380, 420, 400], 128, 2208, 64, 0, False, True, torch.float32),      # 192 outputs a block, the last half full
    ([129] * 3, 128, 1056, 576, 2, False, True, torch.bfloat16)])              # fewer tiles than XCDs
def test_routed_product_of_many_rows_an_expert(ops, counts, tile, n_out, k, act, weigh, gather, out_dtype):
    """As of a decoding batch, in the tiles of a prompt's portion; places of the plan behind its last tile hold anything."""
    g = torch.Generator(device=DEV).manual_seed(64)
    rows, E = sum(counts), len(counts)
    tokens = rows if not gather else rows + 3
    wide = torch.randn(tokens, k + 8, generator=g, device=DEV).to(torch.bfloat16)       # rows with a stride of their own
    a = wide[:, :k]
    w = (torch.randn(E, n_out, k, generator=g, device=DEV) / math.sqrt(k) * 2).to(torch.bfloat16)
    src = torch.randperm(tokens, generator=g, device=DEV)[:rows] if gather else torch.arange(rows, device=DEV)
    row_wt = torch.rand(rows, generator=g, device=DEV) + 0.5 if weigh else None
    tiles, r, ref = [], 0, []
    for e, n in enumerate(counts):
        tiles += [(e, r + o, min(tile, n - o), 0) for o in range(0, n, tile)]
        y = a[src[r:r + n]].double() @ w[e].double().t().contiguous()
        ref.append(y * row_wt[r:r + n, None].double() if weigh else y)
        r += n
    y = torch.cat(ref)
    if act == 1:
        y = y.clamp(min=0) ** 2
    elif act == 2:
        y = torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
    elif act == 3:
        gate, up = y[:, 0::2].clamp(max=1.5), y[:, 1::2].clamp(-1.5, 1.5)
        y = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
    elif act == 4:
        y = torch.nn.functional.gelu(y)
    most = rows // tile + E
    plan = torch.full((4 + 4 * most,), 1 << 20, dtype=torch.int32)
    plan[:4 + 4 * len(tiles)] = torch.tensor([len(tiles), rows, 0, 0] + [v for t in tiles for v in t], dtype=torch.int32)
    out = torch.full((rows, y.shape[1]), float("nan"), dtype=out_dtype, device=DEV)
    for _ in range(2):
        ops.moe_linear(a, src.to(torch.int32) if gather else None, w, plan.to(DEV), most, out, rows, act=act, tile_rows=tile,
                       limit=1.5 if act == 3 else 0.0, row_wt=row_wt)
        assert rel(out, y.cpu().numpy()) < (8 * math.sqrt(k) * 2.0 ** -24 if out_dtype is torch.float32 else 8e-3)


@pytest.mark.parametrize("k", [128, 512, 1160, 1536, 4736])
def test_routed_product_of_a_decoding_batch_is_as_exact_as_of_few_rows(ops, k):
    """No further from the float64 result than the same rows four at a time, which another kernel takes."""
    g = torch.Generator(device=DEV).manual_seed(72)
    rows, n_out = 20, 1024
    a = torch.randn(rows, k, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2, n_out, k, generator=g, device=DEV) / math.sqrt(k)).to(torch.bfloat16)
    plan = lambda *tiles: torch.tensor([len(tiles), 0, 0, 0] + [v for t in tiles for v in t + (0,)], dtype=torch.int32, device=DEV)
    batch, few = torch.empty(rows, n_out, device=DEV), torch.empty(rows, n_out, device=DEV)
    ops.moe_linear(a, None, w, plan((0, 0, 12), (1, 12, 8)), 2, batch, rows)
    for r in range(0, rows, 4):
        ops.moe_linear(a[r:r + 4], None, w, plan((int(r >= 12), 0, 4)), 1, few[r:r + 4], 4)
    want = torch.cat([a[:12].double() @ w[0].double().t(), a[12:].double() @ w[1].double().t()])
    error = [float((v.double() - want).norm()) for v in (batch, few)]
    assert error[0] < 1.03 * error[1], error               # (equal ones differ by 1 / sqrt(2 x 20,480) of themselves)


@pytest.mark.parametrize("tokens,top,experts,n_out,k,streams", [
    (1, 4, 16, 2240, 1536, False), (1, 5, 16, 2240, 1536, False), (1, 7, 16, 2240, 1536, True), (1, 5, 16, 1536, 1024, True),
    (1, 5, 4, 2240, 1536, True), (2, 6, 64, 768, 1536, False), (2, 3, 64, 768, 1536, True), (2, 10, 64, 768, 1536, True),
    (40, 4, 16, 1536, 2240, True), (41, 4, 16, 1536, 2240, False), (64, 4, 16, 1536, 2240, False),
    (96, 1, 8, 3584, 4736, True), (97, 1, 8, 3584, 4736, False), (80, 8, 64, 768, 1536, True), (81, 8, 64, 768, 1536, False),
    (5, 2, 128, 256, 512, True),                 # fewer rows than experts
])
def test_which_routed_products_stream_the_matrices(ops, tokens, top, experts, n_out, k, streams):
    import ctypes
    takes = ops._lib_fn("moe", "li_moe_linear_streams", [ctypes.c_int] * 4, ctypes.c_int)
    assert bool(takes(tokens * top, ops.moe_max_tiles(tokens, top, experts), n_out, k)) == streams


@pytest.mark.parametrize("tokens", [1, 2, 3, 5, 8, 16, 17, 40])        # 1, 2, 4 and 8 tokens a block, whole and cut
@pytest.mark.parametrize("heads,n_out,n_in", [(3, 70, 520), (2, 130, 256), (2, 64, 264), (1, 5, 36)])      # trips of 256 bfloat16 or 128 float32 inputs, whole, cut and one piece over
@pytest.mark.parametrize("kind", ["float32", "bfloat16", "to_float32"])
@pytest.mark.parametrize("gated", [None, "heads", "columns"])
def test_per_head_products_of_few_tokens(ops, tokens, heads, n_out, n_in, kind, gated):
    g = torch.Generator().manual_seed(73)
    dt = torch.float32 if kind == "float32" else torch.bfloat16
    x = torch.randn(tokens, heads, n_in, generator=g).to(dt)
    m = (torch.randn(heads, n_out, n_in, generator=g) / math.sqrt(n_in)).to(dt)
    gate = None if gated is None else torch.randn(tokens, heads * (1 if gated == "heads" else n_out), generator=g)
    want = (x.double()[:, :, None, :] * m.double()[None]).sum(-1)
    if gate is not None:
        want = want * torch.sigmoid(gate.double()).view(tokens, heads, -1)
    out = torch.full((tokens, heads * n_out), float("nan"), dtype=torch.bfloat16 if kind == "bfloat16" else torch.float32, device=DEV)
    ops.headwise_linear(x.view(tokens, -1).to(DEV), heads * n_in, n_in, m.to(DEV), out, heads * n_out, n_out, tokens,
                        gate=None if gate is None else gate.to(DEV), gate_columns=gated == "columns")
    # sums of n_in exact products (of rounded ones in float32), or the rounding to bfloat16
    assert rel(out, want.reshape(tokens, -1).numpy()) < (8e-3 if kind == "bfloat16" else 8 * math.sqrt(n_in) * 2.0 ** -24)


def _one_token_batch(n):
    import types
    at = np.arange(n, dtype=np.int32)
    dev = lambda a: torch.from_numpy(a).to(DEV)
    return types.SimpleNamespace(num_tokens=n, num_segments=n, max_q_len=1, host_state_slots=at[::-1].copy(), state_slots=dev(at[::-1].copy()),
                                 q_start=dev(at), q_len=dev(np.ones(n, dtype=np.int32)))


@pytest.mark.parametrize("n,heads,vdim,n_state,groups", [
    (1, 48, 64, 128, 8),          # few requests: a head's columns over the most lanes
    (3, 6, 20, 100, 2),           # columns and values that fill neither a wave nor the lanes' shares
    (2, 4, 256, 256, 4),
    (5, 2, 4, 12, 1),             # one piece of columns
    (40, 48, 64, 128, 8),         # enough requests: fewer lanes a column
])
@pytest.mark.parametrize("kind", ["ssm", "fixed", "delta"])
def test_recurrences_of_a_decoding_step(ops, kind, n, heads, vdim, n_state, groups):
    """One token a request from its state, in slots in reverse order; against the equations in float64, within the random
    walk of a column's 2 n_state products."""
    g = torch.Generator().manual_seed(64)
    R = lambda *s: torch.randn(*s, generator=g)
    inner, rep = heads * vdim, heads // groups
    ctx = _one_token_batch(n)
    state = R(n + 1, heads, n_state, vdim) * 0.3
    rows = R(n, inner + 2 * groups * n_state)
    aux, bias, a_log, d = R(n, 2 * heads), R(heads) - 2.0, torch.rand(heads, generator=g), R(heads)
    fixed = torch.linspace(0.9, 0.99, heads)
    old = state.double()[torch.arange(n - 1, -1, -1)]
    w = rows.double()
    v = w[:, :inner].view(n, heads, vdim)
    b = w[:, inner:inner + groups * n_state].view(n, groups, n_state).repeat_interleave(rep, 1)
    c = w[:, inner + groups * n_state:].view(n, groups, n_state).repeat_interleave(rep, 1)
    dev_state, y = state.to(DEV), torch.full((n, inner), float("nan"), device=DEV)
    sp = torch.nn.functional.softplus
    if kind == "delta":
        unit = lambda z: z / (z.square().sum(-1, keepdim=True) + 1e-6).sqrt()
        k, q = unit(b), unit(c) * n_state ** -0.5
        beta, decay = torch.sigmoid(aux.double()[:, :heads]), torch.exp(-a_log.double().exp() * sp(aux.double()[:, heads:] + bias.double()))
        new = old * decay[:, :, None, None]
        u = beta[:, :, None] * (v - (new * k[..., None]).sum(2))
        new = new + k[..., None] * u[:, :, None]
        want = (new * q[..., None]).sum(2)
        ops.delta_scan(rows.to(DEV), aux.to(DEV), bias.to(DEV), a_log.to(DEV), dev_state, ctx, y, heads, vdim, n_state, groups, n_state ** -0.5)
    else:
        dt = torch.full((n, heads), 0.3, dtype=torch.float64) if kind == "fixed" else sp(aux.double()[:, :heads] + bias.double())
        decay = fixed.double().expand(n, heads) if kind == "fixed" else torch.exp(-a_log.double().exp() * dt)
        new = old * decay[:, :, None, None] + (dt[:, :, None] * b)[..., None] * v[:, :, None]
        want = (new * c[..., None]).sum(2) + d.double()[None, :, None] * v
        gpu = lambda z: None if kind == "fixed" else z.contiguous().to(DEV)
        ops.ssm_scan(rows.to(DEV), gpu(aux[:, :heads]), gpu(bias), gpu(a_log), d.to(DEV), dev_state, ctx, y, heads, vdim, n_state, groups, None,
                     fixed_decay=fixed.to(DEV) if kind == "fixed" else None, fixed_step=0.3)
    tol_ = 8 * math.sqrt(2 * n_state) * 2.0 ** -24
    assert rel(y, want.reshape(n, -1).numpy()) < tol_
    assert rel(dev_state[torch.arange(n - 1, -1, -1)], new.numpy()) < tol_
    assert torch.equal(dev_state[n].cpu(), state[n])                       # a slot that is not in the batch


@pytest.mark.parametrize("n,heads,vdim,n_state,groups", [(40, 5, 32, 16, 5), (3, 3, 20, 12, 3), (70, 6, 128, 64, 2)])
@pytest.mark.parametrize("kind", ["ssm", "fixed", "delta"])
def test_recurrences_of_a_decoding_step_with_idle_waves(ops, kind, n, heads, vdim, n_state, groups):
    """Heads that fill no whole block: waves without columns, lanes without columns and values."""
    test_recurrences_of_a_decoding_step(ops, kind, n, heads, vdim, n_state, groups)


@pytest.mark.parametrize("lens,heads,vdim,n_state,groups,skip_d", [
    ([65], 6, 64, 128, 2, False),                # a chunk and one token
    ([64, 1, 130, 7], 4, 36, 100, 4, False),     # one whole chunk, one token, a short last chunk, less than a chunk; values that fill no fragment
    ([64, 1, 130, 7], 4, 20, 100, 4, False),     # ... narrow heads with many state values: token by token in chunks
    ([200, 190], 3, 68, 24, 1, True),            # columns over a second block; no term of x
    ([96], 2, 8, 256, 2, False),
    ([96], 2, 72, 252, 2, False),                # four shares of the state values, the last one cut
    ([70], 4, 6, 30, 2, False),                  # not in 16-byte pieces: token by token in chunks
])
def test_state_space_recurrence_of_long_portions(ops, lens, heads, vdim, n_state, groups, skip_d):
    """Against the equations in float64, within the random walk of a column's 2 n_state + 128 products."""
    import types
    g = torch.Generator().manual_seed(65)
    R = lambda *s: torch.randn(*s, generator=g)
    n, T, inner, rep = len(lens), sum(lens), heads * vdim, heads // groups
    starts = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    dev = lambda a: torch.from_numpy(np.asarray(a, dtype=np.int32)).to(DEV)
    slots = list(range(n))[::-1]
    ctx = types.SimpleNamespace(num_tokens=T, num_segments=n, max_q_len=max(lens), host_state_slots=np.array(slots, dtype=np.int32),
                                state_slots=dev(slots), q_start=dev(starts), q_len=dev(lens))
    state, rows, dt = R(n, heads, n_state, vdim) * 0.3, R(T, inner + 2 * groups * n_state), R(T, heads)
    bias, a_log, d = R(heads) - 3.0, 2.0 * torch.rand(heads, generator=g), None if skip_d else R(heads)
    dev_state, y = state.to(DEV), torch.full((T, inner), float("nan"), device=DEV)
    ops.ssm_scan(rows.to(DEV), dt.to(DEV), bias.to(DEV), a_log.to(DEV), None if skip_d else d.to(DEV), dev_state, ctx, y, heads, vdim,
                 n_state, groups, _Lender())
    step = torch.nn.functional.softplus(dt.double() + bias.double())
    decay = torch.exp(-a_log.double().exp() * step)
    tol_ = 8 * math.sqrt(2 * n_state + 128) * 2.0 ** -24
    for i, (o, L) in enumerate(zip(starts, lens)):
        S, out = state[slots[i]].double(), []
        for t in range(o, o + L):
            x, b, c = rows[t].double().split([inner, groups * n_state, groups * n_state])
            x, b, c = x.view(heads, vdim), b.view(groups, n_state).repeat_interleave(rep, 0), c.view(groups, n_state).repeat_interleave(rep, 0)
            S = decay[t][:, None, None] * S + (step[t][:, None] * b)[:, :, None] * x[:, None]
            out.append((S * c[:, :, None]).sum(1) + (0.0 if skip_d else d.double()[:, None] * x))
        assert rel(y[o:o + L], torch.stack(out).reshape(L, -1).numpy()) < tol_, i
        assert rel(dev_state[slots[i]], S.numpy()) < tol_, i


@pytest.mark.parametrize("kind,silu", [("ssm", False), ("fixed", False), ("fixed", True)])
@pytest.mark.parametrize("vdim,n_state", [(64, 128), (132, 40)])
def test_recurrence_of_long_portions_keeps_values_that_are_not_finite_to_their_columns_and_later_tokens(ops, kind, silu, vdim, n_state):
    """Token by token an infinite value reaches its own column's state and outputs from its token on and nothing else: all
    other outputs and states are, bit for bit, those of the same portion without it."""
    import types
    g = torch.Generator().manual_seed(69)
    R = lambda *s: torch.randn(*s, generator=g)
    lens, heads, groups = [130, 40, 64], 4, 4
    n, T, inner = len(lens), sum(lens), heads * vdim
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(num_tokens=T, num_segments=n, max_q_len=max(lens), host_state_slots=np.arange(n, dtype=np.int32),
                                state_slots=dev([0, 1, 2]), q_start=dev([0, 130, 170]), q_len=dev(lens))
    state, rows, dt = R(n, heads, n_state, vdim) * 0.3, R(T, inner + 2 * groups * n_state), R(T, heads).to(DEV)
    bias, a_log, d = (R(heads) - 3.0).to(DEV), torch.rand(heads, generator=g).to(DEV), R(heads).to(DEV)
    fixed = torch.linspace(0.9, 0.99, heads).to(DEV)
    bad = [(0, 20, 5, float("inf")), (0, 63, 0, float("-inf")), (0, 64, vdim - 1, float("nan")), (0, 129, inner - 1, float("inf")),
           (1, 130, 7, float("inf")), (1, 169, 8, float("nan")), (2, 170 + 31, vdim, float("inf")), (2, 170 + 33, vdim, float("inf"))]
    spoilt = rows.clone()
    for _, t, col, v in bad:
        spoilt[t, col] = v

    def run(x):
        s, y = state.to(DEV), torch.zeros(T, inner, device=DEV)
        if kind == "ssm":
            ops.ssm_scan(x.to(DEV), dt, bias, a_log, d, s, ctx, y, heads, vdim, n_state, groups, _Lender())
        else:
            ops.ssm_scan(x.to(DEV), None, None, None, None, s, ctx, y, heads, vdim, n_state, groups, _Lender(), fixed_decay=fixed,
                         fixed_step=0.3, silu_in=silu)
        return y.cpu(), s.cpu()

    (y0, s0), (y1, s1) = run(rows), run(spoilt)
    ends = [130, 170, 234]
    reached, state_reached = torch.zeros(T, inner, dtype=torch.bool), torch.zeros(n, heads, n_state, vdim, dtype=torch.bool)
    for i, t, col, _ in bad:
        reached[t:ends[i], col] = True
        state_reached[i, col // vdim, :, col % vdim] = True
    assert torch.isfinite(y0).all() and torch.isfinite(s0).all()
    assert torch.equal(y1[~reached], y0[~reached]) and not torch.isfinite(y1[reached]).any()
    assert torch.equal(s1[~state_reached], s0[~state_reached]) and not torch.isfinite(s1[state_reached]).any()


@pytest.mark.parametrize("kind", ["ssm", "fixed"])
def test_recurrence_of_long_portions_leaves_requests_without_tokens_alone(ops, kind):
    """A request that brings no tokens, before, between and behind others: no chunk is its own, its state stays as it was, and
    the other requests' outputs and states are those of a step without it."""
    import types
    g = torch.Generator().manual_seed(72)
    R = lambda *s: torch.randn(*s, generator=g)
    heads, vdim, n_state = 3, 36, 20
    T, inner = 230, heads * vdim
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    state, rows, dt = R(5, heads, n_state, vdim), R(T, inner + 2 * heads * n_state).to(DEV), R(T, heads).to(DEV)
    bias, a_log, d = R(heads).to(DEV), torch.rand(heads, generator=g).to(DEV), R(heads).to(DEV)
    fixed = torch.linspace(0.9, 0.99, heads).to(DEV)

    def run(lens, slots):
        starts = [sum(lens[:i]) for i in range(len(lens))]
        ctx = types.SimpleNamespace(num_tokens=T, num_segments=len(lens), max_q_len=max(lens), host_state_slots=np.array(slots, dtype=np.int32),
                                    state_slots=dev(slots), q_start=dev(starts), q_len=dev(lens))
        s, y = state.to(DEV), torch.zeros(T, inner, device=DEV)
        if kind == "ssm":
            ops.ssm_scan(rows, dt, bias, a_log, d, s, ctx, y, heads, vdim, n_state, heads, _Lender())
        else:
            ops.ssm_scan(rows, None, None, None, None, s, ctx, y, heads, vdim, n_state, heads, _Lender(), fixed_decay=fixed, fixed_step=0.3)
        return y.cpu(), s.cpu()

    (y0, s0), (y1, s1) = run([130, 100], [1, 3]), run([0, 130, 0, 100, 0], [0, 1, 2, 3, 4])
    assert torch.equal(y0, y1) and torch.equal(s0, s1)
    assert torch.equal(s1[[0, 2, 4]], state[[0, 2, 4]]) and not torch.equal(s1[1], state[1])


@pytest.mark.parametrize("a_log,dt_raw", [
    (2.0, 100.0),            # a decay of exp(-740): zero in float32
    (60.0, 3.0),             # an exponent of 1e26, beside which the other tokens' vanish
    (80.0, 1.0e4),           # ... that overflows
    (95.0, -2.0),            # a rate that overflows by itself
])
def test_state_space_recurrence_of_long_portions_with_decays_of_zero(ops, a_log, dt_raw):
    """Some tokens multiply the state by zero; the tokens between them decay as usual (heads 1 and 2) or also to zero (head 0)."""
    import types
    g = torch.Generator().manual_seed(70)
    R = lambda *s: torch.randn(*s, generator=g)
    lens, heads, vdim, n_state, groups = [130, 70, 20], 3, 64, 32, 1
    n, T, inner = len(lens), sum(lens), heads * vdim
    starts = [0, 130, 200]
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(num_tokens=T, num_segments=n, max_q_len=max(lens), host_state_slots=np.arange(n, dtype=np.int32),
                                state_slots=dev([0, 1, 2]), q_start=dev(starts), q_len=dev(lens))
    state, rows, dt = R(n, heads, n_state, vdim) * 0.3, R(T, inner + 2 * groups * n_state), R(T, heads)
    bias, rates, d = R(heads) - 3.0, torch.tensor([a_log, 0.5, a_log]), R(heads)
    for t in (5, 40, 41, 64, 127, 150, 199, 203):
        dt[t, :] = torch.tensor([dt_raw, 0.1, dt_raw])
    if a_log > 50:                                             # head 2: exponents near one for the other tokens
        quiet = torch.ones(T, dtype=torch.bool)
        quiet[[5, 40, 41, 64, 127, 150, 199, 203]] = False
        dt[quiet, 2] = -a_log - float(bias[2]) if a_log < 85 else dt[quiet, 2]
    dev_state, y = state.to(DEV), torch.full((T, inner), float("nan"), device=DEV)
    ops.ssm_scan(rows.to(DEV), dt.to(DEV), bias.to(DEV), rates.to(DEV), d.to(DEV), dev_state, ctx, y, heads, vdim, n_state, groups, _Lender())
    raw = (dt + bias).double()
    step = torch.where(raw > 20, raw, torch.log1p(torch.exp(raw.clamp(max=20))))
    decay = torch.exp(-rates.double().exp() * step)
    for i, (o, L) in enumerate(zip(starts, lens)):
        S, out = state[i].double(), []
        for t in range(o, o + L):
            x, b, c = rows[t].double().split([inner, groups * n_state, groups * n_state])
            x, b, c = x.view(heads, vdim), b.expand(heads, -1), c.expand(heads, -1)
            S = decay[t][:, None, None] * S + (step[t][:, None] * b)[:, :, None] * x[:, None]
            out.append((S * c[:, :, None]).sum(1) + d.double()[:, None] * x)
        want = torch.stack(out)
        for h in range(heads):                                 # (each head by itself: their sizes differ)
            got = y[o:o + L].view(L, heads, vdim)[:, h]
            assert rel(got, want[:, h].numpy()) < 8 * math.sqrt(2 * n_state + 128) * 2.0 ** -24, (i, h)
            assert rel(dev_state[i, h], S[h].numpy()) < 8 * math.sqrt(2 * n_state + 128) * 2.0 ** -24, (i, h)


@pytest.mark.parametrize("vdim,n_state", [(64, 128), (128, 256), (36, 100), (64, 132), (16, 252), (8, 128), (32, 36), (32, 32)])
def test_state_space_recurrence_of_long_portions_is_as_exact_as_token_by_token(ops, vdim, n_state):
    """The rule that takes long portions as matrix products, against the form it replaces (which rows that do not lie in
    16-byte pieces still take): no further from the float64 result."""
    import types
    T, heads, groups = 200, 32, 4
    inner, width = heads * vdim, heads * vdim + 2 * groups * n_state
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(num_tokens=T, num_segments=1, max_q_len=T, host_state_slots=np.zeros(1, dtype=np.int32),
                                state_slots=dev([0]), q_start=dev([0]), q_len=dev([T]))
    g = torch.Generator(device=DEV).manual_seed(71)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)
    rows, dt, state = torch.nn.functional.silu(R(T, width)), R(T, heads), R(1, heads, n_state, vdim) * 0.1
    bias, a_log, d = R(heads) * 0.1 - 3.0, 2.0 * torch.rand(heads, generator=g, device=DEV), R(heads)
    step = torch.nn.functional.softplus(dt.double() + bias.double())
    decay = torch.exp(-a_log.double().exp() * step)
    x, b, c = rows.double().split([inner, groups * n_state, groups * n_state], dim=1)
    x = x.view(T, heads, vdim)
    b, c = (v.view(T, groups, n_state).repeat_interleave(heads // groups, 1) for v in (b, c))
    S, want = state[0].double(), []
    for t in range(T):
        S = decay[t][:, None, None] * S + (step[t][:, None] * b[t])[:, :, None] * x[t][:, None]
        want.append((S * c[t][:, :, None]).sum(1) + d.double()[:, None] * x[t])
    want = torch.stack(want).view(T, inner)
    wide = torch.zeros(T, width + 1, device=DEV)
    wide[:, :width] = rows
    errors = []
    for xbc in (rows, wide[:, :width]):
        s, y = state.clone(), torch.empty(T, inner, device=DEV)
        ops.ssm_scan(xbc, dt, bias, a_log, d, s, ctx, y, heads, vdim, n_state, groups, _Lender())
        errors.append([float((v.double() - w).norm() / w.norm()) for v, w in ((y, want), (s[0], S))])
    assert all(product <= 1.01 * tokens for product, tokens in zip(*errors)), errors


@pytest.mark.parametrize("act", ["relu2", "gelu_tanh", "gelu", "xielu"])
@pytest.mark.parametrize("m,n,k,bias,ws", [
    (1, 36, 40, True, True),             # the few-row kernel: a chunk that is not whole, columns that fill no tile
    (8, 9000, 1536, False, True),        # ... many columns
    (24, 301, 520, True, True),          # ... two tiles of rows
    (40, 130, 72, True, True),           # 33 to 64 rows, K no multiple of 64: four tiles of rows
    (50, 300, 1024, True, True),         # K in parts
    (64, 17000, 128, False, True),       # 64-row tiles of 128 columns
    (37, 33000, 64, True, True),         # ... and of 256
    (33, 16387, 64, True, True),         # ... whose sums end inside a piece of four
    (65, 300, 4096, True, True),         # more rows, K in parts
    (300, 2053, 192, True, True),        # tiles whose last columns lie past the end, not in 16-byte pieces
    (1100, 4608, 320, False, True),
    (2050, 264, 64, True, True),
])
def test_linear_with_an_activation_of_its_sums(ops, act, m, n, k, bias, ws):
    g = torch.Generator().manual_seed(67)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * 2 / math.sqrt(k)).to(torch.bfloat16)
    b = torch.randn(n, generator=g) if bias else None
    sp, sq = 0.7, 1.3
    z = x.double() @ w.double().t() + (0 if b is None else b.double())
    want = {"relu2": lambda: z.clamp(min=0) ** 2, "gelu_tanh": lambda: torch.nn.functional.gelu(z, approximate="tanh"),
            "gelu": lambda: torch.nn.functional.gelu(z),
            "xielu": lambda: torch.where(z > 0, sp * z * z, sq * (torch.expm1(z) - z)) + 0.5 * z}[act]()
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    did = ops.linear_act(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), out, act, (sp, sq), _Lender())
    assert did == (m <= 64 or act == "relu2")
    if did:
        assert rel(out, want.numpy()) < 5e-3                       # the rounding to bfloat16
        # value by value: half a bfloat16 step of the value, and what the float32 sums of K products lose in the activation's slope
        slack = want.abs() * 2.0 ** -8 + 8 * math.sqrt(k) * 2.0 ** -24 * (1 + z.abs())
        assert bool(((out.double().cpu() - want).abs() <= slack).all())
    else:
        assert bool(torch.isnan(out.float()).all())


def test_where_the_tanh_form_of_gelu_is_the_gated_products_epilogue(ops):
    """The rule at its lines: a product that is not cut along K always, one that is by the length of K and, for 33 to 64 rows,
    by the matrix."""
    takes = lambda m, n, k: ops.gelu_gate_as_epilogue(m, n, k, torch.bfloat16)
    assert all(takes(m, 8960, 1536) for m in (1, 16, 17, 32, 65, 300, 2048)) and not takes(33, 8960, 1536) and not takes(64, 8960, 1536)
    assert takes(48, 6144, 1536) and takes(48, 14000, 768) and takes(64, 40000, 1024)
    assert takes(1, 2048, 4096) and takes(2048, 37888, 3584) and not any(takes(m, 4096, 4096) for m in (33, 64, 65, 128))
    assert ops.gelu_gate_as_epilogue(48, 8960, 1536, torch.float32)


@pytest.mark.parametrize("m,n,k", [(1, 100, 72), (9, 8960, 1536), (30, 50, 136), (64, 9000, 256), (200, 333, 128), (1030, 1500, 192)])
def test_gated_product_with_the_tanh_form_of_gelu(ops, m, n, k):
    g = torch.Generator().manual_seed(68)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * n, k, generator=g) * 2 / math.sqrt(k)).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    want = torch.nn.functional.gelu(z[:, :n], approximate="tanh") * z[:, n:]
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear_swiglu(x.to(DEV), w.to(DEV), out, limit=ops.GELU_TANH_GATE)
    assert rel(out, want.numpy()) < 5e-3
    if m <= 16:
        out = torch.full((m, n), float("nan"), device=DEV)
        ops.linear_swiglu(x.float().to(DEV), w.float().to(DEV), out, limit=ops.GELU_TANH_GATE)
        assert rel(out, want.numpy()) < 8 * math.sqrt(k) * 2.0 ** -24


@pytest.mark.parametrize("limit", [-1.0, -2.5])
@pytest.mark.parametrize("dtype,m", [(torch.bfloat16, 5), (torch.bfloat16, 40), (torch.bfloat16, 100), (torch.float32, 3)])
def test_gated_product_takes_a_limit_that_is_not_positive_as_none(ops, dtype, m, limit):
    g = torch.Generator().manual_seed(74)
    n, k = 300, 128
    x, w = torch.randn(m, k, generator=g).to(dtype).to(DEV), (torch.randn(2 * n, k, generator=g) * 2 / math.sqrt(k)).to(dtype).to(DEV)
    plain, other = torch.empty(m, n, dtype=dtype, device=DEV), torch.empty(m, n, dtype=dtype, device=DEV)
    ops.linear_swiglu(x, w, plain)
    ops.linear_swiglu(x, w, other, limit=limit)
    assert torch.equal(plain, other)


def test_the_profiler_sees_products_that_may_not_be_taken(ops, monkeypatch):
    """A product with an epilogue of its own is a row of the table like any other call; one that is not taken is none."""
    from litinfer_amd.utils import OpProfiler
    prof = OpProfiler(False)
    prof.enabled, prof.phase = True, "decode"
    monkeypatch.setattr(ops, "profiler", prof)
    bf16 = lambda *s: torch.randn(*s, device=DEV).to(torch.bfloat16)
    out = torch.empty(4, 48, dtype=torch.bfloat16, device=DEV)
    assert ops.linear_act(bf16(4, 64), bf16(48, 64), None, out, "gelu", ws=_Lender())
    assert not ops.linear_act(bf16(100, 64), bf16(48, 64), None, torch.empty(100, 48, dtype=torch.bfloat16, device=DEV), "gelu", ws=_Lender())
    m, n, k = 64, 3584, 18944
    rows, xn = torch.zeros(m, n, device=DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    assert ops.linear_then_norm(bf16(m, k), bf16(n, k), None, rows, torch.ones(n, device=DEV), 1e-6, xn, _Lender())
    assert ops.linear_tanh_norm(bf16(m, k), bf16(n, k), None, rows, 0.5, torch.ones(n, device=DEV), torch.zeros(n, device=DEV), xn, _Lender())
    assert dict(prof.calls) == {("decode", name): 1 for name in ("linear_act", "linear_then_norm", "linear_tanh_norm")}
    assert all(v > 0 for v in prof.total.values())


@pytest.mark.parametrize("vocab", [5 * 8192 + 3, 32 * 8192])
def test_top_p_alone_hands_over_exactly_its_candidates_or_all_above_a_bound(ops, vocab):
    # the latter from 513 tiles of rows on; the same rows in a step of few and in one of many, a prefix within the candidates and one
    # beyond them (flat rows), ties at the threshold
    few, many = 8, -(-513 // -(-vocab // 8192))
    g = torch.Generator().manual_seed(71)
    logits = torch.randn(many, vocab, generator=g) * 6
    logits[1] *= 0.1
    logits[2] = (logits[2] * 2).round() / 2
    logits[3, 100:] = -60.0
    rows = logits[:few].double().numpy()
    for top_p in (0.9, 0.3, 0.999):
        u = torch.rand(many, generator=g).tolist()
        a = _sample(ops, logits[:few], [0.8] * few, [0] * few, [top_p] * few, u[:few])
        b = _sample(ops, logits, [0.8] * many, [0] * many, [top_p] * many, u)
        for r in range(few):
            assert _pick_is_right(rows[r], 0.8, 0, top_p, u[r], a[r]) and _pick_is_right(rows[r], 0.8, 0, top_p, u[r], b[r]), (r, top_p)
