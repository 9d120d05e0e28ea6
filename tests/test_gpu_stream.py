"""The streaming few-row product (`csrc/stream.hpp`) in every weight format, against the f64
product of the exactly dequantized weight: row counts at the edges of its forms (4, 8, 16,
32 rows of x a workgroup, chunks of 32), K that ends inside a wave's share or a 256-input
line, a partial last tile and workgroup, groups within, of and over a 128-input step,
scales and zero points at odd addresses, and rows of x past the last.

Bound: half a unit in the last place of the result (one rounding; one more with a bias),
plus 16 f32 units of the sum of the products' magnitudes as they are added -- int4 codes
carry 128 (f16: 1024) plus the zero point, int8 in bf16 carries 128, until the fold."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from linnet_amd.torch import kernels
from oracle import linear, quant

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}
BF16, F16 = torch.bfloat16, torch.float16


def _x(rows: int, width: int, dtype: torch.dtype) -> torch.Tensor:
    return torch.randn(rows, width, generator=torch.Generator().manual_seed(rows + width)).to(dtype)


def _check(got: torch.Tensor, x: torch.Tensor, w: np.ndarray, carried: np.ndarray, bias: torch.Tensor | None = None) -> None:
    """`w` [Out, In] f64; `carried` the magnitudes the kernel adds up for each weight."""
    xd = x.double().numpy()
    ref = xd @ w.T
    bound = ULP[x.dtype] * np.abs(ref)
    if bias is not None:
        ref = ref + bias.double().numpy()
        bound = bound + ULP[x.dtype] * np.abs(ref)
    bound = bound + 2.0**-20 * (np.abs(xd) @ carried.T) + 2.0**-24
    err = np.abs(got.double().cpu().numpy() - ref)
    print(f"max err / bound {float((err / bound).max()):.3f}", flush=True)
    assert got.shape == ref.shape and np.all(err <= bound)


@pytest.mark.parametrize(("rows", "out", "width", "group", "dtype"), [
    (1, 40, 128, 32, BF16),  # one step, one wave, a partial tile
    (4, 300, 1152, 64, F16),  # 9 steps: an odd last unit; 4-row form
    (5, 2049, 1024, 128, BF16),  # GEMV's rows 5..16, a ragged last workgroup
    (8, 96, 2176, 128, F16),  # 17 groups: scale rows at odd addresses
    (9, 4100, 640, 32, BF16),  # 32 rows a workgroup, its last of 4
    (16, 520, 3072, 384, F16),  # a group of three steps
    (17, 130, 4352, 256, BF16),  # 32-row form, a group of two steps
    (33, 24, 14336, 64, BF16),  # two chunks; long K; 8 rows a workgroup
    (16, 14336, 4096, 64, F16),  # every wave two units, 56 rows a workgroup, one workgroup a CU
    (64, 20000, 256, 64, F16),  # more workgroups than CUs, one unit of weights
    (20, 512, 8192, 32, BF16),  # scales past the LDS beside 32 rows: fewer rows a workgroup
])
def test_int4(rows: int, out: int, width: int, group: int, dtype: torch.dtype) -> None:
    print(f"int4 stream rows={rows} out={out} in={width} group={group} {dtype}", flush=True)
    g = torch.Generator().manual_seed(out + width)
    groups = width // group
    packed = torch.randint(0, 256, (out, groups, group // 2), generator=g, dtype=torch.uint8)
    scale = (torch.rand(out * groups + 1, generator=g) * 0.02 + 0.001).to(dtype)[1:].view(out, groups)
    zero = torch.randint(0, 16, (out * groups + 3,), generator=g, dtype=torch.uint8)[3:].view(out, groups)
    bias = torch.randn(out, generator=g).to(dtype) if rows % 2 else None
    # Contiguous views one scale and three zero points into their buffers on the GPU.
    sd = torch.cat([scale.reshape(-1)[:1], scale.reshape(-1)]).to(DEV)[1:].view(out, groups)
    zd = torch.cat([zero.reshape(-1)[:3], zero.reshape(-1)]).to(DEV)[3:].view(out, groups)
    x = _x(rows, width, dtype)
    got = kernels.int4_linear(x.to(DEV), packed.to(DEV), sd, zd, None if bias is None else bias.to(DEV))
    q = quant.unpack_int4_codes(packed.numpy()).reshape(out, groups, group).astype(np.float64)
    s, z = scale.double().numpy()[..., None], zero.double().numpy()[..., None]
    offset = 128.0 if dtype == BF16 else 1024.0
    _check(got, x, ((q - z) * s).reshape(out, width), ((q + z + 2 * offset) * s).reshape(out, width), bias)


@pytest.mark.parametrize(("out", "width"), [(8192, 48640), (8192, 49024), (6144, 64896), (6144, 65408)])
def test_int4_scales_that_fill_the_lds(out: int, width: int) -> None:
    """Groups of 32 at 4 rows whose scales and zero points take all the LDS that the stages
    leave, against the skinny kernel (f32 sums in another order, one rounding each)."""
    print(f"int4 stream full LDS out={out} in={width}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(width)
    packed = torch.randint(0, 256, (out, width // 32, 16), generator=g, dtype=torch.uint8, device=DEV)
    scale = (torch.rand(out, width // 32, generator=g, device=DEV) * 0.02 + 0.001).to(BF16)
    zero = torch.randint(0, 16, (out, width // 32), generator=g, dtype=torch.uint8, device=DEV)
    x = torch.randn(4, width, generator=g, device=DEV).to(BF16)
    got = kernels.int4_linear(x, packed, scale, zero).double()
    want = kernels.int4_linear(x, packed, scale, zero, kernel="skinny").double()
    # Half a unit in the last place each, and 16 f32 units of the magnitudes added: |x| times
    # codes that carry 128 and the zero point, at most (2 * 128 + 30) * 0.021.
    carried = x.double().abs().sum(1, keepdim=True) * (286 * 0.021)
    assert bool(((got - want).abs() <= 2 * ULP[BF16] * want.abs() + 2.0**-19 * carried).all())


@pytest.mark.parametrize(("rows", "out", "width", "group"), [
    (16, 2048, 512, 128), (24, 4096, 512, 64), (17, 1000, 1024, 128), (64, 4096, 1024, 128), (36, 2048, 2048, 256),
    (48, 4096, 512, 32), (64, 8192, 256, 64), (65, 2048, 1536, 384), (600, 1024, 2176, 2176)])
def test_int4_short_layers_keep_the_skinny_kernel(rows: int, out: int, width: int, group: int) -> None:
    """Where the skinny kernel is the faster one the automatic choice has its bits."""
    print(f"int4 short layer rows={rows} out={out} in={width} group={group}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows)
    packed = torch.randint(0, 256, (out, width // group, group // 2), generator=g, dtype=torch.uint8, device=DEV)
    scale = (torch.rand(out, width // group, generator=g, device=DEV) * 0.02 + 0.001).to(F16)
    zero = torch.randint(0, 16, (out, width // group), generator=g, dtype=torch.uint8, device=DEV)
    x = torch.randn(rows, width, generator=g, device=DEV).to(F16)
    assert torch.equal(kernels.int4_linear(x, packed, scale, zero), kernels.int4_linear(x, packed, scale, zero, kernel="skinny"))


@pytest.mark.parametrize("fp8", [True, False])
@pytest.mark.parametrize(("rows", "out", "width", "group", "row_block", "dtype"), [
    (1, 72, 640, 0, 1, BF16),  # one row, a scale a row, 5 steps
    (3, 5000, 4096, 0, 1, F16),
    (8, 100, 2176, 64, 1, BF16),  # two groups a step
    (16, 264, 1280, 128, 1, F16),
    (31, 48, 3840, 384, 1, BF16),  # a group of three steps
    (33, 60, 1152, 192, 5, F16),  # groups of 1.5 steps, a scale row for 5 weight rows
    (64, 1024, 1024, 128, 128, BF16),  # block scales
    (1, 24, 65664, 0, 1, BF16),  # past the streaming kernel's inputs: the skinny kernel's 16-,
    (20, 40, 65664, 128, 1, F16),  # 32-
    (40, 24, 65664, 64, 1, BF16),  # and 64-row forms
    (130, 300, 1024, 128, 1, F16),  # past 64 rows, where the skinny kernel is the faster one
])
def test_eight_bit(fp8: bool, rows: int, out: int, width: int, group: int, row_block: int, dtype: torch.dtype) -> None:
    print(f"w8 stream fp8={fp8} rows={rows} out={out} in={width} group={group}/{row_block} {dtype}", flush=True)
    g = torch.Generator().manual_seed(out + width)
    if fp8:
        weight = (torch.randn(out, width, generator=g) * 60).clamp(-448, 448).to(torch.float8_e4m3fn)
        w = weight.float().double().numpy()
    else:
        weight = torch.randint(-128, 128, (out, width), generator=g, dtype=torch.int8)
        w = weight.double().numpy()
    shape = (out // row_block, width // group) if group else (out,)
    scale = torch.rand(shape, generator=g) * 0.01 + 0.001
    s = scale.double().numpy()
    s = np.repeat(np.repeat(s, row_block, 0), group, 1) if group else s[:, None]
    x = _x(rows, width, dtype)
    got = kernels.w8a16(x.to(DEV), weight.to(DEV), scale.to(DEV), fp8, group, row_block)
    carried = np.abs(w) + (256.0 if not fp8 and dtype == BF16 else 0.0)
    _check(got, x, w * s, carried * s)


@pytest.mark.parametrize(("rows", "out", "width", "block", "dtype"), [
    (3, 40, 8256, 64, BF16),  # In ends inside a step
    (5, 300, 1088, 64, F16),
    (9, 2050, 4096, 32, BF16),
    (17, 130, 1024, 128, F16),
    (24, 72, 14336, 64, BF16),
    (96, 1000, 1536, 512, BF16),
    (9, 40, 8256, 64, BF16),  # In ends inside a step, long
])
def test_nf4(rows: int, out: int, width: int, block: int, dtype: torch.dtype) -> None:
    print(f"nf4 stream rows={rows} out={out} in={width} block={block} {dtype}", flush=True)
    rng = np.random.default_rng(out + width)
    codes = rng.integers(0, 256, (out, width // 2)).astype(np.uint8)
    absmax = (rng.random((out, width // block)) * 0.1 + 0.01).astype(np.float32)
    x = _x(rows, width, dtype)
    bias = _x(1, out, dtype)[0] if rows % 2 else None
    got = kernels.nf4_linear(x.to(DEV), torch.from_numpy(codes).to(DEV), torch.from_numpy(absmax).to(DEV), block,
                             None if bias is None else bias.to(DEV))
    # The codes' values as the kernel holds them, rounded to x's type.
    values = torch.from_numpy(quant.NF4_VALUES.copy()).to(dtype).double().numpy()
    w = values[np.stack([codes & 15, codes >> 4], axis=-1).reshape(out, width)] * np.repeat(absmax.astype(np.float64), block, 1)
    _check(got, x, w, np.abs(w), bias)


@pytest.mark.parametrize(("rows", "out", "width", "block", "dtype"), [
    (97, 7003, 1856, 64, BF16),  # 29 chunks of 64: the last step holds one; a partial column tile
    (130, 4097, 2048, 128, F16),  # odd rows of y, a block over two chunks
    (64, 14336, 512, 64, BF16),  # the tiles at 33..96 rows
    (257, 5000, 768, 256, BF16),
])
def test_nf4_tiles(rows: int, out: int, width: int, block: int, dtype: torch.dtype) -> None:
    print(f"nf4 tiles rows={rows} out={out} in={width} block={block} {dtype}", flush=True)
    rng = np.random.default_rng(rows)
    codes = rng.integers(0, 256, (out, width // 2)).astype(np.uint8)
    absmax = (rng.random((out, width // block)) * 0.1 + 0.01).astype(np.float32)
    x = _x(rows, width, dtype)
    bias = _x(1, out, dtype)[0] if rows % 2 else None
    strided = torch.zeros(rows, width + 8, dtype=dtype, device=DEV)
    strided[:, :width] = x.to(DEV)
    got = kernels.nf4_linear(strided[:, :width], torch.from_numpy(codes).to(DEV), torch.from_numpy(absmax).to(DEV), block,
                             None if bias is None else bias.to(DEV))
    values = torch.from_numpy(quant.NF4_VALUES.copy()).to(dtype).double().numpy()
    w = values[np.stack([codes & 15, codes >> 4], axis=-1).reshape(out, width)] * np.repeat(absmax.astype(np.float64), block, 1)
    _check(got, x, w, np.abs(w), bias)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize(("rows", "chosen", "count", "out", "width", "skew"), [
    (40, 4, 8, 1500, 2880, False),  # In ends inside a step; 20 pairs an expert on average
    (24, 2, 4, 3000, 1056, True),  # one expert takes most pairs (several passes), some are out of range
    (600, 4, 2, 70, 256, False),  # more pairs than a launch lists
    (16, 4, 16, 2048, 2048, False),  # 4 pairs an expert: 16 a pass
    (11, 4, 16, 2050, 2880, True),  # 8 a pass, several passes of one expert
])
def test_mxfp4_grouped(dtype: torch.dtype, rows: int, chosen: int, count: int, out: int, width: int, skew: bool) -> None:
    print(f"mxfp4 grouped rows={rows} chosen={chosen} E={count} out={out} in={width} {dtype}", flush=True)
    rng = np.random.default_rng(out + width)
    blocks = rng.integers(0, 256, (count, out, width // 32, 16)).astype(np.uint8)
    scales = rng.integers(118, 136, (count, out, width // 32)).astype(np.uint8)
    experts = rng.integers(0, count, (rows, chosen)).astype(np.int64)
    if skew:
        experts[rng.random((rows, chosen)) < 0.8] = 1
        experts[0, 0], experts[3, 1] = -1, count
    x = torch.randn(rows, width, generator=torch.Generator().manual_seed(rows)).to(dtype)
    xs = x.to(DEV)[:, None].expand(rows, chosen, width)
    args = [torch.from_numpy(t).to(DEV) for t in (blocks, scales, experts)]
    got = kernels.mxfp4_experts(xs, *args).cpu()
    for r, k in ((0, 0), (3, 1), (rows // 2, 0), (rows - 1, chosen - 1)):
        e = int(experts[r, k])
        if not 0 <= e < count:
            assert not got[r, k].any()
            continue
        w = quant.dequantize_mxfp4(blocks[e], scales[e]).astype(np.float64)
        _check(got[r, k][None], x[r][None], w, np.abs(w))
    # Every pair against the pair kernel's answer for its row alone (one row's pairs stay on it).
    for r in range(0, rows, max(1, rows // 12)):
        alone = kernels.mxfp4_experts(xs[r:r + 1], args[0], args[1], args[2][r:r + 1]).cpu()[0].double()
        top = alone.abs().amax().item()
        assert (got[r].double() - alone).abs().max().item() <= 2 * ULP[dtype] * top


@pytest.mark.parametrize(("rows", "out", "width", "group", "dtype"), [
    (65, 40, 128, 128, BF16),  # half of the only step, a partial tile, rows past the last
    (66, 130, 384, 64, F16),  # a step and a half, a second column tile of 2
    (129, 384, 1152, 32, BF16),  # two scales a chunk
    (128, 256, 1024, 128, F16),  # 8 groups at once
    (200, 700, 13 * 1024, 128, BF16),  # 52 steps: both scale sets on either side of the unrolled twelve
    (257, 129, 3328, 128, BF16),  # 13 steps, 26 groups: one a step
    (300, 514, 2048, 256, F16),
    (96, 2050, 768, 32, F16),
])
def test_int4_mid(rows: int, out: int, width: int, group: int, dtype: torch.dtype) -> None:
    """The automatic choice at 65 rows up to a tile a CU: products of x and the weight rounded
    to x's type, as the prefill kernels' -- that rounding is in the reference here."""
    print(f"int4 mid rows={rows} out={out} in={width} group={group} {dtype}", flush=True)
    rng = np.random.default_rng(rows + out)
    codes = rng.integers(0, 16, (out, width)).astype(np.uint8)
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4)).reshape(out, width // group, group // 2)
    scale = torch.from_numpy((rng.random((out, width // group)) * 0.02 + 0.001).astype(np.float32)).to(dtype)
    zero = rng.integers(0, 16, (out, width // group)).astype(np.uint8)
    wide = scale.double().numpy().repeat(group, 1) * (codes.astype(np.float64) - zero.repeat(group, 1))
    w = torch.from_numpy(wide).float().to(dtype).double().numpy()
    x = _x(rows, width, dtype)
    bias = _x(1, out, dtype)[0] if rows % 2 else None
    args = [t.to(DEV) for t in (x, torch.from_numpy(packed), scale, torch.from_numpy(zero))]
    bias_d = None if bias is None else bias.to(DEV)
    got = kernels.int4_linear(*args, bias_d)
    _check(got, x, w, np.abs(w), bias)
    _check(kernels.int4_linear(*args, bias_d, kernel="tiled128"), x, w, np.abs(w), bias)


def test_replayed_from_a_graph() -> None:
    """A captured call of each format replays to the eager bits with work between."""
    x = _x(12, 1024, BF16).to(DEV)
    g = torch.Generator().manual_seed(0)
    w8 = torch.randint(-128, 128, (512, 1024), generator=g, dtype=torch.int8).to(DEV)
    s8 = (torch.rand(512, 8, generator=g) * 0.01).to(DEV)
    codes = torch.randint(0, 256, (512, 512), generator=g, dtype=torch.uint8).to(DEV)
    absmax = torch.rand(512, 16, generator=g).to(DEV)
    packed = codes.view(512, 16, 32)
    scale, zero = torch.rand(512, 16, generator=g).to(BF16).to(DEV), torch.randint(0, 16, (512, 16), generator=g, dtype=torch.uint8).to(DEV)
    calls = [lambda: kernels.w8a16(x, w8, s8, False, 128), lambda: kernels.nf4_linear(x, codes, absmax, 64),
             lambda: kernels.int4_linear(x, packed, scale, zero)]
    want = [c().clone() for c in calls]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = [c() for c in calls]
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        torch.randn(1 << 20, device=DEV).sum().item()
