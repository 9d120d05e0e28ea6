"""Which kernel a call takes, asked of the library without a GPU (256 compute units are
assumed there): the lines between kernels at shapes on both sides of them."""

from __future__ import annotations

import ctypes

import pytest

from linnet_amd import _lib

WIDENED, GEMV, STREAM, TILES = _lib.NF4_WIDENED, _lib.NF4_GEMV, _lib.NF4_STREAM, _lib.NF4_TILES


def _nf4(rows: int, out: int, width: int, block: int = 64, stride: int | None = None) -> int:
    chosen = ctypes.c_int32(-1)
    _lib.call("lnq_nf4_linear_plan", rows, width if stride is None else stride, out, width, block, ctypes.byref(chosen))
    return chosen.value


@pytest.mark.parametrize(("out", "width"), [(28672, 4096), (32768, 4096), (28672, 8192), (28672, 14336), (28160, 4096)])
@pytest.mark.parametrize("block", [64, 128])
def test_nf4_few_rows_over_wide_outputs_take_no_tiles(out: int, width: int, block: int) -> None:
    """A 64-row tile is mostly empty there: 4096 -> 28672 at one row 30 us, 18 on the GEMV."""
    for rows in (1, 2):
        assert _nf4(rows, out, width, block) == GEMV
    for rows in (5, 8, 16):
        assert _nf4(rows, out, width, block) == STREAM
    assert _nf4(64, out, width, block) == TILES


@pytest.mark.parametrize(("rows", "out", "width", "block", "want"), [
    (17, 4096, 4096, 64, STREAM), (64, 14336, 4096, 64, TILES), (96, 4096, 14336, 64, STREAM),
    (128, 14336, 4096, 64, TILES), (97, 4096, 14336, 64, STREAM),  # 67 us streamed, 88 in tiles, 75 widened
    (97, 2048, 14336, 64, WIDENED),  # 63 us streamed, 48 widened
    (96, 9216, 3072, 32, WIDENED),  # blocks of 32 have no tiles: 47 us streamed, 39 widened
    (64, 9216, 3072, 32, STREAM), (96, 18944, 3584, 64, WIDENED), (96, 14336, 4096, 32, STREAM), (200, 14336, 4096, 64, WIDENED),  # two tiles a unit
    (17, 64, 65536, 64, WIDENED), (17, 1 << 20, 8192, 64, WIDENED),  # lnq_nf4_linear refuses
    (16, 64, 1024, 16, GEMV), (17, 64, 1024, 16, WIDENED),  # blocks that only the GEMV takes
    (9, 64, 16384, 16, WIDENED)])
def test_nf4_reads_the_stored_weight_where_it_is_faster(rows: int, out: int, width: int, block: int, want: int) -> None:
    assert _nf4(rows, out, width, block) == want


def test_nf4_rows_far_apart_are_widened() -> None:
    """Past the streaming kernel's and the tiles' strides the stored weight would be read
    again for every 8 rows, or the call refused."""
    for stride in (1 << 23, 1 << 28):
        assert _nf4(16, 4096, 4096, 64, stride) == GEMV
        for rows in (17, 64, 128):
            assert _nf4(rows, 4096, 4096, 64, stride) == WIDENED


@pytest.mark.parametrize(("rows", "out", "width", "want"), [
    (5, 1024, 4096, GEMV), (8, 1024, 8192, GEMV), (9, 1024, 4096, STREAM), (5, 1025, 4096, STREAM), (5, 1024, 2048, STREAM),
    (3, 2048, 8192, GEMV), (4, 2049, 8192, STREAM), (3, 1536, 6144, STREAM), (8, 1024, 6144, GEMV),
    (3, 2048, 14336, GEMV), (4, 2049, 14336, STREAM), (5, 512, 14336, STREAM), (3, 1024, 11008, GEMV),
    (3, 1152, 11008, STREAM), (4, 14336, 4096, GEMV), (3, 4096, 14336, STREAM)])
def test_nf4_narrow_outputs_keep_the_gemv(rows: int, out: int, width: int, want: int) -> None:
    """One GEMV pass of at most a workgroup a unit: 4096 -> 1024 at 5 rows 5.0 us, streamed 5.9."""
    assert _nf4(rows, out, width) == want


def test_nf4_outputs_past_the_streaming_grid() -> None:
    """The grid's y holds 65535 steps of eight blocks."""
    assert _nf4(16, 65535 * 64, 64) == STREAM
    assert _nf4(16, 65535 * 64 + 1, 64) == GEMV
    assert _nf4(17, 65535 * 64 + 1, 64) == WIDENED


@pytest.mark.parametrize(("rows", "out", "width", "group", "row_block", "want"), [
    (1, 4096, 4096, 0, 1, _lib.W8_ROW), (1, 4096, 4096, 64, 1, _lib.W8_STREAM), (1, 4112, 4096, 128, 128, None),
    (1, 6144, 4096, 0, 1, _lib.W8_STREAM), (32, 2048, 2048, 0, 1, _lib.W8_STREAM), (33, 4096, 1024, 0, 1, _lib.W8_SKINNY),
    (64, 4096, 4096, 128, 128, _lib.W8_STREAM), (128, 2048, 2048, 128, 1, _lib.W8_SKINNY),
    (512, 14336, 4096, 0, 1, _lib.W8_STREAM), (512, 1024, 14336, 64, 1, _lib.W8_SKINNY),
    (1, 64, 65536, 0, 1, _lib.W8_STREAM), (1, 64, 65664, 0, 1, _lib.W8_SKINNY),
    (1, 65535 * 64 + 1, 128, 0, 1, _lib.W8_SKINNY)])
def test_eight_bit_kernels(rows: int, out: int, width: int, group: int, row_block: int, want: int | None) -> None:
    """`want` None: scale blocks that do not tile the weight are refused."""
    chosen = ctypes.c_int32(-1)
    args = ("lnq_w8a16_plan", rows, out, width, group, row_block, ctypes.byref(chosen))
    if want is None:
        with pytest.raises(_lib.LinnetError):
            _lib.call(*args)
        return
    _lib.call(*args)
    assert chosen.value == want


@pytest.mark.parametrize(("rows", "chosen", "experts", "out", "width", "want"), [
    (1, 4, 32, 5760, 2880, 0), (4, 4, 32, 5760, 2880, 0),  # 32 us a pass a pair, 39 grouped
    (16, 1, 32, 5760, 2880, 0), (12, 1, 32, 5760, 2880, 0), (64, 1, 128, 1536, 4096, 0),  # 40 and 60
    (16, 4, 128, 1536, 4096, 0), (8, 2, 8, 1536, 4096, 0), (8, 8, 128, 1024, 1024, 0), (4, 8, 128, 2880, 2880, 0),
    (12, 4, 32, 5760, 2880, 8), (32, 4, 32, 5760, 2880, 16), (256, 4, 32, 5760, 2880, 32), (64, 1, 32, 5760, 2880, 8),
    (64, 2, 8, 1501, 1056, 32), (64, 4, 128, 1536, 4096, 8), (1024, 1, 4, 1024, 1024, 32)])
def test_mxfp4_pairs_a_pass(rows: int, chosen: int, experts: int, out: int, width: int, want: int) -> None:
    got = ctypes.c_int32(-1)
    _lib.call("lnq_mxfp4_experts_plan", rows, chosen, experts, out, width, ctypes.byref(got))
    assert got.value == want


@pytest.mark.parametrize(("rows", "out", "width", "block", "want"), [
    (48, 14336, 4096, 0, 64), (16, 14336, 4096, 0, 32), (128, 14336, 4096, 0, 64), (256, 4096, 14336, 0, 64), (512, 4096, 14336, 0, 128),
    (160, 12288, 6144, 0, 128),  # 45 us in 256 rows, 54 in 32, 37 in 128
    (1500, 12288, 6144, 0, 256), (777, 14336, 4096, 1, 256), (300, 28672, 8192, 1, 256),  # 115 us, 154 in 64
    (128, 25600, 5120, 1, 128), (64, 28672, 4096, 0, 64), (128, 18944, 3584, 0, 128),
    (257, 28672, 4096, 1, 256), (257, 12288, 6144, 1, 256), (640, 14336, 4096, 1, 256), (33, 2048, 2048, 1, 32)])
def test_eight_bit_tile_rows(rows: int, out: int, width: int, block: int, want: int) -> None:
    got = ctypes.c_int32(-1)
    _lib.call("lnq_mm8_rows_plan", rows, out, width, 1, block, ctypes.byref(got))
    assert got.value == want
