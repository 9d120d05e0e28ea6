"""Which kernel a call takes, asked of the library without a GPU (256 compute units are
assumed there): the lines between kernels at shapes on both sides of them."""

from __future__ import annotations

import ctypes

import pytest

from linnet_amd import _lib

GEMV, STREAM, TILES = 1, 2, 3


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
