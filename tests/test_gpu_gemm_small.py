"""GPU parity of the blockwise-scaled GEMM on the tiles below 256x256, one
shape per tile of the dispatch rule, with ragged last tiles and K ranges that
leave waves without a block.

fp32 output against a float64 product of the operands' q * s values.  Int
grid: a K block's sum is an exact int32, so only the promotion rounds, once
per block and once for its two scales' product: at most (blocks + 2) * 2^-23 of
the sum of the terms' magnitudes.  e4m3: v_mfma_f32_16x16x128_f8f6f4 aligns its
128 products to the largest and drops low bits (1.7e-5 of the norm on the
256x256 tiles at N(0,1) data with outliers), so the path's bar of 1e-3 is held;
a dropped or doubled K block of the 4 to 12 here is above 0.2.
"""

from __future__ import annotations

import pytest
import torch

from _gpu_util import seeded

pytestmark = pytest.mark.gpu

# M, N, K: 16x16 one wave (4 K blocks at most), 16x16, 16x32, 32x32, 32x64,
# 64x64 with four and with two waves, 128x128, and few rows by many columns
SHAPES = [(37, 300, 500), (3, 129, 1500), (18, 4000, 640), (70, 2900, 1152), (120, 4001, 700), (250, 4090, 1300),
          (500, 4000, 770), (1100, 2000, 1200), (9, 17000, 640), (60, 18432, 640)]


def _value(q):
    """the float64 values q * s of a QTensor"""
    from lowbit import ops

    codes = q.codes[:, :q.K]
    v = codes.view(torch.float8_e4m3fn).double() if q.grid == ops.grid_code("e4m3") else codes.view(torch.int8).double()
    r = torch.arange(q.rows, device=codes.device)[:, None] >> q.shift
    kb = torch.arange(q.K, device=codes.device)[None, :] >> 7
    return v * q.scales.flatten()[r * q.s_row + kb * q.s_col].double()


@pytest.mark.parametrize("fmt", ["e4m3", "int_grid"])
@pytest.mark.parametrize("blocks", [True, False])
@pytest.mark.parametrize("mnk", SHAPES)
def test_small_tiles_match_float64(gpu_device, mnk, blocks, fmt):
    from lowbit import ops

    M, N, K = mnk
    x = seeded((M, K), seed=20262001 + M, outliers=0.01).to(gpu_device)
    w = seeded((N, K), seed=20262002 + N, std=0.02).to(gpu_device)
    b = seeded((N,), seed=20262003, dtype=torch.float32).to(gpu_device)
    qx = ops.quant_tile_1x128(x, fmt=fmt, want_nan_rows=True)
    # one B scale per 128x128 block, or one per row and K block
    qw = ops.quant_block_128x128(w, fmt=fmt, want_nan_rows=True)[0] if blocks else \
        ops.quant_tile_1x128(w, fmt=fmt, want_nan_rows=True)
    ref = _value(qx) @ _value(qw).T
    y = ops.gemm_blockscaled(qx, qw, out_dtype=torch.float32).double()
    if fmt == "e4m3":
        assert float((y - ref).norm() / ref.norm()) <= 1e-3
    else:
        mag = _value(qx).abs() @ _value(qw).abs().T
        assert float(((y - ref).abs() / mag).max()) <= (-(-K // 128) + 2) * 2.0 ** -23
    # bias, NaN rows and columns, bf16 output; and the same bits on a second call
    yb = ops.gemm_blockscaled(qx, qw, bias=b)
    assert torch.equal(yb, (y.float() + b).to(torch.bfloat16))
    assert torch.equal(yb, ops.gemm_blockscaled(qx, qw, bias=b))
    qx.nan_rows[M - 1] = 1
    qw.nan_rows[N - 1] = 1
    yn = ops.gemm_blockscaled(qx, qw, bias=b)
    nan = torch.isnan(yn)
    assert nan[M - 1].all() and nan[:, N - 1].all() and int(nan.sum()) == M + N - 1
    assert torch.equal(yn[:M - 1, :N - 1], yb[:M - 1, :N - 1])
