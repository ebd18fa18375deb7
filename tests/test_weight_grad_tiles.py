"""The weight-gradient kernel at the edges of its tiles and plans (GPU): both
output tiles (256 x 256 for long products that fill such tiles, else 128 x 128),
column remainders, a last stage of one row, rows that are not whole 16-byte
pieces or hold none, splits that are not dealt to the XCDs, masks and the
variants without bias sums, against FP64 of the same BF16 operands.

Bound: an output is a chain of at most `rows` FP32 additions of products that
are exact in FP32; for independent zero-mean terms the rounding errors add like
a random walk, so the relative L2 error is at most about 2^-24 sqrt(rows)."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    ("rows", "in_features", "out_features", "g_dtype", "x_dtype", "masked", "pad", "bias"),
    [
        (65537, 264, 520, torch.bfloat16, torch.float16, False, 0, True),     # remainders, odd last stage
        (65537, 264, 520, torch.float16, torch.bfloat16, True, 8, False),
        (131072, 256, 264, torch.float16, torch.float16, True, 0, True),
        (33, 128, 128, torch.bfloat16, torch.bfloat16, False, 0, True),       # one whole small tile, a row past a stage
        (1, 136, 120, torch.float16, torch.bfloat16, False, 0, False),
        (2000, 768, 1344, torch.bfloat16, torch.bfloat16, True, 0, True),     # more tiles than an XCD's workgroups
        (517, 131, 257, torch.bfloat16, torch.float16, False, 0, True),       # pieces aligned to their elements
        (4100, 72, 56, torch.float16, torch.float16, True, 3, False),         # a row stride that is not whole pieces
        (40001, 440, 760, torch.bfloat16, torch.float16, False, 0, True),     # large tile, remainders, odd last stage
        (40001, 440, 760, torch.float16, torch.bfloat16, True, 8, False),
        (40001, 441, 759, torch.float16, torch.bfloat16, True, 0, True),      # large tile, pieces aligned to their elements
        (4700, 1536, 1800, torch.bfloat16, torch.bfloat16, True, 0, True),    # more large tiles than an XCD's workgroups
        (4700, 1537, 1801, torch.bfloat16, torch.float16, False, 1, False),
        (65537, 263, 521, torch.bfloat16, torch.float16, True, 0, True),
        (4100, 5, 300, torch.float16, torch.bfloat16, True, 0, True),         # element loads: rows without a whole piece
        (1000, 300, 7, torch.bfloat16, torch.float16, False, 2, False),
        (65, 1, 1, torch.bfloat16, torch.bfloat16, False, 1, True),
    ],
)
def test_weight_gradient_tiles_match_fp64(
    native, rows, in_features, out_features, g_dtype, x_dtype, masked, pad, bias
) -> None:
    generator = torch.Generator(device="cuda").manual_seed(rows + in_features)

    def matrix(cols, dtype):
        storage = torch.randn(rows, cols + pad, device="cuda", generator=generator)
        return storage.to(dtype)[:, :cols]

    g, x = matrix(out_features, g_dtype), matrix(in_features, x_dtype)
    mask = None
    if masked:
        mask = torch.rand(rows, device="cuda", generator=generator) > 0.3
        g[~mask] = float("nan")
        x[~mask] = float("inf")
    grad_weight, grad_bias = native._weight_gradient(g, x, mask, bias)
    if masked:
        g, x = torch.where(mask[:, None], g, 0), torch.where(mask[:, None], x, 0)
    expected = g.bfloat16().double().t().contiguous() @ x.bfloat16().double()
    limit = 2.0 ** -24 * max(2.0, math.sqrt(rows))
    assert float((grad_weight.double() - expected).norm() / expected.norm()) <= limit
    again, _ = native._weight_gradient(g, x, None, bias)
    assert torch.equal(again, grad_weight)              # zeros in place of the excluded rows: the same sums
    if bias:
        scale = g.double().abs().sum(0)
        assert torch.all((grad_bias.double() - g.double().sum(0)).abs() <= limit * scale)
    else:
        assert grad_bias is None


@pytest.mark.parametrize(("rows", "in_features", "out_features"), ((1, 8, 9), (31, 9, 15), (65, 131, 8), (4097, 250, 130),
                                                                  (40001, 437, 763)))
@pytest.mark.parametrize(("pad", "offset", "masked"), ((0, 1, False), (1, 0, True), (3, 5, False)))
def test_pieces_aligned_to_their_elements_match_whole_pieces(
    native, rows, in_features, out_features, pad, offset, masked
) -> None:
    """Rows, strides and bases that are not whole 16-byte pieces give the sums
    of the same operands padded with zeros to whole pieces, each partial bit for
    bit; the partials' own sums may take another order (by the column count), so
    the two may differ by both sums' bounds.  What lies between the rows and
    around the operands is NaN and must not be read into the result."""

    generator = torch.Generator(device="cuda").manual_seed(rows + in_features + pad)

    def operand(cols, dtype):
        values = torch.randn(rows, cols, device="cuda", generator=generator).to(dtype)
        stride = cols + pad
        storage = torch.full((offset + rows * stride + 16,), float("nan"), device="cuda", dtype=dtype)
        odd = storage[offset:offset + rows * stride].view(rows, stride)[:, :cols]
        odd.copy_(values)
        whole = torch.zeros(rows, -(-cols // 8) * 8, device="cuda", dtype=dtype)
        whole[:, :cols] = values
        return odd, whole

    g, whole_g = operand(out_features, torch.bfloat16)
    x, whole_x = operand(in_features, torch.float16)
    mask = torch.rand(rows, device="cuda", generator=generator) > 0.3 if masked else None
    grad_weight, grad_bias = native._weight_gradient(g, x, mask, True)
    expected_weight, expected_bias = native._weight_gradient(whole_g, whole_x, mask, True)
    limit = 2.0 ** -23 * max(2.0, math.sqrt(rows))
    expected_weight = expected_weight[:out_features, :in_features].double()
    assert float((grad_weight.double() - expected_weight).norm() / expected_weight.norm()) <= limit
    scale = g.double().abs().sum(0)
    assert torch.all((grad_bias.double() - expected_bias[:out_features].double()).abs() <= limit * scale)


def test_strides_past_32_bit_stage_offsets(native) -> None:
    generator = torch.Generator(device="cuda").manual_seed(5)
    rows, stride = 70, (1 << 24) + 8
    x = torch.empty(rows, stride, device="cuda", dtype=torch.bfloat16)[:, :72]
    x.copy_(torch.randn(rows, 72, device="cuda", generator=generator))
    g = torch.randn(rows, 136, device="cuda", generator=generator).bfloat16()
    grad_weight, grad_bias = native._weight_gradient(g, x, None, True)
    expected = g.double().t().contiguous() @ x.double()
    limit = 2.0 ** -24 * math.sqrt(rows)
    assert float((grad_weight.double() - expected).norm() / expected.norm()) <= limit
    assert torch.all((grad_bias.double() - g.double().sum(0)).abs() <= limit * g.double().abs().sum(0))


@pytest.mark.parametrize(("splits", "cols"), ((1, 5), (2, 4), (7, 132), (64, 8), (600, 1024), (33, 1003)))
def test_column_sums_of_few_and_many_splits(native, splits, cols) -> None:
    """The split sums' lane plans (one lane per piece to 32, whole and odd
    pieces) through the one-pass column sums, whose splits follow the rows."""

    rows = splits * 16
    g = torch.randn(rows, cols, device="cuda").bfloat16()
    _, sums = native._grad_columns(g, None, False, True)
    scale = g.double().abs().sum(0)
    assert torch.all((sums.double() - g.double().sum(0)).abs() <= 2.0 ** -24 * math.sqrt(rows) * scale)
