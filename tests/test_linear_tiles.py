"""The projection kernels at the edges of their tiles (GPU): every K tier with
one to several row tiles per workgroup, ragged rows, strided x, masked rows
holding NaN, outputs that are not whole 16-byte pieces, against FP64 of the
same BF16 operands.

Bound: K products (exact in FP32) and the bias added in FP32, at most
2^-24 sqrt(K) relative L2 for independent terms, then one rounding to the
output type (2^-9 for BF16, 2^-12 for FP16, at most)."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


@pytest.mark.parametrize("features", ((64, 64), (100, 52), (128, 264), (192, 448), (256, 640), (384, 90), (392, 256),
                                      (512, 256), (520, 72), (640, 264), (648, 128), (768, 1344), (1344, 136), (770, 50)))
@pytest.mark.parametrize(("rows", "pad", "masked"), ((1, 0, False), (65, 8, True), (700, 0, True), (40001, 0, False),
                                                     (9000, 5, True)))
def test_linear_tiles_match_fp64(native, features, rows, pad, masked) -> None:
    in_features, out_features = features
    generator = torch.Generator(device="cuda").manual_seed(rows + in_features)
    x_dtype, y_dtype = ((torch.float16, torch.bfloat16), (torch.bfloat16, torch.float16))[rows % 2]
    x = torch.randn(rows, in_features + pad, device="cuda", generator=generator).to(x_dtype)[:, :in_features]
    weight = torch.randn(out_features, in_features, device="cuda", generator=generator) / math.sqrt(in_features)
    bias = torch.randn(out_features, device="cuda", generator=generator) if rows != 700 else None
    mask = None
    if masked:
        mask = torch.rand(rows, device="cuda", generator=generator) > 0.3
        x[~mask] = float("nan")
    y = native.linear(x, weight, bias, y_dtype, row_mask=mask)
    expected = x.bfloat16().double() @ weight.bfloat16().double().t()
    if bias is not None:
        expected = expected + bias.double()
    if masked:
        assert torch.count_nonzero(y[~mask]) == 0
        expected = torch.where(mask[:, None], expected, 0)
    error = float((y.double() - expected).norm() / expected.norm().clamp_min(1e-30))
    assert error <= HALF_ULP[y_dtype] + 2.0 ** -24 * math.sqrt(in_features)
    # A row's result does not depend on which tile or workgroup holds it.
    start = min(33, rows - 1)
    again = native.linear(x[start:], weight, bias, y_dtype, row_mask=None if mask is None else mask[start:])
    assert torch.equal(again, y[start:])


@pytest.mark.parametrize("in_features", (1, 3, 7, 8, 9, 15, 60, 100, 130, 250, 257, 300, 380, 391, 510, 636, 641, 700, 1001))
@pytest.mark.parametrize(("rows", "out_features", "pad", "offset"), ((1, 1, 0, 0), (63, 7, 1, 0), (130, 9, 3, 1), (2049, 257, 0, 3),
                                                                     (20000, 321, 2, 1), (77, 264, 8, 1), (300, 100, 0, 0)))
def test_pieces_aligned_to_their_elements_match_whole_pieces(native, in_features, rows, out_features, pad, offset) -> None:
    """Rows, strides, bases and outputs that are not whole 16-byte pieces give
    the bits of the same operands padded with zeros to whole pieces.  What lies
    between the rows and around the operands is NaN and must not be read into
    the result."""

    generator = torch.Generator(device="cuda").manual_seed(rows + in_features)
    x_dtype, y_dtype = ((torch.float16, torch.bfloat16), (torch.bfloat16, torch.float16))[rows % 2]
    stride = in_features + pad
    values = torch.randn(rows, in_features, device="cuda", generator=generator).to(x_dtype)
    storage = torch.full((offset + rows * stride + 16,), float("nan"), device="cuda", dtype=x_dtype)
    x = storage[offset:offset + rows * stride].view(rows, stride)[:, :in_features]
    x.copy_(values)
    weights = torch.randn(out_features, in_features, device="cuda", generator=generator) / math.sqrt(in_features)
    weight_storage = torch.full((offset + weights.numel() + 8,), float("nan"), device="cuda")
    weight = weight_storage[offset:offset + weights.numel()].view(out_features, in_features)
    weight.copy_(weights)
    bias = torch.randn(out_features, device="cuda", generator=generator)
    mask = torch.rand(rows, device="cuda", generator=generator) > 0.3 if rows % 3 == 0 else None

    def whole(value: torch.Tensor, *sizes: int) -> torch.Tensor:
        padded = torch.zeros(*(-(-size // 8) * 8 for size in sizes), device="cuda", dtype=value.dtype)
        padded[tuple(slice(size) for size in sizes)] = value
        return padded

    expected = native.linear(whole(values, rows, in_features)[:rows], whole(weights, out_features, in_features),
                             whole(bias, out_features), y_dtype, row_mask=mask)
    y = native.linear(x, weight, bias, y_dtype, row_mask=mask)
    assert torch.equal(y, expected[:, :out_features])


@pytest.mark.parametrize(("rows", "in_features", "out_features", "stride"), (
    (70, 64, 72, (1 << 23) + 8),            # a tile's rows past 32-bit offsets, resident weights
    (130, 648, 136, (1 << 23) + 8),         # the same, K-streaming
    (9, (1 << 22) + 8, 8, (1 << 22) + 8),   # weight rows past them
))
def test_strides_past_32_bit_tile_offsets(native, rows, in_features, out_features, stride) -> None:
    generator = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.empty(rows, stride, device="cuda", dtype=torch.bfloat16)[:, :in_features]
    x.copy_(torch.randn(rows, in_features, device="cuda", generator=generator))
    weight = torch.randn(out_features, in_features, device="cuda", generator=generator) / math.sqrt(in_features)
    y = native.linear(x, weight, None, torch.bfloat16)
    expected = x.double() @ weight.bfloat16().double().t().contiguous()
    error = float((y.double() - expected).norm() / expected.norm())
    assert error <= HALF_ULP[torch.bfloat16] + 2.0 ** -24 * math.sqrt(in_features)
