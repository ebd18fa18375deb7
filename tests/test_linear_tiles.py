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
