"""Token chunks evened over a sequence and head groups spread over idle CUs
(GPU): lengths around the chunk limits (512 tokens, 1,024 from 4,096 on) and
batches that leave the staged reductions few workgroups, forward and backward
against the FP64 oracle within the module's bars, and a sample's output and
input gradient bitwise the same alone and in a batch (its chunks depend on the
length alone, and the grouping of heads changes no chain)."""

from __future__ import annotations

import pytest
import torch

from lsso_amd import LSSO, LSSOConfig
from oracle import lsso_reference as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("dim", "heads", "rank"), ((128, 4, 32), (256, 4, 48), (384, 6, 64), (384, 12, 48)))
@pytest.mark.parametrize("length", (511, 513, 575, 1025, 1537, 4095, 4097))
def test_lengths_around_the_chunk_limits(native, dim, heads, rank, length) -> None:
    torch.manual_seed(length + rank)
    layer = LSSO(LSSOConfig(dim=dim, num_heads=heads, rank=rank, bias=True)).cuda()
    with torch.no_grad():
        layer.core_base_raw.normal_(std=0.05)
        layer.core_drive_weight.normal_(std=0.05)
    x = torch.randn(3, length, dim, device="cuda", dtype=torch.float16).requires_grad_()
    dy = torch.randn(3, length, dim, device="cuda", dtype=torch.float16)
    y = layer(x, implementation="hip")
    (gx,) = torch.autograd.grad(y, x, dy)
    alone = x.detach()[1:2].clone().requires_grad_()
    y_alone = layer(alone, implementation="hip")
    (gx_alone,) = torch.autograd.grad(y_alone, alone, dy[1:2])
    assert torch.equal(y_alone[0], y[1]) and torch.equal(gx_alone[0], gx[1])
    if length in (513, 1025, 4097):
        params = {name: p.detach().double().cpu() for name, p in layer.named_parameters()}
        leaf = x.detach()[1:2].double().cpu().requires_grad_()
        expected = oracle.lsso_forward(params, {"dim": dim, "num_heads": heads, "rank": rank, "bias": True}, leaf)
        expected.backward(dy[1:2].double().cpu())
        error = (y[1:2].detach().double().cpu() - expected.detach()).norm() / expected.norm()
        grad_error = (gx[1:2].double().cpu() - leaf.grad).norm() / leaf.grad.norm()
        assert error <= 5e-3 and grad_error <= 3e-2
