"""The layer's backward in one native call (GPU): any subset of the gradients
is bitwise that of the full backward, and the full one bitwise that of the
separate projections and mixer, over masks, biases, sizes that the weight
transpose's 32 x 32 tiles do not divide, strided and FP32 upstream gradients."""

from __future__ import annotations

import pytest
import torch

from lsso_amd import LSSO, LSSOConfig

NAMES = ("x", "w_bc.weight", "w_bc.bias", "core_base_raw", "core_drive_weight", "eta_raw", "w_o.weight", "w_o.bias")


def _layer(dim, heads, rank, bias):
    torch.manual_seed(dim + rank)
    layer = LSSO(LSSOConfig(dim=dim, num_heads=heads, rank=rank, bias=bias)).cuda()
    with torch.no_grad():
        layer.core_base_raw.normal_(std=0.05)
        layer.core_drive_weight.normal_(std=0.05)
    return layer


def _separate(native, layer, x, mask, positions, dy):
    centered, counts, mask = layer._native_geometry(x, mask, positions)
    packed = native.linear(x, layer.w_bc.weight, layer.w_bc.bias, torch.bfloat16, row_mask=mask)
    mixed = native.fast_mix(packed, layer.core_base_raw, layer.core_drive_weight, layer.eta_raw, centered, counts)
    return native.linear(mixed, layer.w_o.weight, layer.w_o.bias, x.dtype, row_mask=mask)


@pytest.mark.gpu
@pytest.mark.parametrize(("dim", "heads", "rank", "bias", "masked", "length", "dtype"), (
    (48, 3, 16, True, False, 77, torch.float16),
    (256, 8, 32, True, True, 600, torch.bfloat16),
    (256, 8, 48, False, False, 1100, torch.float16),
    (128, 2, 64, True, True, 130, torch.float16),
))
def test_gradient_subsets_and_separate_calls(native, dim, heads, rank, bias, masked, length, dtype) -> None:
    layer = _layer(dim, heads, rank, bias)
    x = torch.randn(3, length, dim, device="cuda", dtype=dtype).requires_grad_()
    mask = None
    if masked:
        mask = torch.arange(length, device="cuda")[None, :] < torch.tensor([[length], [length // 2], [1]], device="cuda")
    dy = torch.randn(3, length, dim, device="cuda", dtype=dtype)
    tensors = {"x": x, **dict(layer.named_parameters())}
    names = [name for name in NAMES if name in tensors]

    def gradients(wanted, upstream=dy):
        for name, tensor in tensors.items():
            tensor.requires_grad_(name in wanted)
        y = layer(x, valid_mask=mask, implementation="hip")
        return torch.autograd.grad(y, [tensors[name] for name in wanted], upstream)

    full = dict(zip(names, gradients(names)))
    for tensor in tensors.values():
        tensor.requires_grad_(True)
    separate = torch.autograd.grad(_separate(native, layer, x, mask, None, dy), [tensors[n] for n in names], dy)
    for name, grad in zip(names, separate):
        if name == "w_bc.bias" and not masked:
            # One call sums the bias inside the token map, the separate calls in the weight gradient.
            assert float((full[name] - grad).norm() / grad.norm()) <= 1e-5
        else:
            assert torch.equal(full[name], grad), name
    subsets = [[name] for name in names] + [["w_o.weight", "w_o.bias"], ["x", "eta_raw"], ["w_bc.weight", "w_bc.bias"]]
    for wanted in subsets:
        wanted = [name for name in wanted if name in tensors]
        for name, grad in zip(wanted, gradients(wanted)):
            if name.endswith("bias") and len(wanted) == 1:
                # Without its weight, a bias gradient is one column pass instead.
                assert float((full[name] - grad).norm() / grad.norm()) <= 1e-5
            else:
                assert torch.equal(full[name], grad), (name, wanted)
    # A broadcast upstream gradient stands for the dense one.
    row = torch.randn(dim, device="cuda", dtype=dtype)
    for a, b in zip(gradients(names, row.expand(3, length, dim)), gradients(names, row.expand(3, length, dim).contiguous())):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_layers_with_more_parameters_are_checked_in_full(native) -> None:
    layer = _layer(64, 2, 16, True)
    x = torch.randn(1, 40, 64, device="cuda", dtype=torch.float16)
    expected = layer(x, implementation="hip")
    layer.register_parameter("extra", torch.nn.Parameter(torch.zeros(1)))
    with pytest.raises(RuntimeError, match="requires extra on"):
        layer(x, implementation="hip")
    layer.extra.data = layer.extra.data.cuda()
    assert torch.equal(layer(x, implementation="hip"), expected)
    layer.w_o.bias.data = layer.w_o.bias.data.cpu()
    with pytest.raises(RuntimeError, match="requires w_o.bias on"):
        layer(x, implementation="hip")


@pytest.mark.gpu
def test_saved_tensor_hooks(native) -> None:
    """Saved tensors that hooks hand back are read as they are: offloaded and
    strided copies give the same gradients, tensors of another type, size or
    device are refused before any kernel runs."""

    layer = _layer(64, 2, 16, True)
    x = torch.randn(2, 70, 64, device="cuda", dtype=torch.float16).requires_grad_()
    mask = torch.arange(70, device="cuda")[None, :] < torch.tensor([[70], [31]], device="cuda")
    dy = torch.randn_like(x)
    wanted = [x, *layer.parameters()]

    def gradients(pack, unpack):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = layer(x, valid_mask=mask, implementation="hip")
        return torch.autograd.grad(y, wanted, dy)

    expected = gradients(lambda t: t, lambda t: t)

    def strided(t):
        keeps = t.dim() == 1 or t.shape[-1] == 2 * 16 + 64 or t.shape[-1] == 16   # packed, tape and compact parameters
        return t if keeps else t.transpose(-1, -2).contiguous().transpose(-1, -2)

    for pack, unpack in ((lambda t: t.cpu(), lambda t: t.cuda()), (lambda t: t, strided)):
        for a, b in zip(gradients(pack, unpack), expected):
            assert torch.equal(a, b)
    # packed: another type, fewer rows, the host; tape: cut short; W_o: another type; x: another type.
    packed = lambda t: t.dim() == 3 and t.shape[-1] == 2 * 16 + 64
    tape = lambda t: t.dim() == 1 and t.numel() > 2
    changes = (
        (packed, lambda t: t.float()), (packed, lambda t: t[:1]), (packed, lambda t: t.cpu()), (tape, lambda t: t[:-1]),
        (lambda t: tuple(t.shape) == (64, 64), lambda t: t.bfloat16()),
        (lambda t: t.dtype == torch.float16, lambda t: t.float()),
    )
    for match, change in changes:
        with pytest.raises((RuntimeError, TypeError)):
            gradients(lambda t: t, lambda t, m=match, c=change: c(t) if m(t) else t)


def test_saved_extents_are_checked() -> None:
    from lsso_amd.ball import hip

    value = torch.zeros(2, 3)
    assert hip._saved(value, "tape", torch.float32, (2, 3), value.device) is value
    for dtype, sizes, device in ((torch.float16, (2, 3), "cpu"), (torch.float32, (2, 4), "cpu"),
                                 (torch.float32, (2, 3), "meta")):
        with pytest.raises(RuntimeError, match="saved tape"):
            hip._saved(value, "tape", dtype, sizes, torch.device(device))


def test_layer_backward_rejects_bad_arguments() -> None:
    """Host-side validation of the C entry (no launch, no GPU)."""

    import ctypes

    from lsso_amd.ball import hip

    path = hip.default_library_path()
    if not path.is_file():
        import __graft_entry__

        __graft_entry__.build()
    library = hip.open_library(path)
    shape = hip.MixerShape(2, 64, 2, 16, 32)
    size = ctypes.c_size_t()
    assert library.lsso_hip_layer_backward_workspace_bytes(ctypes.byref(shape), 0, ctypes.byref(size)) == 0
    assert library.lsso_hip_layer_backward_workspace_bytes(ctypes.byref(shape), 0, None) == -1
    need = size.value

    def call(grad_y=256, dtype=1, workspace=256, size=need):
        return library.lsso_hip_layer_backward(
            ctypes.byref(shape), grad_y, dtype, 64, 256, 1, 256, None, 256, 256, 256, 256, 256, None, None, 0, None, 256,
            256, None, None, None, None, None, None, None, None, workspace, size, None,
        )

    assert call(grad_y=None) == -1
    assert call(dtype=7) == -2
    assert call(workspace=None) == -1
    assert call(size=need - 1) == -1
