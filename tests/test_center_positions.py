"""Centred positions and valid counts in one native launch (GPU) against the
oracle's FP64 evaluation of the same ids and masks (reference
lsso/ball/model.py:163-243).

Bound: a position is id - anchor (exact or rounded once to FP32), minus an
FP32 mean rounded once, rounded once: three FP32 roundings of values no
larger than the row's spread of valid ids."""

from __future__ import annotations

import pytest
import torch

from lsso_amd import LSSO, LSSOConfig
from oracle import lsso_reference as oracle


def _mask(batch: int, length: int) -> torch.Tensor:
    generator = torch.Generator().manual_seed(length)
    mask = torch.rand(batch, length, generator=generator) < 0.7
    mask[0] = True
    if batch > 1:
        mask[1] = False                       # a sample without a valid token
    if batch > 2:
        mask[2] = torch.arange(length) < (length + 1) // 2
    return mask


def _ids(kind: str, batch: int, length: int):
    generator = torch.Generator().manual_seed(7)
    starts = torch.randint(0, 1 << 20, (batch, 1), generator=generator)
    if kind == "none":
        return None
    if kind == "int64":                        # beyond FP32's integers
        return (1 << 40) + 3 * torch.arange(length)[None, :] + starts
    if kind == "int32":
        return (torch.arange(length)[None, :] + starts).to(torch.int32)
    if kind == "int64_shared":
        return torch.arange(length) * 2 + 5
    if kind == "float64":
        return 1e9 + 0.25 * torch.arange(length, dtype=torch.float64)[None, :] + starts
    if kind == "float32_shared":
        return torch.cat((torch.zeros(1), torch.arange(length - 1, dtype=torch.float32) - 0.5 * (length - 2)))
    if kind == "int64_expanded":               # one row read by every sample
        return (torch.arange(length) + 9)[None, :].expand(batch, length)
    assert kind == "int64_transposed"          # unit batch stride
    return (torch.arange(length)[None, :] + starts).t().contiguous().t()


@pytest.mark.gpu
@pytest.mark.parametrize("masked", (False, True))
@pytest.mark.parametrize("kind", ("none", "int64", "int32", "int64_shared", "float64", "float32_shared",
                                  "int64_expanded", "int64_transposed"))
@pytest.mark.parametrize(("batch", "length"), ((1, 1), (3, 63), (3, 1024), (4, 4097), (2, 65536)))
def test_center_positions_match_fp64(native, batch, length, kind, masked) -> None:
    ids = _ids(kind, batch, length)
    mask = _mask(batch, length) if masked else None
    if ids is None and mask is None:
        assert native.center_positions(None, None, batch, length, torch.device("cuda", 0)) is None
        return
    device_ids = None if ids is None else ids.cuda()
    if kind == "int64_expanded":
        device_ids = ids[0].cuda()[None, :].expand(batch, length)
    if kind == "int64_transposed":
        device_ids = ids.t().contiguous().cuda().t()
    centered, counts = native.center_positions(
        device_ids, None if mask is None else mask.cuda(), batch, length, torch.device("cuda", 0)
    )
    expected = oracle.center_positions(ids, mask, dtype=torch.float64, all_valid=not masked,
                                       batch=batch, length=length)
    shared = not masked and ids.dim() == 1
    assert tuple(centered.shape) == ((length,) if shared else (batch, length))
    spread = float(expected.abs().max()) * 2 + 1
    if shared:
        expected = expected[0]
    assert float((centered.cpu().double() - expected).abs().max()) <= 3 * 2.0 ** -24 * spread
    if masked:
        assert torch.equal(counts.cpu(), mask.sum(-1).clamp_min(1).float())
        assert torch.count_nonzero(centered.cpu()[~mask]) == 0
    else:
        assert counts is None


@pytest.mark.gpu
def test_module_geometry_routes(native) -> None:
    """Ids the kernel does not take keep the tensor path's results and errors."""

    layer = LSSO(LSSOConfig(dim=32, num_heads=2, rank=16)).cuda()
    x = torch.randn(2, 70000, 32, device="cuda", dtype=torch.float16)
    mask = torch.ones(2, 70000, dtype=torch.bool, device="cuda")
    mask[1, 100:] = False
    centered, counts, _ = layer._native_geometry(x, mask, None)      # longer than the kernel's rows
    assert counts.tolist() == [70000.0, 100.0]
    assert float(centered[1, 0]) == -49.5
    x = x[:, :50]
    ids16 = torch.arange(50, dtype=torch.int16, device="cuda")
    centered, counts, _ = layer._native_geometry(x, None, ids16)
    assert counts is None and torch.equal(centered, torch.arange(50.0, device="cuda") - 24.5)
    centered, _, _ = layer._native_geometry(x, None, torch.arange(50))  # ids on the host
    assert centered.device.type == "cuda" and torch.equal(centered.cpu(), torch.arange(50.0) - 24.5)
    for bad, error in ((ids16.half(), TypeError), (ids16.bool(), TypeError), (ids16[:-1].long(), ValueError),
                       (ids16[None].long(), ValueError)):
        with pytest.raises(error):
            layer._native_geometry(x, None, bad)


def test_center_positions_rejects_bad_arguments() -> None:
    """Host-side validation of the C entry (no launch, no GPU)."""

    from lsso_amd.ball import hip

    path = hip.default_library_path()
    if not path.is_file():
        import __graft_entry__

        __graft_entry__.build()
    library = hip.open_library(path)
    call = library.lsso_hip_center_positions
    assert call(None, None, 0, 0, 0, 1, 0, 256, None, None) == -1
    assert call(None, None, 0, 0, 0, 1, 65537, 256, None, None) == -2
    assert call(None, None, 0, 0, 0, 1 << 22, 1, 256, None, None) == -2      # 2^32 threads
    assert call(None, None, 2, 0, 1, 1, 8, 256, None, None) == -1
    assert call(256, None, 0, 0, 0, 1, 8, 256, None, None) == -1
    assert call(None, 256, 9, 0, 1, 1, 8, 256, None, None) == -1


@pytest.mark.parametrize(("mask", "error"), (
    (torch.ones(4, dtype=torch.bool), ValueError),                    # [N], not broadcast
    (torch.ones(1, 4, dtype=torch.bool), ValueError),                 # [1, N], not broadcast
    (torch.ones(3, 2, dtype=torch.bool), ValueError),                 # shorter rows
    (torch.ones(3, 4), ValueError),                                   # read bytewise otherwise
    (torch.ones(3, 4, dtype=torch.int64), ValueError),
    (torch.ones(3, 4, dtype=torch.uint8), ValueError),
    (torch.ones(3, 4, dtype=torch.bool), RuntimeError),               # on the host
))
def test_center_positions_rejects_other_masks(mask, error) -> None:
    """A mask is read as batch x length bytes on the device, so its type,
    shape and device are checked before its pointer is taken (no launch, no
    GPU)."""

    from lsso_amd.ball import hip

    with pytest.raises(error, match="valid_mask"):
        hip.center_positions(None, mask, 3, 4, torch.device("cuda", 0))


def test_center_positions_rejects_other_devices() -> None:
    from lsso_amd.ball import hip

    with pytest.raises(RuntimeError, match="device"):
        hip.center_positions(None, torch.ones(3, 4, dtype=torch.bool), 3, 4, torch.device("cpu"))
    with pytest.raises(RuntimeError, match="device"):
        hip.center_positions(torch.arange(4), None, 3, 4, torch.device("cpu"))


@pytest.mark.gpu
def test_center_positions_takes_a_device_without_index(native) -> None:
    mask = torch.tensor([[True, False, True, True]], device="cuda")
    centered, counts = native.center_positions(None, mask, 1, 4, torch.device("cuda"))
    assert counts.tolist() == [3.0]
    assert torch.allclose(centered.cpu(), torch.tensor([[-5.0, 0.0, 1.0, 4.0]]) / 3.0)
