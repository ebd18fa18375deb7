"""Performance cases of the LSSO mixer layer on one MI355X.

Every case is one call of the public module, ``LSSO(...)(x, valid_mask=...,
position_ids=..., implementation="hip")``: the whole layer from x to y for
inference, and the same call with its first-order backward for training.

A case is a dict of plain values:
  kind       "infer" (forward without gradients) or "train" (forward and the
             gradients of x and of every parameter for a given dy)
  batch, length, dim, heads, rank, bias, dtype
  mask       trailing padding: per-sample valid lengths
  positions  "default" (none given), "shared" (one float32 [N] grid, as the
             vision adapter passes it) or "batched" (int64 [B, N], each sample
             with its own start)
"""

from __future__ import annotations

import math

import torch

from lsso_amd import LSSO, LSSOConfig
from lsso_amd.ball import hip


def _case(name, kind, batch, length, dim, heads, rank, dtype, mask=False, positions="default", bias=True):
    return {
        "name": name, "kind": kind, "batch": batch, "length": length, "dim": dim, "heads": heads,
        "rank": rank, "dtype": dtype, "mask": mask, "positions": positions, "bias": bias,
    }


def listed():
    return [
        # One image of 14 x 14 patches and a class token through the smallest
        # vision layer: the latency of a single request.
        _case("infer_one_image", "infer", 1, 197, 192, 3, 16, "float16", positions="shared"),
        # An evaluation batch of images through a wide vision layer, whose
        # features exceed what the fused projection kernels hold.
        _case("infer_image_batch", "infer", 64, 197, 768, 12, 48, "bfloat16", positions="shared"),
        # A serving batch of requests of different lengths, padded together.
        _case("infer_ragged_requests", "infer", 8, 513, 256, 8, 32, "float16", mask=True),
        # Heads of 24 features and a sequence one past a power of two: shapes
        # that no tile divides; the configuration's default without biases.
        _case("infer_narrow_heads", "infer", 32, 1025, 192, 8, 32, "float16", bias=False),
        # The published forward shell at its shortest and longest sequence.
        _case("infer_l1024", "infer", 64, 1024, 256, 8, 32, "float16"),
        _case("infer_l4096", "infer", 64, 4096, 256, 8, 32, "float16"),
        # Long padded documents in BF16 at the largest rank, every sample with
        # positions of its own.
        _case("infer_masked_r64", "infer", 32, 4096, 384, 6, 64, "bfloat16", mask=True, positions="batched"),
        # A training step of the default layer on a handful of short sequences.
        _case("train_short", "train", 8, 65, 192, 3, 16, "float16", bias=False),
        # Sequence-runner training: padded batches under BF16 autocast.
        _case("train_masked", "train", 16, 1000, 128, 4, 32, "bfloat16", mask=True),
        # The published forward + backward shell at its longest sequence.
        _case("train_l4096", "train", 64, 4096, 256, 8, 32, "float16"),
        # The same layer at rank 48.
        _case("train_r48", "train", 64, 2048, 256, 8, 48, "float16"),
        # A wide layer on two long sequences, as large models train with.
        _case("train_wide", "train", 2, 4096, 768, 12, 48, "bfloat16"),
    ]


# (dim, heads, rank) of the layers that configurations, tests and benchmark use.
_LAYERS = (
    (192, 3, 16), (256, 8, 32), (256, 8, 48), (384, 6, 64), (768, 12, 48), (192, 8, 32),
    (128, 4, 32), (128, 1, 64), (256, 8, 16),
)


def draw(rng):
    kind = rng.choice(("infer", "infer", "train"))
    dim, heads, rank = rng.choice(_LAYERS)
    length = int(round(math.exp(rng.uniform(math.log(48), math.log(4096)))))
    batch = int(round(math.exp(rng.uniform(0.0, math.log(64)))))
    case = {
        "kind": kind, "batch": batch, "length": length, "dim": dim, "heads": heads, "rank": rank,
        "dtype": rng.choice(("float16", "bfloat16")), "mask": rng.random() < 0.4,
        "positions": rng.choice(("default", "default", "shared", "batched")), "bias": rng.random() < 0.7,
    }
    budgets = {c["name"]: work(c) for c in listed() if c["kind"] == kind}
    largest = max(budgets.values(), key=lambda w: w["flops"])
    while case["batch"] > 1:
        needed = work(case)
        if needed["flops"] <= largest["flops"] and needed["bytes"] <= largest["bytes"]:
            break
        case["batch"] -= 1
    return case


def _inputs(case, seed):
    """Parameters, x, mask, positions and dy of a case, from the seed alone."""

    device = torch.device("cuda")
    generator = torch.Generator(device=device).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    batch, length, dim, heads, rank = (case[k] for k in ("batch", "length", "dim", "heads", "rank"))
    dtype = getattr(torch, case["dtype"])
    width = heads * rank + dim

    def uniform(shape, bound):
        return (torch.rand(shape, generator=generator, device=device) * 2.0 - 1.0) * bound

    def normal(shape, std=1.0):
        return torch.randn(shape, generator=generator, device=device) * std

    bound = 1.0 / math.sqrt(dim)
    parameters = {
        "core_base_raw": normal((heads, rank, rank), 0.05),
        "core_drive_weight": normal((heads, dim // heads, rank), 0.05),
        "eta_raw": math.atanh(0.9) + normal((heads,), 0.1),
        "w_bc.weight": uniform((width, dim), bound),
        "w_o.weight": uniform((dim, dim), bound),
    }
    if case["bias"]:
        parameters["w_bc.bias"] = uniform((width,), bound)
        parameters["w_o.bias"] = uniform((dim,), bound)
    x = normal((batch, length, dim)).to(dtype)
    mask = positions = None
    if case["mask"]:
        lengths = torch.randint((length + 1) // 2, length + 1, (batch,), generator=host)
        lengths[0] = length
        mask = torch.arange(length, device=device)[None, :] < lengths.to(device)[:, None]
    if case["positions"] == "shared":
        # A class token at phase zero, then centred patch coordinates.
        patches = torch.arange(length - 1, dtype=torch.float32, device=device) - 0.5 * (length - 2)
        positions = torch.cat((torch.zeros(1, device=device), patches))
    elif case["positions"] == "batched":
        starts = torch.randint(0, 1024, (batch,), generator=host).to(device)
        positions = starts[:, None] + torch.arange(length, device=device)[None, :]
    dy = normal((batch, length, dim)).to(dtype) if case["kind"] == "train" else None
    return parameters, x, mask, positions, dy


def prepare(case, seed):
    hip.load()
    parameters, x, mask, positions, dy = _inputs(case, seed)
    config = LSSOConfig(dim=case["dim"], num_heads=case["heads"], rank=case["rank"], bias=case["bias"])
    with torch.device("cuda"):
        layer = LSSO(config)
    with torch.no_grad():
        for name, parameter in layer.named_parameters():
            parameter.copy_(parameters[name])
    train = case["kind"] == "train"
    layer.train(train)
    if train:
        x.requires_grad_()
    return {"layer": layer, "x": x, "mask": mask, "positions": positions, "dy": dy}


def run(state):
    layer, x = state["layer"], state["x"]
    options = {"valid_mask": state["mask"], "position_ids": state["positions"], "implementation": "hip"}
    if state["dy"] is None:
        with torch.no_grad():
            return {"y": layer(x, **options)}
    y = layer(x, **options)
    names, parameters = zip(*layer.named_parameters())
    grads = torch.autograd.grad(y, (x, *parameters), state["dy"])
    return {"y": y.detach(), "x": grads[0], **dict(zip(names, grads[1:]))}


def work(case):
    batch, length, dim, heads, rank = (case[k] for k in ("batch", "length", "dim", "heads", "rank"))
    head_dim = dim // heads
    width = heads * rank + dim
    tokens = batch * length
    valid = tokens * (0.75 if case["mask"] else 1.0)
    weights = 4.0 * (width * dim + dim * dim + heads * rank * (rank + head_dim) + heads
                     + (width + dim if case["bias"] else 0))
    side = (tokens if case["mask"] else 0) + {"default": 0, "shared": 4 * length, "batched": 8 * tokens}[case["positions"]]
    # Both projections; A^T A, A^T C and the readout A M per token; the
    # factorization, two inverses and products of each compact system.
    flops = valid * (2.0 * dim * width + 2.0 * dim * dim + 2.0 * heads * rank * (rank + 2 * head_dim))
    flops += batch * heads * (3.0 * rank ** 3 + 7.0 * rank * rank * head_dim)
    moved = 2.0 * dim * (valid + tokens) + weights + side
    if case["kind"] == "train":
        # dX and dW of both projections; A^T dY, dY M^T, C E^T, A E and A Gamma
        # per token; the compact problem's VJP.
        flops += valid * (4.0 * dim * width + 4.0 * dim * dim + 2.0 * heads * rank * (rank + 4 * head_dim))
        flops += batch * heads * (8.0 * rank ** 3 + 14.0 * rank * rank * head_dim)
        moved += 2.0 * dim * (valid + tokens) + weights
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # BF16 operands and intermediates with FP32 sums: y and every gradient
    # are about 3e-3 (up to 6e-3) from the 64-bit result.
    return {"rel": 1.2e-2 if case["kind"] == "infer" else 2e-2}


def _centred(case, positions, mask, batch, length, device):
    if positions is None:
        positions = torch.arange(length, device=device)
    positions = positions.double().expand(batch, length)
    keep = torch.ones(batch, length, dtype=torch.float64, device=device) if mask is None else mask.double()
    return (positions - (positions * keep).sum(-1, keepdim=True) / keep.sum(-1, keepdim=True)) * keep


def _forward64(case, p, x, mask, positions):
    """The layer in 64 bits, through the Cholesky factor of I + A^T A."""

    heads, rank, dim = case["heads"], case["rank"], case["dim"]
    head_dim = dim // heads
    batch, length, _ = x.shape
    centred = _centred(case, positions, mask, batch, length, x.device)
    packed = x @ p["w_bc.weight"].mT
    if "w_bc.bias" in p:
        packed = packed + p["w_bc.bias"]
    if mask is not None:
        packed = torch.where(mask[:, :, None], packed, torch.zeros_like(packed))
        count = mask.sum(-1).double()
    else:
        count = torch.full((batch,), float(length), dtype=torch.float64, device=x.device)
    scale = count.sqrt().view(batch, 1, 1, 1)
    relation = packed[..., :heads * rank].view(batch, length, heads, rank).transpose(1, 2)
    content = packed[..., heads * rank:].view(batch, length, heads, head_dim).transpose(1, 2)
    half = rank // 2
    frequency = 10000.0 ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    angle = (centred[:, :, None] * frequency)[:, None]
    cos, sin = angle.cos(), angle.sin()
    even, odd = relation[..., 0::2], relation[..., 1::2]
    a = torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).flatten(-2) / scale
    # The r x r problems on the host: their 64-bit factorizations are small.
    gram, moment, root = (a.mT @ a).cpu(), (a.mT @ content).cpu(), scale.cpu()
    base, drive = p["core_base_raw"].cpu(), p["core_drive_weight"].cpu()
    eye = torch.eye(rank, dtype=torch.float64)
    lower = torch.linalg.cholesky(gram + eye)
    z = torch.linalg.solve_triangular(lower, moment, upper=False)
    theta = base + z @ drive / root
    diagonal = torch.nn.functional.softplus(torch.diagonal(theta, dim1=-2, dim2=-1) + math.log(math.expm1(1.0)))
    factor = torch.tril(theta, -1) + torch.diag_embed(diagonal)
    upper = torch.triu(theta, 1)
    system = eye + factor @ factor.mT + upper - upper.mT
    eta = torch.tanh(p["eta_raw"])
    state = 2.0 * torch.linalg.solve(system, z) - (1.0 + eta.cpu().view(1, heads, 1, 1)) * z
    readout = torch.linalg.solve_triangular(lower.mT, state, upper=True).to(x.device)
    mixed = eta.view(1, heads, 1, 1) * content + a @ readout
    y = mixed.transpose(1, 2).reshape(batch, length, dim) @ p["w_o.weight"].mT
    if "w_o.bias" in p:
        y = y + p["w_o.bias"]
    return y if mask is None else torch.where(mask[:, :, None], y, torch.zeros_like(y))


def exact(case, seed):
    parameters, x, mask, positions, dy = _inputs(case, seed)
    train = case["kind"] == "train"
    p = {name: value.double().requires_grad_(train) for name, value in parameters.items()}
    batch, length, _ = x.shape
    step = max(1, 16384 // length)      # samples a slice, which bounds the memory
    y, grad_x = [], []
    for begin in range(0, batch, step):
        part = slice(begin, min(batch, begin + step))
        xs = x[part].double().requires_grad_(train)
        per_sample = positions is not None and positions.dim() == 2
        with torch.set_grad_enabled(train):
            ys = _forward64(case, p, xs, None if mask is None else mask[part],
                            positions[part] if per_sample else positions)
        y.append(ys.detach())
        if train:
            ys.backward(dy[part].double())
            grad_x.append(xs.grad)
    result = {"y": torch.cat(y)}
    if train:
        result["x"] = torch.cat(grad_x)
        result.update({name: value.grad for name, value in p.items()})
    return result
