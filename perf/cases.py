"""
The work that users of this package have it do, as cases that can be timed and compared.

Everything goes through ``scanscam_amd.scan``: a forward pass alone (inference, prefill), or a training step,
i.e. the forward pass and the gradients of gate and value for a given output gradient. A case's fields:

  layout  "rows": contiguous ``[lead, rows, T]``; "channels_last": ``[lead, C, T]`` stored ``[lead, T, C]``
          (``rows`` is then C); "fused": channels-last halves of one ``[lead, T, 2C]`` projection, taken as views
  dtype   "float32", "float64", "bfloat16" or "float16" storage (16-bit storage is scanned in fp32)
  lead, rows, T
  train   whether the gradients are computed as well
  near_one  gates in U(0.9, 1), a long memory; otherwise sigmoid(N(1, 1))
"""
import math

import torch

from scanscam_amd import scan

_DTYPES = {"float32": torch.float32, "float64": torch.float64, "bfloat16": torch.bfloat16, "float16": torch.float16}
_BYTES = {"float32": 4, "float64": 8, "bfloat16": 2, "float16": 2}

# About four times the largest error of the outputs against the same inputs scanned in float64: over the listed
# and two dozen drawn cases rel 1.3e-7 / max 1.5e-6 in fp32 (long rows of gates near 1), 2.4e-3 / 7.7e-3 in bf16
# (the gate gradient, a product with the stored output), an eighth of that in fp16; float64 is fp32 scaled by the
# ratio of the types' roundings.
_TOLERANCE = {"float32": {"rel": 6e-7, "max": 8e-6}, "float64": {"rel": 2e-15, "max": 2e-14},
              "bfloat16": {"rel": 1e-2, "max": 3e-2}, "float16": {"rel": 1.2e-3, "max": 4e-3}}

# Ranges of draw(): elements per tensor, and the bytes of one pass (below the largest listed case's).
_LEAST_ELEMENTS, _MOST_ELEMENTS = 1 << 16, 1 << 26
_MOST_BYTES = 2_000_000_000


def _case(name, layout, dtype, lead, rows, T, train, near_one=False):
    return {"name": name, "layout": layout, "dtype": dtype, "lead": lead, "rows": rows, "T": T, "train": train,
            "near_one": near_one}


def listed():
    return [
        # A short segment of a small model at inference: the launch and the host's call are all there is.
        _case("short_segment_forward", "rows", "float32", 8, 256, 32, False),
        # One training step of a small model's layer (the smallest benchmark configuration).
        _case("small_layer_step", "rows", "float32", 4, 256, 1024, True),
        # The row shape of the reference's timing tests: a mid-sized layer, all tensors fit the last-level cache.
        _case("mid_layer_step", "rows", "float32", 8, 256, 4096, True),
        # The headline configuration: a state-space layer at training batch size.
        _case("large_layer_step", "rows", "float32", 8, 2048, 4096, True),
        # Long-context sequences, few rows: time has to be spread over the chip.
        _case("long_rows_step", "rows", "float32", 1, 64, 1 << 20, True, near_one=True),
        # The same layer in mixed-precision training.
        _case("bf16_layer_step", "rows", "bfloat16", 16, 1024, 2048, True),
        # Many short sequences (windowed or per-patch scans).
        _case("short_rows_step", "rows", "float32", 256, 512, 64, True),
        # Sequences with one extra token: rows that start at any element.
        _case("odd_rows_bf16_step", "rows", "bfloat16", 40, 1676, 1001, True),
        # What a linear layer's output looks like, small batch: the reference's channels-last timing shape.
        _case("channels_last_step", "channels_last", "float32", 8, 512, 4096, True),
        # Channels-last at training batch size, a channel count off the cache line.
        _case("channels_last_odd_step", "channels_last", "float32", 64, 1001, 2048, True),
        # Few channels (one head, a small state) over a large batch.
        _case("few_channels_bf16_step", "channels_last", "bfloat16", 2048, 40, 512, True),
        # Prefill of a layer whose gate and value come out of one projection: channels-last views, no copy.
        _case("fused_projection_bf16_forward", "fused", "bfloat16", 64, 1024, 2048, False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    layout = rng.choices(("rows", "channels_last", "fused"), (0.5, 0.35, 0.15))[0]
    dtype = rng.choices(("float32", "bfloat16", "float16", "float64"), (0.45, 0.3, 0.15, 0.1))[0]
    train = rng.random() < 0.7
    # Large calls are what takes a user's time, small ones are the most numerous: half and half.
    if rng.random() < 0.5:
        elements = _log_int(rng, _LEAST_ELEMENTS, 1 << 22)
    else:
        elements = _log_int(rng, 1 << 22, _MOST_ELEMENTS)
    elements = min(elements, _MOST_BYTES // (_BYTES[dtype] * (8 if train else 3)))
    if layout == "rows":
        T = _log_int(rng, 32, min(1 << 20, elements // 8))
        count = max(1, elements // T)  # rows in all
        lead = min(_log_int(rng, 1, 64), count)
        rows = max(1, count // lead)
    else:
        rows = _log_int(rng, 8, 4096)
        T = _log_int(rng, 64, min(32768, max(65, elements // rows)))
        lead = max(1, elements // (rows * T))
    if rng.random() < 0.5:  # sizes that models choose: whole vectors and lines
        if layout == "rows" and T >= 64:
            T -= T % 32
        if layout != "rows":
            rows = rows - rows % 32 if rows >= 64 else max(8, rows - rows % 8)
    return {"layout": layout, "dtype": dtype, "lead": lead, "rows": rows, "T": T, "train": train,
            "near_one": T >= 65536 or rng.random() < 0.2}


def prepare(case, seed):
    """Gate and value (leaves that require gradients in training) and the gradient of the output, on the GPU."""
    dtype, lead, rows, T = _DTYPES[case["dtype"]], case["lead"], case["rows"], case["T"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.float64 if dtype is torch.float64 else torch.float32
    stored = (lead, rows, T) if case["layout"] == "rows" else (lead, T, rows)

    def gates(shape):
        if case["near_one"]:
            return torch.rand(shape, generator=gen, device="cuda", dtype=wide).mul_(0.1).add_(0.9)
        return torch.randn(shape, generator=gen, device="cuda", dtype=wide).add_(1.0).sigmoid_()

    def normal(shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=wide)

    if case["layout"] == "fused":
        projection = torch.empty((lead, T, 2 * rows), device="cuda", dtype=dtype)
        a, b = projection.chunk(2, dim=2)
        a.copy_(gates(stored))
        b.copy_(normal(stored))
    else:
        a, b = gates(stored).to(dtype), normal(stored).to(dtype)
    if case["layout"] != "rows":
        a, b = a.mT, b.mT
    state = {"gate": a.requires_grad_(case["train"]), "value": b.requires_grad_(case["train"])}
    if case["train"]:
        grad = normal(stored).to(dtype)
        state["output_grad"] = grad.mT if case["layout"] != "rows" else grad
    return state


def run(state):
    if "output_grad" not in state:
        return {"output": scan(state["gate"], state["value"])}
    output = scan(state["gate"], state["value"])
    gate_grad, value_grad = torch.autograd.grad(output, (state["gate"], state["value"]), state["output_grad"])
    return {"output": output.detach(), "gate_grad": gate_grad, "value_grad": value_grad}


def work(case):
    """Each input read once, each output written once: forward a, b -> h; backward a, h, gh -> ga, gb."""
    n = case["lead"] * case["rows"] * case["T"]
    return {"bytes": n * _BYTES[case["dtype"]] * (8 if case["train"] else 3), "flops": n * (5 if case["train"] else 2)}


def tolerance(case):
    return _TOLERANCE[case["dtype"]]


def _scan64(a, b):
    """``h[t] = a[t] * h[t-1] + b[t]`` along the last dimension, by doubling spans (no code of this package)."""
    a, b, span = a.clone(), b.clone(), 1
    while span < a.shape[-1]:
        b = torch.cat((b[..., :span], torch.addcmul(b[..., span:], a[..., span:], b[..., :-span])), dim=-1)
        a = torch.cat((a[..., :span], a[..., span:] * a[..., :-span]), dim=-1)
        span *= 2
    return b


def exact(case, seed):
    """What run() returns for these inputs, carried in 64 bits from the stored inputs on."""
    state = prepare(case, seed)
    a, b = (state[k].detach().double().contiguous() for k in ("gate", "value"))
    h = _scan64(a, b)
    if not case["train"]:
        return {"output": h}
    g = state["output_grad"].double().contiguous()
    none = torch.zeros_like(g[..., :1])
    value_grad = _scan64(torch.cat((none, a[..., 1:].flip(-1)), dim=-1), g.flip(-1)).flip(-1)
    return {"output": h, "gate_grad": value_grad * torch.cat((none, h[..., :-1]), dim=-1), "value_grad": value_grad}
