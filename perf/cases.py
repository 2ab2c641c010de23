"""The work the quantized-matmul path is used for, as cases that can be timed.

A case is a dict of plain values; `prepare` builds what a program holds before the call
(device tensors, packed matrices, a recorded execution), `run` makes one pass through
the public entry points of `ferrum_amd.api`, `work` says what the pass cannot do without.

Five kinds of pass cover the path from end to end:

* ``project``  one dense projection, called from the host each time;
* ``layer``    the projections of dense transformer blocks with what stands between them:
               residual add + RMSNorm, attention-sized projection, residual add + RMSNorm,
               gate|up, SiLU*up, down;
* ``head``     the output matrix of a vocabulary and the greedy choice over its logits;
* ``moe``      the routed FFN with its shared expert in one call;
* ``hybrid``   the hybrid engine's routed FFN in its own id / weight arrays (f32 rows),
               its per-route branch for a few tokens and its expert-sorted branch for prompts.
"""
import random

import torch

from ferrum_amd import api

# what one block of each format weighs: (weights, bytes)
BLOCKS = {"Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210), "IQ4_XS": (256, 136), "Q8_0": (32, 34)}
SIZE = {"F32": 4, "F16": 2, "BF16": 2}
TORCH = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}


def listed():
    return [
        # one attention-sized projection of one token: the smallest call, where the host and the launch count
        {"name": "project_1x4096x4096_f32", "kind": "project", "format": "Q4_K", "n": 4096, "k": 4096, "tokens": 1,
         "dtype": "F32"},
        # token-by-token decode of a 27B-class dense model in a Q4_K_M mix, as a recorded execution
        {"name": "decode_layers_5120_f32", "kind": "layer", "format": "Q4_K", "down": "Q6_K", "hidden": 5120,
         "inter": 17408, "tokens": 1, "layers": 2, "dtype": "F32", "recorded": True},
        # the same model's output head and greedy choice
        {"name": "head_151936x5120_f32", "kind": "head", "format": "Q6_K", "n": 151936, "k": 5120, "tokens": 1,
         "dtype": "F32"},
        # a speculative tree's verification block
        {"name": "verify_8_layers_5120_f16", "kind": "layer", "format": "Q4_K", "down": "Q4_K", "hidden": 5120,
         "inter": 17408, "tokens": 8, "layers": 2, "dtype": "F16", "recorded": True},
        # a batch of sequences decoded together by an f32 model
        {"name": "batch_24_layer_4096_f32", "kind": "layer", "format": "Q4_K", "down": "Q6_K", "hidden": 4096,
         "inter": 14336, "tokens": 24, "layers": 1, "dtype": "F32", "recorded": False},
        # prefill chunks of the dense model: the short one, the long one, and a whole prompt of odd length
        {"name": "prefill_128_layer_5120_bf16", "kind": "layer", "format": "Q4_K", "down": "Q6_K", "hidden": 5120,
         "inter": 17408, "tokens": 128, "layers": 1, "dtype": "BF16", "recorded": False},
        {"name": "prefill_512_layer_5120_f16", "kind": "layer", "format": "Q4_K", "down": "Q4_K", "hidden": 5120,
         "inter": 17408, "tokens": 512, "layers": 1, "dtype": "F16", "recorded": False},
        {"name": "prefill_1999_layer_5120_bf16", "kind": "layer", "format": "Q4_K", "down": "Q6_K", "hidden": 5120,
         "inter": 17408, "tokens": 1999, "layers": 1, "dtype": "BF16", "recorded": False},
        # a 35B-A3B style model's FFN: one token, a batch of sequences, a prefill chunk
        {"name": "moe_1_f16", "kind": "moe", "format": "Q4_K", "down": "Q4_K", "hidden": 2048, "inter": 512,
         "experts": 256, "top_k": 8, "shared": True, "tokens": 1, "dtype": "F16", "recorded": True},
        {"name": "moe_16_bf16", "kind": "moe", "format": "Q4_K", "down": "Q4_K", "hidden": 2048, "inter": 512,
         "experts": 256, "top_k": 8, "shared": True, "tokens": 16, "dtype": "BF16", "recorded": False},
        {"name": "moe_512_f16", "kind": "moe", "format": "Q4_K", "down": "Q4_K", "hidden": 2048, "inter": 512,
         "experts": 256, "top_k": 8, "shared": True, "tokens": 512, "dtype": "F16", "recorded": False},
        # the same FFN through the hybrid engine's steps, on the format its published file has
        {"name": "hybrid_prompt_200_f32", "kind": "hybrid", "format": "IQ4_XS", "down": "IQ4_XS", "hidden": 2048,
         "inter": 512, "experts": 256, "top_k": 8, "shared": True, "tokens": 200, "dtype": "F32", "recorded": False},
    ]


def _log_uniform(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng: random.Random):
    largest = max((work(c) for c in listed()), key=lambda w: w["flops"])["flops"]
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= largest and _weight_bytes(case) <= 800 << 20:
            return case


def _draw(rng):
    kind = rng.choices(["project", "layer", "head", "moe", "hybrid"], [30, 30, 5, 20, 15])[0]
    form = rng.choices(list(BLOCKS), [50, 12, 18, 10, 10])[0]
    dtype = rng.choices(list(SIZE), [20, 40, 40])[0]
    # an f32 model's batches end where prompts are rounded to 16 bits by its own engine
    tokens = _log_uniform(rng, 1, 64 if dtype == "F32" else 2048)
    unit = BLOCKS[form][0]
    if kind == "project":
        return {"kind": kind, "format": form, "n": _log_uniform(rng, 512, 32768),
                "k": unit * max(1, _log_uniform(rng, 512, 17408) // unit), "tokens": tokens, "dtype": dtype}
    if kind == "head":
        return {"kind": kind, "format": rng.choice(["Q6_K", "Q8_0", "Q4_K"]), "n": _log_uniform(rng, 32000, 152000),
                "k": 256 * rng.randint(8, 20), "tokens": rng.choice([1, 1, 1, 2, 4, 8]), "dtype": dtype}
    down = "Q6_K" if form == "Q4_K" and rng.random() < 0.5 else form
    if kind == "layer":
        hidden = 256 * rng.randint(4, 24)
        inter = 256 * max(1, round(hidden * rng.uniform(2.0, 3.6) / 256))
        return {"kind": kind, "format": form, "down": down, "hidden": hidden, "inter": inter, "tokens": tokens,
                "layers": 1, "dtype": dtype, "recorded": tokens <= 16 and rng.random() < 0.7}
    experts = rng.choice([32, 64, 128, 256])
    case = {"kind": kind, "format": form, "down": down, "hidden": 256 * rng.randint(4, 12),
            "inter": 256 * rng.randint(2, 7 if experts <= 64 else 3), "experts": experts,
            "top_k": rng.choice([4, 6, 8]), "shared": True, "tokens": tokens, "dtype": dtype, "recorded": False}
    if kind == "moe":
        case["shared"] = rng.random() < 0.7
        case["recorded"] = tokens <= 16 and rng.random() < 0.7
    else:
        case["dtype"] = "F32"
        case["tokens"] = _log_uniform(rng, 1, 1024)
    return case


# ---- what a program has in hand ----------------------------------------------------------

_DEVICE = None


def _device():
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = api.Device.new(0)
    return _DEVICE


class _Memory:
    """A device buffer as torch sees one (and what keeps it alive)."""

    def __init__(self, tensor):
        self.tensor = tensor
        kind = "<i4" if tensor.dtype == api.DType.F32 else "<i2"
        self.__cuda_array_interface__ = {"shape": tuple(tensor.shape()), "typestr": kind, "version": 2,
                                         "data": (tensor.buffer.device_ptr() + tensor.offset, False),
                                         "strides": None}


def _seen(tensor, bits=False):
    """The framework's tensor as a torch tensor on the same memory."""
    t = torch.as_tensor(_Memory(tensor), device="cuda")
    return t if bits else t.view(TORCH[tensor.dtype.name])


def _zeros(shape, dtype):
    return api.Tensor.zeros(_device(), shape, api.DType[dtype])


def _normal(shape, dtype, gen, scale=1.0):
    t = _zeros(shape, dtype)
    _device().synchronize()
    _seen(t).copy_(torch.randn(shape, generator=gen, device="cuda") * scale)
    torch.cuda.synchronize()
    return t


def _packed(form, rows, cols, gen):
    """GGUF blocks whose weights have mean near 0 and a spread of 1 / sqrt(cols): uniform quants and
    sub-block scales, block scales between half and one and a half times what that spread asks for."""
    weights, size = BLOCKS[form]
    count = rows * cols // weights
    blocks = torch.randint(0, 256, (count, size), dtype=torch.uint8, device="cuda", generator=gen)

    def half(values):
        return values.to(torch.float16).view(torch.uint8).reshape(count, 2)

    unit = (0.5 + torch.rand(count, device="cuda", generator=gen)) / cols ** 0.5
    if form in ("Q4_K", "Q5_K"):
        top = 15 if form == "Q4_K" else 31
        d = unit / (14.7 * top)
        blocks[:, 0:2] = half(d)
        blocks[:, 2:4] = half(d * (top / 2))
    elif form == "Q6_K":
        blocks[:, 192:208] = torch.randint(-64, 64, (count, 16), dtype=torch.int8, device="cuda",
                                           generator=gen).view(torch.uint8)
        blocks[:, 208:210] = half(unit / 680)
    elif form == "IQ4_XS":
        blocks[:, 0:2] = half(unit / 1250)
    else:
        blocks[:, 0:2] = half(unit / 74)
    return blocks.reshape(-1).cpu().numpy()


def _matrix(form, rows, cols, gen):
    return api.QuantizedMatrix.from_bytes(_device(), rows, cols, api.QuantizationFormat[form],
                                          _packed(form, rows, cols, gen))


def _experts(form, experts, rows, cols, gen):
    return api.QuantizedExpertMatrix.new(_device(), _packed(form, experts * rows, cols, gen),
                                         api.QuantizationFormat[form], experts, rows, cols)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    state = {"project": _prepare_project, "head": _prepare_project, "layer": _prepare_layer, "moe": _prepare_moe,
             "hybrid": _prepare_hybrid}[case["kind"]](case, gen)
    state["kind"], state["case"], state["graph"] = case["kind"], case, None
    torch.cuda.synchronize()
    if case.get("recorded"):
        enqueue = {"layer": _run_layer, "moe": _run_moe}[case["kind"]]
        enqueue(state)                      # sizes the library's own workspaces
        _device().synchronize()
        with _device().execution() as recording:
            enqueue(state)
        state["graph"] = recording.graph
        state["graph"].launch()
        _device().synchronize()
    return state


def _prepare_project(case, gen):
    y = _zeros((case["tokens"], case["n"]), case["dtype"])
    return {"x": _normal((case["tokens"], case["k"]), case["dtype"], gen), "y": y, "out": _seen(y),
            "w": _matrix(case["format"], case["n"], case["k"], gen)}


def _prepare_layer(case, gen):
    t, h, i, dtype = case["tokens"], case["hidden"], case["inter"], case["dtype"]
    first, stream = _normal((t, h), dtype, gen), _normal((t, h), dtype, gen)
    layers = []
    for _ in range(case["layers"]):
        layers.append({"attention": _matrix(case["format"], h, h, gen), "up": _matrix(case["format"], 2 * i, h, gen),
                       "down": _matrix(case["down"], h, i, gen),
                       "norm1": _normal((h,), dtype, gen, 0.1), "norm2": _normal((h,), dtype, gen, 0.1),
                       "sum1": _zeros((t, h), dtype), "normed1": _zeros((t, h), dtype),
                       "projected": _zeros((t, h), dtype), "sum2": _zeros((t, h), dtype),
                       "normed2": _zeros((t, h), dtype), "packed": _zeros((t, 2 * i), dtype),
                       "activated": _zeros((t, i), dtype), "out": _zeros((t, h), dtype)})
        for name in ("norm1", "norm2"):
            _seen(layers[-1][name]).add_(1.0)
    torch.cuda.synchronize()
    last = layers[-1]
    return {"layers": layers, "first": first, "stream": stream,
            "outputs": [_seen(last[name]) for name in ("sum2", "packed", "out")]}


def _prepare_moe(case, gen):
    t, h, i, e, dtype = case["tokens"], case["hidden"], case["inter"], case["experts"], case["dtype"]
    shared = (_matrix(case["format"], 2 * i, h, gen), _matrix(case["down"], h, i, gen)) if case["shared"] else (None, None)
    ffn = api.SparseMoe(_device(), _experts(case["format"], e, 2 * i, h, gen), _experts(case["down"], e, h, i, gen),
                        api.MoeRoutingPolicy(e, case["top_k"]), shared_input=shared[0], shared_output=shared[1])
    out = _zeros((t, h), dtype)
    return {"ffn": ffn, "x": _normal((t, h), dtype, gen), "logits": _normal((t, e), "F32", gen), "y": out,
            "out": _seen(out)}


def _prepare_hybrid(case, gen):
    t, h, i, e = case["tokens"], case["hidden"], case["inter"], case["experts"]
    return {"x": _normal((t, h), "F32", gen), "logits": _normal((t, e), "F32", gen),
            "gate": _normal((h,), "F32", gen, h ** -0.5), "policy": api.MoeRoutingPolicy(e, case["top_k"]),
            "up": _experts(case["format"], e, 2 * i, h, gen), "down": _experts(case["down"], e, h, i, gen),
            "shared_up": _matrix(case["format"], 2 * i, h, gen), "shared_down": _matrix(case["down"], h, i, gen)}


# ---- one pass ------------------------------------------------------------------------------

def run(state):
    return {"project": _run_project, "head": _run_head, "layer": _run_layer, "moe": _run_moe,
            "hybrid": _run_hybrid}[state["kind"]](state)


def _run_project(state):
    _device().project_quantized(state["x"], state["w"], out=state["y"])
    return state["out"]


def _run_head(state):
    _device().project_quantized(state["x"], state["w"], out=state["y"])
    return state["out"], _seen(_device().argmax_rows(state["y"]), bits=True)


def _run_layer(state):
    if state.get("graph") is not None:
        state["graph"].launch()
        return state["outputs"]
    device, inter = _device(), state["case"]["inter"]
    total, branch = state["stream"], state["first"]
    for layer in state["layers"]:
        device.add_rmsnorm(total, branch, layer["norm1"], 1e-6, residual=layer["sum1"], normed=layer["normed1"])
        device.project_quantized(layer["normed1"], layer["attention"], out=layer["projected"])
        device.add_rmsnorm(layer["sum1"], layer["projected"], layer["norm2"], 1e-6, residual=layer["sum2"],
                           normed=layer["normed2"])
        device.project_quantized(layer["normed2"], layer["up"], out=layer["packed"])
        if state["case"]["tokens"] == 1:
            device.project_quantized(layer["packed"], layer["down"], out=layer["out"], silu_mul=True)
        else:
            device.expert_silu_mul(layer["packed"], inter, out=layer["activated"])
            device.project_quantized(layer["activated"], layer["down"], out=layer["out"])
        total, branch = layer["sum2"], layer["out"]
    return state["outputs"]


def _run_moe(state):
    if state.get("graph") is not None:
        state["graph"].launch()
    else:
        state["ffn"].forward_in_one_call(state["x"], state["logits"], out=state["y"])
    return state["out"]


def _run_hybrid(state):
    device, case = _device(), state["case"]
    used, tokens, inter, x = case["top_k"], case["tokens"], case["inter"], state["x"]
    routes = tokens * used
    ids, weights, gate = device.hybrid_moe_route(state["logits"], state["policy"], x, state["gate"])
    if routes <= 32:    # the engine's per-route branch
        packed, shared = device.hybrid_project_id_with_shared(state["up"], state["shared_up"], x, ids, routes, used,
                                                              tokens)
        down, shared_down = device.hybrid_project_id_with_shared(
            state["down"], state["shared_down"], device.expert_silu_mul(packed, inter), ids, routes, 1, tokens,
            shared_x=device.expert_silu_mul(shared, inter))
        position = None
    else:
        offsets, order, position = device.hybrid_moe_map(ids, case["experts"])
        sorted_rows = device.hybrid_moe_gather(x, order, used)
        packed, shared = device.hybrid_project_mm_id_with_shared(state["up"], state["shared_up"], sorted_rows, offsets, x)
        down, shared_down = device.hybrid_project_mm_id_with_shared(
            state["down"], state["shared_down"], device.expert_silu_mul(packed, inter), offsets,
            device.expert_silu_mul(shared, inter))
    out = device.hybrid_moe_combine(down, weights, position, shared_down, gate, used)
    return _seen(out), _seen(ids, bits=True), _seen(weights)


# ---- what a pass cannot do without ---------------------------------------------------------

def _bytes_of(form, rows, cols):
    weights, size = BLOCKS[form]
    return rows * cols // weights * size


def _weight_bytes(case):
    if case["kind"] in ("project", "head"):
        return _bytes_of(case["format"], case["n"], case["k"])
    h, i = case["hidden"], case["inter"]
    if case["kind"] == "layer":
        return case["layers"] * (_bytes_of(case["format"], h + 2 * i, h) + _bytes_of(case["down"], h, i))
    per = _bytes_of(case["format"], 2 * i, h) + _bytes_of(case["down"], h, i)
    return per * (case["experts"] + (1 if case["shared"] else 0))


def work(case):
    t = case["tokens"]
    if case["kind"] in ("project", "head"):
        size, n, k = SIZE[case["dtype"]], case["n"], case["k"]
        return {"bytes": _bytes_of(case["format"], n, k) + t * (k + n) * size, "flops": 2 * t * n * k}
    h, i, size = case["hidden"], case["inter"], SIZE[case["dtype"]]
    if case["kind"] == "layer":
        # the two streams come in; the sum, the packed rows and the branch go out
        return {"bytes": _weight_bytes(case) + t * (4 * h + 2 * i) * size,
                "flops": case["layers"] * 2 * t * (h * h + 3 * h * i)}
    per = _bytes_of(case["format"], 2 * i, h) + _bytes_of(case["down"], h, i)
    e, k = case["experts"], case["top_k"]
    hit = e * (1 - (1 - k / e) ** t)      # experts that at least one of t tokens chooses
    shared = 1 if case["shared"] else 0
    return {"bytes": (hit + shared) * per + t * (2 * h * size + 4 * e), "flops": 2 * t * (k + shared) * 3 * h * i}


def tolerance(case):
    if case["kind"] == "hybrid":
        # f32 results of rows and weights rounded to f16 on the way into the tiles, twice over
        return {"rel": 2e-3, "max": 0.02, "differ": 0.002}
    # Against the same pass in 64 bits one projection is off by 1.6e-6 / 2.9e-4 / 2.4e-3 (f32 / f16 / bf16
    # rows: tile weights and results are rounded to the row's type), the chain of projections of two
    # blocks by 9e-6 / 1.2e-3 / 9e-3.
    chained = case["kind"] in ("layer", "moe")
    rel = {"F32": 1e-5, "F16": 1e-3, "BF16": 8e-3}[case["dtype"]] * (3 if chained else 1)
    # "differ": a logit's neighbour may win a near tie
    return {"rel": rel, "max": min(0.5, 40 * rel), "differ": 0.01}
