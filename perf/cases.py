"""What a user of this package has it do, as cases that can be timed and whose results can be compared.

A case is a dict of plain values.  ``listed()`` names the ones that stand for everyday use,
``draw(rng)`` gives further ones of the same ranges, ``prepare(case, seed)`` builds what a program
has in hand before the call, ``run(state)`` makes one pass through the public entry points and
returns its outputs, ``work(case)`` says what the pass cannot do without and ``tolerance(case)``
how far another correct implementation of the same precision may be away.

Six kinds of work:

* ``layers``: the packed linear layers of decoder blocks (q / k / v / o, gate / up / down) at 1 to
  2048 activation rows: token by token, a batch of sequences, a prompt;
* ``head``: a tied output head and its embedding table, both read from the same packed codes;
* ``round``: rounding a weight matrix to nearest, with its packed stream and reconstruction;
* ``gptq``: error feedback over scalar grids from a calibration Hessian;
* ``ldlq``: error feedback over vector grids (the E8P lattice, a codebook of 8-vectors);
* ``incoherent``: rounding in a randomly rotated basis.
"""

import math

import torch
from torch import nn

import mlkit_amd as mk

SEVEN_VALUES = (-1.0, -0.5, -0.25, 0.0, 0.25, 0.5, 1.0)

# name -> (bits per code, columns per scale, side values per scale group, quantizer)
FORMATS = {
    "int4": (4, 128, 1, lambda: mk.int(4, 128)),
    "int4-asym": (4, 128, 2, lambda: mk.int(4, 128, asym=True)),
    "int2": (2, 64, 1, lambda: mk.int(2, 64)),
    "int3": (3, 64, 1, lambda: mk.int(3, 64)),
    "int8": (8, 128, 1, lambda: mk.int(8, 128)),
    "nf4": (4, 64, 1, lambda: mk.nf4(64)),
    "codebook": (3, 64, 1, lambda: mk.scaled(mk.grid.values(list(SEVEN_VALUES), bits=3), group=64, scale="mse")),
}

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}


def listed():
    return [
        # One token of one sequence through a 0.5B-class decoder block, layer by layer from Python: the smallest
        # calls there are, where the cost of a call and of a launch is what counts.
        {"name": "decode-896-m1", "kind": "layers", "format": "int4", "dtype": "fp16", "rows": 1, "blocks": 1,
         "hidden": 896, "kv": 128, "mlp": 4864, "bias": True, "rotated": False, "graph": False},
        # One token through 8B-class decoder blocks as a serving loop runs them: captured once, replayed per token,
        # siblings in shared launches, o and down with their online rotation.  Three blocks' weights (340 MB) do
        # not stay in the 256 MB cache, as a model's do not.
        {"name": "decode-4096-m1-graph", "kind": "layers", "format": "int4", "dtype": "fp16", "rows": 1, "blocks": 3,
         "hidden": 4096, "kv": 1024, "mlp": 14336, "bias": False, "rotated": True, "graph": True},
        # Eight sequences decoding together, on the normal-float codebook.
        {"name": "decode-4096-nf4-m8", "kind": "layers", "format": "nf4", "dtype": "bf16", "rows": 8, "blocks": 3,
         "hidden": 4096, "kv": 1024, "mlp": 14336, "bias": False, "rotated": False, "graph": False},
        # Thirty-two sequences decoding together (or a short prompt), weights with offsets.
        {"name": "batch-4096-m32", "kind": "layers", "format": "int4-asym", "dtype": "bf16", "rows": 32, "blocks": 3,
         "hidden": 4096, "kv": 1024, "mlp": 14336, "bias": False, "rotated": False, "graph": False},
        # A prompt of 2048 tokens through one block.
        {"name": "prompt-4096-m2048", "kind": "layers", "format": "int4", "dtype": "bf16", "rows": 2048, "blocks": 1,
         "hidden": 4096, "kv": 1024, "mlp": 14336, "bias": False, "rotated": False, "graph": False},
        # The first and the last layer of a tied 0.5B-class decoder: embedding rows and logits of four sequences.
        {"name": "tied-head-151936-m4", "kind": "head", "format": "int4", "dtype": "fp16", "rows": 4, "vocabulary": 151936,
         "hidden": 896},
        # Converting a checkpoint without calibration: one 8B-class weight to codes, scales, offsets, the packed
        # stream and the reconstruction that replaces the weight.
        {"name": "round-int4-4096x14336", "kind": "round", "format": "int4-asym", "dtype": "fp16", "rows": 4096,
         "width": 14336},
        # The same with scales searched for least squared error, on a codebook.
        {"name": "round-codebook-4096x4096", "kind": "round", "format": "codebook", "dtype": "fp16", "rows": 4096,
         "width": 4096},
        # Calibrated conversion of a small layer, columns in order of activation.
        {"name": "gptq-4864x896-order", "kind": "gptq", "format": "int4-asym", "dtype": "fp16", "rows": 4864, "width": 896,
         "order": True},
        # Calibrated conversion of a large layer.
        {"name": "gptq-4096x11008", "kind": "gptq", "format": "int4", "dtype": "fp16", "rows": 4096, "width": 11008,
         "order": False},
        # Calibrated conversion to two bits per weight on the E8P lattice.
        {"name": "ldlq-e8p-2048x2048", "kind": "ldlq", "grid": "e8p", "dtype": "fp16", "rows": 2048, "width": 2048},
        # Conversion in a rotated basis: a down projection whose 14336 columns rotate as 28 blocks of 512.
        {"name": "incoherent-4096x14336", "kind": "incoherent", "format": "int4", "dtype": "bf16", "rows": 4096,
         "width": 14336},
    ]


# -- drawn cases ---------------------------------------------------------------------------------


def _size(rng, low, high, units):
    """A size between ``low`` and ``high``, even over its logarithm, a multiple of one of ``units``."""
    unit = rng.choice(units)
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high // unit * unit, max(-(-low // unit) * unit, round(value / unit) * unit))


LAYER_WORK = 2048 * 218_103_808   # activation rows x weights of the listed prompt


def draw(rng):
    kind = rng.choice(["layers", "layers", "layers", "layers", "head", "round", "gptq", "ldlq", "incoherent"])
    if kind == "layers":
        hidden = _size(rng, 256, 8192, (8, 64, 128, 256))
        mlp = _size(rng, 2 * hidden, min(28672, 4 * hidden), (8, 64, 128, 256))
        kv = max(32, hidden // rng.choice((1, 2, 4, 8)) - rng.choice((0, 0, 1, 3)))
        weights = 2 * hidden * (hidden + kv) + 3 * hidden * mlp
        regime = rng.choice(("decode", "batch", "prompt"))
        low, high = {"decode": (1, 8), "batch": (9, 128), "prompt": (129, 2048)}[regime]
        rows = _size(rng, low, max(low, min(high, LAYER_WORK // weights)), (1,))
        formats = list(FORMATS) if hidden % 32 == 0 and mlp % 32 == 0 else ["int4", "int4-asym", "int8", "nf4"]
        dtype = rng.choice(("fp16", "bf16", "fp32") if regime == "decode" else ("fp16", "bf16"))
        return {"kind": kind, "format": rng.choice(formats), "dtype": dtype, "rows": rows, "blocks": 1, "hidden": hidden,
                "kv": kv, "mlp": mlp, "bias": rng.random() < 0.3,
                "rotated": regime != "prompt" and dtype != "fp32" and hidden % 64 == 0 and mlp % 64 == 0 and rng.random() < 0.3,
                "graph": regime == "decode" and rng.random() < 0.4}
    if kind == "head":
        return {"kind": kind, "format": rng.choice(("int4", "int8", "int4-asym")), "dtype": rng.choice(("fp16", "bf16")),
                "rows": _size(rng, 1, 64, (1,)), "vocabulary": _size(rng, 16000, 151936, (1, 2, 128)),
                "hidden": _size(rng, 512, 2048, (64, 128))}
    if kind == "round":
        return {"kind": kind, "format": rng.choice(list(FORMATS)), "dtype": rng.choice(("fp16", "bf16", "fp32")),
                "rows": _size(rng, 128, 8192, (1, 8, 128)), "width": _size(rng, 256, 14336, (1, 8, 64, 128))}
    if kind == "gptq":
        return {"kind": kind, "format": rng.choice(("int4", "int4-asym", "int3", "nf4")),
                "dtype": rng.choice(("fp16", "bf16")), "rows": _size(rng, 128, 4096, (1, 8, 128)),
                "width": _size(rng, 384, 8192, (1, 8, 128)), "order": rng.random() < 0.4}
    if kind == "ldlq":
        return {"kind": kind, "grid": rng.choice(("e8p", "vector")), "dtype": rng.choice(("fp16", "bf16")),
                "rows": _size(rng, 128, 4096, (1, 8, 128)), "width": _size(rng, 384, 4096, (8, 128))}
    return {"kind": kind, "format": rng.choice(("int4", "int4-asym", "int3", "nf4")), "dtype": rng.choice(("fp16", "bf16")),
            "rows": _size(rng, 256, 8192, (64, 128, 256)), "width": _size(rng, 512, 14336, (64, 128, 512))}


# -- what a program has in hand ------------------------------------------------------------------


class _Attention(nn.Module):
    def __init__(self, hidden, kv, bias):
        super().__init__()
        self.q_proj = nn.Linear(hidden, hidden, bias=bias)
        self.k_proj = nn.Linear(hidden, kv, bias=bias)
        self.v_proj = nn.Linear(hidden, kv, bias=bias)
        self.o_proj = nn.Linear(hidden, hidden, bias=False)

    def forward(self, entering, attended):
        return self.q_proj(entering), self.k_proj(entering), self.v_proj(entering), self.o_proj(attended)


class _Mlp(nn.Module):
    def __init__(self, hidden, mlp):
        super().__init__()
        self.gate_proj = nn.Linear(hidden, mlp, bias=False)
        self.up_proj = nn.Linear(hidden, mlp, bias=False)
        self.down_proj = nn.Linear(mlp, hidden, bias=False)

    def forward(self, entering, gated):
        return self.gate_proj(entering), self.up_proj(entering), self.down_proj(gated)


class _Blocks(nn.Module):
    """The linear layers of decoder blocks; what lies between them (attention, activation, norms) is not this
    package's work, so each layer's input is given."""

    def __init__(self, case):
        super().__init__()
        self.blocks = nn.ModuleList()
        for _ in range(case["blocks"]):
            block = nn.Module()
            block.self_attn = _Attention(case["hidden"], case["kv"], case["bias"])
            block.mlp = _Mlp(case["hidden"], case["mlp"])
            self.blocks.append(block)

    def forward(self, entering, attended, normed, gated):
        return [output for block in self.blocks
                for output in (*block.self_attn(entering, attended), *block.mlp(normed, gated))]


class _TiedHead(nn.Module):
    def __init__(self, case):
        super().__init__()
        self.embed_tokens = nn.Embedding(case["vocabulary"], case["hidden"])
        self.lm_head = nn.Linear(case["hidden"], case["vocabulary"], bias=False)
        self.lm_head.weight = self.embed_tokens.weight

    def forward(self, tokens, hidden):
        return self.embed_tokens(tokens), self.lm_head(hidden)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(rows, width, dtype, generator, outliers):
    """N(0, 0.02^2); with ``outliers`` one input channel in a thousand twenty times as large."""
    weight = torch.randn((rows, width), generator=generator, device="cuda") * 0.02
    if outliers:
        large = torch.rand((width,), generator=generator, device="cuda") < 1e-3
        weight = torch.where(large, weight * 20, weight)
    return weight.to(dtype)


def _hessian(width, generator):
    """``X^T X / n`` of fp16 activations, one channel in a hundred thirty times as large."""
    tokens = max(1024, min(16384, 2 * width))
    inputs = torch.randn((tokens, width), generator=generator, device="cuda")
    large = torch.rand((width,), generator=generator, device="cuda") < 1e-2
    inputs = torch.where(large, inputs * 30, inputs).half().float()
    return inputs.T @ inputs / tokens


def _module_on_gpu(build, case, generator):
    with torch.device("meta"):
        module = build(case)
    module = module.to_empty(device="cuda").to(DTYPES[case["dtype"]])
    if isinstance(module, _TiedHead):
        module.lm_head.weight = module.embed_tokens.weight
    with torch.no_grad():
        for parameter in module.parameters():
            if parameter.dim() == 2:
                parameter.copy_(_weight(*parameter.shape, parameter.dtype, generator, True))
            else:
                parameter.copy_(torch.randn(parameter.shape, generator=generator, device="cuda") * 0.1)
    return module


def _normal(rows, width, case, generator):
    return torch.randn((rows, width), generator=generator, device="cuda").to(DTYPES[case["dtype"]])


def prepare(case, seed):
    generator = _generator(seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("layers", "head"):
        quantization = FORMATS[case["format"]][3]()
        module = _module_on_gpu(_Blocks if kind == "layers" else _TiedHead, case, generator)
        if kind == "layers":
            if case["rotated"]:
                mk.rotate(seed=1)(module)
            served = mk.optimize(mk.quantize(module, quantization), "packed", inplace=True, group_siblings=case["graph"])
            hidden, mlp, rows = case["hidden"], case["mlp"], case["rows"]
            inputs = [_normal(rows, width, case, generator) for width in (hidden, hidden, hidden, mlp)]
        else:
            served = mk.optimize(mk.quantize(module, quantization, head=quantization), "packed", inplace=True)
            inputs = [torch.randint(case["vocabulary"], (case["rows"],), generator=generator, device="cuda"),
                      _normal(case["rows"], case["hidden"], case, generator)]
        state.update(module=served.module, inputs=inputs)
        if case.get("graph"):
            state.update(_captured(served.module, inputs))
        return state
    state["weight"] = _weight(case["rows"], case["width"], DTYPES[case["dtype"]], generator, kind == "round")
    if kind == "ldlq":
        if case["grid"] == "e8p":
            grid = mk.grid.e8p()
        else:
            grid = mk.grid.vector(torch.randn((256, 8), generator=generator, device="cuda").cpu())
        state["quantizer"] = mk.ldlq(mk.scaled(grid, group=128), step=8, refit=128)
    else:
        inner = FORMATS[case["format"]][3]()
        if kind == "round":
            state["quantizer"], state["bits"] = inner, FORMATS[case["format"]][0]
        elif kind == "gptq":
            state["quantizer"] = mk.gptq(inner, act_order=case["order"])
        else:
            state["quantizer"] = mk.incoherent(inner)
    if kind in ("gptq", "ldlq"):
        state["context"] = mk.Ctx("blocks.0.layer", H=_hessian(case["width"], generator), device="cuda")
    else:
        state["context"] = mk.Ctx("blocks.0.layer", device="cuda")
    return state


def _captured(module, inputs):
    """The pass over ``module`` as a HIP graph, the way a serving loop keeps it."""
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            module(*inputs)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = module(*inputs)
    return {"graph": graph, "outputs": outputs}


# -- one pass ------------------------------------------------------------------------------------


def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if "graph" in state:
            state["graph"].replay()
            return state["outputs"]
        if kind in ("layers", "head"):
            return state["module"](*state["inputs"])
        quantized = state["quantizer"](state["weight"], state["context"])
        outputs = {"codes": quantized.codes}
        outputs.update({name: value for name, value in quantized.params.items()
                        if name.removeprefix("inner_") in ("scales", "zero", "permutation")})
        if kind in ("round", "incoherent"):   # what a conversion writes back into the model
            outputs["weight"] = quantized.w.to(state["weight"].dtype)
        if kind == "round":
            outputs["packed"] = mk.pack(quantized.codes, state["bits"])
        return outputs


# -- what a pass cannot do without ---------------------------------------------------------------


def _packed_bytes(rows, width, format_name):
    bits, group, side, _ = FORMATS[format_name]
    return rows * width * bits / 8 + rows * -(-width // group) * side * 2


def work(case):
    kind, element = case["kind"], BYTES[case["dtype"]]
    if kind == "layers":
        hidden, kv, mlp, rows = case["hidden"], case["kv"], case["mlp"], case["rows"]
        linears = [(hidden, hidden), (kv, hidden), (kv, hidden), (hidden, hidden), (mlp, hidden), (mlp, hidden), (hidden, mlp)]
        total = sum(_packed_bytes(n, k, case["format"]) + rows * n * element for n, k in linears)
        return {"bytes": case["blocks"] * total + rows * (3 * hidden + mlp) * element,
                "flops": case["blocks"] * 2.0 * rows * sum(n * k for n, k in linears)}
    if kind == "head":
        rows, hidden, vocabulary = case["rows"], case["hidden"], case["vocabulary"]
        return {"bytes": _packed_bytes(vocabulary, hidden, case["format"]) + rows * (vocabulary + 2 * hidden) * element + 8 * rows,
                "flops": 2.0 * rows * hidden * vocabulary}
    rows, width = case["rows"], case["width"]
    weight = rows * width
    if kind == "ldlq":
        # the weight in, a 32-bit code per eight weights out, scales, the Hessian
        return {"bytes": weight * element + weight / 2 + rows * -(-width // 128) * 4 + 4.0 * width * width,
                "flops": width**3 / 3 + float(rows) * width * width}
    _, group, side, _ = FORMATS[case["format"]]
    total = weight * element + weight + rows * -(-width // group) * side * 4
    if kind == "gptq":
        return {"bytes": total + 4.0 * width * width, "flops": width**3 / 3 + float(rows) * width * width}
    total += weight * element   # the reconstruction
    if kind == "round":
        return {"bytes": total + weight * FORMATS[case["format"]][0] / 8, "flops": 0}
    # two butterfly transforms of every element, there and back
    return {"bytes": total, "flops": 2.0 * weight * (math.log2(rows) + math.log2(width))}


def tolerance(case):
    """About four times what two correct ways of the same precision were measured to differ by."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "round":
        return "exact"
    if kind in ("layers", "head"):
        # against products in 64 bits, with the decoded weight kept exact and rounded to the activations' type:
        # fp16 up to 3.7e-4 (largest 1.6e-3), bf16 2.9e-3 (1.6e-2), fp32 7e-7 (3e-6)
        return {"fp16": {"rel": 1.5e-3, "max": 6e-3}, "bf16": {"rel": 1.2e-2, "max": 6e-2},
                "fp32": {"rel": 4e-6, "max": 2e-5}}[dtype]
    if kind == "incoherent":
        # against rotations in 64 bits: 4e-6 of the codes (a value next to a rounding boundary), weights
        # 6e-4 (fp16) and 9e-4 (bf16), the largest difference one step of their type
        return {"differ": 2e-5, **{"fp16": {"rel": 2.4e-3, "max": 6e-3}, "bf16": {"rel": 4e-3, "max": 3.2e-2},
                                   "fp32": {"rel": 2.4e-3, "max": 6e-3}}[dtype]}
    # against coefficients from a factorisation in 64 bits.  A code next to a rounding boundary flips and the columns
    # after it in that row follow: gptq up to 5.8e-4 of the codes, scales 1.5e-3 (largest 0.18), offsets 8e-3 (0.66);
    # ldlq 2e-4 of the codes, scales 6e-4 (0.09)
    if kind == "gptq":
        return {"differ": 2.4e-3, "rel": 3e-2, "max": 0.99} if "asym" in case["format"] else {"differ": 2.4e-3, "rel": 6e-3, "max": 0.7}
    return {"differ": 8e-4, "rel": 2.4e-3, "max": 0.36}
