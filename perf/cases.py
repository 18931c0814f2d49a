"""The work that a user of this package has it do, as a list of measurable cases.

A case is a dict of plain values.  `listed()` gives the named ones, `draw(rng)` one more of the same
ranges, `prepare(case, seed)` what a program holds before the call (layers with quantized weights and
inputs, on the GPU, made from the seed), `run(state)` one pass through the public entry points and its
outputs, `work(case)` the bytes and operations one pass cannot do without, and `tolerance(case)` how far
another correct implementation of the same precision may be off.

Kinds of work:
  linear   one `OrbitLinear` forward: quantize the tokens, multiply with the packed weight
  mlp      two of them with the GELU between them fused into the first (`fuse_output_activation`)
  block    the linears of a transformer block: q, k, v of one input (as an `OrbitLinearGroup`, or one fused
           matrix), the output projection, and the MLP; the attention between them is the model's own.
           `graph`: the pass is a captured HIP graph, as decoding programs launch it
  adaln    one `RTNInt4Linear` forward (the INT4 modulation linear of DiT blocks)
  native   the kernel package's W4A4 pair: `quantize_activations_packed_w4`, `matmul_packed_w4a4_int8`
  values   the kernel package's `matmul_packed_weight`: floating activations times the packed weight
  convert  a weight taken into the packed format on the GPU and read back as the matrix it now stands for
"""

from __future__ import annotations

import math

import torch

import orbitquant_packed_matmul as native_package
from orbitquant_amd import OrbitLinear, OrbitLinearGroup, OrbitQuantConfig, RTNInt4Linear, get_codebook, get_rpbh_rotation, ops

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ADALN_GROUP = 64


def listed() -> list[dict]:
    return [
        # the smallest call: one token through one projection, as a decoding program issues it eagerly
        {"name": "token linear", "kind": "linear", "m": 1, "k": 4096, "n": 4096, "wbits": 4, "abits": 4, "dtype": "bf16",
         "bias": False, "outliers": "none"},
        # one token through a layer of the mixed-width decode stack (q, k at two bits, the rest at three), as a graph
        {"name": "decode block", "kind": "block", "m": 1, "hidden": 4096, "kv": 4096, "ffn": 14336, "wqk": 2, "wvo": 3, "wmlp": 3,
         "abits": 4, "dtype": "bf16", "fused": False, "graph": True, "outliers": "none"},
        # sixteen sequences decoded together through one of the stack's four-bit layers
        {"name": "batch decode block", "kind": "block", "m": 16, "hidden": 4096, "kv": 4096, "ffn": 14336, "wqk": 4, "wvo": 4,
         "wmlp": 4, "abits": 4, "dtype": "bf16", "fused": False, "graph": False, "outliers": "none"},
        # the modulation of a DiT-XL/2 block, one conditioning row per image of a batch of eight
        {"name": "adaln modulation", "kind": "adaln", "m": 8, "k": 1152, "n": 6912},
        # an attention projection of DiT-XL/2 in fp32, blocks of 64 values
        {"name": "fp32 projection", "kind": "linear", "m": 256, "k": 1152, "n": 1152, "wbits": 4, "abits": 4, "dtype": "fp32",
         "bias": True, "outliers": "entries"},
        # a prompt of a few hundred tokens (prefill) in fp16, a ragged token count
        {"name": "prompt linear", "kind": "linear", "m": 333, "k": 4096, "n": 14336, "wbits": 4, "abits": 4, "dtype": "fp16",
         "bias": True, "outliers": "none"},
        # the DiT-XL/2 MLP pair, eight images of 256 patches
        {"name": "dit mlp", "kind": "mlp", "m": 2048, "k": 1152, "n": 4608, "wbits": 4, "abits": 4, "dtype": "bf16", "outliers": "columns"},
        # the linears of a Flux-style block in the three-bit recipe: 4096 image tokens and 512 text tokens
        {"name": "flux block", "kind": "block", "m": 4608, "hidden": 3072, "kv": 3072, "ffn": 12288, "wqk": 3, "wvo": 3, "wmlp": 3,
         "abits": 3, "dtype": "bf16", "fused": True, "graph": False, "outliers": "heavy"},
        # the largest: the FFN of a video DiT, 21 latent frames of 30 x 52 patches, six-bit activations
        {"name": "video ffn", "kind": "mlp", "m": 32760, "k": 5120, "n": 13824, "wbits": 4, "abits": 6, "dtype": "bf16", "outliers": "entries"},
        # the kernel package's W4A4 pair on the wide projection it is quoted on
        {"name": "native w4a4", "kind": "native", "m": 4608, "k": 4096, "n": 36864, "dtype": "bf16", "outliers": "none"},
        # the kernel package's floating-activation matmul, half precision
        {"name": "native values", "kind": "values", "m": 512, "k": 3072, "n": 12288, "wbits": 4, "dtype": "fp16", "bias": False},
        # the largest matrix of the decode stack taken into the packed format, and read back
        {"name": "convert weight", "kind": "convert", "n": 14336, "k": 4096, "wbits": 4, "dtype": "bf16"},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def _width(rng, low: int, high: int, step: int) -> int:
    """A layer width: a multiple of `step`, spread over the logarithm of the range."""
    return max(low, _log_int(rng, low, high) // step * step)


def draw(rng) -> dict:
    kind = rng.choices(["linear", "mlp", "block", "adaln", "native", "values", "convert"], [5, 3, 4, 2, 2, 2, 2])[0]
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    outliers = rng.choice(["none", "entries", "columns", "heavy"])
    wbits, abits = rng.choice([(4, 4), (4, 4), (3, 3), (2, 4), (2, 3), (4, 6)])
    if kind == "adaln":
        return {"kind": kind, "m": _log_int(rng, 1, 64), "k": _width(rng, 256, 6144, 64), "n": _width(rng, 1024, 36864, 8)}
    if kind == "convert":
        return {"kind": kind, "n": _width(rng, 256, 14336, 8), "k": _width(rng, 256, 14336, 64), "wbits": wbits, "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "native":
        return {"kind": kind, "m": _log_int(rng, 1, 4608), "k": _width(rng, 512, 8192, 64), "n": _width(rng, 512, 18432, 8), "dtype": dtype,
                "outliers": outliers}
    if kind == "values":
        return {"kind": kind, "m": _log_int(rng, 1, 4608), "k": _width(rng, 512, 8192, 64), "n": _width(rng, 512, 12288, 8), "wbits": rng.choice([2, 3, 4, 4, 6]),
                "dtype": dtype, "bias": rng.random() < 0.5}
    if kind == "linear":
        if rng.random() < 0.15:
            dtype = "fp32"
        k = rng.choice([768, 1152, 3072, 4096, 5120]) if abits > 4 else _width(rng, 256, 12288, 64)
        return {"kind": kind, "m": _log_int(rng, 1, 8192), "k": k, "n": _width(rng, 256, 14336, 8), "wbits": wbits, "abits": abits,
                "dtype": dtype, "bias": rng.random() < 0.5, "outliers": outliers}
    if kind == "mlp":
        k = rng.choice([768, 1152, 3072, 5120]) if abits > 4 else _width(rng, 512, 5120, 64)
        n = 4 * k if abits > 4 else _width(rng, 2 * k, 4 * k, 64)
        return {"kind": kind, "m": _log_int(rng, 64, 16384), "k": k, "n": n, "wbits": wbits, "abits": abits, "dtype": dtype, "outliers": outliers}
    hidden = _width(rng, 768, 5120, 128)
    decode = rng.random() < 0.6
    kv = hidden if rng.random() < 0.5 else max(128, hidden // 4 // 64 * 64)
    wqk, wvo = (2, 3) if rng.random() < 0.4 else (wbits, wbits)
    return {"kind": kind, "m": _log_int(rng, 1, 64) if decode else _log_int(rng, 65, 6144), "hidden": hidden, "kv": kv,
            "ffn": _width(rng, 2 * hidden, min(4 * hidden, 14336), 64), "wqk": wqk, "wvo": wvo, "wmlp": wvo, "abits": min(abits, 4), "dtype": dtype,
            "fused": not decode and kv == hidden and wqk == wvo, "graph": decode and rng.random() < 0.5, "outliers": outliers}


# ---------------------------------------------------------------- inputs and layers

def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _tokens(g, m: int, k: int, dtype: str, outliers: str = "none") -> torch.Tensor:
    """Activations: N(0, 1), with the outliers that diffusion transformers and language models show."""
    x = torch.randn(m, k, generator=g, device="cuda")
    if outliers == "entries":      # one value in a hundred, twenty times as large
        x = torch.where(torch.rand(m, k, generator=g, device="cuda") < 0.01, x * 20, x)
    elif outliers == "columns":    # a few channels, thirty times as large
        channels = torch.randperm(k, generator=g, device="cuda")[: max(1, math.ceil(0.005 * k))]
        x[:, channels] *= 30
    elif outliers == "heavy":      # Student-t with four degrees of freedom
        chi = torch.zeros_like(x)
        for _ in range(4):
            chi += torch.randn(m, k, generator=g, device="cuda").square_()
        x = x / torch.sqrt(chi / 4)
    return x.to(DTYPES[dtype])


def _weight(g, n: int, k: int, dtype: str = "bf16") -> torch.Tensor:
    return (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(DTYPES[dtype])


def _layer(g, k: int, n: int, wbits: int, abits: int, dtype: str, bias: bool = False) -> OrbitLinear:
    config = OrbitQuantConfig(weight_bits=wbits, activation_bits=abits)
    b = (torch.randn(n, generator=g, device="cuda") * 0.02).to(DTYPES[dtype]) if bias else None
    return OrbitLinear.from_weight(_weight(g, n, k), bias=b, config=config)


def _mlp(g, k: int, n: int, wbits: int, abits: int, dtype: str, bias: bool) -> tuple[OrbitLinear, OrbitLinear]:
    up = _layer(g, k, n, wbits, abits, dtype, bias)
    up.fuse_output_activation(torch.nn.functional.gelu, dtype=DTYPES[dtype])
    return up, _layer(g, n, k, wbits, abits, dtype, bias)


def _int8_codes(centroids: torch.Tensor) -> tuple[torch.Tensor, float]:
    """A codebook as the int8 table and scale that the W4A4 entry point takes."""
    scale = float(centroids.abs().max()) / 127
    return torch.round(centroids / scale).to(torch.int8), scale


def prepare(case: dict, seed: int) -> dict:
    g, c = _generator(seed), dict(case)
    kind = c["kind"]
    state = {"case": c}
    if kind == "linear":
        state["layer"] = _layer(g, c["k"], c["n"], c["wbits"], c["abits"], c["dtype"], c["bias"])
        state["x"] = _tokens(g, c["m"], c["k"], c["dtype"], c["outliers"])
    elif kind == "mlp":
        state["up"], state["down"] = _mlp(g, c["k"], c["n"], c["wbits"], c["abits"], c["dtype"], True)
        state["x"] = _tokens(g, c["m"], c["k"], c["dtype"], c["outliers"])
    elif kind == "block":
        h, kv = c["hidden"], c["kv"]
        if c["fused"]:
            state["qkv"] = _layer(g, h, h + 2 * kv, c["wqk"], c["abits"], c["dtype"], True)
        else:
            state["qkv"] = OrbitLinearGroup(_layer(g, h, h, c["wqk"], c["abits"], c["dtype"]), _layer(g, h, kv, c["wqk"], c["abits"], c["dtype"]),
                                            _layer(g, h, kv, c["wvo"], c["abits"], c["dtype"]))
        state["out"] = _layer(g, h, h, c["wvo"], c["abits"], c["dtype"], c["fused"])
        state["up"], state["down"] = _mlp(g, h, c["ffn"], c["wmlp"], c["abits"], c["dtype"], c["fused"])
        for name in ("attention_input", "attention_output", "mlp_input"):
            state[name] = _tokens(g, c["m"], h, c["dtype"], c["outliers"])
        if c["graph"]:
            _capture(state)
    elif kind == "adaln":
        state["layer"] = RTNInt4Linear.from_weight(_weight(g, c["n"], c["k"]), bias=torch.randn(c["n"], generator=g, device="cuda").to(torch.bfloat16),
                                                   config=OrbitQuantConfig(adaln_group_size=ADALN_GROUP))
        state["x"] = torch.nn.functional.silu(_tokens(g, c["m"], c["k"], "bf16"))
    elif kind == "native":
        layer = _layer(g, c["k"], c["n"], 4, 4, c["dtype"])
        state["x"] = _tokens(g, c["m"], c["k"], c["dtype"], c["outliers"])
        codes, scale = _int8_codes(layer._activation_codebook_centroids)   # (both sides are four bits wide: one codebook)
        state.update(layer=layer, codes=codes, scale=scale)
    elif kind == "values":
        state["layer"] = _layer(g, c["k"], c["n"], c["wbits"], 4, c["dtype"], c["bias"])
        state["x"] = _tokens(g, c["m"], c["k"], c["dtype"])
    else:
        state["weight"] = _weight(g, c["n"], c["k"], c["dtype"])
        state["config"] = OrbitQuantConfig(weight_bits=c["wbits"])
        get_rpbh_rotation(c["k"], 0, "paper")      # the constants of a width are made once in a program
        get_codebook(c["k"], c["wbits"]), get_codebook(c["k"], 4)
    return state


def _capture(state: dict) -> None:
    """The pass as a HIP graph on the state's own inputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            _block(state)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = _block(state)
    state["graph"], state["graph_outputs"] = graph, outputs


# ---------------------------------------------------------------- one pass

def _block(state: dict) -> dict:
    qkv = state["qkv"](state["attention_input"])
    out = state["out"](state["attention_output"])
    return {"qkv": qkv, "out": out, "mlp": state["down"](state["up"](state["mlp_input"]))}


def run(state: dict):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear" or kind == "adaln":
        return state["layer"](state["x"])
    if kind == "mlp":
        return state["down"](state["up"](state["x"]))
    if kind == "block":
        if c["graph"]:
            state["graph"].replay()
            return state["graph_outputs"]
        return _block(state)
    if kind == "native":
        layer = state["layer"]
        packed, norms = native_package.quantize_activations_packed_w4(
            state["x"], layer._rotation_permutation, layer._rotation_signs, layer._activation_codebook_boundaries, eps=1e-10,
            inv_sqrt_block=layer.rotation.normalization, block_size=layer.rotation.block_size)
        out = native_package.matmul_packed_w4a4_int8(
            packed, layer.packed_weight_indices, norms, layer.row_norms, state["codes"], state["codes"], activation_scale=state["scale"],
            weight_scale=state["scale"], out_features=c["n"], in_features=c["k"], output_dtype=state["x"].dtype)
        return {"packed": packed, "norms": norms, "out": out}
    if kind == "values":
        layer = state["layer"]
        return native_package.matmul_packed_weight(state["x"], layer.packed_weight_indices, layer.row_norms, layer._weight_codebook_centroids,
                                                   bits=c["wbits"], out_features=c["n"], in_features=c["k"], bias=layer.bias)
    layer = OrbitLinear.from_weight(state["weight"], bias=None, config=state["config"])
    dense = ops.dequantize_packed_weight(layer.packed_weight_indices, layer.row_norms, layer._weight_codebook_centroids, bits=c["wbits"],
                                         out_features=c["n"], in_features=c["k"], dtype=state["weight"].dtype)
    return {"packed": layer.packed_weight_indices, "row_norms": layer.row_norms, "dense": dense}


# ---------------------------------------------------------------- what a pass costs and how exact it is

def _element(dtype: str) -> int:
    return 4 if dtype == "fp32" else 2


def _matrix_bytes(k: int, n: int, bits: int) -> int:
    return (n * k * bits + 7) // 8 + 2 * n


def work(case: dict) -> dict:
    c = case
    kind = c["kind"]
    if kind == "convert":
        e = _element(c["dtype"])
        return {"bytes": 2 * c["n"] * c["k"] * e + _matrix_bytes(c["k"], c["n"], c["wbits"]), "flops": c["n"] * c["k"] * math.log2(c["k"] & -c["k"])}
    if kind == "block":
        h, kv, f, m = c["hidden"], c["kv"], c["ffn"], c["m"]
        matrices = [(h, h, c["wqk"]), (h, kv, c["wqk"]), (h, kv, c["wvo"]), (h, h, c["wvo"]), (h, f, c["wmlp"]), (f, h, c["wmlp"])]
        tokens = m * (3 * h + (h + 2 * kv) + h + h) * _element(c["dtype"])
    elif kind == "mlp":
        matrices = [(c["k"], c["n"], c["wbits"]), (c["n"], c["k"], c["wbits"])]
        tokens = 2 * c["m"] * c["k"] * _element(c["dtype"])
    elif kind == "adaln":
        groups = -(-c["k"] // ADALN_GROUP)
        return {"bytes": c["n"] * groups * (ADALN_GROUP // 2 + 2) + 2 * c["n"] + 2 * c["m"] * (c["k"] + c["n"]), "flops": 2 * c["m"] * c["n"] * c["k"]}
    else:
        matrices = [(c["k"], c["n"], c.get("wbits", 4))]
        tokens = c["m"] * (c["k"] + c["n"]) * _element(c["dtype"])
        if kind == "native":   # the codes and norms are results too
            tokens += c["m"] * (c["k"] // 2 + 4)
    return {"bytes": tokens + sum(_matrix_bytes(k, n, b) for k, n, b in matrices), "flops": sum(2 * c["m"] * n * k for k, n, _ in matrices)}


def tolerance(case: dict):
    """Measured as the difference between two summation orders of the same operands (other tiles, another split of K),
    times four.  A pass without a second quantization differs by the sums' last bits and by the 16-bit outputs these
    move across a rounding midpoint.  Behind such an output a second quantizer (mlp, block) may take the
    neighbouring code, one step of a three- or four-bit codebook.  Codes, indices and conversions are exact."""
    kind = case["kind"]
    if kind == "convert":
        return "exact"
    if kind in ("mlp", "block"):
        return {"rel": 1e-2, "max": 0.3}
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 4e-4, "max": 0.03}


# ---------------------------------------------------------------- the same in 64 bits

def _indices(packed: torch.Tensor, bits: int, n: int, k: int) -> torch.Tensor:
    """The indices of a packed weight: one little-endian bit stream over the matrix in row-major order."""
    shifts = torch.arange(8, device=packed.device, dtype=torch.uint8)
    stream = ((packed.flatten()[:, None] >> shifts) & 1).flatten()[: n * k * bits].view(n * k, bits)
    index = torch.zeros(n * k, dtype=torch.int64, device=packed.device)
    for b in range(bits):
        index += stream[:, b].to(torch.int64) << b
    return index.view(n, k)


def _weight64(layer, table: torch.Tensor) -> torch.Tensor:
    """The matrix that a packed weight stands for, `table[index] * row norm`."""
    index = _indices(layer.packed_weight_indices, layer.weight_bits, layer.out_features, layer.in_features)
    return table.double()[index] * layer.row_norms.double()[:, None]


def _quantized64(x: torch.Tensor, layer, table: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(codes, what they stand for, norms) of the tokens: unit norm, permute, sign, Hadamard blocks, nearest centroid."""
    x = x.double()
    norm = x.square().sum(-1, keepdim=True).sqrt()
    y = (x / (norm + layer.activation_eps))[:, layer.rotation.permutation.to(x.device)] * layer.rotation.signs.to(x.device, torch.float64)
    h = layer.rotation.block_size
    y = y.reshape(-1, h)
    distance = 1
    while distance < h:
        pairs = y.view(-1, h // (2 * distance), 2, distance)
        y = torch.stack((pairs[:, :, 0] + pairs[:, :, 1], pairs[:, :, 0] - pairs[:, :, 1]), dim=2).view(-1, h)
        distance *= 2
    codes = torch.bucketize((y / math.sqrt(h)).view(x.shape), layer._activation_codebook_boundaries.double())
    return codes, table.double()[codes] * norm, norm.squeeze(-1)


def _linear64(x: torch.Tensor, layer) -> torch.Tensor:
    y = _quantized64(x, layer, layer._activation_codebook_centroids)[1] @ _weight64(layer, layer._weight_codebook_centroids).T
    return y if layer.bias is None else y + layer.bias.double()


def _mlp64(x: torch.Tensor, up, down) -> torch.Tensor:
    """The MLP; what one layer hands to the next has the tokens' type."""
    h = torch.nn.functional.gelu(_linear64(x, up).to(x.dtype))
    return _linear64(h, down)


def exact(case: dict, seed: int):
    """What `run` returns, in 64 bits, from the packed weights and codebooks that the layers hold."""
    kind, s = case["kind"], prepare({**case, "graph": False}, seed)
    if kind == "linear":
        return _linear64(s["x"], s["layer"])
    if kind == "mlp":
        return _mlp64(s["x"], s["up"], s["down"])
    if kind == "block":
        linears = getattr(s["qkv"], "linears", None)
        qkv = _linear64(s["attention_input"], s["qkv"]) if linears is None else tuple(_linear64(s["attention_input"], l) for l in linears)
        return {"qkv": qkv, "out": _linear64(s["attention_output"], s["out"]), "mlp": _mlp64(s["mlp_input"], s["up"], s["down"])}
    if kind == "adaln":
        l = s["layer"]
        padded = l.num_groups * l.group_size
        w = (_indices(l.packed_weight, 4, l.out_features, padded) - 8).double() * l.scales.double().repeat_interleave(l.group_size, dim=1)
        return s["x"].double() @ w[:, : l.in_features].T + l.bias.double()
    if kind == "native":
        table = s["codes"].double() * s["scale"]
        _, values, norms = _quantized64(s["x"], s["layer"], table)
        return {"packed": None, "norms": norms, "out": values @ _weight64(s["layer"], table).T}
    if kind == "values":
        l = s["layer"]
        y = s["x"].double() @ _weight64(l, l._weight_codebook_centroids).T
        return y if l.bias is None else y + l.bias.double()
    return None   # (indices and a table lookup: compared bit for bit)
