"""Performance cases of the quantized-linear path: what a program that uses the package has it do, through
`Bitween.quantize`, `QuantizedLinear` (forward and backward), `quantize_rtn` and `dequantize_rtn`.

A case is a plain dict; `path` says which work it is:

  linear    one QuantizedLinear: K = k, N = n
  mlp       gate, up (hidden -> inter) and down (inter -> hidden) of one decoder MLP
  decoder   q, k, v, o, gate, up, down of `blocks` decoder blocks, one call per module as a model makes them; `attention_bits` / `low_down`
            give the attention another width and the first `low_down` down projections 2 bits at g32, as a per-layer precision map does;
            `siblings`: q/k/v and gate/up share a launch (fuse_sibling_linears); `graph`: the calls replayed as one HIP graph
  quantize  Bitween(...).quantize of a model that is one decoder block of linears
  codec     quantize_rtn of one weight tensor and dequantize_rtn of the result

`rows` is the number of rows of activations (batch x tokens), `dtype` theirs (or the weight tensor's, for quantize and codec);
`backward` adds the gradient with respect to the activations of every call.
"""
import torch
import torch.nn as nn

from bitween_amd import Bitween, QuantizedLinear, dequantize_rtn, fuse_sibling_linears, quantize_rtn

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


def listed():
    return [
        # The smallest call: an OPT-125m fc1 for one token, from eager code.  Latency of one call is all there is.
        {"name": "fc1-one-row", "path": "linear", "k": 768, "n": 3072, "rows": 1, "bits": 4, "group": 128, "dtype": "float16", "bias": True},
        # Odd sizes through forward and backward: a head with an odd number of outputs on a width that is no multiple of 128.
        {"name": "ragged-head-train", "path": "linear", "k": 2880, "n": 3001, "rows": 333, "bits": 4, "group": 64, "dtype": "float16",
         "bias": True, "backward": True},
        # One token through the linears of eight Llama-2-7B blocks (more bytes than the Infinity Cache holds), launches in a HIP graph: the
        # serving loop of the repository's headline benchmark.
        {"name": "token-graph-w4", "path": "decoder", "hidden": 4096, "inter": 11008, "blocks": 8, "rows": 1, "bits": 4, "group": 128,
         "dtype": "float16", "graph": True},
        # The same token from eager code (model.generate) with the mixed precision map: attention W8, MLP W4, one down projection W2.
        {"name": "token-eager-mixed", "path": "decoder", "hidden": 4096, "inter": 11008, "blocks": 4, "rows": 1, "bits": 4, "group": 128,
         "attention_bits": 8, "low_down": 1, "dtype": "float16"},
        # A decode step of 16 sequences, eager.
        {"name": "batch-16-eager", "path": "decoder", "hidden": 4096, "inter": 11008, "blocks": 4, "rows": 16, "bits": 4, "group": 128,
         "dtype": "float16"},
        # A serving batch of 40 sequences in bfloat16, W4 g64, siblings fused, launches in a HIP graph.
        {"name": "batch-40-graph-fused", "path": "decoder", "hidden": 4096, "inter": 11008, "blocks": 4, "rows": 40, "bits": 4, "group": 64,
         "dtype": "bfloat16", "graph": True, "siblings": True},
        # Prefill of Llama-3-8B MLP shapes in bfloat16: a short prompt, and a long one.
        {"name": "prefill-128", "path": "mlp", "hidden": 4096, "inter": 14336, "rows": 128, "bits": 4, "group": 128, "dtype": "bfloat16"},
        {"name": "prefill-2048", "path": "mlp", "hidden": 4096, "inter": 14336, "rows": 2048, "bits": 4, "group": 128, "dtype": "bfloat16"},
        # A prompt of an odd length at the package's default precision, 8 bits in groups of 32.
        {"name": "prefill-509-w8", "path": "mlp", "hidden": 4096, "inter": 11008, "rows": 509, "bits": 8, "group": 32, "dtype": "float16"},
        # Forward and backward of a frozen MLP under adapter training.
        {"name": "train-2048", "path": "mlp", "hidden": 4096, "inter": 14336, "rows": 2048, "bits": 4, "group": 128, "dtype": "float16",
         "backward": True},
        # Quantizing one Llama-2-7B block the way a whole model is quantized.
        {"name": "quantize-block", "path": "quantize", "hidden": 4096, "inter": 11008, "bits": 4, "group": 128, "dtype": "float16"},
        # The functional pair on a float32 master weight, 2 bits g32: quantize and pack, then back to float32.
        {"name": "codec-w2", "path": "codec", "n": 11008, "k": 4096, "bits": 2, "group": 32, "dtype": "float32"},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, uniform over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def _width(rng, lo, hi, unit):
    return max(unit, _log(rng, lo, hi) // unit * unit)


def draw(rng):
    path = rng.choice(["linear"] * 4 + ["mlp"] * 3 + ["decoder"] * 3 + ["quantize", "codec"])
    bits, group = rng.choice([(4, 128), (4, 128), (4, 64), (4, 32), (8, 32), (8, 64), (8, 128), (2, 32), (2, 64), (2, 128)])
    unit = 128 if group == 128 or rng.random() < 0.7 else 64
    case = {"path": path, "bits": bits, "group": group}
    if path == "codec":
        case.update(k=_width(rng, 512, 14336, unit), n=_log(rng, 512, 11008), dtype=rng.choice(["float32", "float16", "bfloat16"]))
    elif path == "quantize":
        case.update(hidden=_width(rng, 512, 4096, unit), inter=_width(rng, 1024, 14336, unit), dtype=rng.choice(["float32", "float16", "bfloat16"]))
    elif path == "linear":
        n = _log(rng, 512, 14336)
        case.update(k=_width(rng, 512, 14336, unit), n=n if rng.random() < 0.3 else max(16, n // 16 * 16), rows=_log(rng, 1, 2048),
                    bias=rng.random() < 0.5, dtype=rng.choice(["float16", "bfloat16"]), backward=rng.random() < 0.3)
    elif path == "mlp":
        case.update(hidden=_width(rng, 512, 4096, unit), inter=_width(rng, 1024, 14336, unit), rows=_log(rng, 16, 2048),
                    dtype=rng.choice(["float16", "bfloat16"]), backward=rng.random() < 0.5)
    else:
        case.update(hidden=_width(rng, 512, 4096, unit), inter=_width(rng, 1024, 11008, unit), blocks=rng.randint(1, 8), rows=_log(rng, 1, 64),
                    dtype=rng.choice(["float16", "bfloat16"]), graph=rng.random() < 0.5, siblings=rng.random() < 0.4)
    return case


class _MLP(nn.Module):
    def __init__(self, hidden, inter, **kw):
        super().__init__()
        self.gate_proj = nn.Linear(hidden, inter, bias=False, **kw)
        self.up_proj = nn.Linear(hidden, inter, bias=False, **kw)
        self.down_proj = nn.Linear(inter, hidden, bias=False, **kw)

    def calls(self, x):
        """(module, its input) of one pass: x["hidden"] stands for the normalised block input, x["inter"] for the activation's output."""
        return [(self.gate_proj, x["hidden"]), (self.up_proj, x["hidden"]), (self.down_proj, x["inter"])]


class _Block(nn.Module):
    def __init__(self, hidden, inter, **kw):
        super().__init__()
        self.q_proj = nn.Linear(hidden, hidden, bias=False, **kw)
        self.k_proj = nn.Linear(hidden, hidden, bias=False, **kw)
        self.v_proj = nn.Linear(hidden, hidden, bias=False, **kw)
        self.o_proj = nn.Linear(hidden, hidden, bias=False, **kw)
        self.mlp = _MLP(hidden, inter, **kw)

    def calls(self, x):
        attention = [(p, x["hidden"]) for p in (self.q_proj, self.k_proj, self.v_proj)] + [(self.o_proj, x["attention"])]
        return attention + self.mlp.calls(x)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _init(model, gen):
    """Weights N(0, 0.02) with one in a thousand ten times larger."""
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() > 1:
                p.normal_(0, 0.02, generator=gen)
                p[:, ::1000] *= 10
            else:
                p.normal_(0, 0.1, generator=gen)
    return model


def _forward(calls):
    return [module(x) for module, x in calls]


def prepare(case, seed):
    gen = _generator(seed)
    path, bits, group, dtype = case["path"], case["bits"], case["group"], DTYPES[case["dtype"]]
    state = {"path": path}
    if path == "codec":
        w = torch.empty(case["n"], case["k"], device="cuda", dtype=dtype)
        state.update(weight=w.normal_(0, 0.02, generator=gen), bits=bits, group=group)
        return state
    if path == "quantize":
        model = _init(_Block(case["hidden"], case["inter"], device="cuda", dtype=dtype), gen)
        state.update(model=model, quantizer=Bitween(model, bits=bits, group_size=group))
        return state

    def activations(width):
        return torch.randn(1, case["rows"], width, device="cuda", generator=gen).to(dtype)

    if path == "linear":
        layer = _init(nn.Linear(case["k"], case["n"], bias=case["bias"], device="cuda", dtype=torch.float16), gen)
        calls = [(QuantizedLinear.from_float(layer, bits, group), activations(case["k"]))]
    else:
        make, count = (_MLP, 1) if path == "mlp" else (_Block, case["blocks"])
        model = nn.ModuleList([_init(make(case["hidden"], case["inter"], device="cuda", dtype=torch.float16), gen) for _ in range(count)])
        precision = {}
        for i in range(count):
            if case.get("attention_bits"):
                precision.update({"%d.%s_proj" % (i, p): (case["attention_bits"], group) for p in "qkvo"})
            if i < case.get("low_down", 0):
                precision["%d.mlp.down_proj" % i] = (2, 32)
        model = Bitween(model, bits=bits, group_size=group).quantize(rtn=True, verbose=False, layer_config=precision)
        if case.get("siblings"):
            fuse_sibling_linears(model)
        inputs = {"hidden": activations(case["hidden"]), "inter": activations(case["inter"])}
        if path == "decoder":
            inputs["attention"] = activations(case["hidden"])
        calls = [call for block in model for call in block.calls(inputs)]
        state["model"] = model
    state["calls"] = calls
    if case.get("backward"):
        for _, x in calls:
            x.requires_grad_(True)
        state["grads"] = [torch.randn(1, case["rows"], m.out_features, device="cuda", generator=gen).to(torch.float16) for m, _ in calls]
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.no_grad():
            _forward(calls)                                # every launch path is warm before the capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]), torch.no_grad():
            state["outputs"] = _forward(calls)
    return state


def run(state):
    path = state["path"]
    if path == "codec":
        q, scale, zero, group = quantize_rtn(state["weight"], state["bits"], state["group"])
        return [q, scale, zero, dequantize_rtn(q, scale, zero, group, state["bits"])]
    if path == "quantize":
        model = state["quantizer"].quantize(rtn=True, verbose=False)
        return [t for m in model.modules() if isinstance(m, QuantizedLinear) for t in (m.qweight, m.scale, m.zero_point)]
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if "grads" in state:
        out = []
        for (module, x), grad in zip(state["calls"], state["grads"]):
            y = module(x)
            out += [y.detach(), torch.autograd.grad(y, x, grad)[0]]
        return out
    with torch.no_grad():
        return _forward(state["calls"])


def _shapes(case):
    """(K, N, bits, group) of every linear of a pass."""
    bits, group = case["bits"], case["group"]
    if case["path"] in ("linear", "codec"):
        return [(case["k"], case["n"], bits, group)]
    hidden, inter = case["hidden"], case["inter"]
    shapes = []
    for i in range(case.get("blocks", 1)):
        if case["path"] != "mlp":
            shapes += [(hidden, hidden, case.get("attention_bits") or bits, group)] * 4
        shapes += [(hidden, inter, bits, group)] * 2
        shapes.append((inter, hidden, 2, 32) if i < case.get("low_down", 0) else (inter, hidden, bits, group))
    return shapes


def work(case):
    """Packed weights, scales and zero points (float16), activations and gradients read once, outputs written once; 2 K N flops a row."""
    size = DTYPES[case["dtype"]].itemsize
    total, flops = 0, 0
    for k, n, bits, group in _shapes(case):
        packed, groups = n * k * bits // 8, n * (k // group)
        if case["path"] == "quantize":
            total += n * k * size + packed + groups * 4
        elif case["path"] == "codec":
            total += n * k * size + 2 * (packed + groups * (size + 4)) + n * k * 4
        else:
            rows, passes = case["rows"], 2 if case.get("backward") else 1
            total += passes * (packed + groups * 4) + rows * k * size * passes + rows * n * 2 * passes + (2 * n if case.get("bias") else 0)
            flops += passes * 2 * rows * n * k
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Packed integers, scales and reconstructed weights are exact.  Products accumulate in float32 and round once to float16 (2^-12 of a
    value on average); whether the group's scale multiplies the weight (rounded to float16) or the partial sum is the implementation's
    choice and costs about as much again.  A gradient handed back to bfloat16 activations is rounded to bfloat16."""
    if case["path"] in ("quantize", "codec"):
        return "exact"
    return {"rel": 1e-2 if case.get("backward") and case["dtype"] == "bfloat16" else 1e-3}
