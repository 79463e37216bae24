"""Performance cases of the W4A16 framework: what a serving engine has it do.

Every case goes through the layer interface an engine calls.  Four kinds:

* ``step``: two consecutive decoder layers' linear work (norm + QKV, q/k norm, O, norm +
  gate_up + SiLU * up, down) captured in a HIP graph as engines capture their decode and
  verify steps, one replay per pass.  Attention itself is not part of the framework: its
  output is an input here.  Two layers are 200 MB of weights, so replays over a few states
  stream them from HBM.
* ``linear``: one projection called eagerly.
* ``mlp``: the eager prefill block: norm + gate_up + SiLU * up in one call, then down.
* ``quantize`` / ``load``: the producer of the AWQ tensors and their preparation at model
  load.

Layer shapes are those of the tests and the benchmark (hidden size, QKV width, intermediate
size); ``q8`` is the benchmark's.
"""
import importlib
import math

import torch
from torch import nn

pkg = importlib.import_module("llm-serve_amd")
linear = importlib.import_module("llm-serve_amd.layers.linear")
layernorm = importlib.import_module("llm-serve_amd.layers.layernorm")
awq = importlib.import_module("llm-serve_amd.layers.quantization.awq")
calibration = importlib.import_module("llm-serve_amd.quantization.awq_calibration")

GROUP = 128
HEAD = 128
EPS = 1e-6
STEP_LAYERS = 2
# hidden size, query heads, kv heads, intermediate size
MODELS = {"q8": (4096, 32, 8, 12288), "q14": (5120, 40, 8, 17408), "q4": (2560, 32, 8, 9728)}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SHIFTS = (0, 16, 4, 20, 8, 24, 12, 28)  # bit offset of logical column c of an AutoAWQ word


def listed():
    return [
        # one token through one projection, called eagerly: the smallest call there is
        {"name": "o_eager_m1", "kind": "linear", "model": "q8", "proj": "o", "m": 1, "epilogue": "plain"},
        # a single user's decode step
        {"name": "step_m1", "kind": "step", "model": "q8", "m": 1},
        # a few users: the norms split across the projections around them
        {"name": "step_m4", "kind": "step", "model": "q8", "m": 4},
        # an ordinary decode batch
        {"name": "step_m16", "kind": "step", "model": "q8", "m": 16},
        # a full decode batch
        {"name": "step_m64", "kind": "step", "model": "q8", "m": 64},
        # speculative verification of a batch, a ragged number of rows
        {"name": "step_m150", "kind": "step", "model": "q8", "m": 150},
        # a mixed batch: decode tokens, verify rows and a short prefill chunk
        {"name": "mixed_mlp_m497", "kind": "mlp", "model": "q8", "m": 497},
        # an odd-sized prompt's norm + QKV
        {"name": "prefill_qkv_m1331", "kind": "linear", "model": "q8", "proj": "qkv", "m": 1331, "epilogue": "norm"},
        # a chunked-prefill chunk
        {"name": "prefill_mlp_m2048", "kind": "mlp", "model": "q8", "m": 2048},
        # half of the engine's largest packed batch
        {"name": "prefill_mlp_m8192", "kind": "mlp", "model": "q8", "m": 8192},
        # producing a checkpoint: the largest projection quantized
        {"name": "quantize_gate_up", "kind": "quantize", "model": "q8", "proj": "gate_up", "dtype": "bf16", "group": 128},
        # loading a checkpoint: the largest projection prepared for the kernels
        {"name": "load_gate_up", "kind": "load", "model": "q8", "proj": "gate_up"},
    ]


def shape(case):
    """(K, N) of the case's projection."""
    hidden, heads, kv, inter = MODELS[case["model"]]
    return {"qkv": (hidden, (heads + 2 * kv) * HEAD), "o": (heads * HEAD, hidden),
            "gate_up": (hidden, 2 * inter), "down": (inter, hidden)}[case["proj"]]


def draw(rng):
    def rows(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["step", "step", "linear", "linear", "mlp", "mlp", "quantize", "load"])
    if kind == "step":
        return {"kind": kind, "model": "q8", "m": rows(1, 512)}
    if kind == "linear":
        proj = rng.choice(["qkv", "o", "gate_up", "down"])
        epilogue = {"qkv": ["plain", "norm"], "o": ["plain", "residual"], "gate_up": ["silu", "norm_silu"],
                    "down": ["plain", "residual"]}[proj]
        return {"kind": kind, "model": rng.choice(["q8", "q8", "q14", "q4"]), "proj": proj, "m": rows(1, 4096),
                "epilogue": rng.choice(epilogue)}
    if kind == "mlp":
        return {"kind": kind, "model": rng.choice(["q8", "q8", "q14", "q4"]), "m": rows(192, 4096)}
    proj = rng.choice(["qkv", "o", "gate_up", "down"])
    case = {"kind": kind, "model": rng.choice(["q8", "q14", "q4"]), "proj": proj}
    if kind == "quantize":
        case["dtype"] = rng.choice(["bf16", "f16", "f32"])
        case["group"] = rng.choice([128, 128, 64, 32])
    return case


# ------------------------------------------------------------------- inputs
def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def awq_tensors(gen, k, n):
    """AutoAWQ tensors as a quantizer leaves them: normally distributed weights around a
    zero point near the middle of the range, scales spread over a factor of ten."""
    q = (torch.randn(k, n // 8, 8, generator=gen, device="cuda") * 2.7 + 7.5).round_().clamp_(0, 15).to(torch.int32)
    z = (torch.randn(k // GROUP, n // 8, 8, generator=gen, device="cuda") + 7.5).round_().clamp_(0, 15).to(torch.int32)

    def pack(v):
        out = torch.zeros(v.shape[:2], dtype=torch.int32, device="cuda")
        for c in range(8):
            out |= v[:, :, c] << SHIFTS[c]
        return out

    s = torch.empty(k // GROUP, n, device="cuda").uniform_(0.002, 0.02, generator=gen).to(torch.bfloat16)
    return pack(q), pack(z), s


def activations(gen, m, k):
    """Normal activations with one input channel in a hundred 20 times as large."""
    x = torch.randn(m, k, generator=gen, device="cuda")
    x[:, torch.randperm(k, generator=gen, device="cuda")[: k // 100]] *= 20
    return x.to(torch.bfloat16)


def norm_weight(gen, k):
    return (1 + 0.1 * torch.randn(k, generator=gen, device="cuda")).to(torch.bfloat16)


def config():
    return awq.AWQRuntimeConfig(bits=4, group_size=GROUP, zero_point=True, version="gemm", backend="autoawq",
                                activation_dtype=torch.bfloat16)


def projection(gen, model, proj):
    """A layer of the engine's model, its weights loaded and processed."""
    hidden, heads, kv, inter = MODELS[model]
    cfg = config()
    with torch.device("cuda"):
        if proj == "qkv":
            layer = linear.QKVParallelLinear(hidden, HEAD, heads, kv, quant_config=cfg)
        elif proj == "o":
            layer = linear.RowParallelLinear(heads * HEAD, hidden, quant_config=cfg)
        elif proj == "gate_up":
            layer = linear.MergedColumnParallelLinear(hidden, [inter, inter], quant_config=cfg)
        else:
            layer = linear.RowParallelLinear(inter, hidden, quant_config=cfg)
    k, n = shape({"model": model, "proj": proj})
    for param, value in zip((layer.qweight, layer.qzeros, layer.scales), awq_tensors(gen, k, n)):
        param.data.copy_(value)
    layer.quant_method.process_weights_after_loading(layer)
    return layer


def norm_layer(gen, k):
    with torch.device("cuda"):
        norm = layernorm.RMSNorm(k, EPS)
    norm.weight.data.copy_(norm_weight(gen, k))
    return norm


# --------------------------------------------------------------------- step
def split_norms(m):
    """Batches whose norms an engine splits across the projections around them."""
    return 2 <= m <= 4


def step_state(case, seed):
    gen = generator(seed)
    hidden, heads, kv, _ = MODELS[case["model"]]
    m = case["m"]
    layers = []
    for _ in range(STEP_LAYERS):
        layers.append({
            "qkv": projection(gen, case["model"], "qkv"), "o": projection(gen, case["model"], "o"),
            "gate_up": projection(gen, case["model"], "gate_up"), "down": projection(gen, case["model"], "down"),
            "norm1": norm_layer(gen, hidden), "norm2": norm_layer(gen, hidden),
            "q_norm": norm_layer(gen, HEAD), "k_norm": norm_layer(gen, HEAD),
            "attn": activations(gen, m, heads * HEAD)})
    state = {"case": case, "layers": layers, "h": activations(gen, m, hidden), "residual": activations(gen, m, hidden)}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step_forward(state)
    torch.cuda.current_stream().wait_stream(side)
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        state["out"] = step_forward(state)
    return state


def step_forward(state):
    hidden, heads, kv, _ = MODELS[state["case"]["model"]]
    m = state["case"]["m"]
    split = split_norms(m)
    h, residual, inp = state["h"], state["residual"], None
    outs = []
    for layer in state["layers"]:
        if inp is None:
            qkv, residual = layer["qkv"].forward_rmsnorm(layer["norm1"], h, residual)
        else:
            qkv = layer["qkv"].forward_rmsnorm_stats(layer["norm1"], inp)
        q, k, _ = qkv.split([heads * HEAD, kv * HEAD, kv * HEAD], dim=-1)
        q = layer["q_norm"](q.view(-1, heads, HEAD))
        k = layer["k_norm"](k.view(-1, kv, HEAD))
        if split:
            inp, residual = layer["o"].forward_residual_stats(layer["attn"], residual)
            act = layer["gate_up"].forward_rmsnorm_stats_silu_and_mul(layer["norm2"], inp)
            inp, residual = layer["down"].forward_residual_stats(act, residual)
            h = inp.s
        else:
            o = layer["o"](layer["attn"])
            act, residual = layer["gate_up"].forward_rmsnorm_silu_and_mul(layer["norm2"], o, residual)
            h = layer["down"](act)
        outs.append({"qkv": qkv, "q": q, "k": k, "act": act, "h": h, "residual": residual})
    return outs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return step_state(case, seed)
    gen = generator(seed)
    model = case["model"]
    hidden = MODELS[model][0]
    state = {"case": case}
    if kind == "mlp":
        state["gate_up"] = projection(gen, model, "gate_up")
        state["down"] = projection(gen, model, "down")
        state["norm"] = norm_layer(gen, hidden)
        state["x"] = activations(gen, case["m"], hidden)
        state["residual"] = activations(gen, case["m"], hidden)
        return state
    k, n = shape(case)
    if kind == "linear":
        state["layer"] = projection(gen, model, case["proj"])
        state["x"] = activations(gen, case["m"], k)
        if case["epilogue"] == "residual":
            state["residual"] = activations(gen, case["m"], n)
        if case["epilogue"].startswith("norm"):
            state["norm"] = norm_layer(gen, k)
            state["residual"] = activations(gen, case["m"], k)
    elif kind == "quantize":
        state["weight"] = (torch.randn(n, k, generator=gen, device="cuda") * 0.02).to(DTYPES[case["dtype"]])
    else:
        state["tensors"] = awq_tensors(gen, k, n)
        state["method"] = awq.AWQLinearMethod(config())
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["out"]
    if kind == "mlp":
        act, residual = state["gate_up"].forward_rmsnorm_silu_and_mul(state["norm"], state["x"], state["residual"])
        return {"act": act, "residual": residual, "h": state["down"](act)}
    if kind == "linear":
        layer, x = state["layer"], state["x"]
        if case["epilogue"] == "plain":
            return {"y": layer(x)}
        if case["epilogue"] == "residual":
            return {"y": layer.forward_residual(x, state["residual"])}
        if case["epilogue"] == "silu":
            return {"y": layer.forward_silu_and_mul(x)}
        forward = layer.forward_rmsnorm if case["epilogue"] == "norm" else layer.forward_rmsnorm_silu_and_mul
        y, residual = forward(state["norm"], x, state["residual"])
        return {"y": y, "residual": residual}
    if kind == "quantize":
        packed = calibration.quantize_awq_weight(state["weight"], case["group"])
        return {"qweight": packed.qweight, "qzeros": packed.qzeros, "scales": packed.scales}
    layer = nn.Module()
    for name, value in zip(("qweight", "qzeros", "scales"), state["tensors"]):
        setattr(layer, name, nn.Parameter(value, requires_grad=False))
    state["method"].process_weights_after_loading(layer)
    return {"qweight": layer.awq_qweight, "qzeros": layer.awq_qzeros}


# --------------------------------------------------------------------- work
def weight_bytes(k, n):
    return k * n / 2 + k * n / (2 * GROUP) + 2 * k * n / GROUP


def work(case):
    kind = case["kind"]
    hidden, heads, kv, inter = MODELS[case["model"]]
    if kind in ("step", "mlp"):
        m = case["m"]
        projs = [(hidden, 2 * inter), (inter, hidden)]
        # x, residual, new residual, act written and read, h
        act = m * (3 * hidden + 2 * inter + hidden) * 2
        if kind == "step":
            qkv = (heads + 2 * kv) * HEAD
            projs += [(hidden, qkv), (heads * HEAD, hidden)]
            # norm + QKV (x, residual, new residual, qkv); q and k read and written; O
            act += m * (3 * hidden + qkv + 2 * (heads + kv) * HEAD + heads * HEAD + hidden) * 2
        times = STEP_LAYERS if kind == "step" else 1
        return {"bytes": times * (act + sum(weight_bytes(k, n) for k, n in projs)),
                "flops": times * sum(2 * m * k * n for k, n in projs)}
    k, n = shape(case)
    if kind == "linear":
        m = case["m"]
        n_out = n // 2 if case["epilogue"] in ("silu", "norm_silu") else n
        extra = {"residual": m * n, "norm": 2 * m * k, "norm_silu": 2 * m * k}.get(case["epilogue"], 0)
        return {"bytes": weight_bytes(k, n) + 2 * (m * k + m * n_out + extra), "flops": 2 * m * k * n}
    if kind == "quantize":
        size = 4 if case["dtype"] == "f32" else 2
        groups = k // case["group"]
        return {"bytes": k * n * size + k * n / 2 + groups * n / 2 + groups * n * size, "flops": 0}
    return {"bytes": k * n, "flops": 0}


def tolerance(case):
    if case["kind"] in ("quantize", "load"):
        return "exact"
    # A projection's bf16 result lies 1.7e-3 (one rounding) from its 64-bit value, the chained
    # ones (act, h, the second layer) up to 5e-3.
    return {"rel": 2e-2 if case["kind"] == "step" else 1e-2}


# -------------------------------------------------------------------- exact
def unpack64(packed):
    shifts = torch.tensor(SHIFTS, dtype=torch.int32, device=packed.device)
    return ((packed.unsqueeze(-1) >> shifts) & 15).flatten(1)


def weight64(tensors):
    """The bf16 weight an AutoAWQ checkpoint stands for, in 64 bits."""
    qweight, qzeros, scales = tensors
    q = unpack64(qweight)
    z = unpack64(qzeros).repeat_interleave(GROUP, 0)
    w = (q - z).float() * scales.float().repeat_interleave(GROUP, 0)
    return w.to(torch.bfloat16).double()


def rms64(s, weight):
    return s * torch.rsqrt(s.square().mean(-1, keepdim=True) + EPS) * weight.double()


def silu64(gate_up):
    g, u = gate_up.chunk(2, -1)
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    kind = case["kind"]
    if kind == "load":
        return None
    gen = generator(seed)
    hidden, heads, kv, inter = MODELS[case["model"]]
    if kind == "quantize":
        k, n = shape(case)
        weight = (torch.randn(n, k, generator=gen, device="cuda") * 0.02).to(DTYPES[case["dtype"]]).double()
        groups = weight.view(n, -1, case["group"])
        scales = (groups.amax(-1) - groups.amin(-1)).clamp(min=1e-5) / 15
        return {"qweight": None, "qzeros": None, "scales": scales.t().contiguous()}

    def tensors(proj):
        return awq_tensors(gen, *shape({"model": case["model"], "proj": proj}))

    # the tensors are drawn in prepare()'s order
    if kind == "step":
        m = case["m"]
        drawn = []
        for _ in range(STEP_LAYERS):
            layer = {p: tensors(p) for p in ("qkv", "o", "gate_up", "down")}
            layer.update(norm1=norm_weight(gen, hidden), norm2=norm_weight(gen, hidden), q_norm=norm_weight(gen, HEAD),
                         k_norm=norm_weight(gen, HEAD), attn=activations(gen, m, heads * HEAD).double())
            drawn.append(layer)
        h, residual = activations(gen, m, hidden).double(), activations(gen, m, hidden).double()
        split = split_norms(m)
        outs = []
        for layer in drawn:
            if not split or not outs:
                residual = residual + h
            qkv = rms64(residual, layer["norm1"]) @ weight64(layer["qkv"])
            q, k, _ = qkv.split([heads * HEAD, kv * HEAD, kv * HEAD], dim=-1)
            q = rms64(q.reshape(-1, heads, HEAD), layer["q_norm"])
            k = rms64(k.reshape(-1, kv, HEAD), layer["k_norm"])
            residual = residual + layer["attn"] @ weight64(layer["o"])
            act = silu64(rms64(residual, layer["norm2"]) @ weight64(layer["gate_up"]))
            h = act @ weight64(layer["down"])
            if split:
                residual = residual + h
            outs.append({"qkv": qkv, "q": q, "k": k, "act": act, "h": residual if split else h, "residual": residual})
        return outs
    if kind == "mlp":
        gate_up, down = tensors("gate_up"), tensors("down")
        weight = norm_weight(gen, hidden)
        x = activations(gen, case["m"], hidden).double()
        s = x + activations(gen, case["m"], hidden).double()
        act = silu64(rms64(s, weight) @ weight64(gate_up))
        return {"act": act, "residual": s, "h": act @ weight64(down)}
    k, n = shape(case)
    packed = tensors(case["proj"])
    x = activations(gen, case["m"], k).double()
    w = weight64(packed)
    if case["epilogue"] == "plain":
        return {"y": x @ w}
    if case["epilogue"] == "residual":
        return {"y": x @ w + activations(gen, case["m"], n).double()}
    if case["epilogue"] == "silu":
        return {"y": silu64(x @ w)}
    weight = norm_weight(gen, k)
    s = x + activations(gen, case["m"], k).double()
    y = rms64(s, weight) @ w
    return {"y": y if case["epilogue"] == "norm" else silu64(y), "residual": s}
