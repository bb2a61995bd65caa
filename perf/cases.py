"""Performance cases of the AWQ W4A16 engine: what a serving program has it do.

Four kinds of work, each through the layer objects that a model is built of:

  linear  one row-parallel projection called eagerly: the smallest call, where
          launch latency and the host path count
  decode  the AWQ linears of a stack of decoder layers (fused qkv with or
          without bias, o, gated MLP) at decode batch sizes, captured in one
          graph as a serving program runs its decode step; the stack's weights
          are larger than the Infinity Cache, so they come from HBM
  prefill the same linears of one layer, called eagerly on a prompt chunk
  moe     whole expert blocks (routing, alignment, grouped GEMMs, combine) of
          AWQ experts: a stack of blocks in one graph at decode batch sizes,
          one block called eagerly on longer chunks

Weights follow the distributions of the engine's benchmark: uniform nibbles,
uniform zero points, scales uniform in [0.002, 0.02]; activations N(0, 1);
router logits N(0, 1) in the activation dtype, as a router linear gives them.
"""

import math

import torch

from sglite_amd.linear import QKVParallelLinear, RowParallelLinear
from sglite_amd.mlp import GatedMLP
from sglite_amd.moe import AWQMoELayer
from sglite_amd.quantization import get_quantization_config

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
AWQ_ORDER = (0, 4, 1, 5, 2, 6, 3, 7)  # nibble of column 8j + i in word j

# Largest batch that a serving program captures; longer inputs run eagerly.
GRAPH_MAX = 160


def _dense(name, kind, dims, M, layers, dtype="fp16", group=128, bias=False):
    hidden, qkv, attn, inter = dims
    return {"name": name, "kind": kind, "hidden": hidden, "qkv": qkv, "attn": attn, "inter": inter, "M": M,
            "layers": layers, "dtype": dtype, "group": group, "bias": bias}


def _moe(name, E, top_k, hidden, inter, T, layers, dtype="fp16", group=128):
    return {"name": name, "kind": "moe", "E": E, "top_k": top_k, "hidden": hidden, "inter": inter, "M": T,
            "layers": layers, "dtype": dtype, "group": group}


# (hidden, qkv columns, attention width, intermediate): Qwen3-4B, Llama-3-8B
# and one GPU's share of tensor-parallel Llama-3.1-70B (TP8) and Llama-3-8B.
QWEN3_4B = (2560, 6144, 4096, 9728)
LLAMA3_8B = (4096, 6144, 4096, 14336)
LLAMA3_70B_TP8 = (8192, 1280, 1024, 3584)
LLAMA3_8B_TP2 = (4096, 3072, 2048, 7168)
LLAMA3_8B_TP4 = (4096, 1536, 1024, 3584)
DENSE = (QWEN3_4B, LLAMA3_8B, LLAMA3_70B_TP8, LLAMA3_8B_TP2, LLAMA3_8B_TP4)


def listed():
    return [
        # One o projection for one token, called eagerly.
        _dense("linear_m1", "linear", QWEN3_4B, 1, 1),
        # Decode of a single sequence, the headline decode configuration.
        _dense("decode_4b_m1", "decode", QWEN3_4B, 1, 8),
        # A small batch of sequences.
        _dense("decode_4b_m8", "decode", QWEN3_4B, 8, 8),
        # A full small batch in bf16.
        _dense("decode_4b_m32_bf16", "decode", QWEN3_4B, 32, 8, dtype="bf16"),
        # A large captured decode batch.
        _dense("decode_8b_m64", "decode", LLAMA3_8B, 64, 4),
        # The ragged last chunk of a prompt; group size 64, biased qkv.
        _dense("prefill_4b_m333_g64", "prefill", QWEN3_4B, 333, 1, group=64, bias=True),
        # A prompt chunk, the headline prefill configuration.
        _dense("prefill_8b_m2048", "prefill", LLAMA3_8B, 2048, 1),
        # The largest prefill chunk the scheduler forms, in bf16.
        _dense("prefill_8b_m8192_bf16", "prefill", LLAMA3_8B, 8192, 1, dtype="bf16"),
        # Qwen3-30B-A3B-shaped experts: one token, a decode batch, a short
        # chunk (the engine's MoE benchmark) and a long one.
        _moe("moe_t1", 128, 8, 2048, 768, 1, 4),
        _moe("moe_t24_bf16", 128, 8, 2048, 768, 24, 3, dtype="bf16"),
        _moe("moe_t512", 128, 8, 2048, 768, 512, 1),
        _moe("moe_t4096_bf16", 128, 8, 2048, 768, 4096, 1, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))))))


def draw(rng):
    dtype = rng.choice(("fp16", "bf16"))
    group = rng.choice((128, 128, 128, 64, 64, 32))
    if rng.random() < 0.5:
        dims = rng.choice(DENSE)
        M = _log_int(rng, 1, 8192)
        if rng.random() < 0.1:
            c = _dense("", "linear", dims, min(M, 32), 1, dtype, group, rng.random() < 0.5)
        elif M <= GRAPH_MAX:
            hidden, qkv, attn, inter = dims
            layers = max(2, min(8, round(420e6 / (0.52 * (hidden * (qkv + 3 * inter) + attn * hidden)))))
            c = _dense("", "decode", dims, M, layers, dtype, group, rng.random() < 0.5)
        else:
            c = _dense("", "prefill", dims, M, 1, dtype, group, rng.random() < 0.5)
    else:
        E = rng.choice((16, 32, 64, 128))
        top_k = rng.choice((2, 4, 6, 8))
        hidden = rng.choice((1024, 2048, 4096))
        inter = rng.choice((384, 512, 768, 1024, 1408, 1536))
        while E * hidden * inter > 128 * 4096 * 768:
            E //= 2
        T = _log_int(rng, 1, 4096)
        layers = 1
        if T <= GRAPH_MAX:
            layers = max(2, min(6, round(900e6 / (1.56 * E * hidden * inter))))
        c = _moe("", E, top_k, hidden, inter, T, layers, dtype, group)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs, from the seed alone.
# ---------------------------------------------------------------------------

def _awq(gen, lead, K, N, group, dtype):
    def words(*shape):
        return torch.randint(-2 ** 31, 2 ** 31, lead + shape, generator=gen, device=DEVICE, dtype=torch.int32)

    scales = torch.rand(lead + (K // group, N), generator=gen, device=DEVICE) * 0.018 + 0.002
    return {"qweight": words(K, N // 8), "qzeros": words(K // group, N // 8), "scales": scales.to(dtype)}


def _rows(gen, M, K, dtype):
    return torch.randn((M, K), generator=gen, device=DEVICE).to(dtype)


def _layers(case, seed):
    """Checkpoint tensors and activations, one layer after the other."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt, G, M, H = DTYPES[case["dtype"]], case["group"], case["M"], case["hidden"]
    for _ in range(case["layers"]):
        if case["kind"] == "moe":
            E, I = case["E"], case["inter"]
            yield {"gate_up_proj": _awq(gen, (E,), H, 2 * I, G, dt), "down_proj": _awq(gen, (E,), I, H, G, dt),
                   "x": _rows(gen, M, H, dt), "logits": _rows(gen, M, E, dt)}
            continue
        d = {"o": _awq(gen, (), case["attn"], H, G, dt), "a": _rows(gen, M, case["attn"], dt)}
        if case["kind"] != "linear":
            d["qkv"] = _awq(gen, (), H, case["qkv"], G, dt)
            d["x"], d["y"] = _rows(gen, M, H, dt), _rows(gen, M, H, dt)
            d["mlp"] = {"gate_up_proj": _awq(gen, (), H, 2 * case["inter"], G, dt),
                        "down_proj": _awq(gen, (), case["inter"], H, G, dt)}
        if case["bias"]:
            n = H if case["kind"] == "linear" else case["qkv"]
            d["bias"] = torch.randn(n, generator=gen, device=DEVICE).to(dt)
        yield d


# ---------------------------------------------------------------------------
# The program: layers as a model holds them, called as a model calls them.
# ---------------------------------------------------------------------------

def _flat(prefix, tensors):
    return {f"{prefix}.{k}": v for k, v in tensors.items()}


def _build(case, d):
    """The layer's modules with their weights loaded (repacked on the device)."""
    H, G = case["hidden"], case["group"]
    if case["kind"] == "moe":
        moe = AWQMoELayer(case["E"], case["top_k"], H, case["inter"], group_size=G, params_dtype=DTYPES[case["dtype"]])
        moe.load_state_dict({**_flat("gate_up_proj", d["gate_up_proj"]), **_flat("down_proj", d["down_proj"])})
        return {"moe": moe, "x": d["x"], "logits": d["logits"]}
    method = get_quantization_config("awq").from_config(
        {"bits": 4, "group_size": G, "zero_point": True, "quant_method": "awq"}).get_linear_method()
    before = torch.get_default_dtype()
    torch.set_default_dtype(DTYPES[case["dtype"]])
    try:
        with torch.device(DEVICE):
            linear = case["kind"] == "linear"
            bias = {"bias": d["bias"]} if case["bias"] else {}
            o = RowParallelLinear(case["attn"], H, linear and case["bias"], method)
            o.load_state_dict({**d["o"], **(bias if linear else {})})
            if linear:
                return {"o": o, "a": d["a"]}
            # The fused projection as 128-wide heads, a quarter of the rest of
            # the columns each for keys and values.
            heads = case["qkv"] // 128
            kv = max(1, heads // 6)
            qkv = QKVParallelLinear(H, 128, heads - 2 * kv, kv, case["bias"], method)
            qkv.load_state_dict({**d["qkv"], **bias})
            mlp = GatedMLP(H, case["inter"], "silu", method)
            mlp.load_state_dict({**_flat("gate_up_proj", d["mlp"]["gate_up_proj"]),
                                 **_flat("down_proj", d["mlp"]["down_proj"])})
    finally:
        torch.set_default_dtype(before)
    return {"qkv": qkv, "o": o, "mlp": mlp, "x": d["x"], "a": d["a"], "y": d["y"]}


def _forward(layers):
    out = []
    for m in layers:
        if "moe" in m:
            # The block writes its result over its input.
            out.append(m["moe"].forward(m["x"].clone(), m["logits"]))
        elif "qkv" in m:
            out += [m["qkv"].forward(m["x"]), m["o"].forward(m["a"]), m["mlp"].forward(m["y"])]
        else:
            out.append(m["o"].forward(m["a"]))
    return out


def prepare(case, seed):
    state = {"layers": [_build(case, d) for d in _layers(case, seed)], "graph": None}
    if case["kind"] == "decode" or (case["kind"] == "moe" and case["M"] <= GRAPH_MAX):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _forward(state["layers"])
        torch.cuda.current_stream().wait_stream(stream)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _forward(state["layers"])
    return state


def run(state):
    if state["graph"] is None:
        return _forward(state["layers"])
    state["graph"].replay()
    return state["out"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what its results are.
# ---------------------------------------------------------------------------

def _weight_bytes(K, N, group):
    return K * N / 2 + (K // group) * N / 2 + (K // group) * N * 2


def work(case):
    M, H, G = case["M"], case["hidden"], case["group"]
    if case["kind"] == "moe":
        E, k, I = case["E"], case["top_k"], case["inter"]
        # Expected number of experts that M tokens of k distinct, equally
        # likely experts reach.
        touched = E * (1.0 - (1.0 - k / E) ** M)
        b = touched * (_weight_bytes(H, 2 * I, G) + _weight_bytes(I, H, G)) + 2 * M * (2 * H + E)
        f = 2.0 * M * k * 3 * H * I
    else:
        shapes = [(case["attn"], H)]
        if case["kind"] != "linear":
            shapes += [(H, case["qkv"]), (H, 2 * case["inter"]), (case["inter"], H)]
        b = sum(_weight_bytes(K, N, G) for K, N in shapes)
        b += 2 * M * (case["attn"] + H)
        if case["kind"] != "linear":
            b += 2 * M * (H + case["qkv"] + H + H)
        f = sum(2.0 * M * K * N for K, N in shapes)
    return {"bytes": b * case["layers"], "flops": f * case["layers"]}


def tolerance(case):
    # Outputs are rounded to 11 (fp16) or 8 (bf16) bits, after weights that may
    # be rounded to as many and, in the gated blocks, one or two rounded
    # intermediates.  Measured against 64 bits: 2e-4 to 7e-4 in fp16, 2.3e-3
    # to 4.8e-3 in bf16; two implementations differ by up to both errors.
    return {"rel": 1.5e-3, "max": 0.012} if case["dtype"] == "fp16" else {"rel": 1.2e-2, "max": 0.08}


def _nibbles(words, cols):
    shift = torch.tensor([4 * p for p in AWQ_ORDER], dtype=torch.int32, device=words.device)
    return ((words.unsqueeze(-1) >> shift) & 0xF).reshape(words.shape[:-1] + (cols,))


def _dense64(t, group):
    """(q - z) * s in 64 bits."""
    N = t["scales"].shape[-1]
    q = _nibbles(t["qweight"], N).double()
    z = _nibbles(t["qzeros"], N).double().repeat_interleave(group, 0)
    return (q - z) * t["scales"].double().repeat_interleave(group, 0)


def _gated64(x, gate_up, down, group):
    g, u = (x @ _dense64(gate_up, group)).chunk(2, -1)
    return (torch.nn.functional.silu(g) * u) @ _dense64(down, group)


def _moe64(case, d):
    x, k = d["x"].double(), case["top_k"]
    p, ids = torch.sort(torch.softmax(d["logits"].double(), -1), dim=-1, descending=True, stable=True)
    w = p[:, :k] / (p[:, :k].sum(-1, keepdim=True) + 1e-8)
    out = torch.zeros_like(x)
    for e in range(case["E"]):
        t, j = torch.nonzero(ids[:, :k] == e, as_tuple=True)
        if t.numel():
            pick = [{n: v[e] for n, v in d[m].items()} for m in ("gate_up_proj", "down_proj")]
            out.index_add_(0, t, _gated64(x[t], pick[0], pick[1], case["group"]) * w[t, j, None])
    return out


def exact(case, seed):
    G, out = case["group"], []
    for d in _layers(case, seed):
        if case["kind"] == "moe":
            out.append(_moe64(case, d))
            continue
        o = d["a"].double() @ _dense64(d["o"], G)
        if case["kind"] == "linear":
            out.append(o + d["bias"].double() if case["bias"] else o)
            continue
        qkv = d["x"].double() @ _dense64(d["qkv"], G)
        out.append(qkv + d["bias"].double() if case["bias"] else qkv)
        out += [o, _gated64(d["y"].double(), d["mlp"]["gate_up_proj"], d["mlp"]["down_proj"], G)]
    return out
