"""The work whose speed counts: decode, batched decode, prefill and LoRA training through the public modules.

Every case is one of four kinds:

  "layer"        one 4-bit linear layer without gradients: a projection called on its own, from a single decoded row to
                 a prefill of some thousand rows
  "decode"       one step of a stack of decoder blocks without gradients, 1..16 rows (one token of as many sequences):
                 q|k|v and gate|up grouped in place, optionally adapters on q and v (inference with a LoRA), optionally
                 replayed as a HIP graph (the serving loop)
  "train_layer"  forward + backward of one 4-bit linear layer with a LoRA adapter
  "train_block"  forward + backward of the seven linear layers of one decoder block, adapters on q and v

Feature counts are those of the 7B and 13B decoder layers and, in drawn cases, any multiple of 128 between 2048 and 13824;
rows are arbitrary.  Attention itself and the embeddings are not this package's work: in a block, attention is stood for
by v * sigmoid(q + k), which keeps every projection's output and gradient in use.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from alpaca_lora_4bit_amd.autograd_4bit import Autograd4bitQuantLinear
from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp, make_quant_attn
from alpaca_lora_4bit_amd.models import inject_lora_layers

#: (hidden size, MLP size) of the 7B and 13B decoder layers
WIDTHS = {"7b": (4096, 11008), "13b": (5120, 13824)}


def listed():
    return [
        # one attention projection of one decoded token: the smallest product, latency
        {"name": "layer_1_7b_q", "kind": "layer", "rows": 1, "k": 4096, "n": 4096, "groupsize": 128, "act_order": False},
        # one decoded token through an act-order checkpoint's gate projection
        {"name": "layer_1_13b_gate_actorder", "kind": "layer", "rows": 1, "k": 5120, "n": 13824, "groupsize": 128, "act_order": True},
        # 48 sequences decoded together, or a short prompt: gate projection
        {"name": "layer_48_7b_gate", "kind": "layer", "rows": 48, "k": 4096, "n": 11008, "groupsize": 128, "act_order": False},
        # prefill of 512 tokens on an act-order checkpoint
        {"name": "layer_512_13b_gate_actorder", "kind": "layer", "rows": 512, "k": 5120, "n": 13824, "groupsize": 128, "act_order": True},
        # prefill of 2048 tokens
        {"name": "layer_2048_7b_gate", "kind": "layer", "rows": 2048, "k": 4096, "n": 11008, "groupsize": 128, "act_order": False},
        # one token of one sequence, the serving loop's replayed graph
        {"name": "decode_1_7b_graph", "kind": "decode", "rows": 1, "h": 4096, "i": 11008, "groupsize": 128, "blocks": 8, "lora_r": 0, "graph": True},
        # one token of a beam of 4 with the trained adapter on q and v, called as generate() does
        {"name": "decode_4_7b_lora", "kind": "decode", "rows": 4, "h": 4096, "i": 11008, "groupsize": 128, "blocks": 8, "lora_r": 8, "graph": False},
        # one token of 16 sequences
        {"name": "decode_16_7b_graph", "kind": "decode", "rows": 16, "h": 4096, "i": 11008, "groupsize": 128, "blocks": 8, "lora_r": 0, "graph": True},
        # finetuning with the default micro-batch of one sample, not padded to a round length
        {"name": "train_block_200_7b", "kind": "train_block", "rows": 200, "h": 4096, "i": 11008, "groupsize": 128, "lora_r": 8, "dropout": 0.05},
        # finetuning, 4 samples of 256 tokens
        {"name": "train_block_1024_7b", "kind": "train_block", "rows": 1024, "h": 4096, "i": 11008, "groupsize": 128, "lora_r": 8, "dropout": 0.05},
        # q projection of 8 samples of 256 tokens
        {"name": "train_layer_2048_7b_q", "kind": "train_layer", "rows": 2048, "k": 4096, "n": 4096, "groupsize": 128, "lora_r": 8, "dropout": 0.0},
        # the largest: one 13B block, 4096 tokens
        {"name": "train_block_4096_13b", "kind": "train_block", "rows": 4096, "h": 5120, "i": 13824, "groupsize": 128, "lora_r": 8, "dropout": 0.05},
    ]


def _log_between(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _features(rng):
    """(in, out) of one layer: a projection of the 7B / 13B layers, or any multiples of 128."""
    h, i = WIDTHS[rng.choice(["7b", "13b"])]
    return rng.choice([(h, h), (h, i), (i, h), (128 * _log_between(rng, 16, 108), 128 * _log_between(rng, 16, 108))])


def draw(rng):
    """One more case of the same ranges.  Group sizes: mostly 128, as published checkpoints have, sometimes 64 or 32."""
    groupsize = rng.choice([128] * 6 + [64, 32])
    kind = rng.choice(["layer", "layer", "layer", "decode", "train_layer", "train_layer", "train_block"])
    if kind == "layer":
        k, n = _features(rng)
        act_order = groupsize == 128 and rng.random() < 0.25
        return {"kind": kind, "rows": _log_between(rng, 1, 4096), "k": k, "n": n, "groupsize": groupsize, "act_order": act_order}
    if kind == "decode":
        h, i = WIDTHS[rng.choice(["7b", "13b"])]
        lora_r = rng.choice([0, 0, 8, 16])
        return {"kind": kind, "rows": _log_between(rng, 1, 16), "h": h, "i": i, "groupsize": groupsize, "blocks": rng.randint(4, 8), "lora_r": lora_r, "graph": lora_r == 0 and rng.random() < 0.5}
    dropout, lora_r = rng.choice([0.0, 0.05]), rng.choice([8, 8, 16, 32, 64])
    if kind == "train_layer":
        k, n = _features(rng)
        return {"kind": kind, "rows": _log_between(rng, 64, 4096), "k": k, "n": n, "groupsize": groupsize, "lora_r": lora_r, "dropout": dropout}
    h, i = WIDTHS[rng.choice(["7b", "13b"])]
    return {"kind": kind, "rows": _log_between(rng, 64, 2048), "h": h, "i": i, "groupsize": groupsize, "lora_r": lora_r, "dropout": dropout}


# ---------------------------------------------------------------------------------------------------- inputs
class _Source:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return (torch.randn(shape, device="cuda", generator=self.gen) * scale).half()

    def linear(self, k, n, groupsize, act_order=False):
        """A quantized layer as a checkpoint gives it: uniform codes, zero points about the middle of the range, scales
        that give the weights the spread of a trained projection (outputs of unit size for inputs of unit size)."""
        groups = k // groupsize
        layer = Autograd4bitQuantLinear(k, n, groupsize=groupsize)
        lo, hi = -2 ** 31, 2 ** 31 - 1
        layer.qweight = torch.randint(lo, hi, (k // 8, n), device="cuda", dtype=torch.int32, generator=self.gen)
        zero = torch.randint(0, 2, (groups, n // 8, 8), device="cuda", dtype=torch.int32, generator=self.gen) + 6
        layer.qzeros = (zero << (4 * torch.arange(8, device="cuda", dtype=torch.int32))).sum(-1, dtype=torch.int32)
        mean = (64.0 / k) ** 0.5 / 32.0                      # codes have a standard deviation of 4.6
        layer.scales = (mean * (0.5 + torch.rand((groups, n), device="cuda", generator=self.gen))).half()
        layer.bias = torch.zeros(n, dtype=torch.float16, device="cuda")
        order = torch.arange(k, device="cuda")
        if act_order:
            order = torch.randperm(k, device="cuda", generator=self.gen)
        layer.g_idx = (order // groupsize).to(torch.int32)
        return layer

    def adapters(self, layers):
        """Trained adapters: lora_A as initialised, lora_B no longer zero."""
        for layer in layers:
            for a in layer.lora_A.values():
                r, k = a.weight.shape
                a.weight.data = (torch.rand((r, k), device="cuda", generator=self.gen) * 2 - 1) * (6.0 / k) ** 0.5 / 2.5
            for b in layer.lora_B.values():
                b.weight.data = torch.randn(b.weight.shape, device="cuda", generator=self.gen) * 0.02


class _Attention(nn.Module):
    def __init__(self, src, h, groupsize):
        super().__init__()
        self.q_proj, self.k_proj, self.v_proj, self.o_proj = (src.linear(h, h, groupsize) for _ in range(4))

    def forward(self, x):
        q, k, v = self.q_proj(x), self.k_proj(x), self.v_proj(x)
        return self.o_proj(v * torch.sigmoid(q + k))


class _MLP(nn.Module):
    def __init__(self, src, h, i, groupsize):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = src.linear(h, i, groupsize), src.linear(h, i, groupsize), src.linear(i, h, groupsize)
        self.act_fn = nn.SiLU()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))


class _Block(nn.Module):
    def __init__(self, src, h, i, groupsize):
        super().__init__()
        self.self_attn, self.mlp = _Attention(src, h, groupsize), _MLP(src, h, i, groupsize)

    def forward(self, x):
        x = x + self.self_attn(F.rms_norm(x, x.shape[-1:]))
        return x + self.mlp(F.rms_norm(x, x.shape[-1:]))


def _lora(model, src, r, dropout):
    layers = list(inject_lora_layers(model, ("q_proj", "v_proj"), r=r, lora_alpha=2 * r, lora_dropout=dropout).values())
    src.adapters(layers)
    return layers


def prepare(case, seed):
    src = _Source(seed)
    state = {"kind": case["kind"], "seed": seed}
    if case["kind"] == "layer":
        state["model"] = src.linear(case["k"], case["n"], case["groupsize"], case["act_order"])
        state["x"] = src.normal(case["rows"], case["k"])
        return state
    if case["kind"] == "train_layer":
        holder = nn.Module()
        holder.q_proj = src.linear(case["k"], case["n"], case["groupsize"])
        lora = _lora(holder, src, case["lora_r"], case["dropout"])
        state["model"] = holder.q_proj.cuda().train()
        state["x"] = src.normal(case["rows"], case["k"]).requires_grad_(True)
        state["dy"] = src.normal(case["rows"], case["n"])
        state["params"] = [p for m in lora for p in (m.lora_A["default"].weight, m.lora_B["default"].weight)]
        return state
    blocks = nn.Sequential(*[_Block(src, case["h"], case["i"], case["groupsize"]) for _ in range(case.get("blocks", 1))])
    lora = _lora(blocks, src, case["lora_r"], case.get("dropout", 0.0)) if case["lora_r"] else []
    make_quant_attn(blocks)
    make_fused_mlp(blocks)
    state["model"] = blocks.cuda().train(case["kind"] == "train_block")
    state["x"] = src.normal(case["rows"], case["h"])
    if case["kind"] == "train_block":
        state["x"].requires_grad_(True)
        state["dy"] = src.normal(case["rows"], case["h"])
        state["params"] = [p for m in lora for p in (m.lora_A["default"].weight, m.lora_B["default"].weight)]
    elif case["graph"]:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.no_grad(), torch.cuda.stream(stream):
            for _ in range(2):
                blocks(state["x"])
        torch.cuda.current_stream().wait_stream(stream)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.no_grad(), torch.cuda.graph(state["graph"], stream=stream):
            state["y"] = blocks(state["x"])
    return state


def run(state):
    if state["kind"] in ("layer", "decode"):
        if "graph" in state:
            state["graph"].replay()
            return state["y"]
        with torch.no_grad():
            return state["model"](state["x"])
    torch.default_generator.manual_seed(state["seed"])       # the dropout masks of this pass
    x, params = state["x"], state["params"]
    for t in [x] + params:
        t.grad = None
    with torch.amp.autocast("cuda", dtype=torch.float16):
        y = state["model"](x)
    y.backward(state["dy"])
    return [y.detach(), x.grad] + [p.grad for p in params]


# ---------------------------------------------------------------------------------------------------- what it takes
def _linear_bytes(k, n, groupsize, act_order=False):
    groups = k // groupsize
    return k * n // 2 + groups * n // 2 + 2 * groups * n + (4 * k if act_order else 0)


def work(case):
    rows, gs = case["rows"], case["groupsize"]
    if case["kind"] == "layer":
        k, n = case["k"], case["n"]
        return {"bytes": _linear_bytes(k, n, gs, case["act_order"]) + 2 * rows * (k + n), "flops": 2 * rows * k * n}
    r = case["lora_r"]
    if case["kind"] == "train_layer":
        k, n = case["k"], case["n"]
        # x, dy in, y, dx out; adapters in, their gradients out
        return {"bytes": _linear_bytes(k, n, gs) + 4 * rows * (k + n) + 8 * r * (k + n),
                "flops": 4 * rows * k * n + 8 * rows * r * (k + n)}
    h, i = case["h"], case["i"]
    weights = 4 * _linear_bytes(h, h, gs) + 2 * _linear_bytes(h, i, gs) + _linear_bytes(i, h, gs)
    products = 4 * h * h + 3 * h * i
    adapter = 2 * r * 2 * h                                  # elements of the adapters on q and v
    if case["kind"] == "decode":
        return {"bytes": case["blocks"] * (weights + 4 * adapter) + 4 * rows * h,
                "flops": case["blocks"] * 2 * rows * (products + adapter)}
    # x, dy in, y, dx out; what forward keeps for backward (x, q, k, v, the MLP's input, gate, up) written and read once
    return {"bytes": weights + 8 * adapter + 8 * rows * h + 4 * rows * (5 * h + 2 * i),
            "flops": 4 * rows * products + 8 * rows * adapter}


def tolerance(case):
    """About four times what the present code is off from the same sums in 64 bits (fp16 inputs, weights and outputs,
    32-bit sums); blocks pass fp16 intermediates on, one after the other."""
    return {"rel": {"layer": 2e-3, "train_layer": 1.5e-3, "train_block": 4.5e-3, "decode": 1e-2}[case["kind"]]}


# ---------------------------------------------------------------------------------------------------- in 64 bits
def _dense64(layer):
    """The layer's weights, scale * (code - zero - 1), in 64 bits."""
    shifts = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
    codes = ((layer.qweight.unsqueeze(1) >> shifts.view(1, 8, 1)) & 15).reshape(-1, layer.qweight.shape[1])
    zeros = ((layer.qzeros.unsqueeze(2) >> shifts) & 15).reshape(layer.qzeros.shape[0], -1) + 1
    g = layer.g_idx.long()
    return layer.scales.double()[g] * (codes - zeros[g]).double()


def _keep64(rows, cols, seed, p):
    """The adapter's dropout factors: 0 where the 15-bit draw of (seed, row, column) lies below p, else 1 / (1 - p)."""
    m32 = 0xFFFFFFFF

    def mul(a, b):                                           # 32-bit product without leaving 64-bit integers
        return ((a & 0xFFFF) * b + ((((a >> 16) * b) & 0xFFFF) << 16)) & m32
    row = (mul(torch.arange(rows, device="cuda"), 0x9E3779B1) + (seed & m32)) & m32
    pair = (mul(torch.arange(cols // 2, device="cuda"), 0x85EBCA6B) + ((seed >> 32) & m32)) & m32
    h = row.view(-1, 1) ^ pair
    h = mul(h ^ (h >> 16), 0x7FEB352D)
    h = mul(h ^ (h >> 15), 0x846CA68B)
    h = h ^ (h >> 16)
    draws = torch.stack([h & 0x7FFF, (h >> 16) & 0x7FFF], dim=-1).view(rows, cols)
    threshold = round(p * 32768)
    return (draws >= threshold).double() / (1.0 - threshold / 32768.0)


def exact(case, seed):
    """What `run` returns, from the same inputs with every weight, product and sum in 64 bits."""
    state = prepare({**case, "graph": False}, seed)
    training = case["kind"].startswith("train")
    x = state["x"].detach().double().requires_grad_(training)
    params = [p.detach().double().requires_grad_(True) for p in state.get("params", [])]
    left = list(params)
    p = case.get("dropout", 0.0)
    torch.default_generator.manual_seed(seed)

    def linear(layer, t):
        y = t @ _dense64(layer)
        if hasattr(layer, "lora_A"):
            a, b = (left.pop(0), left.pop(0)) if training else (m["default"].weight.detach().double() for m in (layer.lora_A, layer.lora_B))
            if training and p > 0.0:
                t = t * _keep64(t.shape[0], t.shape[1], int(torch.randint(0, 2 ** 62, (1,)).item()), p)
            y = y + layer.scaling["default"] * ((t @ a.t()) @ b.t())
        return y

    def block(m, t):
        n, attn, mlp = F.rms_norm(t, t.shape[-1:], eps=torch.finfo(torch.float32).eps), m.self_attn, m.mlp
        q, k, v = linear(attn.q_proj, n), linear(attn.k_proj, n), linear(attn.v_proj, n)
        t = t + linear(attn.o_proj, v * torch.sigmoid(q + k))
        n = F.rms_norm(t, t.shape[-1:], eps=torch.finfo(torch.float32).eps)
        return t + linear(mlp.down_proj, F.silu(linear(mlp.gate_proj, n)) * linear(mlp.up_proj, n))

    with torch.set_grad_enabled(training):
        y = x
        if "layer" in case["kind"]:
            y = linear(state["model"], y)
        else:
            for m in state["model"]:
                y = block(m, y)
    if not training:
        return y
    y.backward(state["dy"].double())
    return [y.detach(), x.grad] + [t.grad for t in params]
