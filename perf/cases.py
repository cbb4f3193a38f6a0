"""Performance cases of the MoE sparse block: what a serving engine asks of it.

A case is one call of a public entry point on resident weights: a block forward
(`SparseMoe.forward`), the forward of a float32 checkpoint's block (`SparseMoeF32.forward`), or a
stack of MoE layers (`MoeStack.forward_`). The ranges are the batch sizes an engine sends, from one
decoded token through continuous batching and short prompts to long prefill chunks, over the
checkpoint formats the library loads: 4-bit group-64 and group-32 experts, 8-bit experts, 8-bit
routers, dense bf16 experts and all-f32 blocks, at the Qwen3.6-35B-A3B-like and
Qwen3-Coder-480B-A35B-like shapes.

The weights are random but distributed as trained and quantized ones are: codes uniform, group
scales |N(0, 0.02)| / 7.5 (4-bit) or / 127.5 (8-bit), biases that centre each group on zero, router
rows N(0, 0.02), activations N(0, 1).
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from mrun_amd import _lib, synth
from mrun_amd import moe as M

SHAPES = {"qwen36": synth.QWEN36, "coder": synth.CODER}

# Largest batches drawn, by kind: no drawn case costs more than the largest listed one.
MAX_TOKENS = {"qwen36": 4096, "coder": 3000, "f32": 128, "stack": 512}


def _case(name, kind, tokens, shape="qwen36", bits=4, group=64, router="dense", layers=1):
    case = {"kind": kind, "shape": shape, "tokens": tokens, "bits": bits, "group": group,
            "router": router, "layers": layers}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # one token for one user: the latency of an interactive reply
        _case("decode_1", "block", 1),
        # a few concurrent users on an mlx-community conversion (8-bit router and shared gate)
        _case("decode_6_router8", "block", 6, router="q8"),
        # continuous batching: a full decode batch
        _case("decode_24", "block", 24),
        # a short prompt, or a decode batch with speculative tokens to verify
        _case("prompt_90", "block", 90),
        # a prefill chunk under a skewed router (some experts far hotter than others)
        _case("prefill_2048_zipf", "block", 2048, router="zipf"),
        # a medium prompt on an 8-bit conversion (8-bit experts, router and shared gate)
        _case("prefill_1000_8bit", "block", 1000, bits=8, router="q8"),
        # a medium prompt on a 4-bit group-32 conversion
        _case("prefill_700_group32", "block", 700, group=32, router="q8"),
        # a prompt on an unquantized bf16 checkpoint
        _case("prefill_300_bf16", "block", 300, bits=16),
        # a small batch on an all-float32 checkpoint
        _case("batch_40_f32", "f32", 40, bits=32),
        # the Coder shape: two users decoding
        _case("coder_decode_2", "block", 2, shape="coder"),
        # the Coder shape: a prefill chunk
        _case("coder_prefill_3000", "block", 3000, shape="coder"),
        # several layers with their norms and residuals around the blocks, one decoded token
        _case("stack_6_layers_1", "stack", 1, layers=6),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.08:
        return _case(None, "f32", _log_int(rng, 1, MAX_TOKENS["f32"]), bits=32)
    if pick < 0.18:
        return _case(None, "stack", _log_int(rng, 1, MAX_TOKENS["stack"]), layers=rng.randint(2, 6))
    if pick < 0.32:
        return _case(None, "block", _log_int(rng, 1, MAX_TOKENS["coder"]), shape="coder")
    tokens = _log_int(rng, 1, MAX_TOKENS["qwen36"])
    fmt = rng.random()
    if fmt < 0.55:
        return _case(None, "block", tokens, router=rng.choice(["dense", "zipf", "q8"]))
    if fmt < 0.72:
        return _case(None, "block", tokens, bits=8, router=rng.choice(["dense", "q8"]))
    if fmt < 0.88:
        return _case(None, "block", tokens, group=rng.choice([32, 128]),
                     router=rng.choice(["dense", "q8"]))
    return _case(None, "block", tokens, bits=16)


# ---- inputs, made on the device from the seed

class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std, dtype=torch.bfloat16):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=self.g)
        return t.to(dtype)

    def quantized(self, experts, out, in_, bits, group):
        """(codes, scales, biases); dense weights (bits 16 and 32) are the codes alone."""
        if bits == 16:
            return torch.empty(experts, out, in_, dtype=torch.bfloat16,
                               device="cuda").normal_(0.0, 0.01, generator=self.g), None, None
        if bits == 32:
            return torch.empty(experts, out, in_, dtype=torch.float32,
                               device="cuda").normal_(0.0, 0.01, generator=self.g), None, None
        levels = (1 << bits) - 1
        codes = torch.randint(-2 ** 31, 2 ** 31, (experts, out, in_ * bits // 32),
                              dtype=torch.int32, device="cuda", generator=self.g)
        scales = (self.normal((experts, out, in_ // group), 0.02, torch.float32).abs()
                  / (levels / 2)).to(torch.bfloat16)
        return codes, scales, (scales.float() * (-levels / 2)).to(torch.bfloat16)


def _weights(gen, case):
    """The tensors of one block, each projection as (codes, scales, biases)."""
    s, bits, group = SHAPES[case["shape"]], case["bits"], case["group"]
    f32 = bits == 32
    w = SimpleNamespace(shape=s, router_bias=None)

    def linear(out):
        if case["router"] == "q8":
            codes, scales, biases = gen.quantized(1, out, s.hidden, 8, 64)
            return codes, scales, biases
        return gen.normal((out, s.hidden), 0.02, torch.float32 if f32 else torch.bfloat16)

    w.router = linear(s.experts)
    if case["router"] == "zipf":
        bias, _ = synth.zipf_bias(int(torch.randint(0, 2 ** 31, (1,), device="cuda",
                                                    generator=gen.g)), s.experts)
        w.router_bias = M.bf16_tensor(bias)
    w.gate = gen.quantized(s.experts, s.intermediate, s.hidden, bits, group)
    w.up = gen.quantized(s.experts, s.intermediate, s.hidden, bits, group)
    w.down = gen.quantized(s.experts, s.hidden, s.intermediate, bits, group)
    if s.shared:
        w.sh_gate = gen.quantized(1, s.shared, s.hidden, bits, group)
        w.sh_up = gen.quantized(1, s.shared, s.hidden, bits, group)
        w.sh_down = gen.quantized(1, s.hidden, s.shared, bits, group)
        w.sh_expert_gate = linear(1)
    return w


def _inputs(case, seed):
    gen = _Gen(seed)
    s = SHAPES[case["shape"]]
    layers = [_weights(gen, case) for _ in range(case["layers"])]
    norms = [1.0 + gen.normal((s.hidden,), 0.1, torch.float32) for _ in layers]
    norms = [n.to(torch.bfloat16) for n in norms]
    x = gen.normal((case["tokens"], s.hidden), 1.0,
                   torch.float32 if case["kind"] == "f32" else torch.bfloat16)
    return layers, norms, x


def _block(w, case):
    s, bits, group = w.shape, case["bits"], case["group"]

    def q(t, in_, n_bits, n_group):
        codes, scales, biases = t
        return M.DeviceQTensor.from_tensors(codes, scales, biases, codes.shape[0], codes.shape[1],
                                            in_, n_group if n_bits < 16 else 0, n_bits)

    lin = lambda t: q(t, s.hidden, 8, 64) if isinstance(t, tuple) else t
    hb = SimpleNamespace(shape=s, router=lin(w.router), router_bias=w.router_bias,
                         gate_proj=q(w.gate, s.hidden, bits, group),
                         up_proj=q(w.up, s.hidden, bits, group),
                         down_proj=q(w.down, s.intermediate, bits, group))
    if s.shared:
        hb.sh_gate_proj = q(w.sh_gate, s.hidden, bits, group)
        hb.sh_up_proj = q(w.sh_up, s.hidden, bits, group)
        hb.sh_down_proj = q(w.sh_down, s.shared, bits, group)
        hb.sh_expert_gate = lin(w.sh_expert_gate)
    return M.SparseMoe(hb)


def _block_f32(w):
    s = w.shape
    quant = lambda t: _lib.Quantized(t.data_ptr(), None, None, t.shape[0] if t.dim() == 3 else 1,
                                     t.shape[-2], t.shape[-1], 0, 32)
    lin = lambda t: _lib.Linear(None, quant(t), None, t.shape[-2], t.shape[-1])
    c = _lib.SparseMoe()
    c.cfg = _lib.MoeConfig(s.hidden, s.experts, s.top_k, s.intermediate, int(s.norm_topk), s.shared)
    c.gate = lin(w.router)
    c.switch_gate_proj, c.switch_up_proj = quant(w.gate[0]), quant(w.up[0])
    c.switch_down_proj = quant(w.down[0])
    c.shared_gate_proj, c.shared_up_proj = lin(w.sh_gate[0]), lin(w.sh_up[0])
    c.shared_down_proj, c.shared_expert_gate = lin(w.sh_down[0]), lin(w.sh_expert_gate)
    return M.SparseMoeF32.from_view(c, owner=w)


def prepare(case, seed):
    layers, norms, x = _inputs(case, seed)
    if case["kind"] == "f32":
        return {"kind": "f32", "block": _block_f32(layers[0]), "x": x}
    blocks = [_block(w, case) for w in layers]
    if case["kind"] == "stack":
        # the residual stream is updated in place: each pass starts from a copy of the embeddings
        return {"kind": "stack", "stack": M.MoeStack(blocks, norms), "x": x,
                "stream": torch.empty_like(x)}
    return {"kind": "block", "block": blocks[0], "x": x}


def run(state):
    if state["kind"] == "stack":
        state["stream"].copy_(state["x"])
        return state["stack"].forward_(state["stream"])
    return state["block"].forward(state["x"])


# ---- costs and tolerances

def _projection_bytes(out, in_, bits, group):
    n = out * in_
    return n * bits / 8 + (n / group * 4 if bits < 16 else 0)


def work(case):
    s, T, bits, group = SHAPES[case["shape"]], case["tokens"], case["bits"], case["group"]
    act = 4 if case["kind"] == "f32" else 2
    D, I, S, E, k = s.hidden, s.intermediate, s.shared, s.experts, s.top_k
    distinct = E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens choose, on average
    expert = 2 * _projection_bytes(I, D, bits, group) + _projection_bytes(D, I, bits, group)
    gates = _projection_bytes(E + (1 if S else 0), D, 8 if case["router"] == "q8" else 8 * act, 64)
    total = distinct * expert + gates
    flops = 2.0 * T * (3 * k * D * I + D * E)
    if S:
        total += 2 * _projection_bytes(S, D, bits, group) + _projection_bytes(D, S, bits, group)
        flops += 2.0 * T * (3 * D * S + D)
    layers = case["layers"]
    return {"bytes": layers * total + 2 * act * T * D, "flops": layers * flops}


def tolerance(case):
    # Measured against exact(): f32 blocks 2.2e-7; bf16 blocks 4.9e-3 to 7.2e-3 (the output's and
    # the intermediate rows' bf16 roundings); a stack 1.7e-3 to 1.9e-3 at a few layers, but with
    # many rows a near tie in a later layer's router may choose another expert for a row.
    if case["kind"] == "f32":
        return {"rel": 1e-6}
    if case["kind"] == "stack":
        return {"rel": 2e-2}
    return {"rel": 1.2e-2}


# ---- the same results in 64 bits

def _bf16(t):
    return t.to(torch.bfloat16).to(torch.float64)


def _dequant(t, e, bits, group):
    """Expert e's weight [out, in] in float64."""
    codes, scales, biases = t
    if scales is None:
        return codes[e].double()
    shifts = torch.arange(0, 32, bits, dtype=torch.int32, device=codes.device)
    q = ((codes[e].unsqueeze(-1) >> shifts) & ((1 << bits) - 1)).flatten(1).double()
    q = q.view(q.shape[0], -1, group)
    return (q * scales[e].double().unsqueeze(-1) + biases[e].double().unsqueeze(-1)).flatten(1)


def _silu(z):
    return z * torch.sigmoid(z)


def _exact_block(w, case, x):
    """x [T, hidden] float64 -> the block's output. The router's choice follows the stored
    precision of its logits and gates (bf16, equal gates by lower id); everything else is
    unrounded."""
    s, bits, group = w.shape, case["bits"], case["group"]
    stored = (lambda t: t) if case["kind"] == "f32" else _bf16
    linear = lambda t: _dequant(t, 0, 8, 64) if isinstance(t, tuple) else t.double()
    exact_logits = x @ linear(w.router).T
    logits = stored(exact_logits)
    if w.router_bias is not None:
        exact_logits = exact_logits + w.router_bias.double()
        logits = stored(logits + w.router_bias.double())
    order = torch.sort(stored(torch.softmax(logits, -1)), dim=-1, descending=True, stable=True)[1]
    ids = order[:, :s.top_k]
    scores = torch.gather(torch.softmax(exact_logits, -1), 1, ids)
    if s.norm_topk:
        scores = scores / scores.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(s.experts):
        t, j = (ids == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        xe = x[t]
        act = _silu(xe @ _dequant(w.gate, e, bits, group).T) * (xe @ _dequant(w.up, e, bits, group).T)
        out.index_add_(0, t, (act @ _dequant(w.down, e, bits, group).T) * scores[t, j, None])
    if s.shared:
        act = _silu(x @ _dequant(w.sh_gate, 0, bits, group).T)
        act = act * (x @ _dequant(w.sh_up, 0, bits, group).T)
        gate = torch.sigmoid(x @ linear(w.sh_expert_gate).T)
        out += gate * (act @ _dequant(w.sh_down, 0, bits, group).T)
    return out


def exact(case, seed):
    layers, norms, x = _inputs(case, seed)
    x = x.double()
    if case["kind"] != "stack":
        return _exact_block(layers[0], case, x)
    # between the ops of a stack stand bf16 tensors: the residual stream and the normalised rows
    for w, n in zip(layers, norms):
        h = _bf16(_bf16(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)) * n.double())
        x = _bf16(x + _exact_block(w, case, h))
    return x
