"""The work that a user of this provider has it do, as cases of one timed pass each.

A pass is made of MatMulNBits nodes of decoder-model shapes (the repository's own benchmark shapes), called through the
provider's public interface: `get_kernel`, `set_constant_inputs`, `execute`, and for decode steps `capture_begin` /
`capture_end` / `replay`. What `prepare` builds is what a session holds: weights on the GPU, one kernel object per node,
activation and output buffers, and for a decode loop the recorded graph.

The nets:
  proj     one node, `k` -> `n`
  mlp      gate/up and down of one layer
  layer    qkv, o, gate/up, down of one layer
  step     `layers` layers and the output head: one token step of a decode loop

`fused` nets carry the nodes as the graph optimizer leaves them: RMS normalization before qkv and gate/up inside the node, gate
and up with SwiGLU as one node, the residual in the bias slot of o and down. The others are plain nodes; what other
providers compute between them (attention, SwiGLU) is an input. Each node reads what the node before it wrote where the
model does that.
"""
import math

import torch

from onnx_genai_amd import ep as E

# hidden, q + k + v columns (None: three nodes of their own), k / v columns, intermediate, vocabulary
MODELS = {
    "0.5b": (896, None, 128, 4864, 151936),
    "7b": (3584, 4608, 512, 18944, 152064),
    "8b": (4096, 6144, 1024, 14336, 128256),
    "70b": (8192, 10240, 1024, 28672, 128256),
}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
CODE = {"f32": E.F32, "f16": E.F16, "bf16": E.BF16}

_provider = None


def provider():
    """One provider per process and GPU, as a session has it."""
    global _provider
    if _provider is None:
        _provider = E.RocmExecutionProvider(0)
    return _provider


def _case(name, net, rows, dtype, block, *, model="", k=0, n=0, layers=1, bits=4, zero_points=True, act_order=False, accuracy=0, fused=False, graph=False):
    return {"name": name, "net": net, "model": model, "k": k, "n": n, "layers": layers, "rows": rows, "dtype": dtype, "block": block, "bits": bits,
            "zero_points": zero_points, "act_order": act_order, "accuracy": accuracy, "fused": fused, "graph": graph}


def listed():
    return [
        # the smallest call there is: one eager f32 node of a 0.5B model, one row
        _case("one_node_f32", "proj", 1, "f32", 32, k=896, n=4864, zero_points=False),
        # a 0.5B assistant generating for one user, model exported without fusion: 169 short nodes in a recorded step
        _case("step_0.5b_f16", "step", 1, "f16", 32, model="0.5b", layers=24, graph=True),
        # a 7B model generating for one user
        _case("step_7b_bf16", "step", 1, "bf16", 128, model="7b", layers=28, fused=True, graph=True),
        # the same model serving a batch of sixteen sequences
        _case("step_7b_bf16_batch16", "step", 16, "bf16", 128, model="7b", layers=28, fused=True, graph=True),
        # the MLP of an 8B model over a prompt of ordinary length, ragged
        _case("prompt_8b_f16_777", "mlp", 777, "f16", 32, model="8b", zero_points=False, fused=True),
        # the same over a long prompt
        _case("prompt_8b_f16_8192", "mlp", 8192, "f16", 32, model="8b", zero_points=False, fused=True),
        # a 70B layer of a model exported with accuracy_level 4 (int8 activations), one token
        _case("int8_70b_token", "layer", 1, "f16", 64, model="70b", accuracy=4, graph=True),
        # and a long prompt through its MLP
        _case("int8_70b_4096", "mlp", 4096, "f16", 64, model="70b", accuracy=4),
        # an f32 export of a 0.5B model over a short prompt
        _case("prompt_0.5b_f32_200", "layer", 200, "f32", 32, model="0.5b", zero_points=False),
        # the 8-bit output head that mixed 4 / 8-bit exports have, four sequences
        _case("head_7b_8bit_4", "proj", 4, "bf16", 128, k=3584, n=152064, bits=8, graph=True),
        # a layer with act-order (g_idx) weights, one token
        _case("act_order_7b_token", "layer", 1, "f16", 128, model="7b", act_order=True, graph=True),
        # the MLP of an 8-bit model over a ragged prompt
        _case("prompt_7b_8bit_500", "mlp", 500, "bf16", 128, model="7b", bits=8),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    """A case of the ranges around the listed ones: rows over their whole range, 16-bit types, block sizes, options."""
    kind = rng.choice(["step", "step", "prompt", "prompt", "int8", "int8", "f32", "nbits", "act_order"])
    dtype = rng.choice(["f16", "bf16"])
    block = rng.choice([32, 64, 128])
    if kind == "step":
        model = rng.choice(["0.5b", "7b"])
        c = _case("", "step", _log_int(rng, 1, 64), dtype, block, model=model, layers=rng.randint(4, 24), fused=model == "7b", graph=True,
                  zero_points=rng.random() < 0.7)
    elif kind == "prompt":
        c = _case("", "mlp", _log_int(rng, 17, 8192), dtype, block, model=rng.choice(["0.5b", "7b", "8b"]), fused=True, zero_points=rng.random() < 0.5)
    elif kind == "int8":
        rows = _log_int(rng, 1, 4096)
        c = _case("", rng.choice(["mlp", "layer"]) if rows <= 2048 else "mlp", rows, dtype, block, model=rng.choice(["7b", "8b", "70b"]), accuracy=4, graph=rows <= 16,
                  zero_points=rng.random() < 0.7)
    elif kind == "f32":
        c = _case("", rng.choice(["mlp", "layer"]), _log_int(rng, 1, 512), "f32", block, model="0.5b", zero_points=rng.random() < 0.5)
    elif kind == "nbits":
        rows = _log_int(rng, 1, 2048)
        c = _case("", "mlp", rows, dtype, block, model=rng.choice(["7b", "8b"]), bits=rng.choice([2, 8, 8]), graph=rows <= 16, zero_points=rng.random() < 0.7)
    else:
        rows = _log_int(rng, 1, 2048)
        c = _case("", rng.choice(["mlp", "layer"]), rows, dtype, block, model=rng.choice(["7b", "8b"]), act_order=True, graph=rows <= 16, zero_points=rng.random() < 0.7)
    del c["name"]
    return c


def _nodes(case):
    """[(name, kind, k, n)] of a pass in order; kind: plain | norm (RMS prologue) | residual (per-token bias) | swiglu (pair with prologue)."""
    if case["net"] == "proj":
        return [("proj", "plain", case["k"], case["n"])]
    h, qkv, kv, inter, vocab = MODELS[case["model"]]
    fused = case["fused"]
    layer = []
    if case["net"] != "mlp":
        if fused:
            layer.append(("qkv", "norm", h, qkv))
        elif qkv:
            layer.append(("qkv", "plain", h, qkv))
        else:
            layer += [("q", "plain", h, h), ("k", "plain", h, kv), ("v", "plain", h, kv)]
        layer.append(("o", "residual" if fused else "plain", h, h))
    if fused:
        layer.append(("gate_up", "swiglu", h, inter))
    elif qkv:
        layer.append(("gate_up", "plain", h, 2 * inter))
    else:
        layer += [("gate", "plain", h, inter), ("up", "plain", h, inter)]
    layer.append(("down", "residual" if fused else "plain", inter, h))
    nodes = layer * case["layers"]
    if case["net"] == "step":
        nodes.append(("head", "norm" if fused else "plain", h, vocab))
    return nodes


class Weights:
    """One projection's packed weights, scales and zero points in the ONNX layout, from the generator alone."""

    def __init__(self, g, k, n, case):
        bits, block = case["bits"], case["block"]
        kb = -(-k // block)
        self.b = torch.randint(-2**63, 2**63 - 1, (n * kb * block * bits // 64,), dtype=torch.int64, device="cuda", generator=g).view(torch.uint8)
        # columns of unit gain: |q - zp| is about 2^bits * 0.41 with random zero points, 0.29 without
        spread = (0.41 if case["zero_points"] else 0.29) * 2 ** bits
        self.scales = ((torch.rand((n, kb), device="cuda", generator=g) + 0.5) / (spread * math.sqrt(k))).to(TORCH[case["dtype"]])
        self.zp = torch.randint(0, 256, (n, (kb * bits + 7) // 8), dtype=torch.uint8, device="cuda", generator=g) if case["zero_points"] else None
        self.g_idx = None
        if case["act_order"]:
            order = torch.randperm(k, device="cuda", generator=g)
            self.g_idx = torch.empty(k, dtype=torch.int32, device="cuda")
            self.g_idx[order] = (torch.arange(k, device="cuda") // block).to(torch.int32)
        dt = CODE[case["dtype"]]
        self.b_view = E.TensorView(self.b.data_ptr(), E.U8, (n, kb, block * bits // 8))
        self.s_view = E.TensorView(self.scales.data_ptr(), dt, (n, kb))
        self.z_view = E.TensorView(self.zp.data_ptr(), E.U8, tuple(self.zp.shape)) if self.zp is not None else E.TensorView.absent(E.U8)
        self.g_view = E.TensorView(self.g_idx.data_ptr(), E.I32, (k,)) if self.g_idx is not None else E.TensorView.absent(E.I32)


class Node:
    """A MatMulNBits node with its weights, as a session keeps it; calling it enqueues one execute."""

    def __init__(self, g, kind, k, n, case):
        self.k, self.n, self.kind, self.code = k, n, kind, CODE[case["dtype"]]
        self.w = Weights(g, k, n, case)
        attrs = {"K": k, "N": n, "bits": case["bits"], "block_size": case["block"], "accuracy_level": case["accuracy"]}
        if kind in ("norm", "swiglu"):
            self.gamma = (torch.rand(k, device="cuda", generator=g) * 0.5 + 0.75).to(TORCH[case["dtype"]])
            gamma = E.TensorView(self.gamma.data_ptr(), self.code, (k,))
            attrs.update(rmsnorm_prologue=1, rmsnorm_epsilon=1e-6)
        w = self.w
        if kind == "swiglu":
            self.up = u = Weights(g, k, n, case)
            attrs.update(gate_up_swiglu=1)
            self.rest = [w.b_view, w.s_view, u.b_view, u.s_view, gamma] + ([w.z_view, u.z_view] if w.zp is not None else [])
        elif kind == "norm":
            self.rest = [w.b_view, w.s_view, w.z_view, w.g_view, E.TensorView.absent(self.code), gamma]
        else:
            self.rest = [w.b_view, w.s_view] + ([w.z_view] if w.zp is not None or w.g_idx is not None or kind == "residual" else [])
            if w.g_idx is not None or kind == "residual":
                self.rest.append(w.g_view)
        self.kernel = provider().get_kernel(attrs)
        self.kernel.set_constant_inputs([False] + [True] * len(self.rest) if kind != "residual" else [False, True, True, True, True, False])

    def __call__(self, x, y, residual=None):
        inputs = [E.TensorView(x.data_ptr(), self.code, (x.shape[0], self.k))] + self.rest
        if residual is not None:
            inputs.append(E.TensorView(residual.data_ptr(), self.code, (x.shape[0], self.n)))
        self.kernel.execute(inputs, [E.TensorView(y.data_ptr(), self.code, (x.shape[0], self.n))])


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dt, m = TORCH[case["dtype"]], case["rows"]
    randn = lambda *shape: torch.randn(shape, device="cuda", generator=g, dtype=torch.float32).to(dt)  # noqa: E731
    nodes = [(name, Node(g, kind, k, n, case)) for name, kind, k, n in _nodes(case)]
    h = MODELS[case["model"]][0] if case["model"] else case["k"]
    layers = case["layers"]
    state = {"nodes": nodes, "x": randn(m, h), "out": {}}
    if case["net"] in ("layer", "step"):
        state["attention"] = randn(layers, m, h)
    if not case["fused"] and case["net"] != "proj":
        state["act"] = randn(layers, m, MODELS[case["model"]][3])
    for name, node in nodes:
        if name not in state["out"]:
            count = 1 if name in ("head", "proj") else layers
            state["out"][name] = torch.empty((count, m, node.n), dtype=dt, device="cuda")
    torch.cuda.synchronize()
    if case["graph"]:
        # a decode loop runs its step once, then records it
        _enqueue(state)
        ep = provider()
        ep.sync()
        ep.capture_begin()
        _enqueue(state)
        state["graph"] = ep.capture_end()
    return state


def _enqueue(s):
    x, out, layer = s["x"], s["out"], 0
    after_o = x                                           # what gate/up reads; an mlp net has no o in front of it
    for name, node in s["nodes"]:
        if name in ("proj", "head"):
            node(x, out[name][0])
            continue
        y = out[name][layer]
        residual = node.kind == "residual"
        if name == "o":
            node(s["attention"][layer], y, x if residual else None)
            after_o = y
        elif name == "gate_up" or name == "gate" or name == "up":
            node(after_o, y)
        elif name == "down":
            node(out["gate_up"][layer] if residual else s["act"][layer], y, after_o if residual else None)
            x = after_o = y
            layer += 1
        else:
            node(x, y)


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        _enqueue(state)
    return state["out"]


def work(case):
    m, item = case["rows"], 4 if case["dtype"] == "f32" else 2
    nbytes = flops = 0
    for _, kind, k, n in _nodes(case):
        kb = -(-k // case["block"])
        columns = 2 * n if kind == "swiglu" else n
        nbytes += columns * (kb * case["block"] * case["bits"] // 8 + kb * item + ((kb * case["bits"] + 7) // 8 if case["zero_points"] else 0))
        nbytes += m * (k + n * (2 if kind == "residual" else 1)) * item
        nbytes += (k * item if kind in ("norm", "swiglu") else 0) + (k * 4 if case["act_order"] else 0)
        flops += 2 * m * k * columns
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what a pass differs by from its float64 evaluation with the same roundings between nodes (worst output):
    f32 2.2e-7 (longer chains of sums reach 1e-6); f16 4.7e-4 (weights rounded to f16 in tall calls), 28 normalized layers
    about an eighth of bf16's; bf16 2.6e-3 for one node, 1.0e-2 (largest 0.15) behind 28 normalized layers, where every
    rounding of the residual stream feeds the layers after it."""
    if case["dtype"] == "f32":
        return {"rel": 4e-6}
    deep = case["net"] == "step" and case["fused"]
    if case["dtype"] == "f16":
        return {"rel": 5e-3 if deep else 2e-3}
    return {"rel": 3e-2, "max": 0.6} if deep else {"rel": 1e-2}
