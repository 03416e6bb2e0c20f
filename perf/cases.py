"""Cases of the MoE-layer path, from a decode token to a large skewed prefill.

A case is one pass of a program's own work through the public entry points:
``layer.moe_forward`` over experts that are resident in HBM (the whole layer:
router, grouping, SwiGLU experts, weighted merge), or one
``PDScopeCudaRuntime.forward`` call.  Shapes are the two that
``pdscope_amd.synthetic`` names and two smaller ones of the tests; weights and
tokens are its seeded synthetic layers (experts and routers N(0, 0.02),
activations N(0, 1), all bf16).

Decode-sized batches (up to 64 tokens) run as a serving loop runs them: the
layers of the pass are captured in one graph when the program starts, and a
pass replays it.  Their pass covers several layers, so that a layer's weights
come from HBM as they do in a deep stack and not from the cache that the last
pass left.  Larger batches are one eager call.
"""
import math

import torch

from pdscope_amd import layer, ops, synthetic
from pdscope_amd.cache import ExpertKey
from pdscope_amd.executor import masters_from_block
from pdscope_amd.pdscope_runtime import PDScopeCudaRuntime

DEV = "cuda"

SHAPES = {
    # Qwen3-30B-A3B layer and DeepSeek-V2-Lite layer (2 shared experts as one 2816-wide MLP)
    "qwen": dict(H=2048, I=768, E=128, k=8, normalize=True, shared_I=0),
    "dsv2": dict(H=2048, I=1408, E=64, k=6, normalize=False, shared_I=2816),
    # smaller layers: fewer experts, a narrower hidden size
    "small": dict(H=1024, I=512, E=64, k=4, normalize=True, shared_I=0),
    "narrow": dict(H=1536, I=384, E=96, k=6, normalize=True, shared_I=0),
}
GRAPH_MAX_T = 64


def listed():
    return [
        # one token of one request through 8 resident layers: the decode step
        # of a single user, where latency counts
        dict(name="decode_qwen_t1", path="layer", shape="qwen", T=1, layers=8, merge="fused", zipf=False),
        # the same for a model with always-on shared experts
        dict(name="decode_dsv2_t1", path="layer", shape="dsv2", T=1, layers=6, merge="fused", zipf=False),
        # decode steps of a few concurrent requests: each token picks its own
        # experts, so most expert rows are alone
        dict(name="decode_qwen_t4", path="layer", shape="qwen", T=4, layers=4, merge="fused", zipf=False),
        dict(name="decode_qwen_t17", path="layer", shape="qwen", T=17, layers=2, merge="reference", zipf=False),
        # the decode half of a mixed serving batch, 48 requests
        dict(name="decode_dsv2_t48", path="layer", shape="dsv2", T=48, layers=2, merge="fused", zipf=False),
        # a short prompt, an odd length
        dict(name="prefill_qwen_t201", path="layer", shape="qwen", T=201, layers=1, merge="reference", zipf=False),
        # a prompt through the small layer
        dict(name="prefill_small_t777", path="layer", shape="small", T=777, layers=1, merge="fused", zipf=False),
        # the prefill of a medium prompt: every expert has a few dozen rows
        dict(name="prefill_qwen_t512", path="layer", shape="qwen", T=512, layers=1, merge="fused", zipf=False),
        # a mixed batch of decode tokens and two prompt chunks (48 + 256 + 1000)
        dict(name="mixed_dsv2_t1304", path="layer", shape="dsv2", T=1304, layers=1, merge="fused", zipf=False),
        # long prompts: uniform routing, and a skewed one where a few experts
        # take most of the tokens
        dict(name="prefill_qwen_t4096", path="layer", shape="qwen", T=4096, layers=1, merge="reference", zipf=False),
        dict(name="prefill_qwen_t4096_zipf", path="layer", shape="qwen", T=4096, layers=1, merge="fused", zipf=True),
        # the whole runtime call of a prompt (routing, ledger, launches, trace
        # row) with every expert resident
        dict(name="runtime_qwen_t512", path="runtime", shape="qwen", T=512, layers=1, merge="reference", zipf=False),
    ]


def draw(rng):
    path = "runtime" if rng.random() < 0.1 else "layer"
    lo = 16 if path == "runtime" else 1
    hi = 2048 if path == "runtime" else 4096
    T = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    shape = "qwen" if path == "runtime" else rng.choice(["qwen", "qwen", "dsv2", "small", "narrow"])
    layers = 1
    if path == "layer" and T <= GRAPH_MAX_T:
        layers = 8 if T == 1 else 4 if T <= 8 else 2
    return dict(path=path, shape=shape, T=T, layers=layers, merge=rng.choice(["fused", "reference"]),
                zipf=path == "layer" and rng.random() < 0.25)


def _make(case, seed, i):
    """Layer i of a case: its synthetic weights, tokens and router bias."""
    s = SHAPES[case["shape"]]
    base = 1_000_003 * (int(seed) % 1_000_000) + 101 * i
    lay = synthetic.make_layer(s["H"], s["I"], s["E"], s["k"], s["normalize"], seed=base, device=DEV,
                               shared_I=s["shared_I"] or None)
    x = synthetic.make_tokens(case["T"], s["H"], seed=base + 7, device=DEV)
    bias = synthetic.zipf_bias(s["E"], 1.1, seed=base + 11, device=DEV)[0] if case["zipf"] else None
    return lay, x, bias


class _Layers:
    """Resident layers with their slot tables and workspaces, captured in one
    graph for decode-sized batches."""

    def __init__(self, case, seed):
        s = SHAPES[case["shape"]]
        T = case["T"]
        self.merge = case["merge"]
        self.items = []
        for i in range(case["layers"]):
            lay, x, bias = _make(case, seed, i)
            slots = ops.slot_table([lay.experts[e] for e in range(s["E"])], DEV)
            shared = ops.slot_table([lay.shared], DEV) if s["shared_I"] else None
            ws = layer.MoEWorkspace(T, s["H"], s["I"], s["E"], s["k"], DEV, shared_I=s["shared_I"] or None)
            self.items.append((lay, x, bias, slots, shared, ws))
        self.graph = None
        if T <= GRAPH_MAX_T:
            cur, side = torch.cuda.current_stream(), torch.cuda.Stream()
            side.wait_stream(cur)
            with torch.cuda.stream(side):
                self.eager()
            cur.wait_stream(side)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                self.outputs = self.eager()
            self.graph = graph

    def eager(self):
        return [layer.moe_forward(x, lay.gate, slots, ws, normalize=lay.normalize, bias=bias, shared_slot=shared,
                                  merge=self.merge)
                for lay, x, bias, slots, shared, ws in self.items]

    def run(self):
        if self.graph is None:
            return self.eager()
        self.graph.replay()
        return self.outputs


class _Runtime:
    """One layer behind PDScopeCudaRuntime, every expert resident; each pass
    is the prefill of a new request."""

    def __init__(self, case, seed):
        s = SHAPES[case["shape"]]
        lay, self.x, _ = _make(case, seed, 0)
        masters = masters_from_block(0, lay.experts, s["E"], s["H"], s["I"])
        self.gate, self.k, self.normalize = lay.gate, s["k"], s["normalize"]
        del lay
        hot = [ExpertKey(0, e, "bf16") for e in range(s["E"])]
        self.rt = PDScopeCudaRuntime(masters, hot_keys=hot, speculative_slots=0, demand_slots=8,
                                     device=torch.device("cuda", torch.cuda.current_device()), diagnostics=False,
                                     merge=case["merge"])
        self.requests = 0

    def run(self):
        self.requests += 1
        out, routing, _ = self.rt.forward(self.x, self.gate, layer=0, step=0, request=f"r{self.requests}",
                                          top_k=self.k, normalize=self.normalize, prefetch=False)
        return [(out, routing.logits, routing.selected, routing.weights)]

    def __del__(self):
        rt = getattr(self, "rt", None)
        if rt is not None:
            rt.close()


def prepare(case, seed):
    return (_Runtime if case["path"] == "runtime" else _Layers)(case, seed)


def run(state):
    return state.run()


def work(case):
    """Router and touched expert weights, tokens in and results out, once
    each; the multiply-adds of the router, the routed rows and the shared
    experts.  Touched experts: the expected number for uniform routing, or for
    Zipf(1.1) shares of k draws without replacement (approximated)."""
    s = SHAPES[case["shape"]]
    H, I, E, k, T = s["H"], s["I"], s["E"], s["k"], case["T"]
    if case["zipf"]:
        p = [r ** -1.1 for r in range(1, E + 1)]
        total = sum(p)
        hit = [1 - (1 - v / total) ** k for v in p]
    else:
        hit = [k / E] * E
    touched = sum(1 - (1 - h) ** T for h in hit)
    if T == 1:
        touched = k
    expert = 3 * H * I * 2
    byts = touched * expert + E * H * 2 + 2 * T * H * 2 + T * E * 2 + T * k * 6 + 3 * s["shared_I"] * H * 2
    flops = 2.0 * T * H * (E + 3 * I * k + 3 * s["shared_I"])
    return {"bytes": byts * case["layers"], "flops": flops * case["layers"]}


def exact(case, seed):
    """The layer in 64 bits.  The router's logits are bf16 by definition
    (the selection is made on the rounded values, equal ones in order of the
    expert id), so the selection uses the rounded logits; every other value
    is not rounded at all."""
    s = SHAPES[case["shape"]]
    H, I, E, k = s["H"], s["I"], s["E"], s["k"]
    results = []

    def mlp(rows, block, width):
        g = block[:width * H].view(width, H).double()
        u = block[width * H:2 * width * H].view(width, H).double()
        d = block[2 * width * H:].view(H, width).double()
        return (torch.nn.functional.silu(rows @ g.T) * (rows @ u.T)) @ d.T

    for i in range(case["layers"]):
        lay, x, bias = _make(case, seed, i)
        xd = x.double()
        logits = xd @ lay.gate.double().T
        seen = logits.to(torch.bfloat16).double()
        if bias is not None:
            seen = seen + bias.double()
        p = torch.softmax(seen, dim=1)
        order = torch.sort(p, dim=1, descending=True, stable=True)
        w, ids = order.values[:, :k], order.indices[:, :k]
        if s["normalize"]:
            w = w / w.sum(dim=1, keepdim=True)
        out = mlp(xd, lay.shared, s["shared_I"]) if s["shared_I"] else torch.zeros_like(xd)
        for e in range(E):
            t, slot = torch.nonzero(ids == e, as_tuple=True)
            if t.numel():
                out.index_add_(0, t, mlp(xd[t], lay.experts[e], I) * w[t, slot][:, None])
        results.append((out, logits, None, w))
        del lay, x
    return results


def tolerance(case):
    # bf16 results of bf16 operands: every expert value is rounded four times
    # on its way (gate, up, their product, the expert's row) and the merged
    # sum once more; the reference merge rounds after each of its k adds.
    # Ids differ where two rounded logits tie.
    return {"rel": 0.015 if case["merge"] == "reference" else 0.01, "max": 0.25, "differ": 0.002}
