"""Timed cases of the routed-expert MoE layer, each through the package's public entry points.

A case is one layer configuration (widths, experts, quantization, activation, routing rule), a
token count and the way a program calls it:

  block   `MoELayer(x)`, fully resident experts, `layers` layers called one after another
  graph   `brx_moe_block_forward_noalloc` of `layers` layers captured in a HIP graph, one replay
          a pass (a decode step of a stack; every layer has its own input, as attention sits
          between a model's MoE layers)
  rows    `StreamingSwitchGLU(x, indices)`: the unreduced rows for a routing the caller made
  pool    `MoELayer(x)` token after token over a pool that holds `capacity` of the experts, the
          misses copied in from pinned host memory

Weights are N(0, 0.02), quantized here; router weights N(0, 0.02), inputs N(0, 1), and a Zipf
bias on the router where `zipf` is set (a few experts take most of the tokens, as in a trained
model). Everything is made on the GPU from the seed alone.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from bigrig_amd import formats as F
from bigrig_amd import lib as L
from bigrig_amd.layer import MoELayer, StreamingSwitchGLU
from bigrig_amd.pool import ExpertPool, HostStore, PinnedFetcher
from bigrig_amd.spec import LayerSpec

DEV = "cuda"

# The layer shapes of the package's own configurations.
_QWEN3 = dict(hidden=2048, inter=768, experts=128, top_k=8, mode="affine", bits=4, group=64,
              f16=False, bias=False, act="swiglu", route="softmax_topk_renorm", router_f32=False,
              shared=0, n_group=0, topk_group=0, zipf=1.1, capacity=0)
_OLMOE = dict(_QWEN3, inter=1024, experts=64, route="softmax_topk", router_f32=True, zipf=0.0)
_E256 = dict(_QWEN3, inter=512, experts=256, shared=512)
_GPTOSS = dict(_QWEN3, hidden=2880, inter=2880, top_k=4, mode="mxfp4", group=32, bias=True,
               act="swiglu_clamped", route="topk_softmax", zipf=0.0)


def _case(name, kind, shape, tokens, layers=1, **kw):
    return dict(shape, **kw, name=name, kind=kind, tokens=tokens, layers=layers)


def listed():
    return [
        # one token through one layer, called eagerly: the smallest call, launches and host time
        _case("decode1-eager", "block", _QWEN3, 1),
        # single-user generation: one token through a stack of layers, replayed as a graph (the
        # layers' hit experts together exceed the last-level cache, as a whole model's do)
        _case("decode1-stack", "graph", _QWEN3, 1, 16),
        # the same with large MXFP4 experts
        _case("decode1-mxfp4", "graph", _GPTOSS, 1, 8),
        # a few users, or a short speculative step: 3 tokens, fp32 router
        _case("decode3-f32router", "graph", _OLMOE, 3, 8),
        # 8 users of a many-expert layer with an always-on shared expert
        _case("decode8-shared", "graph", _E256, 8, 8),
        # a server's decode step for 32 users, two layers
        _case("batch32", "block", _QWEN3, 32, 2),
        # a short prompt through large MXFP4 experts: every expert hit by few tokens
        _case("prefill512-mxfp4", "block", _GPTOSS, 512),
        # an ordinary prompt chunk
        _case("prefill2048", "block", _QWEN3, 2048),
        # the bare operator in 3 bits on an odd chunk, the program routing and combining itself
        _case("rows777-3bit", "rows", _QWEN3, 777, bits=3),
        # an odd chunk of a sigmoid, group-limited layer in 8 bits with fp16 scales
        _case("prefill301-sigmoid-8bit", "block", _E256, 301, bits=8, f16=True,
              route="sigmoid_topk_renorm", n_group=8, topk_group=4, zipf=0.0),
        # a long chunk of an unquantized layer
        _case("prefill4096-bf16", "block", _QWEN3, 4096, mode="none", bits=16, group=0),
        # generation with a quarter of the experts resident: 64 tokens, misses over the bus
        _case("pool-decode64-3bit", "pool", _QWEN3, 64, bits=3, capacity=32),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the listed ones' ranges: decode steps of 1 to 8 tokens, batches and chunks of 9
    to 4096, the package's shapes or others of their range, every quantization."""
    shape = dict(rng.choice([_QWEN3, _QWEN3, _OLMOE, _E256, _GPTOSS]))
    if rng.random() < 0.6:      # widths and expert counts of the same range
        shape.update(hidden=64 * rng.randint(8, 45), inter=64 * rng.randint(3, 45),
                     experts=rng.choice([8, 16, 32, 60, 64, 96, 128, 160, 256]))
        shape["top_k"] = min(shape["top_k"], shape["experts"])
        if shape["shared"]:
            shape["shared"] = 64 * rng.randint(3, 32)
    if shape["mode"] == "affine":
        q = rng.choice([(4, 64), (4, 64), (3, 64), (2, 64), (6, 64), (8, 64), (4, 128), (16, 0)])
        if q[1] == 128 and (shape["hidden"] | shape["inter"] | shape["shared"]) % 128:
            q = (q[0], 64)
        shape.update(bits=q[0], group=q[1], mode="none" if q[0] == 16 else "affine")
        shape["f16"] = shape["mode"] == "affine" and rng.random() < 0.3
    if shape["route"] == "softmax_topk_renorm" and rng.random() < 0.2:
        shape.update(route="sigmoid_topk_renorm", zipf=0.0)
    kind = rng.choice(["graph", "block", "block", "rows"])
    if kind == "graph":
        tokens = rng.randint(1, 8)
        while tokens * shape["top_k"] > 64:
            tokens -= 1
        layers = 8
    else:
        tokens = _log_int(rng, 1, 4096)
        layers = 1
    c = dict(shape, kind=kind, tokens=tokens, layers=layers)
    # no more weight than 8 layers of the largest listed stack, no more arithmetic than the
    # longest listed chunk
    while c["layers"] > 1 and c["layers"] * c["experts"] * _expert_bytes(c) > 13e9:
        c["layers"] //= 2
    while work(c)["flops"] > 300e9:
        c["tokens"] = c["tokens"] * 3 // 4
    return c


# ------------------------------------------------------------------ weights
def _spec(c):
    quant = F.QuantSpec(c["bits"], c["group"], c["mode"], "float16" if c["f16"] else "bfloat16")
    return LayerSpec(c["hidden"], c["inter"], c["experts"], c["top_k"], quant=quant,
                     has_bias=c["bias"], act=c["act"], route=c["route"],
                     router_dtype="float32" if c["router_f32"] else "bfloat16",
                     shared_inter=c["shared"], n_group=c["n_group"], topk_group=c["topk_group"])


def _expert_bytes(c, shared=False):
    inter = c["shared"] if shared else c["inter"]
    n = c["hidden"] * inter
    per = n * c["bits"] // 8
    if c["mode"] == "affine":
        per += n // c["group"] * 4
    elif c["mode"] == "mxfp4":
        per += n // 32
    b = 2 * (2 * inter + c["hidden"]) if c["bias"] else 0
    return 3 * per + b


def _gen(seed, *tags):
    g = torch.Generator(device=DEV)
    v = seed & 0xFFFFFFFF
    for t in tags:
        v = (v * 1000003 + t + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(v)
    return g


_FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _quantize(w, c):
    """w [n, N, K] fp32 -> (list of byte tensors [n, bytes] in the packed order, a function of an
    index that gives that expert's dequantized weight in fp64)."""
    n, N, K = w.shape
    as_bytes = lambda t: t.contiguous().view(torch.uint8).reshape(n, -1)  # noqa: E731
    if c["mode"] == "none":
        wb = w.to(torch.bfloat16)
        return [as_bytes(wb)], lambda i: wb[i].double()
    if c["mode"] == "mxfp4":
        g = w.view(n, N, K // 32, 32)
        e = (torch.floor(torch.log2(g.abs().amax(-1).clamp_min(1e-30))) - 2).clamp(-127, 127)
        a = g * torch.exp2(-e)[..., None]
        mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
        code = torch.bucketize(a.abs(), mid, out_int32=True).to(torch.uint8)
        code |= (a < 0).to(torch.uint8) << 3
        pairs = code.view(n, N, K // 2, 2)
        packed = pairs[..., 0] | (pairs[..., 1] << 4)
        sc = (e + 127).to(torch.uint8)

        def deq(i):
            q = code[i].int()
            v = torch.tensor(_FP4, device=DEV, dtype=torch.float64)[(q & 7).long()]
            v = torch.where(q >= 8, -v, v) * torch.exp2(e[i].double())[..., None]
            return v.reshape(N, K)
        return [as_bytes(packed), as_bytes(sc)], deq
    G, b = c["group"], c["bits"]
    sdt = torch.float16 if c["f16"] else torch.bfloat16
    top = float((1 << b) - 1)
    g = w.view(n, N, K // G, G)
    lo, hi = g.amin(-1), g.amax(-1)
    step = ((hi - lo) / top).clamp_min(1e-7)
    down = hi.abs() >= lo.abs()          # codes count down from the end of larger magnitude
    s = torch.where(down, -step, step).to(sdt)
    o = torch.where(down, hi, lo).to(sdt)
    code = torch.round((g - o.float()[..., None]) / s.float()[..., None]).clamp_(0, top)
    code = code.to(torch.uint8).view(n, N, K)
    if b == 8:
        packed = code
    else:                                # 8 codes a run of b bytes, least significant bits first
        run = torch.zeros((n, N, K // 8), dtype=torch.int64, device=DEV)
        c8 = code.view(n, N, K // 8, 8)
        for j in range(8):
            run |= c8[..., j].long() << (b * j)
        packed = torch.stack([(run >> (8 * j)).to(torch.uint8) for j in range(b)], -1)

    def deq(i):
        q = code[i].view(N, K // G, G).double()
        return (q * s[i].double()[..., None] + o[i].double()[..., None]).view(N, K)
    return [as_bytes(packed), as_bytes(s), as_bytes(o)], deq


def _experts(c, seed, layer, shared=False):
    """The layer's experts in runs: yields (first expert, packed bytes [n, bytes], dequantizers
    of gate, up and down, their biases)."""
    E = 1 if shared else c["experts"]
    inter = c["shared"] if shared else c["inter"]
    H = c["hidden"]
    step = max(1, min(E, (1 << 25) // (H * inter)))
    for e0 in range(0, E, step):
        n = min(step, E - e0)
        parts, deqs, biases = [], [], []
        for p, (N, K) in enumerate([(inter, H), (inter, H), (H, inter)]):
            g = _gen(seed, layer, e0 + (100000 if shared else 0), p)
            w = torch.randn((n, N, K), generator=g, device=DEV) * 0.02
            by, dq = _quantize(w, c)
            parts += by
            deqs.append(dq)
            if c["bias"]:
                bv = (torch.randn((n, N), generator=g, device=DEV) * 0.02).to(torch.bfloat16)
                parts.append(bv.view(torch.uint8).reshape(n, -1))
                biases.append(bv)
        yield e0, torch.cat(parts, 1), deqs, biases


def _inputs(c, seed, layer):
    """(x [T, H] bf16, router weight, router bias or None, shared gate row or None)."""
    H, E = c["hidden"], c["experts"]
    g = _gen(seed, layer, 777777)
    x = torch.randn((c["tokens"], H), generator=g, device=DEV).to(torch.bfloat16)
    wr = torch.randn((E, H), generator=g, device=DEV) * 0.02
    if not c["router_f32"]:
        wr = wr.to(torch.bfloat16)
    bias = None
    if c["zipf"]:
        rank = torch.randperm(E, generator=g, device=DEV).double()
        bias = (-c["zipf"] * torch.log(rank + 1.0)).float()
    elif c["route"].startswith("sigmoid"):
        bias = torch.rand(E, generator=g, device=DEV) * 0.2     # a score-correction bias
    sgw = (torch.randn(H, generator=g, device=DEV) * 0.02).to(torch.bfloat16) if c["shared"] else None
    return x, wr, bias, sgw


def _indices(c, seed):
    """A routing [T, k] int32, drawn without repeats from the Zipf-weighted experts."""
    E = c["experts"]
    g = _gen(seed, 888888)
    z = -(c["zipf"] or 0.0) * torch.log(torch.randperm(E, generator=g, device=DEV).double() + 1.0)
    u = torch.rand((c["tokens"], E), generator=g, device=DEV, dtype=torch.float64)
    z = z - torch.log(-torch.log(u.clamp(1e-12, 1 - 1e-12)))
    return z.topk(c["top_k"], -1).indices.int().contiguous()


def _resident_layer(c, seed, layer):
    spec = _spec(c)
    pool = ExpertPool(layer, spec, c["experts"]).build()
    for e0, by, _, _ in _experts(c, seed, layer):
        for i in range(by.shape[0]):
            pool.touch([e0 + i], [0])
            pool.admit_device(e0 + i, by[i].data_ptr())
        pool.device.sync()
    return spec, pool


def _shared(c, seed, layer):
    if not c["shared"]:
        return None
    return next(_experts(c, seed, layer, shared=True))[1][0].contiguous()


class _State:
    """What a program holds between calls. The pools are closed with it."""

    def __init__(self, kind):
        self.kind = kind
        self.pools, self.layers, self.xs, self.keep = [], [], [], []
        self.graph = self.outs = self.indices = None

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.graph = None
            for p in self.pools:
                p.close()
        except Exception:
            pass


def prepare(case, seed):
    c = case
    L.init(0)
    st = _State(c["kind"])
    if c["kind"] == "pool":
        spec = _spec(c)
        per = _expert_bytes(c)
        host = torch.empty((c["experts"], per), dtype=torch.uint8, pin_memory=True)
        for e0, by, _, _ in _experts(c, seed, 0):
            host[e0:e0 + by.shape[0]].copy_(by)
        store = HostStore()
        store.add_layer_tensor(0, host)
        pool = ExpertPool(0, spec, c["capacity"]).build()
        sw = StreamingSwitchGLU(pool, PinnedFetcher(store))
        sw.refresh()
        x, wr, bias, _ = _inputs(c, seed, 0)
        st.pools.append(pool)
        st.layers.append(MoELayer(spec, wr, sw, router_bias=bias))
        st.xs = [x[t:t + 1] for t in range(c["tokens"])]
        torch.cuda.synchronize()
        return st
    for l in range(c["layers"]):
        spec, pool = _resident_layer(c, seed, l)
        shared = _shared(c, seed, l)
        x, wr, bias, sgw = _inputs(c, seed, l)
        sw = StreamingSwitchGLU(pool, None, shared=shared)
        sw.refresh()
        st.pools.append(pool)
        st.layers.append(MoELayer(spec, wr, sw, router_bias=bias, shared_gate_w=sgw))
        st.xs.append(x)
        pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    if c["kind"] == "rows":
        st.indices = _indices(c, seed)
    if c["kind"] == "graph":
        _capture(st, c)
    torch.cuda.synchronize()
    return st


def _capture(st, c):
    lib = L.load()
    st.outs = [torch.empty((c["tokens"], c["hidden"]), dtype=torch.bfloat16, device=DEV)
               for _ in st.layers]
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731

    def step():
        sp = torch.cuda.current_stream().cuda_stream
        for m, x, out in zip(st.layers, st.xs, st.outs):
            d = m.spec.desc()
            st.keep.append(d)
            L.check(lib.brx_moe_block_forward_noalloc(
                ctypes.byref(d), m.switch._pool.device.handle, x.data_ptr(), m.router_w.data_ptr(),
                ptr(m.router_bias), ptr(m.shared_gate_w), ptr(m.switch.shared), c["tokens"],
                out.data_ptr(), None, None, L.FWD_FORCE_DECODE, sp))
    step()
    torch.cuda.synchronize()
    st.graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st.graph):
        step()
    torch.cuda.synchronize()


def run(state):
    if state.kind == "graph":
        state.graph.replay()
        return state.outs
    if state.kind == "rows":
        return state.layers[0].switch(state.xs[0], state.indices)
    if state.kind == "pool":
        m = state.layers[0]
        return [m(x) for x in state.xs]
    return [m(x) for m, x in zip(state.layers, state.xs)]


# ------------------------------------------------------------------ what a pass has to do
def _distinct(c):
    """Experts a layer's tokens hit, for logits of the drawn distribution (a fixed sample)."""
    E, k, T = c["experts"], c["top_k"], c["tokens"]
    rng = np.random.default_rng(5)
    z = -c["zipf"] * np.log(np.arange(E) + 1.0)
    hit = np.zeros(E, bool)
    z = rng.standard_normal((T, E)) * (0.02 * math.sqrt(c["hidden"])) + z
    hit[np.argpartition(-z, k - 1, 1)[:, :k].reshape(-1)] = True
    return int(hit.sum())


def work(case):
    c = case
    H, I, T, k, E = c["hidden"], c["inter"], c["tokens"], c["top_k"], c["experts"]
    by = _distinct(c) * _expert_bytes(c) + 2 * T * H
    fl = 6 * T * k * H * I
    if c["kind"] == "rows":
        by += 2 * T * k * H + 4 * T * k
    else:
        by += 2 * T * H + E * H * (4 if c["router_f32"] else 2)
        fl += 2 * T * E * H
        if c["shared"]:
            by += _expert_bytes(c, shared=True) + 2 * H
            fl += 6 * T * H * c["shared"]
    return {"bytes": by * c["layers"], "flops": fl * c["layers"]}


def tolerance(case):
    # bf16 activations between the two projections and bf16 results; prefill also rounds the
    # dequantized weights to bf16. Measured against 64 bits: 2.7e-3 to 4.1e-3.
    return {"rel": 1.6e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _route64(c, x, wr, bias):
    """(indices, weights) of the layer's rule."""
    lg = x.double() @ wr.double().T
    k = c["top_k"]
    if c["route"].startswith("sigmoid"):
        s = torch.sigmoid(lg)
        sel = s + bias.double() if bias is not None else s
        if c["n_group"] > 1:
            g = sel.view(sel.shape[0], c["n_group"], -1)
            keep = g.topk(2, -1).values.sum(-1).topk(c["topk_group"], -1).indices
            m = torch.zeros(g.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, keep, True)
            sel = torch.where(m[..., None], g, torch.zeros_like(g)).view_as(sel)
        idx = sel.topk(k, -1).indices
        w = s.gather(1, idx)
        return idx, w / w.sum(-1, keepdim=True) if c["route"].endswith("renorm") else w
    if bias is not None:
        lg = lg + bias.double()
    v, idx = lg.topk(k, -1)
    if c["route"] == "topk_softmax":
        return idx, torch.softmax(v, -1)
    w = torch.softmax(lg, -1).gather(1, idx)
    return idx, w / w.sum(-1, keepdim=True) if c["route"].endswith("renorm") else w


def _mlp64(c, x, i, deqs, biases):
    g = x @ deqs[0](i).T
    u = x @ deqs[1](i).T
    if biases:
        g, u = g + biases[0][i].double(), u + biases[1][i].double()
    if c["act"] == "swiglu_clamped":
        g = g.clamp(max=7.0)
        u = u.clamp(-7.0, 7.0) + 1.0
        h = g * torch.sigmoid(1.702 * g) * u
    else:
        h = g * torch.sigmoid(g) * u
    y = h @ deqs[2](i).T
    return y + biases[2][i].double() if biases else y


def exact(case, seed):
    c = case
    outs = []
    for l in range(c["layers"]):
        x, wr, bias, sgw = _inputs(c, seed, l)
        if c["kind"] == "rows":
            idx, w = _indices(c, seed).long(), None
        else:
            idx, w = _route64(c, x, wr, bias)
        x64 = x.double()
        y = torch.zeros((c["tokens"], c["top_k"], c["hidden"]), dtype=torch.float64, device=DEV)
        for e0, by, deqs, biases in _experts(c, seed, l):
            for i in range(by.shape[0]):
                t, j = (idx == e0 + i).nonzero(as_tuple=True)
                if t.numel():
                    y[t, j] = _mlp64(c, x64[t], i, deqs, biases)
        if w is None:
            return y
        out = (y * w[..., None]).sum(1)
        if c["shared"]:
            _, _, deqs, biases = next(_experts(c, seed, l, shared=True))
            gate = torch.sigmoid(x64 @ sgw.double())
            out += gate[:, None] * _mlp64(c, x64, 0, deqs, biases)
        outs.append(out)
    if c["kind"] == "pool":
        return [outs[0][t:t + 1] for t in range(c["tokens"])]
    return outs
