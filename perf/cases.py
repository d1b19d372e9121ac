"""Performance cases: the work that programs have this package do, each through public entry points.

Five kinds of pass, at Qwen2.5-1.5B and 7B sizes (and, drawn, at others of the same range):

- serve:     one decoder layer's projections of a serving loop (q/k/v with biases in one call, o,
             the MLP), captured once in a HIP graph and replayed, as such a loop runs them; decode
             with one or a few sequences, batched decode, a short prefill chunk.
- linear:    a single NF4 projection through the autograd op that bitsandbytes' patched Linear4bit
             calls, eager, forward alone or forward and input gradient.
- mlp:       forward and backward of the Qwen2 MLP in QLoRA training, as the patched Qwen2MLP runs.
- attention: forward and backward of a layer's q/k/v/o with LoRA, dropout masks and RoPE.
- dequant:   the fp16 weights of a layer (merging or exporting a model, a fallback path).

Weights: four-bit codes of normally distributed values (NF4's quantiles make them equally likely),
64-element blocks whose absmax spreads around 2.4 standard deviations, double-quantized in groups
of 256 unless a case says otherwise. Activations are unit normal (norm outputs), gradients small.
"""

import math

import torch

from decik_amd import nf4
from decik_amd.lora import pack_keep, qkv_rope_projection
from decik_amd.mlp import FusedMLP, mlp_forward
from decik_amd.quant import QuantState, State2

# The NF4 code book (a data format).
CODES = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
         -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
         0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
         0.7229568362236023, 1.0]
GROUP = 256       # blocks per group of the second quantization
LORA_SCALE = 2.0  # alpha / r of the adapters


def listed():
    return [
        # chat on one stream: every projection of a 7B layer for a single token
        dict(name="decode_7b_1", kind="serve", m=1, hidden=3584, kv=512, inter=18944, layers=1),
        # a small model with a few streams; four layers, since one fits the caches
        dict(name="decode_1p5b_4", kind="serve", m=4, hidden=1536, kv=256, inter=8960, layers=4),
        # batched decode of a 7B model
        dict(name="decode_7b_16", kind="serve", m=16, hidden=3584, kv=512, inter=18944, layers=1),
        # a prefill chunk, or a large decode batch
        dict(name="prefill_7b_64", kind="serve", m=64, hidden=3584, kv=512, inter=18944, layers=1),
        # the smallest call there is: one token through a k or v projection, eager
        dict(name="linear_kv_1", kind="linear", m=1, n=256, k=1536, bias=True, grad=False, blocksize=64, nested=True),
        # odd sizes: rows that no tile divides, blocks that straddle weight rows, plain statistics
        dict(name="linear_ragged", kind="linear", m=333, n=2056, k=1120, bias=True, grad=True, blocksize=64,
             nested=False),
        # a short training batch through the largest 7B projection, both directions
        dict(name="linear_7b_512", kind="linear", m=512, n=18944, k=3584, bias=False, grad=True, blocksize=64,
             nested=True),
        # the fine-tuning step's attention projections at its usual packed length
        dict(name="attention_1p5b_830", kind="attention", m=830, heads=12, kv_heads=2, head_dim=128, rank=16,
             dropout=True),
        # the fine-tuning step's MLP, gate and up recomputed in the backward (the default)
        dict(name="mlp_1p5b_830", kind="mlp", m=830, hidden=1536, inter=8960, recompute=True),
        # a 7B MLP at a longer packed length, gate and up kept
        dict(name="mlp_7b_2048", kind="mlp", m=2048, hidden=3584, inter=18944, recompute=False),
        # long-context training or a large prefill: the largest call
        dict(name="linear_7b_8192", kind="linear", m=8192, n=3584, k=18944, bias=False, grad=True, blocksize=64,
             nested=True),
        # every weight of a 7B layer to fp16
        dict(name="dequant_7b", kind="dequant", hidden=3584, kv=512, inter=18944),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["serve", "serve", "serve", "linear", "linear", "linear", "mlp", "mlp", "attention", "dequant"])
    if kind == "linear":
        n, k = 8 * _log(rng, 16, 2368), 32 * _log(rng, 8, 592)
        m = _log(rng, 1, max(1, min(8192, 8192 * 18944 * 3584 // (n * k))))
        blocksize = rng.choice([64, 64, 64, 128])
        if (64 * k) % blocksize:
            blocksize = 64
        return dict(kind=kind, m=m, n=n, k=k, bias=rng.random() < 0.5, grad=rng.random() < 0.6, blocksize=blocksize,
                    nested=rng.random() < 0.8)
    if kind == "attention":
        heads, head_dim = rng.randint(4, 32), rng.choice([64, 128])
        kv_heads = rng.choice([h for h in (1, 2, 4, 8) if h <= heads])
        return dict(kind=kind, m=_log(rng, 16, 2048), heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                    rank=rng.choice([16, 16, 32]), dropout=rng.random() < 0.7)
    heads = rng.randint(4, 28)
    hidden, kv = 128 * heads, 128 * rng.choice([h for h in (1, 2, 4, 8) if h <= heads])
    inter = 64 * _log(rng, 16, 296)
    if kind == "dequant":
        return dict(kind=kind, hidden=hidden, kv=kv, inter=inter)
    if kind == "serve":
        return dict(kind=kind, m=_log(rng, 1, 192), hidden=hidden, kv=kv, inter=inter, layers=1)
    return dict(kind=kind, m=_log(rng, 16, 2048), hidden=hidden, inter=inter, recompute=rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------------------------

class _Source:
    """Random tensors on the GPU, made from the seed alone."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float16):
        return (torch.randn(shape, generator=self.g, device=self.dev) * std).to(dtype)

    def weight(self, n, k, blocksize=64, nested=True, std=0.02):
        """An NF4 weight as plain tensors: packed bytes and statistics."""
        blocks = -(-n * k // blocksize)
        w = dict(n=n, k=k, blocksize=blocksize, code=torch.tensor(CODES, device=self.dev),
                 packed=torch.randint(0, 256, (n * k // 2, 1), generator=self.g, device=self.dev, dtype=torch.uint8))
        absmax = (std * (2.4 + 0.35 * torch.randn(blocks, generator=self.g, device=self.dev))).clamp_(min=std)
        if not nested:
            return dict(w, absmax=absmax)
        # second quantization: signed distances from the mean on a 256-entry map, finer near zero
        steps = torch.logspace(-6, 0, 127, base=10.0, dtype=torch.float32).tolist()
        code2 = torch.tensor([-s for s in reversed(steps)] + [0.0, 1e-7] + steps, device=self.dev)
        offset = absmax.mean()
        groups = -(-blocks // GROUP)
        d = torch.zeros(groups * GROUP, device=self.dev)
        d[:blocks] = absmax - offset
        d = d.view(groups, GROUP)
        absmax2 = d.abs().amax(dim=1)
        near = torch.bucketize((d / absmax2[:, None]).reshape(-1)[:blocks].contiguous(), (code2[:-1] + code2[1:]) / 2)
        return dict(w, absmax=near.to(torch.uint8), absmax2=absmax2, code2=code2, offset=offset)


def _layer(src, hidden, kv, inter):
    shapes = dict(q=(hidden, hidden), k=(kv, hidden), v=(kv, hidden), o=(hidden, hidden), gate=(inter, hidden),
                  up=(inter, hidden), down=(hidden, inter))
    return {name: src.weight(*s) for name, s in shapes.items()}


def _inputs(case, seed):
    """Everything a pass reads, as plain tensors."""
    src, kind = _Source(seed), case["kind"]
    if kind == "dequant":
        return dict(weights=list(_layer(src, case["hidden"], case["kv"], case["inter"]).values()))
    m = case["m"]
    if kind == "linear":
        n, k = case["n"], case["k"]
        return dict(w=src.weight(n, k, case["blocksize"], case["nested"]), x=src.normal(m, k), dy=src.normal(m, n, std=1e-2),
                    bias=src.normal(n, std=0.5) if case["bias"] else None)
    if kind == "serve":
        hidden, kv = case["hidden"], case["kv"]
        return dict(layers=[dict(_layer(src, hidden, kv, case["inter"]), x=src.normal(m, hidden),
                                 attn=src.normal(m, hidden, std=0.3), x2=src.normal(m, hidden),
                                 biases=[src.normal(n, std=0.5) for n in (hidden, kv, kv)])
                            for _ in range(case["layers"])])
    if kind == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        return dict(gate=src.weight(inter, hidden), up=src.weight(inter, hidden), down=src.weight(hidden, inter),
                    x=src.normal(m, hidden, dtype=torch.float32), dy=src.normal(m, hidden, std=1e-2))
    heads, kv_heads, d, r = case["heads"], case["kv_heads"], case["head_dim"], case["rank"]
    hidden, kv = heads * d, kv_heads * d
    inv = 1e6 ** (-torch.arange(0, d, 2, device=src.dev, dtype=torch.float64) / d)
    angle = torch.arange(m, device=src.dev, dtype=torch.float64)[:, None] * torch.cat([inv, inv])
    keep = [torch.rand((m, hidden), generator=src.g, device=src.dev) >= 0.05 for _ in range(2)]
    return dict(
        q=src.weight(hidden, hidden), k=src.weight(kv, hidden), v=src.weight(kv, hidden), o=src.weight(hidden, hidden),
        biases=[src.normal(n, std=0.5) for n in (hidden, kv, kv)], x=src.normal(m, hidden, dtype=torch.float32),
        attn=src.normal(m, hidden, std=0.3), cos=angle.cos().float(), sin=angle.sin().float(),
        adapters=[src.normal(*s, std=t, dtype=torch.float32) for s, t in (((r, hidden), 0.02), ((hidden, r), 0.02),
                                                                         ((r, hidden), 0.02), ((kv, r), 0.02))],
        keep=keep if case["dropout"] else None,
        grads=[src.normal(1, heads, m, d, std=1e-2), src.normal(1, kv_heads, m, d, std=1e-2), src.normal(m, kv, std=1e-2),
               src.normal(m, hidden, std=1e-2)])


def _state(w):
    """(packed, QuantState) of a weight, as the loader of a quantized checkpoint leaves them."""
    state2 = State2(w["absmax2"], w["code2"], GROUP) if "absmax2" in w else None
    return w["packed"], QuantState(absmax=w["absmax"], shape=(w["n"], w["k"]), code=w["code"], blocksize=w["blocksize"],
                                   offset=w.get("offset"), state2=state2)


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "dequant":
        return dict(kind=kind, pairs=[_state(w) for w in t["weights"]])
    if kind == "linear":
        packed, qs = _state(t["w"])
        return dict(kind=kind, x=t["x"].requires_grad_(case["grad"]), packed=packed, qs=qs, bias=t["bias"],
                    dy=t["dy"] if case["grad"] else None)
    if kind == "serve":
        layers = [dict(L, **{n: _state(L[n]) for n in ("q", "k", "v", "o", "gate", "up", "down")}) for L in t["layers"]]
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _serve(layers)  # first calls: workspaces
        with torch.cuda.graph(graph, stream=stream):
            outputs = _serve(layers)
        return dict(kind=kind, graph=graph, layers=layers, outputs=outputs)
    if kind == "mlp":
        weights = [v for n in ("gate", "up", "down") for v in _state(t[n])]
        return dict(kind=kind, x=t["x"].requires_grad_(), weights=weights, dy=t["dy"], recompute=case["recompute"])
    adapters = [a.requires_grad_() for a in t["adapters"]]
    projections = [dict(zip(("packed", "qs"), _state(t[n])), bias=b) for n, b in zip("qkv", t["biases"])]
    projections[0].update(lora_a=adapters[0], lora_b=adapters[1], scaling=LORA_SCALE)
    projections[2].update(lora_a=adapters[2], lora_b=adapters[3], scaling=LORA_SCALE)
    if t["keep"] is not None:
        scale = torch.full((1,), 1.0 / 0.95, device=t["x"].device)
        for p, bits in zip((projections[0], projections[2]), pack_keep(*t["keep"])):
            p.update(keep_bits=bits, keep_scale=scale, p=0.05)
    return dict(kind=kind, x=t["x"].requires_grad_(), attn=t["attn"].requires_grad_(), projections=tuple(projections),
                o=_state(t["o"]), cos=t["cos"], sin=t["sin"], heads=case["heads"], kv_heads=case["kv_heads"],
                adapters=adapters, grads=t["grads"])


# ---- passes --------------------------------------------------------------------------------------

def _serve(layers):
    outputs = []
    for L in layers:
        qkv = nf4.linear_forward(L["x"], [dict(packed=L[n][0], qs=L[n][1], bias=b) for n, b in zip("qkv", L["biases"])])
        (o,) = nf4.linear_forward(L["attn"], [dict(packed=L["o"][0], qs=L["o"][1])])
        y, _, _ = mlp_forward(L["x2"], L["gate"], L["up"], L["down"], keep_gate_up=False)
        outputs.append(dict(q=qkv[0], k=qkv[1], v=qkv[2], o=o, mlp=y))
    return outputs


def run(state):
    kind = state["kind"]
    if kind == "dequant":
        return nf4.dequantize_nf4_many(state["pairs"])
    if kind == "serve":
        state["graph"].replay()
        return state["outputs"]
    if kind == "linear":
        y = nf4.NF4Linear.apply(state["x"], state["packed"], state["bias"], state["qs"])
        if state["dy"] is None:
            return dict(y=y)
        (dx,) = torch.autograd.grad(y, state["x"], state["dy"])
        return dict(y=y, dx=dx)
    if kind == "mlp":
        y = FusedMLP.apply(state["x"], *state["weights"], state["recompute"])
        (dx,) = torch.autograd.grad(y, state["x"], state["dy"])
        return dict(y=y, dx=dx)
    q, k, v = qkv_rope_projection(state["x"], state["projections"], state["cos"], state["sin"], state["heads"],
                                  state["kv_heads"])
    o = nf4.NF4Linear.apply(state["attn"], state["o"][0], None, state["o"][1])
    grads = torch.autograd.grad((q, k, v, o), (state["x"], state["attn"], *state["adapters"]), state["grads"])
    return dict(q=q, k=k, v=v, o=o, **dict(zip(("dx", "dattn", "da_q", "db_q", "da_v", "db_v"), grads)))


# ---- what a pass cannot do without ----------------------------------------------------------------

def _weight_bytes(n, k, blocksize=64, nested=True):
    blocks = n * k / blocksize
    return n * k / 2 + (blocks + 4 * blocks / GROUP if nested else 4 * blocks)


def work(case):
    kind, m = case["kind"], case.get("m", 0)
    if kind == "linear":
        n, k = case["n"], case["k"]
        passes = 2 if case["grad"] else 1
        return dict(bytes=_weight_bytes(n, k, case["blocksize"], case["nested"]) + passes * 2 * m * (n + k)
                    + (2 * n if case["bias"] else 0), flops=passes * 2 * m * n * k)
    if kind == "attention":
        hidden, kv, r = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["rank"]
        base = 2 * hidden * hidden + 2 * kv * hidden
        lora = (r * hidden + hidden * r) + (r * hidden + kv * r)
        return dict(bytes=_weight_bytes(1, base) + 2 * 4 * lora + 2 * 4 * m * hidden + 2 * 2 * m * hidden
                    + 2 * 2 * m * (2 * hidden + 2 * kv) + 8 * m * case["head_dim"]
                    + (2 * m * hidden / 8 if case["dropout"] else 0), flops=2 * 2 * m * base + 3 * 2 * m * lora)
    hidden, inter = case["hidden"], case["inter"]
    mlp = 3 * hidden * inter
    if kind == "mlp":
        return dict(bytes=_weight_bytes(1, mlp) + m * hidden * (4 + 2 + 2 + 4), flops=2 * 2 * m * mlp)
    kv = case["kv"]
    layer = mlp + 2 * hidden * hidden + 2 * kv * hidden
    if kind == "dequant":
        return dict(bytes=_weight_bytes(1, layer) + 2 * layer, flops=0)
    return dict(bytes=case["layers"] * (_weight_bytes(1, layer) + 2 * m * (6 * hidden + 2 * kv)),
                flops=case["layers"] * 2 * m * layer)


def tolerance(case):
    """Four times the distance measured from exact(): single products rounded once to fp16 (2.1e-4 in
    the 2-norm), products of operands that were themselves rounded (attention: 2.9e-4 with RoPE and
    the adapters' gradients; MLP: 4.4e-4 with the fp16 gate, up and hidden values). "max" allows a few
    units in fp16's last place (9.8e-4 of a value)."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "linear":
        return {"rel": 8.4e-4, "max": 4e-3}
    return {"rel": 1.2e-3, "max": 1e-2} if kind == "attention" else {"rel": 1.8e-3, "max": 1e-2}


# ---- the same in 64 bits --------------------------------------------------------------------------

def _dequant(w):
    """fp16 weights [n, k]: the format's two fp32 roundings of the scale and one to fp16."""
    scale = w["absmax"]
    if "absmax2" in w:
        group = torch.arange(scale.numel(), device=scale.device) // GROUP
        scale = w["code2"][scale.long()] * w["absmax2"][group]
        scale = scale + w["offset"]
    b = w["packed"].reshape(-1)
    value = torch.stack([w["code"][(b >> 4).int()], w["code"][(b & 15).int()]], dim=1).reshape(-1)
    n = value.numel()
    pad = -n % w["blocksize"]
    value = torch.nn.functional.pad(value, (0, pad)).view(-1, w["blocksize"]) * scale[:, None]
    return value.reshape(-1)[:n].view(w["n"], w["k"]).to(torch.float16)


def _w64(w):
    return _dequant(w).double()


def _silu(x):
    return x * torch.sigmoid(x)


def _rope(x, cos, sin, heads):
    """[m, heads * d] -> rotated [1, heads, m, d]."""
    m, d = cos.shape
    x = x.view(m, heads, d).transpose(0, 1)
    half = torch.cat([-x[..., d // 2:], x[..., :d // 2]], dim=-1)
    return (x * cos + half * sin)[None]


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "dequant":
        return [_dequant(w) for w in t["weights"]]
    if kind == "linear":
        w, x = _w64(t["w"]), t["x"].double()
        y = x @ w.T + (0 if t["bias"] is None else t["bias"].double())
        return dict(y=y, dx=t["dy"].double() @ w) if case["grad"] else dict(y=y)
    if kind == "serve":
        outputs = []
        for L in t["layers"]:
            x, x2 = L["x"].double(), L["x2"].double()
            qkv = [x @ _w64(L[n]).T + b.double() for n, b in zip("qkv", L["biases"])]
            h = _silu(x2 @ _w64(L["gate"]).T) * (x2 @ _w64(L["up"]).T)
            outputs.append(dict(q=qkv[0], k=qkv[1], v=qkv[2], o=L["attn"].double() @ _w64(L["o"]).T,
                                mlp=h @ _w64(L["down"]).T))
        return outputs
    if kind == "mlp":
        x = t["x"].half().double().requires_grad_()
        gate, up, down = (_w64(t[n]) for n in ("gate", "up", "down"))
        y = (_silu(x @ gate.T) * (x @ up.T)) @ down.T
        (dx,) = torch.autograd.grad(y, x, t["dy"].double())
        return dict(y=y.detach(), dx=dx)
    x = t["x"].half().double().requires_grad_()
    adapters = [a.half().double().requires_grad_() for a in t["adapters"]]
    cos, sin = t["cos"].double(), t["sin"].double()
    keep = t["keep"] or (None, None)
    y = {n: x @ _w64(t[n]).T + b.double() for n, b in zip("qkv", t["biases"])}
    for n, a, b, mask in (("q", *adapters[:2], keep[0]), ("v", *adapters[2:], keep[1])):
        branch = x
        if mask is not None:  # the branch's input is rounded after the dropout, as the base's before
            kept = (t["x"] * (mask.float() * torch.tensor(1.0 / 0.95, device=mask.device))).half().double()
            branch = x * mask.double() / 0.95
            branch = branch + (kept - branch).detach()
        y[n] = y[n] + LORA_SCALE * ((branch @ a.T) @ b.T)
    q, k = _rope(y["q"], cos, sin, case["heads"]), _rope(y["k"], cos, sin, case["kv_heads"])
    attn = t["attn"].double().requires_grad_()
    o = attn @ _w64(t["o"]).T
    grads = torch.autograd.grad((q, k, y["v"], o), (x, attn, *adapters), [g.double() for g in t["grads"]])
    return dict(q=q.detach(), k=k.detach(), v=y["v"].detach(), o=o.detach(),
                **dict(zip(("dx", "dattn", "da_q", "db_q", "da_v", "db_v"), grads)))
