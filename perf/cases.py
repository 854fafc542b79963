"""Performance cases of the sparse projection-and-pool layer: the work a program has it do.

Every case builds a layer through its public constructor, keeps it (with its optimizer) as a
training or serving program does, and runs one pass of one of three modes:

* ``infer``: the forward under ``torch.no_grad()``; returns y;
* ``grads``: forward and backward with persistent fp32 ``main_grad`` buffers, or, with
  ``main_grad`` False, with gradients that autograd returns; returns y and every gradient;
* ``train``: forward, backward and the fused AdamW step; returns y, dX, the updated parameters
  and both moments.

Indices, weights and inputs come from the case's seed: indices uniform and distinct per neuron (or
drawn from one window of the inputs per pool), W ~ N(0, 1/K), X and dY ~ N(0, 1).
"""
import math

import torch

from granulelayer_amd import CoverTopK16Layer, FusedAdamW, PhysicalPlan, SparsePoolingLayer

DEVICE = "cuda"
LR, BETAS, EPS = 1e-3, (0.9, 0.999), 1e-8

# Defaults of a case's fields; a case names what differs.
BASE = dict(mode="grads", pool="sum", act="relu", k=0, param=0.0, shard=0, dtype="fp32", x_dtype="fp32", fan_in=8,
            window=0, cover=False, main_grad=True, moments="fp32", relu_bits="recompute")


def listed():
    return [
        # the smallest training step: a layer that fits a test or a notebook, where launches and
        # the host path are all there is
        dict(name="tiny_train", mode="train", pool="mean", D=256, H=6000, G=12, B=40),
        # serving a handful of tokens through a 1M-neuron bf16 layer: latency of one forward
        dict(name="serve_few", mode="infer", pool="mean", dtype="bf16", x_dtype="bf16", D=1024, H=1048576, G=4096,
             B=4),
        # the benchmark's small training step (1M neurons, 64 tokens)
        dict(name="train_1m", mode="train", D=1024, H=1048576, G=4096, B=64),
        # the benchmark's headline forward: 100M neurons, 256 tokens
        dict(name="forward_100m", mode="infer", D=4096, H=100663296, G=98304, B=256),
        # the benchmark's full training step: 100M neurons, 1024 bf16 tokens, ReLU bits kept
        dict(name="train_100m", mode="train", D=8192, H=100663296, G=98304, B=1024, x_dtype="bf16",
             relu_bits="keep"),
        # locality: every pool reads one 256-wide window of the inputs, bf16 tokens
        dict(name="windows", D=4096, H=25165824, G=24576, B=256, x_dtype="bf16", window=256),
        # the constructor's own defaults: max pooling, bf16 parameters, 1024 inputs and outputs, the
        # optimizer with bf16 moments; pools of about ten thousand neurons
        dict(name="max_defaults", mode="train", pool="max", act="identity", dtype="bf16", x_dtype="bf16", D=1024,
             H=10000000, G=1024, B=256, moments="bf16"),
        # top-8 mean pooling, gradients of the selected neurons
        dict(name="topk8", pool="topk_mean", act="identity", k=8, D=4096, H=12582912, G=12288, B=256),
        # LogMeanExp, the smooth maximum: every neuron has a gradient
        dict(name="logmeanexp", pool="logmeanexp", param=0.5, D=4096, H=12582912, G=12288, B=256),
        # two-level pooling: means over shards of 256 neurons, LogMeanExp over a pool's 4 shards
        dict(name="two_level", pool="mean", shard=256, D=4096, H=12582912, G=12288, B=256),
        # Cover-TopK/16: 16 neurons share one fan-in-16 record
        dict(name="cover_k16", pool="mean", fan_in=16, cover=True, D=4096, H=12582912, G=24576, B=512),
        # ragged sizes: odd widths, pools that differ by one neuron, fan-in 16, 77 tokens, a smooth
        # pool over identity neurons, gradients returned by autograd
        dict(name="ragged", pool="softmax_weighted", act="identity", param=1.0, fan_in=16, D=1000, H=777777, G=1009,
             B=77, main_grad=False),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the listed ones' ranges: every mode, pool, dtype and index structure, 1 to 1024
    tokens, 64 to 8192 inputs, 2,000 to 33M neurons."""
    kind = rng.choice(["sum", "sum", "mean", "mean", "max", "max", "topk_mean", "logmeanexp", "power_mean",
                       "softmax_weighted", "shards", "window", "cover"])
    c = dict(mode=rng.choice(["infer", "grads", "grads", "train"]), B=_spread(rng, 1, 1024), D=_spread(rng, 64, 8192))
    c["x_dtype"] = rng.choice(["fp32", "bf16"])
    pool_size = _spread(rng, 24, 4000)
    most = 60e9  # edge-tokens
    c["pool"] = kind
    if kind in ("sum", "mean"):
        c["act"] = rng.choice(["relu", "relu", "relu", "identity", "gelu"])
        c["relu_bits"] = rng.choice(["keep", "recompute"])
        c["fan_in"] = rng.choice([8, 8, 8, 16])
        most = 200e9 if c["act"] != "gelu" else 60e9
    elif kind == "max":
        c["act"] = rng.choice(["identity", "identity", "relu"])
        c["fan_in"] = rng.choice([8, 8, 8, 16])
        pool_size = _spread(rng, 24, 50000)
        most = 200e9
    elif kind == "topk_mean":
        c["act"] = "identity"
        c["k"] = rng.choice([4, 8, 8, 16])
    elif kind in ("logmeanexp", "softmax_weighted"):
        c["act"] = rng.choice(["relu", "identity"])
        c["param"] = rng.choice([0.5, 1.0])
        c["fan_in"] = rng.choice([8, 16])
    elif kind == "power_mean":
        c["param"] = rng.choice([2.0, 4.0])
    elif kind == "shards":
        c["pool"], c["shard"] = "mean", rng.choice([64, 256])
        pool_size = c["shard"] * rng.randint(2, 8)
    elif kind == "window":
        c["pool"], c["window"] = "sum", min(rng.choice([128, 256]), c["D"])
        pool_size = _spread(rng, 200, 4000)
    else:
        c["pool"], c["cover"], c["fan_in"] = "mean", True, 16
        c["x_dtype"] = "fp32"
        pool_size = 64 * rng.randint(2, 16)
    if kind != "cover" and c["x_dtype"] == "bf16" and rng.random() < 0.5:
        c["dtype"] = "bf16"
    c["moments"] = rng.choice(["fp32", "bf16"])
    c["main_grad"] = c["mode"] == "train" or rng.random() < 0.7
    H = _spread(rng, 2000, min(33e6, most / (c["B"] * c.get("fan_in", 8))))
    G = max(1, H // pool_size)
    if kind == "shards" or kind == "cover":
        H = G * pool_size  # whole shards, whole 16-neuron rows
    c["H"], c["G"] = max(H, G), G
    return c


# ---------------------------------------------------------------------------- inputs
def _dtype(name):
    return torch.float32 if name == "fp32" else torch.bfloat16


def _pooling(c):
    if c["shard"]:
        return {"levels": [{"type": c["pool"], "neurons_per_shard": c["shard"], "activation": c["act"]},
                           {"type": "logmeanexp"}]}
    spec = {"type": c["pool"], "activation": c["act"]}
    if c["pool"] == "topk_mean":
        spec["k"] = c["k"]
    name = {"logmeanexp": "temperature", "power_mean": "p", "softmax_weighted": "beta"}.get(c["pool"])
    if name:
        spec[name] = c["param"]
    return spec


def _window_indices(layer, c, gen):
    """Indices of every pool from one window of the inputs at a random offset."""
    G, K, W = c["G"], c["fan_in"], c["window"]
    lo = torch.randint(0, c["D"] - W + 1, (G,), generator=gen, device=DEVICE, dtype=torch.int32)
    with torch.no_grad():
        # K distinct offsets in ascending order: one from each of K equal parts of the window
        shape = layer.indices.shape
        step = W // K
        rec = torch.randint(0, step, shape, generator=gen, device=DEVICE, dtype=torch.int32)
        rec += torch.arange(K, device=DEVICE, dtype=torch.int32) * step
        rec += lo.view(G, *([1] * (len(shape) - 1)))
        slots = shape[1] * shape[2]
        valid = torch.arange(slots, device=DEVICE) < _counts(c)[:, None]
        layer.indices.copy_(rec * valid.view(*shape[:3], 1))


def _cover_layer(c, gen):
    G, n = c["G"], c["H"] // c["G"]
    NB = -(-n // 256)  # records of 256 neurons per output
    env = torch.randint(0, c["D"], (G, NB, 64), generator=gen, device=DEVICE, dtype=torch.int32)
    part = c["D"] // 64  # 64 distinct candidates: one from each of 64 equal parts of the inputs
    env = env % part + torch.arange(64, device=DEVICE, dtype=torch.int32) * part
    w = torch.randn((G, NB, 256, 64), generator=gen, device=DEVICE) / 4.0
    b = torch.zeros((G, NB, 256), device=DEVICE)
    return CoverTopK16Layer.from_envelope(w, b, env, input_dim=c["D"], hidden_dim=c["H"], output_dim=G,
                                          pooling=_pooling(c), plan=PhysicalPlan(relu_bits=c["relu_bits"]))


def prepare(case, seed):
    """The layer (its one-time setup done by a one-token step), its optimizer, tokens and dY."""
    c = {**BASE, **case}
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    if c["cover"]:
        layer = _cover_layer(c, gen)
    else:
        layer = SparsePoolingLayer(c["D"], c["H"], c["G"], fan_in=c["fan_in"], shared_neurons=None,
                                   pooling=_pooling(c), dtype=_dtype(c["dtype"]), device=DEVICE, seed=seed,
                                   plan=PhysicalPlan(relu_bits=c["relu_bits"]))
        if c["window"]:
            _window_indices(layer, c, gen)
    x = torch.randn((c["B"], c["D"]), generator=gen, device=DEVICE).to(_dtype(c["x_dtype"]))
    dy = torch.randn((c["B"], c["G"]), generator=gen, device=DEVICE)
    state = dict(case=c, layer=layer, x=x, dy=dy, opt=None)
    if c["mode"] == "infer":
        with torch.no_grad():
            layer(x[:1])
        return state
    if c["main_grad"]:
        layer.enable_main_grad()
    layer(x[:1]).sum().backward()
    layer.zero_main_grad()
    layer.zero_grad(set_to_none=True)
    if c["mode"] == "train":
        state["opt"] = FusedAdamW(layer.parameters(), lr=LR, betas=BETAS, eps=EPS, moments=c["moments"])
    x.requires_grad_(True)
    return state


# ---------------------------------------------------------------------------- one pass
def run(state):
    c, layer, x = state["case"], state["layer"], state["x"]
    if c["mode"] == "infer":
        with torch.no_grad():
            return {"y": layer(x)}
    x.grad = None
    if state["opt"] is None:
        if c["main_grad"]:
            layer.zero_main_grad()
        else:
            layer.zero_grad(set_to_none=True)
    y = layer(x)
    y.backward(state["dy"])
    out = {"y": y.detach(), "dx": x.grad}
    if state["opt"] is None:
        for name, p in (("dw", layer.weight), ("db", layer.bias)):
            out[name] = p.main_grad if c["main_grad"] else p.grad
        return out
    state["opt"].step()
    for name, p in (("w", layer.weight), ("b", layer.bias)):
        s = state["opt"].state[p]
        out[name], out[name + "_m"], out[name + "_v"] = p.detach(), s["m"], s["v"]
    return out


def work(case):
    c = {**BASE, **case}
    B, D, G, H, K = c["B"], c["D"], c["G"], c["H"], c["fan_in"]
    E = H * K
    ps, xs = (4 if c["dtype"] == "fp32" else 2), (4 if c["x_dtype"] == "fp32" else 2)
    params = (E // 16 if c["cover"] else E) * 4 + (E + H) * ps
    nbytes, flops = params + B * D * xs + 4 * B * G, 2 * B * E
    if c["mode"] == "infer":
        return {"bytes": nbytes, "flops": flops}
    # backward: parameters and tokens again, dY, dX, dW and db written once
    gs = 4 if c["main_grad"] else ps
    nbytes += params + 2 * B * D * xs + 4 * B * G + (E + H) * gs
    selected = B * G * c["k"] if c["pool"] == "topk_mean" else B * G if c["pool"] == "max" else B * H
    flops += 4 * selected * K
    if c["mode"] == "train":  # gradient read and cleared, parameter and both moments read and written
        ms = 4 if c["moments"] == "fp32" else 2
        nbytes += (E + H) * (8 + 2 * ps + 4 * ms)
        flops += 12 * (E + H)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from the 64-bit results, measured over the cases."""
    c = {**BASE, **case}
    if c["mode"] != "infer" and ("bf16" in (c["dtype"], c["x_dtype"]) or (c["mode"] == "train" and c["moments"] == "bf16")):
        return {"rel": 7e-3, "max": 0.9}  # gradients or moments rounded to bf16 (2^-9 each)
    if c["mode"] == "infer":
        return {"rel": 2e-6}
    if c["pool"] in ("max", "topk_mean"):
        return {"rel": 2e-3, "max": 0.9}  # a near-tie may select the other neuron
    if c["act"] == "relu":
        return {"rel": 5e-4, "max": 0.9}  # a z within rounding of 0 may count or not
    return {"rel": 2e-5, "max": 0.01}


# ---------------------------------------------------------------------------- 64-bit results
def _counts(c):
    g = torch.arange(c["G"], device=DEVICE)
    return c["H"] // c["G"] + (g < c["H"] % c["G"]).long()


def _act(z, name):
    if name == "relu":
        return torch.relu(z)
    return torch.nn.functional.gelu(z) if name == "gelu" else z


def _pool(z, valid, c):
    """[pools, slots, tokens] -> [pools, tokens]."""
    a, m = _act(z, c["act"]), valid[..., None]
    n = valid.sum(1).to(z.dtype)[:, None]
    none = torch.full((), -math.inf, dtype=z.dtype, device=z.device)
    p = c["pool"]
    if p in ("sum", "mean"):
        s = torch.where(m, a, torch.zeros_like(a)).sum(1)
        return s if p == "sum" else s / n
    if p == "max":
        a = torch.where(m, a, none)
        return a.gather(1, a.argmax(1, keepdim=True)).squeeze(1)
    if p == "topk_mean":
        k = min(c["k"], z.shape[1])
        top = torch.where(m, z.detach(), none).topk(k, dim=1).indices
        got = m.expand_as(z).gather(1, top)
        return torch.where(got, a.gather(1, top), torch.zeros_like(got, dtype=z.dtype)).sum(1) / got.sum(1)
    if p == "logmeanexp":
        return c["param"] * (torch.logsumexp(torch.where(m, a / c["param"], none), 1) - n.log())
    if p == "softmax_weighted":
        return (torch.softmax(torch.where(m, c["param"] * a, none), 1) * a).sum(1)
    s = (torch.where(m, a, torch.zeros_like(a)) ** c["param"]).sum(1) / n
    return s ** (1.0 / c["param"])


def exact(case, seed):
    """What run() returns, in float64 torch: pools in blocks, forward and then backward by autograd
    through the pooling and by hand through the sparse projection."""
    c = {**BASE, **case}
    K, B, G = c["fan_in"], c["B"], c["G"]
    if B * c["H"] * K > 55e9:
        return None
    s = prepare(case, seed)
    layer = s["layer"]
    x, dy = s["x"].detach().double(), s["dy"].double()
    if c["dtype"] == "bf16":
        x = s["x"].detach().to(torch.bfloat16).double()
    xt = x.t().contiguous()
    w, b = layer.weight.detach().reshape(G, -1, K), layer.bias.detach().reshape(G, -1)
    S = b.shape[1]
    idx = layer.indices.reshape(G, -1, K)
    idx = idx.repeat_interleave(S // idx.shape[1], 1)
    counts = _counts(c)
    # a pool's slots, cut into shards for a two-level layer
    nps = c["shard"] or S
    parts = -(-int(counts.max()) // nps)
    valid = torch.arange(S, device=DEVICE) < counts[:, None]
    step = max(1, int(2**26 // (S * B)))

    def projected(g0, g1):
        z = b[g0:g1].double()[..., None].expand(-1, -1, B).clone()
        for k in range(K):
            z += w[g0:g1, :, k].double()[..., None] * xt[idx[g0:g1, :, k].long()]
        return z

    def pooled(z, g0, g1):
        out = [_pool(z[:, p * nps:(p + 1) * nps], valid[g0:g1, p * nps:(p + 1) * nps], c) for p in range(parts)]
        return torch.stack(out, 1)  # [pools, parts, tokens]

    pre = torch.cat([pooled(projected(g, min(G, g + step)), g, min(G, g + step)) for g in range(0, G, step)])
    pre.requires_grad_(c["mode"] != "infer")
    f = pre
    if c["pool"] in ("max", "topk_mean"):
        f = torch.relu(f) if layer.cfg.levels[0].out_activation == "relu" else f
    y = (torch.logsumexp(f, 1) - math.log(parts) if c["shard"] else f.squeeze(1)).t()
    if c["mode"] == "infer":
        return {"y": y}
    g_pre, = torch.autograd.grad(y, pre, dy)
    dxt = torch.zeros_like(xt)
    dw = torch.zeros((G, S, K), dtype=torch.float64, device=DEVICE)
    db = torch.zeros((G, S), dtype=torch.float64, device=DEVICE)
    for g0 in range(0, G, step):
        g1 = min(G, g0 + step)
        z = projected(g0, g1).requires_grad_(True)
        dz, = torch.autograd.grad(pooled(z, g0, g1), z, g_pre[g0:g1])
        dz = torch.where(valid[g0:g1, :, None], dz, torch.zeros_like(dz))
        db[g0:g1] = dz.sum(2)
        for k in range(K):
            at = idx[g0:g1, :, k].long()
            dw[g0:g1, :, k] = (dz * xt[at]).sum(2)
            dxt.index_add_(0, at.reshape(-1), (dz * w[g0:g1, :, k].double()[..., None]).reshape(-1, B))
    dw, db = dw.view(layer.weight.shape), db.view(layer.bias.shape)
    out = {"y": y.detach(), "dx": dxt.t()}
    if c["mode"] == "grads":
        return {**out, "dw": dw, "db": db}
    for name, p, grad in (("w", layer.weight, dw), ("b", layer.bias, db)):
        m, v = (1 - BETAS[0]) * grad, (1 - BETAS[1]) * grad * grad
        new = p.detach().double() - LR * (m / (1 - BETAS[0])) / ((v / (1 - BETAS[1])).sqrt() + EPS)
        # a bf16 parameter is rounded stochastically: it has no 64-bit value
        out[name], out[name + "_m"], out[name + "_v"] = (new if c["dtype"] == "fp32" else None), m, v
    return out
