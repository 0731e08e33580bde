"""What is timed of this framework: its ChannelMix layers as a program calls
them, from one generated token to a long training batch.

Shapes are those of ``rwkv_mlx_amd.workloads`` and of ``RWKVConfig``'s
defaults (dim_ffn 3.5x), or lie in the same ranges.  Values follow
``workloads.make_inputs``: x ~ N(0,1), weights ~ N(0, 1/sqrt(fan_in)), B ~
N(0, 0.02), a Zipf bias where routing is skewed; they are drawn on the GPU
from the seed.

Kinds of case
  step     ``channel_mixing_rnn``: one token for each of `batch` sequences
  layer    ``LoRAMoE_CMix`` forward (inference, prefill, evaluation); with
           `block` the Block's form x + ffn(ln2(x))
  dense    ``RWKV_CMix_x070`` forward, the layers without experts
  train    ``LoRAMoE_CMix`` forward and backward with the aux, z and
           orthogonality losses; with `fp32_adapters` the fine-tune layer (a
           16-bit base with the fp32 router and adapters)
  experts  ``MoE_CMix`` forward (E full experts)
  experts_train  ``MoE_CMix`` forward and backward
"""
import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "rwkv-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# loss coefficients of a training step (RWKVConfig's defaults) and the top
# gradient's scale
AUX_COEFF, Z_COEFF, ORTHO_COEFF = 0.01, 0.001, 0.001


def _case(name, kind, dtype, batch, seq, d, f, e=0, k=0, r=0, **more):
    c = dict(kind=kind, dtype=dtype, batch=batch, seq=seq, d_model=d, d_ffn=f, experts=e, top_k=k, rank=r,
             block=False, skewed=False, fp32_adapters=False)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # generating one stream of text: every layer is called for a single token
        _case("step-1", "step", "f16", 1, 1, 768, 3072, 8, 2, 16, block=True),
        # batched generation, the decode workload
        _case("step-64", "step", "f16", 64, 1, 768, 3072, 8, 2, 16),
        # a server's decode batch on the wide layer
        _case("step-200-wide", "step", "bf16", 200, 1, 2048, 8192, 16, 2, 32),
        # the small fp32 layer, one sequence: numerics work and small models
        _case("layer-512-f32", "layer", "f32", 1, 512, 512, 2048, 4, 1, 8),
        # the 184M model's layer on an evaluation batch (the headline workload)
        _case("layer-4096", "layer", "f16", 8, 512, 768, 3072, 8, 2, 16),
        # prefill of a few prompts of an odd length, in the Block's form, with the default dim_ffn
        _case("block-ragged", "layer", "bf16", 3, 677, 1024, 3584, 8, 2, 32, block=True),
        # many experts, one of them popular
        _case("layer-skewed", "layer", "f16", 8, 1024, 1024, 4096, 32, 4, 16, skewed=True),
        # the wide bf16 layer on a large batch
        _case("layer-wide", "layer", "bf16", 16, 1024, 2048, 8192, 16, 2, 32),
        # a training step of the adapters and the router, all in fp16
        _case("train-4096", "train", "f16", 8, 512, 768, 3072, 8, 2, 16),
        # the fine-tuning script's step: an fp16 base, fp32 router and adapters, 2 x 512 tokens
        _case("finetune-1024", "train", "f16", 2, 512, 768, 2688, 8, 2, 32, fp32_adapters=True),
        # full experts: evaluation, and a training step of every parameter
        _case("experts-4096", "experts", "f16", 8, 512, 768, 3072, 8, 2),
        _case("experts-train-2048", "experts_train", "bf16", 4, 512, 768, 3072, 8, 2),
    ]


def draw(rng):
    kind = rng.choice(["step", "layer", "layer", "layer", "dense", "train", "train", "experts", "experts_train"])
    dtype = rng.choice(["f16", "bf16"])
    d = rng.choice([512, 640, 768, 896, 1024, 1280, 1536, 2048])
    block = fp32_adapters = skewed = False
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if kind == "step":
        batch, seq = log(1, 512), 1
        block = rng.random() < 0.5
    else:
        batch, seq = rng.choice([1, 2, 3, 4, 6, 8]), log(64, 1024)
    if kind == "layer":
        block = rng.random() < 0.5
        skewed = rng.random() < 0.25
        if rng.random() < 0.2:
            dtype, d, batch = "f32", rng.choice([512, 640, 768]), min(batch, 2)
    if kind == "train" and rng.random() < 0.5:
        dtype, fp32_adapters = "f16", True
    if kind in ("train", "experts", "experts_train"):
        d = min(d, 1024)
    f = rng.choice([4 * d, int(3.5 * d) // 64 * 64])
    if kind == "dense":
        return _case(None, kind, dtype, batch, seq, d, f)
    e, k = rng.choice([(4, 1), (4, 2), (8, 2), (8, 2), (16, 2), (16, 4)] + ([] if "exp" in kind else [(32, 4)]))
    r = 0 if "exp" in kind else rng.choice([8, 16, 32])
    return _case(None, kind, dtype, batch, seq, d, f, e, k, r, block=block, skewed=skewed,
                 fp32_adapters=fp32_adapters)


def _inputs(case, seed):
    """Every tensor of the case as plain torch on the GPU, in its own dtype."""
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(int(seed))
    dt = DTYPES[case["dtype"]]
    pt = torch.float32 if case["fp32_adapters"] else dt
    B, T, C, F, E, r = (case[n] for n in ("batch", "seq", "d_model", "d_ffn", "experts", "rank"))
    normal = lambda shape, scale, t=dt: (torch.randn(shape, generator=g, device=dev) * scale).to(t)
    t = {"x": normal((B, T, C), 1.0)}
    many = (E,) if "experts" in case["kind"] else ()
    t["x_k"] = torch.rand(many + (1, 1, C), generator=g, device=dev).to(dt)
    t["key"] = normal(many + (F, C), 1 / math.sqrt(C))
    t["value"] = normal(many + (C, F), 1 / math.sqrt(F))
    if E:
        t["gate"] = normal((E, C), 1 / math.sqrt(C), pt)
    if r:
        t["A"] = normal((E, C, r), 1 / math.sqrt(C), pt)
        t["B"] = normal((E, r, C), 0.02, pt)
    if case["skewed"]:
        p = torch.arange(1, E + 1, device=dev, dtype=torch.float64) ** -1.2
        t["bias"] = torch.log(p / p.sum()).float()
    if case["kind"] == "step":
        t["x_prev"] = normal((B, C), 1.0)
    if case["block"]:
        t["ln_w"] = (1 + 0.1 * torch.randn(C, generator=g, device=dev)).to(dt)
        t["ln_b"] = normal((C,), 0.1)
    if "train" in case["kind"]:
        # the fine-tune layer's output is fp32, and so is its cotangent
        t["d_out"] = normal((B, T, C), 1.0, pt)
    return t


def prepare(case, seed):
    from torch import nn

    from rwkv_mlx_amd import LoRAMoE_CMix, MoE_CMix, RWKV_CMix_x070, RWKVConfig

    t = _inputs(case, seed)
    kind = case["kind"]
    cfg = RWKVConfig(n_embd=case["d_model"], dim_ffn=case["d_ffn"])
    with torch.device("meta"):  # the parameters come from the seed
        if "experts" in kind:
            layer = MoE_CMix(cfg, 0, case["experts"], case["top_k"])
            names = {"x_k": "x_k", "expert_key": "key", "expert_val": "value", "router.gate.weight": "gate"}
        elif kind == "dense":
            layer = RWKV_CMix_x070(cfg, 0)
            names = {"x_k": "x_k", "key.weight": "key", "value.weight": "value"}
        else:
            layer = LoRAMoE_CMix(RWKV_CMix_x070(cfg, 0), case["experts"], case["rank"], case["top_k"])
            names = {"base.x_k": "x_k", "base.key.weight": "key", "base.value.weight": "value",
                     "router.gate.weight": "gate", "lora_A": "A", "lora_B": "B"}
    layer.load_state_dict({n: t[s] for n, s in names.items()}, assign=True)
    if "bias" in t:
        layer.router.logit_bias = t["bias"]
    state = {"case": case, "layer": layer, "x": t["x"], "ln": None}
    if case["block"]:
        state["ln"] = (t["ln_w"], t["ln_b"])
    if kind == "step":
        state["x"], state["x_prev"] = t["x"][:, 0].contiguous(), t["x_prev"]
    if "train" in kind:
        f32 = lambda v: torch.tensor(v, dtype=torch.float32, device=t["x"].device)
        for p in layer.parameters():
            p.requires_grad_(True)
        state["x"].requires_grad_(True)
        state["cotangents"] = [t["d_out"], f32(AUX_COEFF), f32(Z_COEFF)]
        if kind == "train":
            for p in layer.base.parameters():
                p.requires_grad_(False)
            state["params"] = [layer.lora_A, layer.lora_B, layer.router.gate.weight]
            state["cotangents"].append(f32(ORTHO_COEFF))
        else:
            state["params"] = [layer.x_k, layer.expert_key, layer.expert_val, layer.router.gate.weight]
    else:
        layer.requires_grad_(False)
    return state


def run(state):
    kind, layer, x, ln = state["case"]["kind"], state["layer"], state["x"], state["ln"]
    if "train" in kind:
        outs = list(layer(x))
        if kind == "train":
            outs.append(layer.orthogonal_loss())
        grads = torch.autograd.grad(outs, [x] + state["params"], state["cotangents"])
        return [o.detach() for o in outs] + list(grads)
    with torch.no_grad():
        if kind == "step":
            from rwkv_mlx_amd import channel_mixing_rnn
            return channel_mixing_rnn(x, state["x_prev"], layer, ln=ln)
        if kind == "layer" and ln is not None:
            return layer(x, residual=x, ln=ln)
        return layer(x)


def work(case):
    B, T, C, F, E, k, r = (case[n] for n in ("batch", "seq", "d_model", "d_ffn", "experts", "top_k", "rank"))
    N, s = B * T, DTYPES[case["dtype"]].itemsize
    a = 4 if case["fp32_adapters"] else s
    full = "experts" in case["kind"]
    # a few tokens reach only their own experts' weights
    live = min(E, N * k) if E else 0
    rows = N * k if full else N
    base_w = (live if full else 1) * 2 * F * C * s
    small_w = C * s + E * C * a + live * 2 * C * r * a
    flops = 4 * rows * F * C + 2 * N * C * E + 4 * N * k * C * r
    nbytes = base_w + small_w + N * C * (s + a)
    if case["kind"] == "step":
        nbytes += N * C * s
    if case["kind"] == "train":
        # dU, dx of the adapters, dA, dB; d gate and the router's dx
        flops += 8 * N * k * C * r + 4 * N * C * E + 4 * E * (E - 1) // 2 * r * r * C
        nbytes += N * C * (a + s) + E * C * a + 2 * E * C * r * a
    if case["kind"] == "experts_train":
        flops += 8 * rows * F * C + 4 * N * C * E
        nbytes += 2 * N * C * s + E * 2 * F * C * s + 2 * E * C * s
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # the outputs are rounded to the dtype once, and so are the hidden rows
    # and gradients on their way
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}


def _shift(x, prev):
    first = torch.zeros_like(x[:, :1]) if prev is None else prev[:, None]
    return torch.cat([first, x[:, :-1]], 1)


def _cmix(xk, key, value):
    return torch.relu(xk @ key.T) ** 2 @ value.T


def exact(case, seed):
    kind, k = case["kind"], case["top_k"]
    train = "train" in kind
    t = {n: v.double() for n, v in _inputs(case, seed).items()}
    B, T, C = t["x"].shape
    leaves = []
    if train:
        names = ["x", "A", "B", "gate"] if kind == "train" else ["x", "x_k", "key", "value", "gate"]
        leaves = [t[n].requires_grad_(True) for n in names]
    with torch.set_grad_enabled(train):
        x, x0 = t["x"], t["x"]
        if case["block"]:
            x = torch.nn.functional.layer_norm(x, (C,), t["ln_w"], t["ln_b"], 1e-5)
        sh = _shift(x, t.get("x_prev"))
        flat = x.reshape(-1, C)
        if kind == "dense":
            return _cmix(x + (sh - x) * t["x_k"], t["key"], t["value"])
        logits = flat @ t["gate"].T
        if "bias" in t:
            logits = logits + t["bias"]
        E = case["experts"]
        z = torch.logsumexp(logits, -1).square().mean()
        top, inds = logits.topk(k, -1)
        w = torch.zeros_like(logits).scatter(1, inds, top.softmax(-1))
        share = torch.zeros_like(logits).scatter(1, inds, 1.0).mean(0)
        aux = E * (share / k * logits.softmax(-1).mean(0)).sum()
        if "experts" in kind:
            out = torch.zeros_like(flat)
            mixed = sh.reshape(-1, C) - flat
            for e in range(E):
                at = (inds == e).any(1).nonzero()[:, 0]
                y = _cmix(flat[at] + mixed[at] * t["x_k"][e, 0, 0], t["key"][e], t["value"][e])
                out = out.index_add(0, at, w[at, e:e + 1] * y)
        else:
            with torch.no_grad():
                out = _cmix(x + (sh - x) * t["x_k"], t["key"], t["value"]).reshape(-1, C)
            for e in range(E):
                out = out + w[:, e:e + 1] * (flat @ t["A"][e] @ t["B"][e])
        out = out.reshape(B, T, C)
        if kind == "step":
            return out[:, 0], x[:, 0]
        if case["block"]:
            out = x0 + out
        outs = [out, aux, z]
        if not train:
            return tuple(outs)
        cot = [t["d_out"], *(torch.tensor(c, dtype=torch.float64, device=x.device) for c in (AUX_COEFF, Z_COEFF))]
        if kind == "train":
            gram = torch.einsum("icr,jcs->ijrs", t["A"], t["A"])
            pairs = torch.triu(torch.ones(E, E, device=x.device, dtype=torch.float64), 1)
            outs.append((gram.square().sum((2, 3)) * pairs).sum())
            cot.append(torch.tensor(ORTHO_COEFF, dtype=torch.float64, device=x.device))
        grads = torch.autograd.grad(outs, leaves, cot)
        return [o.detach() for o in outs] + list(grads)
