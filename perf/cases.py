"""Performance cases of the MoE layer: the calls that a program makes, over the range it makes them in.

A case is a dict of plain values:
  kind    "fwd": a forward-only call (decoding, prefill, evaluation) through Plan.forward
          "train": a forward and a backward through Plan.forward and Plan.backward, as a trainer
          with weights and gradient buffers of its own calls them
          "layer": the same step through the autograd module MoeLayer
          "block": the same step through MoeBlock (RMSNorm, layer, residual), activations recomputed
  T, H, E, k, I, S   tokens, hidden size, experts, experts per token, expert width, shared width
  dtype   "bf16" or "f32"
  skew    "none", "zipf" or "lognormal": how uneven the experts' loads are (oxidizr_amd.synth)
  norm, bias   renormalised routing weights; a router bias that is trained

Inputs are made on the GPU from the seed alone: x and the upstream gradient N(0, 1), as after a norm;
weights N(0, std^2) with std 0.02, or 0.006 for the widest layer.
"""
import math

import torch

from oxidizr_amd import synth
from oxidizr_amd.moe import MoeBlock, MoeConfig, MoeLayer, Plan

LB_ALPHA, Z_ALPHA = 0.01, 1e-3  # the trainer's loss coefficients: d(aux), d(z) of a step


def case_of(kind, T, H, E, k, I, S, dtype="bf16", skew="none", norm=False, bias=False):
    return {"kind": kind, "T": T, "H": H, "E": E, "k": k, "I": I, "S": S, "dtype": dtype,
            "skew": skew, "norm": norm, "bias": bias}


def listed():
    named = {
        # one sequence decoding: latency, launches, and the weights of k experts
        "decode_1": case_of("fwd", 1, 2048, 64, 6, 1408, 2816),
        # a few sequences decoding on a layer of few experts
        "decode_16": case_of("fwd", 16, 2048, 16, 2, 1408, 2816),
        # a serving batch that touches nearly every expert: the weights' stream (config 4)
        "decode_64": case_of("fwd", 64, 4096, 128, 8, 1536, 0),
        # a larger serving batch, or a short ragged prompt, on the same layer
        "decode_200": case_of("fwd", 200, 4096, 128, 8, 1536, 0, norm=True),
        # a prompt, and evaluation without gradients
        "prefill_1500": case_of("fwd", 1500, 2048, 64, 6, 1408, 2816),
        # a small fp32 training step (config 1)
        "train_f32_1k": case_of("train", 1024, 384, 8, 2, 1024, 0, dtype="f32"),
        # fp32 at odd sizes, with every router option
        "train_f32_odd": case_of("train", 1999, 776, 12, 3, 1368, 680, dtype="f32",
                                 norm=True, bias=True),
        # a micro-batch of fine-tuning
        "train_500": case_of("train", 500, 2048, 16, 2, 1408, 2816),
        # a training step through the autograd module (config 2)
        "train_8k": case_of("layer", 8192, 2048, 16, 2, 1408, 2816),
        # the decoder block's whole MoE half with activation checkpointing
        "block_4k": case_of("block", 4096, 2048, 16, 2, 1408, 2816),
        # many experts, skewed loads, an empty expert (config 3)
        "train_16k_zipf": case_of("train", 16384, 2048, 64, 6, 1408, 2816, skew="zipf", bias=True),
        # the largest layer: 256 wide experts, uneven loads (config 5)
        "train_8k_wide": case_of("train", 8192, 7168, 256, 8, 2048, 2048, skew="lognormal",
                                 bias=True),
    }
    return [dict(c, name=n) for n, c in named.items()]


def draw(rng):
    """A case of the listed ones' ranges: sizes spread over their logarithm, odd ones among them."""
    def size(lo, hi, step):
        return max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)

    while True:
        kind = rng.choice(("fwd", "fwd", "fwd", "train", "train", "train", "layer", "block"))
        dtype = "f32" if kind == "train" and rng.random() < 0.4 else "bf16"
        E = rng.choice((8, 12, 16) if kind in ("layer", "block") or dtype == "f32"
                       else (8, 12, 16, 24, 32, 64, 64, 128, 128, 256))
        T = size(1, 2048, 1) if kind == "fwd" else size(256, 16384, 1)
        H = size(384, 7168, rng.choice((8, 128)))
        I = size(512, 2048, rng.choice((8, 64)))
        k = min(E, rng.choice((1, 2, 2, 3, 4, 6, 8)))
        S = rng.choice((0, 0, I, 2 * I))
        skew = rng.choice(("none", "none", "none", "lognormal")) if kind == "train" else "none"
        norm = rng.random() < 0.3
        bias = skew != "none" or (kind == "train" and rng.random() < 0.2)
        c = case_of(kind, T, H, E, k, I, S, dtype, skew, norm, bias)
        w = work(c)
        # within the largest listed case's work (fp32 runs at 1/16 of the bf16 rate)
        if w["bytes"] < 2e10 and w["flops"] < (4e11 if dtype == "f32" else 4e12):
            return c


def work(case):
    T, H, E, k, I, S = (case[n] for n in "THEkIS")
    b = 4 if case["dtype"] == "f32" else 2
    touched = E * (1.0 - (1.0 - k / E) ** T)  # experts that a balanced routing reaches
    weights = b * (3.0 * touched * I * H + 3.0 * S * H + E * H)
    flops = 2.0 * T * H * E + 6.0 * T * k * H * I + 6.0 * T * H * S
    if case["kind"] == "fwd":
        return {"bytes": weights + 2.0 * b * T * H, "flops": flops}
    return {"bytes": 2.0 * weights + 4.0 * b * T * H, "flops": 3.0 * flops}


def tolerance(case):
    # Measured against exact(): 32-bit sums are up to 1.1e-6 off, bf16 (which rounds x W, silu(g) u
    # and their gradients once per GEMM) up to 3.5e-3
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 1e-2}


def inputs(case, seed):
    """Every input tensor of a case, by name; expert weights packed [E, ...]."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    T, H, E, k, I, S = (case[n] for n in "THEkIS")
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    std = 0.006 if H > 4096 else 0.02

    def normal(shape, scale):
        t = torch.empty(shape, dtype=dt, device=dev)
        return t.normal_(0.0, scale, generator=g)

    p = {"x": normal((T, H), 1.0), "router": normal((E, H), std), "gate": normal((E, I, H), std),
         "up": normal((E, I, H), std), "down": normal((E, H, I), std)}
    if S:
        p.update(shared_gate=normal((S, H), std), shared_up=normal((S, H), std),
                 shared_down=normal((H, S), std))
    if case["kind"] != "fwd":
        p["dout"] = normal((T, H), 1.0)
    if case["kind"] == "block":
        p["norm_w"] = 1.0 + normal((H,), 0.1)
    if case["skew"] != "none":
        p["bias"] = synth.skew_bias(T, k, E, case["skew"], p["x"], p["router"])[0].contiguous()
    elif case["bias"]:
        p["bias"] = torch.empty(E, device=dev).normal_(0.0, 0.1, generator=g)
    return p


def config(case):
    return MoeConfig(hidden_size=case["H"], num_experts=case["E"], experts_per_tok=case["k"],
                     intermediate_size=case["I"], shared_expert_enabled=case["S"] > 0,
                     shared_intermediate_size=case["S"] or None, norm_topk_prob=case["norm"],
                     router_bias=case["bias"], recompute_activations=case["kind"] == "block")


def prepare(case, seed):
    p = inputs(case, seed)
    dev, dt = p["x"].device, p["x"].dtype
    T, H, E, S = (case[n] for n in "THES")
    s = {"kind": case["kind"], "S": S, "d_aux": torch.tensor(LB_ALPHA, device=dev),
         "d_z": torch.tensor(Z_ALPHA, device=dev)}
    if case["kind"] in ("layer", "block"):
        module = (MoeBlock if case["kind"] == "block" else MoeLayer)(config(case), dt, dev)
        layer = module.ffn if case["kind"] == "block" else module
        with torch.no_grad():
            for name, param in module.trainable_parameters():
                part = name.split(".")
                if part[0] == "experts":
                    param.copy_(p[part[2].replace("_proj", "")][int(part[1])])
                elif part[0] == "shared_expert":
                    param.copy_(p["shared_" + part[1].replace("_proj", "")])
                elif part[0] == "router":
                    param.copy_(p["bias" if part[-1] == "bias" else "router"])
                else:
                    param.copy_(p["norm_w"])
        s.update(module=module, layer=layer, x=p["x"].view(1, T, H).requires_grad_(),
                 dout=p["dout"].view(1, T, H))
        return s
    plan = Plan(config(case), dt, dev)
    shared = tuple(p["shared_" + n] for n in ("gate", "up", "down")) if S else None
    tables = [list(p[n].unbind(0)) for n in ("gate", "up", "down")]
    s["w"], s["w_tables"] = plan.weights_struct(p["router"], *tables, p.get("bias"), shared)
    s.update(plan=plan, p=p)
    if case["kind"] == "train":
        grads = {n: torch.zeros_like(v) for n, v in p.items() if n not in ("x", "dout")}
        g_shared = tuple(grads["shared_" + n] for n in ("gate", "up", "down")) if S else None
        g_tables = [list(grads[n].unbind(0)) for n in ("gate", "up", "down")]
        s["g"], s["g_tables"] = plan.grads_struct(grads["router"], *g_tables, grads.get("bias"),
                                                  g_shared)
        s.update(grads=grads, has_grad=torch.zeros(E, dtype=torch.uint8, device=dev))
    return s


def run(s):
    if s["kind"] == "fwd":
        out, aux, z, _ = s["plan"].forward(s["p"]["x"], s["w"], need_grad=False)
        return {"out": out, "aux": aux, "z": z}
    if s["kind"] == "train":
        plan, x = s["plan"], s["p"]["x"]
        out, aux, z, saved = plan.forward(x, s["w"])
        dx = plan.backward(x, s["p"]["dout"], s["w"], s["g"], saved, d_aux=s["d_aux"],
                           d_z=s["d_z"], has_grad=s["has_grad"])
        return {"out": out, "aux": aux, "z": z, "dx": dx, "has_grad": s["has_grad"],
                "grads": s["grads"]}
    module, layer, x = s["module"], s["layer"], s["x"]
    x.grad = None
    module.zero_grad(set_to_none=True)
    out, aux, z = module(x)
    torch.autograd.backward((out, aux, z), (s["dout"], s["d_aux"], s["d_z"]))
    experts = layer.experts
    grads = {"gate": [e.gate_proj.weight.grad for e in experts],
             "up": [e.up_proj.weight.grad for e in experts],
             "down": [e.down_proj.weight.grad for e in experts],
             "router": layer.router.gate.weight.grad}
    if s["S"]:
        sh = layer.shared_expert
        grads.update(shared_gate=sh.gate_proj.weight.grad, shared_up=sh.up_proj.weight.grad,
                     shared_down=sh.down_proj.weight.grad)
    if s["kind"] == "block":
        grads["norm_w"] = module.post_attention_layernorm.weight.grad
    return {"out": out.detach(), "aux": aux.detach(), "z": z.detach(), "dx": x.grad,
            "grads": grads}


def swiglu(x, gate, up, down, dy):
    """(y, dx, d_gate, d_up, d_down) of one SwiGLU expert in float64 (the last four None without dy)."""
    gate, up, down = gate.double(), up.double(), down.double()
    g, u = x @ gate.t(), x @ up.t()
    sg = torch.sigmoid(g)
    a = g * sg * u
    y = a @ down.t()
    if dy is None:
        return y, None, None, None, None
    dy = dy(y)
    da = dy @ down
    dg, du = da * u * (sg * (1.0 + g * (1.0 - sg))), da * g * sg
    return y, dg @ gate + du @ up, dg.t() @ x, du.t() @ x, dy.t() @ a


def exact(case, seed):
    """What run() returns, in float64 from the same inputs."""
    p = inputs(case, seed)
    T, H, E, k, S = (case[n] for n in "THEkS")
    back = case["kind"] != "fwd"
    h = x = p["x"].double()
    if case["kind"] == "block":
        rstd = torch.rsqrt(h.square().mean(1, keepdim=True) + 1e-6)
        nw = p["norm_w"].double()
        x = (h * rstd * nw).to(p["x"].dtype).double()  # the layer's input has the layer's dtype
    wr = p["router"].double()
    logits = x @ wr.t()
    if "bias" in p:
        logits = logits + p["bias"].double()
    probs = torch.softmax(logits, 1)
    lse = torch.logsumexp(logits, 1)
    idx = torch.topk(logits, k, dim=1).indices
    top = torch.gather(probs, 1, idx)
    w = top / top.sum(1, keepdim=True) if case["norm"] else top
    counts = torch.bincount(idx.flatten(), minlength=E)
    f, mean_p = counts.double() / (T * k), probs.mean(0)
    res = {"aux": E * ((f * mean_p).sum() + mean_p.square().sum()), "z": lse.square().mean()}
    out = torch.zeros_like(x)
    if back:
        dout = p["dout"].double()
        dx, dw = torch.zeros_like(x), torch.zeros_like(w)
        grads = {n: torch.zeros(p[n].shape, dtype=torch.float64, device=x.device)
                 for n in ("gate", "up", "down")}
    for e in range(E):
        t, j = torch.nonzero(idx == e, as_tuple=True)
        if t.numel() == 0:
            continue
        we = w[t, j].unsqueeze(1)

        def upstream(y):
            dw[t, j] = (dout[t] * y).sum(1)
            return we * dout[t]
        y, dxe, *de = swiglu(x[t], p["gate"][e], p["up"][e], p["down"][e],
                             upstream if back else None)
        out.index_add_(0, t, we * y)
        if back:
            dx.index_add_(0, t, dxe)
            for n, d in zip(("gate", "up", "down"), de):
                grads[n][e] = d
    if S:
        y, dxe, *de = swiglu(x, p["shared_gate"], p["shared_up"], p["shared_down"],
                             (lambda y: dout) if back else None)
        out += y
        if back:
            dx += dxe
            grads.update(zip(("shared_gate", "shared_up", "shared_down"), de))
    res["out"] = out + h if case["kind"] == "block" else out
    if not back:
        return res
    if case["norm"]:
        dw = (dw - (dw * w).sum(1, keepdim=True)) / top.sum(1, keepdim=True)
    dp = (LB_ALPHA * E / T * (f + 2.0 * mean_p)).expand(T, E).clone()
    dp.scatter_add_(1, idx, dw)
    dl = probs * (dp - (probs * dp).sum(1, keepdim=True))
    dl += Z_ALPHA * 2.0 / T * lse.unsqueeze(1) * probs
    grads["router"] = dl.t() @ x
    dx += dl @ wr
    if "bias" in p:
        grads["bias"] = dl.sum(0)
    if case["kind"] == "block":
        xh = h * rstd
        grads["norm_w"] = (dx * xh).sum(0)
        dx = dout + rstd * (nw * dx - xh * (xh * nw * dx).mean(1, keepdim=True))
    res["dx"] = dx
    if case["kind"] in ("layer", "block"):
        routed = (counts > 0).tolist()
        for n in ("gate", "up", "down"):
            grads[n] = [d if r else None for d, r in zip(grads[n], routed)]
        res["dx"] = dx.view(1, T, H)
        res["out"] = res["out"].view(1, T, H)
    if case["kind"] == "train":
        res["has_grad"] = (counts > 0).to(torch.uint8)
    res["grads"] = grads
    return res
