"""Performance cases of the MoE expert path: what users of the layer run, through its public entry points.

Each case is a dict of plain values; ``prepare`` makes its inputs and module on
the GPU, ``run`` makes one pass, ``exact`` gives the same outputs in 64 bits
with plain torch. The kinds:

* ``train``: forward and backward of ``MoELayer`` from given router logits
  (output, and gradients of the tokens, the logits and both weights);
* ``infer``: forward of ``MoELayer`` with its router, without gradients (decode
  and prefill);
* ``fp8_infer``: the same with blockwise-FP8 experts and sigmoid,
  group-limited routing;
* ``fp8_train``: forward and backward with FP8 experts and bf16 master weights;
* ``requantize``: the masters written back to e4m3 and block scales, as after
  every optimizer step;
* ``lora``: forward and backward of the layer with per-expert LoRA adapters
  over frozen experts and a frozen router;
* ``router``: forward and backward of ``TopKRouter`` with its losses.

Sizes are those of the package's workloads (``torchturbo_amd.configs``) and
generic ones around them.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import torchturbo_amd
from torchturbo_amd.moe import (Fp8GroupedMLP, GroupedMLP, MoEConfig, MoELayer, MoESubmodules,
                                ModuleSpec, TopKRouter)
from torchturbo_amd.moe.lora import GroupedMLPLoRA

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(name, kind, tokens, hidden, experts, topk, ffn, **more):
    case = {"name": name, "kind": kind, "tokens": tokens, "hidden": hidden, "experts": experts,
            "topk": topk, "ffn": ffn, "dtype": "bf16", "act": "silu", "skew": False, "groups": 0,
            "group_topk": 0, "rank": 0}
    case.update(more)
    return case


def listed():
    return [
        # Training step of the headline layer: many small experts, skewed loads.
        _case("train_16k", "train", 16384, 2048, 128, 8, 768, skew=True),
        # The largest: few large experts, a long batch.
        _case("train_8x14k", "train", 8192, 4096, 8, 2, 14336),
        # A short, ragged micro batch in f16 with a capped gate.
        _case("train_ragged_f16", "train", 1531, 1024, 64, 6, 704, dtype="f16", act="capped"),
        # The fp32 layer of a unit-sized model.
        _case("train_toy_f32", "train", 512, 256, 8, 2, 512, dtype="f32"),
        # Decode of one sequence: the smallest call, latency and launches.
        _case("decode_1", "infer", 1, 2048, 128, 8, 768),
        # Decode of a batch: a few rows for each expert, bound by its weights.
        _case("decode_48", "infer", 48, 2048, 128, 8, 768),
        # Prefill of one prompt.
        _case("prefill_1000", "infer", 1000, 2048, 128, 8, 768),
        # FP8 decode: large experts, weights read once.
        _case("fp8_decode_24", "fp8_infer", 24, 7168, 256, 8, 2048, groups=8, group_topk=4),
        # FP8 training with master weights, about 128 rows for each expert.
        _case("fp8_train_1k", "fp8_train", 1024, 7168, 64, 8, 2048, groups=8, group_topk=4),
        # The masters quantised again after an optimizer step.
        _case("fp8_requantize", "requantize", 0, 7168, 64, 8, 2048),
        # Adapter fine-tuning of the headline layer.
        _case("lora_2k_r16", "lora", 2048, 2048, 128, 8, 768, rank=16),
        # Router of a layer of many experts, with expert bias and both losses.
        _case("router_4k", "router", 4096, 7168, 256, 8, 0, groups=8, group_topk=4),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["train", "train", "infer", "infer", "fp8_infer", "fp8_train", "requantize",
                       "lora", "router"])
    while True:
        if kind == "train":
            dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
            experts = rng.choice([8, 16, 32, 60, 64, 128])
            case = _case("", kind, _log(rng, 256, 16384), 64 * _log(rng, 4, 64), experts,
                         rng.choice([1, 2, 4, 6, 8]), 32 * _log(rng, 8, 448), dtype=dtype,
                         act=rng.choice(["silu", "silu", "silu", "gelu", "capped"]),
                         skew=rng.random() < 0.5)
            rows = case["tokens"] * case["topk"]
            flops = 18.0 * rows * case["hidden"] * case["ffn"]
            weights = 3.0 * experts * case["hidden"] * case["ffn"]
            # At most the work of the largest listed case, at fp32's lower rate.
            fits = flops < (2e11 if dtype == "f32" else 1.2e13) and weights < 1.5e9
        elif kind == "infer":
            case = _case("", kind, _log(rng, 1, 4096), 64 * _log(rng, 16, 64),
                         rng.choice([32, 60, 64, 96, 128, 256]), rng.choice([2, 4, 6, 8]),
                         32 * _log(rng, 12, 96))
            fits = True
        elif kind == "fp8_infer":
            case = _case("", kind, _log(rng, 1, 2048), 128 * _log(rng, 16, 56),
                         rng.choice([64, 128, 256]), 8, 128 * _log(rng, 6, 16), groups=8,
                         group_topk=4)
            fits = True
        elif kind == "fp8_train":
            case = _case("", kind, _log(rng, 128, 2048), 128 * _log(rng, 8, 56),
                         rng.choice([16, 32, 64]), 8, 128 * _log(rng, 4, 16), groups=8,
                         group_topk=4)
            fits = True
        elif kind == "requantize":
            case = _case("", kind, 0, 128 * _log(rng, 8, 56), rng.randint(8, 64), 8,
                         128 * _log(rng, 4, 16))
            fits = True
        elif kind == "lora":
            case = _case("", kind, _log(rng, 256, 4096), 64 * _log(rng, 16, 40),
                         rng.choice([32, 64, 128]), rng.choice([2, 4, 8]), 32 * _log(rng, 12, 48),
                         rank=rng.choice([8, 16, 32, 64]))
            fits = True
        else:
            grouped = rng.random() < 0.5
            case = _case("", kind, _log(rng, 128, 16384), 64 * _log(rng, 16, 112),
                         rng.choice([64, 128, 256]), 8, 0, groups=8 if grouped else 0,
                         group_topk=4 if grouped else 0)
            fits = case["tokens"] * case["hidden"] < 5e7
        if fits:
            del case["name"]
            return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _normal(shape, g, std=1.0, dtype=torch.bfloat16):
    out = torch.empty(shape, dtype=dtype, device=DEV)
    if len(shape) == 3:  # one slice at a time: the fp32 values of one only
        for part in out:
            part.copy_(torch.empty(part.shape, device=DEV).normal_(0.0, std, generator=g))
        return out
    return out.copy_(torch.empty(shape, device=DEV).normal_(0.0, std, generator=g))


def _quantize(weight):
    """One expert's ``[R, C]`` weight in e4m3 with bf16 scales of 128 x 128 blocks."""
    R, C = weight.shape
    blocks = weight.float().view(R // 128, 128, C // 128, 128)
    amax = blocks.abs().amax(dim=(1, 3))
    scale = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax)).bfloat16()
    q = blocks / scale.float()[:, None, :, None]
    return q.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(R, C), scale


def _activation(case):
    return F.gelu if case["act"] == "gelu" else F.silu


def _config(case, dtype, **more):
    fp8 = case["groups"] > 0
    return MoEConfig(
        hidden_size=case["hidden"], num_moe_experts=case["experts"],
        moe_ffn_hidden_size=case["ffn"] or None, gated_linear_unit=True,
        activation_func=_activation(case), moe_router_topk=case["topk"],
        moe_router_score_function="sigmoid" if fp8 else "softmax",
        moe_router_num_groups=case["groups"] or None,
        moe_router_group_topk=case["group_topk"] or None,
        moe_router_topk_scaling_factor=2.5 if fp8 else None,
        moe_router_enable_expert_bias=fp8, moe_router_dtype="fp32", params_dtype=dtype,
        moe_swiglu_limit=[7.0] if case["act"] == "capped" else None, **more)


def _logits(case, g):
    T, E = case["tokens"], case["experts"]
    logits = torch.empty((T, E), device=DEV).normal_(generator=g)
    if case["skew"]:  # a Zipf(1.1) prior on the experts' loads
        rank = torch.randperm(E, generator=g, device=DEV) + 1.0
        logits -= 1.1 * torch.log(rank)
    return logits


def prepare(case, seed):
    torchturbo_amd.init_ops()
    kind = case["kind"]
    T, H, E, Fi = case["tokens"], case["hidden"], case["experts"], case["ffn"]
    dtype = DTYPES[case["dtype"]]
    g = torch.Generator(device=DEV).manual_seed(seed)
    state = {"case": case}
    with torch.device(DEV):
        if kind == "router":
            module = TopKRouter(_config(case, dtype, moe_aux_loss_coeff=1e-3, moe_z_loss_coeff=1e-3))
        elif kind == "requantize":
            module = Fp8GroupedMLP(E, False, _config(case, dtype))
        else:
            fp8 = kind in ("fp8_infer", "fp8_train")
            spec = ModuleSpec(module=Fp8GroupedMLP if fp8 else GroupedMLP,
                              params={"with_master": kind == "fp8_train"} if fp8 else {})
            module = MoELayer(_config(case, dtype), None, MoESubmodules(experts=spec),
                              layer_number=0)
    router = module if kind == "router" else getattr(module, "router", None)
    experts = module if kind == "requantize" else getattr(module, "experts", None)
    with torch.no_grad():
        if router is not None:
            router.weight.copy_(_normal((E, H), g, 0.02))
            if router.expert_bias is not None:
                router.expert_bias.normal_(0.0, 0.01, generator=g)
        if isinstance(experts, GroupedMLP):
            experts.weight1.view(E, H, 2 * Fi).copy_(_normal((E, H, 2 * Fi), g, 0.02, dtype))
            experts.weight2.view(E, Fi, H).copy_(_normal((E, Fi, H), g, 0.02, dtype))
        elif experts is not None:
            for q, s, m in ((experts.q1, experts.s1, experts.master1),
                            (experts.q2, experts.s2, experts.master2)):
                for e in range(E):
                    w = torch.empty(q.shape[1:], device=DEV).normal_(0.0, 0.02, generator=g)
                    if m is not None:
                        m[e].copy_(w)
                    if kind != "requantize":  # a step's masters are not quantised yet
                        q[e], s[e] = _quantize(w.bfloat16())
    if kind == "lora":
        module.requires_grad_(False)
        module.experts = GroupedMLPLoRA(experts, "default", r=case["rank"],
                                        lora_alpha=2 * case["rank"])
        with torch.no_grad():  # as some steps in: B is no longer zero
            for name, p in module.experts.named_parameters():
                if "lora_A" in name:
                    p.copy_(_normal(tuple(p.shape), g, 1.0 / math.sqrt(p.shape[1]), p.dtype))
                elif "lora_B" in name:
                    p.copy_(_normal(tuple(p.shape), g, 0.01, p.dtype))
    state["module"] = module
    if kind == "requantize":
        return state
    state["x"] = _normal((T, H), g, 1.0, dtype)
    if kind in ("train", "fp8_train", "lora"):
        state["grad"] = _normal((T, H), g, 1.0, dtype)
    if kind in ("train", "fp8_train"):
        state["logits"] = _logits(case, g)
    if kind == "router":
        state["grad"] = torch.empty((T, E), device=DEV).normal_(generator=g)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
ADAPTERS = ("lora_A", "lora_B", "lora_A2", "lora_B2")


def run(state):
    case, module = state["case"], state["module"]
    kind = case["kind"]
    if kind == "requantize":
        module.requantize()
        return {"q1": module.q1.view(torch.uint8), "s1": module.s1,
                "q2": module.q2.view(torch.uint8), "s2": module.s2}
    if kind in ("infer", "fp8_infer"):
        with torch.no_grad():
            out, logits = module(state["x"])
        return {"out": out, "router_logits": logits}
    x = state["x"].detach().requires_grad_()
    if kind == "router":
        probs, routing_map, _, logits = module(x)
        counts = getattr(module, "local_tokens_per_expert", None)
        result = {"probs": probs.detach(), "map": routing_map, "router_logits": logits.detach()}
        if counts is not None:  # this step's loads, taken and cleared for the next
            result["counts"] = counts.clone()
            counts.zero_()
        result["d_x"], result["d_weight"] = torch.autograd.grad(
            probs, (x, module.weight), state["grad"])
        return result
    if kind == "lora":
        out, _ = module(x)
        weights = [getattr(module.experts, n)["default"].weight for n in ADAPTERS]
        grads = torch.autograd.grad(out, (x, *weights), state["grad"])
        return {"out": out.detach(), "d_x": grads[0],
                **{"d_" + n: v for n, v in zip(ADAPTERS, grads[1:])}}
    logits = state["logits"].detach().requires_grad_()
    experts = module.experts
    weights = ((experts.weight1, experts.weight2) if kind == "train"
               else (experts.master1, experts.master2))
    out = module.forward_with_logits(x, logits)
    d_x, d_logits, d_w1, d_w2 = torch.autograd.grad(out, (x, logits, *weights), state["grad"])
    return {"out": out.detach(), "d_x": d_x, "d_logits": d_logits, "d_w1": d_w1, "d_w2": d_w2}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _choose(case, scores):
    """Ids of the selected experts, as the router's rule takes them."""
    if not case["group_topk"]:
        return torch.topk(scores, case["topk"], dim=1).indices
    T, E = scores.shape
    groups = scores.view(T, case["groups"], -1)
    value = groups.topk(case["topk"] // case["group_topk"], dim=-1).values.sum(-1)
    keep = torch.zeros_like(value, dtype=torch.bool).scatter_(
        1, value.topk(case["group_topk"], dim=1).indices, True)
    scores = groups.masked_fill(~keep.unsqueeze(-1), -math.inf).view(T, E)
    return torch.topk(scores, case["topk"], dim=1).indices


def _route(case, logits, bias):
    """(ids [T, k], probabilities [T, k]) of 64-bit logits."""
    if case["groups"]:
        scores = torch.sigmoid(logits)
        ids = _choose(case, (scores + bias.double()).detach())
        chosen = scores.gather(1, ids)
        return ids, chosen / (chosen.sum(1, keepdim=True) + 1e-20) * 2.5
    ids = _choose(case, logits.detach())
    return ids, torch.softmax(logits.gather(1, ids), dim=1)


def _gate(case, h):
    gate, up = h.chunk(2, dim=1)
    if case["act"] == "capped":
        gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
    return _activation(case)(gate) * up


def _weights(state, e):
    """The leaves of expert e in 64 bits, and the function of them that gives (W1 [H, 2F], W2 [F, H])."""
    case, experts = state["case"], state["module"].experts
    E, H = case["experts"], case["hidden"]
    if isinstance(experts, GroupedMLPLoRA):
        base, scale = experts.base_layer, experts.scaling["default"]
        w1, w2 = (w.view(E, -1, w.shape[1])[e].double() for w in (base.weight1, base.weight2))
        leaves = [getattr(experts, n)["default"].weight[e].detach().double() for n in ADAPTERS]
        return leaves, lambda a, b, a2, b2: (w1 + scale * (a @ b), w2 + scale * (a2 @ b2))
    if isinstance(experts, Fp8GroupedMLP):
        leaves = []
        for q, s in ((experts.q1, experts.s1), (experts.q2, experts.s2)):
            full = s[e].float().repeat_interleave(128, 0).repeat_interleave(128, 1)
            leaves.append((q[e].float() * full).bfloat16().double())  # the format's value
        return leaves, lambda q1, q2: (q1.t(), q2.t())
    leaves = [w.detach().view(E, -1, w.shape[1])[e].double()
              for w in (experts.weight1, experts.weight2)]
    return leaves, lambda w1, w2: (w1, w2)


def _experts(state, x, ids, probs, grad):
    """The experts' output and, with ``grad``, its gradients of x, probs and each expert's leaves."""
    case = state["case"]
    out, dx, dp = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(probs)
    dw = None
    for e in range(case["experts"]):
        t, j = (ids == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        leaves, build = _weights(state, e)
        rows, p = x[t], probs[t, j]
        if grad is not None:
            for v in (rows, p, *leaves):
                v.requires_grad_()
        w1, w2 = build(*leaves)
        y = (_gate(case, rows @ w1) * p.unsqueeze(1)) @ w2
        out.index_add_(0, t, y.detach())
        if grad is not None:
            got = torch.autograd.grad(y, (rows, p, *leaves), grad[t])
            dx.index_add_(0, t, got[0])
            dp[t, j] = got[1]
            if dw is None:
                dw = [torch.zeros((case["experts"], *v.shape), dtype=v.dtype, device=DEV)
                      for v in leaves]
            for full, v in zip(dw, got[2:]):
                full[e] = v
    return out, dx, dp, dw


def exact(case, seed):
    state = prepare(case, seed)
    module, kind = state["module"], case["kind"]
    if kind == "requantize":
        result = {}
        for n, m in (("1", module.master1), ("2", module.master2)):
            E, R, C = m.shape
            amax = torch.stack([w.double().view(R // 128, 128, C // 128, 128).abs().amax((1, 3))
                                for w in m.detach()])
            result["q" + n], result["s" + n] = None, amax / 448.0
        return result
    x = state["x"].double()
    if "logits" in state:
        router, weight, bias = module.router, None, module.router.expert_bias
        logits = state["logits"].double().requires_grad_()
    else:
        router = module if kind == "router" else module.router
        weight, bias = router.weight.detach().double().requires_grad_(), router.expert_bias
        x.requires_grad_()
        logits = x @ weight.t()
    ids, probs = _route(case, logits, bias)
    if kind == "router":
        T, E = case["tokens"], case["experts"]
        dense = torch.zeros_like(logits).scatter(1, ids, probs)
        chosen = torch.zeros_like(logits).scatter(1, ids, 1.0).detach()
        scores = torch.sigmoid(logits) if case["groups"] else torch.softmax(logits, dim=1)
        if case["groups"]:
            scores = scores / (scores.sum(1, keepdim=True) + 1e-20)
        top = torch.topk(scores.detach(), case["topk"], dim=1).indices
        load = torch.zeros_like(scores).scatter(1, top, 1.0).detach().sum(0)
        total = load.sum() / case["topk"]
        aux = 1e-3 * (scores.sum(0) * load).sum() * E / (case["topk"] * total * total)
        z = 1e-3 * torch.logsumexp(logits, dim=1).square().mean()
        loss = (dense * state["grad"].double()).sum() + aux + z
        d_x, d_weight = torch.autograd.grad(loss, (x, weight))
        result = {"probs": dense.detach(), "map": None, "router_logits": logits.detach(),
                  "d_x": d_x, "d_weight": d_weight}
        if bias is not None:
            result["counts"] = chosen.sum(0)
        return result
    grad = state["grad"].double() if "grad" in state else None
    out, dx, dp, dw = _experts(state, x.detach(), ids, probs.detach(), grad)
    if grad is None:
        return {"out": out, "router_logits": logits.detach()}
    if kind == "lora":
        dx = dx + torch.autograd.grad(probs, x, dp)[0]
        return {"out": out, "d_x": dx, **{"d_" + n: v for n, v in zip(ADAPTERS, dw)}}
    (d_logits,) = torch.autograd.grad(probs, logits, dp)
    if kind == "train":  # the layer's parameters hold all experts' rows in two dimensions
        dw = [v.view(-1, v.shape[2]) for v in dw]
    return {"out": out, "d_x": dx, "d_logits": d_logits, "d_w1": dw[0], "d_w2": dw[1]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    T, H, E, k, Fi = (case[n] for n in ("tokens", "hidden", "experts", "topk", "ffn"))
    b = 4 if case["dtype"] == "f32" else 2
    weights = 3.0 * H * Fi  # of one expert
    if kind == "requantize":
        return {"bytes": 3.0 * E * weights, "flops": 2.0 * E * weights}
    rows = T * k
    gemm = 2.0 * rows * weights
    used = E * (1.0 - (1.0 - k / E) ** T)  # experts that some token takes
    router = 2.0 * T * H * E
    gating = E * H * 2.0 + T * E * 4.0
    if kind == "router":
        # x, the weight and the gradient in; probabilities, map, logits and both gradients out.
        return {"bytes": 2.0 * T * H * b + 2.0 * E * H * b + T * E * (4 + 4 + 4 + 1),
                "flops": 3.0 * router}
    if kind == "infer":
        return {"bytes": 2.0 * T * H * b + used * weights * b + gating, "flops": gemm + router}
    if kind == "fp8_infer":
        return {"bytes": 2.0 * T * H * 2 + used * weights + gating, "flops": gemm + router}
    if kind == "fp8_train":
        return {"bytes": 4.0 * T * H * 2 + 2.0 * T * E * 4 + used * weights + E * weights * 2,
                "flops": 3.0 * gemm}
    if kind == "lora":
        r = case["rank"]
        adapters = r * (2.0 * H + 3.0 * Fi)  # of one expert
        return {"bytes": 4.0 * T * H * b + used * weights * b + 2.0 * E * adapters * 4 + gating,
                "flops": 2.0 * gemm + 6.0 * rows * adapters + 2.0 * router}
    return {"bytes": 4.0 * T * H * b + 2.0 * T * E * 4 + used * weights * b + E * weights * b,
            "flops": 3.0 * gemm}


def tolerance(case):
    if case["kind"] == "requantize":
        return "exact"  # bytes and scales of a format, each rounded once
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["dtype"] == "f16":
        return {"rel": 2e-3, "max": 0.08}
    # 16-bit activations between the layer's products; near ties of the router may be
    # taken the other way where its fp32 sums run in another order.
    return {"rel": 1e-2, "max": 0.4, "differ": 1e-3}
