"""The work that users of this package have it do, at the sizes they have it do it: LoRA fine-tuning over frozen packed
GGUF weights (forward and backward of the dense and the expert projections, the loss through the packed lm_head), and the
forward passes of evaluating and sampling from the adapted model, down to one token at a time.

A case is one call sequence of a training step or of a forward pass on one layer:

  linear_step / linear_forward      ``FastGGUFLoraLinear`` with its adapter active
  experts_step / experts_forward    ``FastGGUFMoeLora`` over packed experts; the forward passes select the experts with the
                                    package's router, the training steps are handed the selection and its weights
  loss_step                         ``packed_linear_cross_entropy`` and the gradient of the hidden states
  head_forward                      the lm_head as a layer (``GGUFLinear``), for logits

Weights are drawn from N(0, 0.02^2) and quantized, activations and cotangents from N(0, 1), LoRA factors as an adapter in
training holds them (A of norm one per row, B small and non-zero)."""

from __future__ import annotations

import torch

import __graft_entry__

Q8_0, Q2_K, Q4_K, Q6_K, IQ2_XXS = 8, 10, 12, 14, 16
# (elements, bytes) of a block
BLOCKS = {Q8_0: (32, 34), Q2_K: (256, 84), Q4_K: (256, 144), Q6_K: (256, 210), IQ2_XXS: (256, 66)}
DEVICE = "cuda"


# ------------------------------------------------------------------------------------------------
# the cases
def _linear(kind, tokens, in_features, out_features, quant, rank=16):
    return dict(kind=kind, tokens=tokens, in_features=in_features, out_features=out_features, quant=quant, rank=rank)


def _experts(kind, tokens, hidden, inter, experts, top_k, quant, down_quant, rank=16):
    return dict(kind=kind, tokens=tokens, hidden=hidden, inter=inter, experts=experts, top_k=top_k, quant=quant, down_quant=down_quant, rank=rank)


def _head(kind, tokens, hidden, vocab, quant, chunk=0):
    return dict(kind=kind, tokens=tokens, hidden=hidden, vocab=vocab, quant=quant, chunk=chunk)


def listed():
    cases = {
        # one token through an attention projection while sampling: the smallest call there is
        "linear_decode_q4k": _linear("linear_forward", 1, 2048, 4096, Q4_K),
        # a short sequence through a square Q8_0 projection, forward and backward
        "linear_step_q8_0": _linear("linear_step", 512, 2048, 2048, Q8_0),
        # a batch of four sequences of 1024 through an attention projection, forward and backward
        "linear_step_q4k": _linear("linear_step", 4096, 2048, 4096, Q4_K),
        # an unpadded sequence through a narrow (key / value) projection: ragged rows, few output columns, a smaller rank
        "linear_step_q6k_ragged": _linear("linear_step", 1021, 2048, 512, Q6_K, rank=8),
        # the next token's logits while sampling: one row against the whole packed vocabulary
        "head_decode_q6k": _head("head_forward", 1, 2048, 151936, Q6_K),
        # one token through the router and eight of 256 experts while sampling
        "experts_decode_q4k": _experts("experts_forward", 1, 2048, 512, 256, 8, Q4_K, Q4_K),
        # evaluation or the prompt of a sample: a few rows for every expert, forward only
        "experts_prompt_q4k": _experts("experts_forward", 515, 2048, 512, 256, 8, Q4_K, Q4_K),
        # training on one short unpadded sequence
        "experts_step_q4k_short": _experts("experts_step", 997, 2048, 512, 256, 8, Q4_K, Q4_K),
        # the training step that bench.py times
        "experts_step_q4k": _experts("experts_step", 4096, 2048, 512, 256, 8, Q4_K, Q4_K),
        # the large expert layer at two bits per weight
        "experts_step_iq2xxs": _experts("experts_step", 2048, 4096, 2048, 256, 8, IQ2_XXS, IQ2_XXS),
        # the loss of one short unpadded sequence with the default chunk
        "loss_q6k_short": _head("loss_step", 701, 2048, 151936, Q6_K, chunk=256),
        # the loss of the whole batch, and the gradient of its hidden states
        "loss_q6k": _head("loss_step", 4096, 2048, 151936, Q6_K, chunk=1024),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, low, high):
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear_forward", "linear_step", "linear_step", "experts_forward", "experts_step", "experts_step", "head_forward", "loss_step"])
    if kind.startswith("linear"):
        # a few rows while sampling (one per sequence) up to a prompt; training sequences and batches of them
        tokens = _log_int(rng, 1, 2048) if kind == "linear_forward" else _log_int(rng, 128, 4096)
        return _linear(kind, tokens, 256 * rng.randint(4, 16), 32 * _log_int(rng, 8, 256), rng.choice([Q8_0, Q4_K, Q6_K]),
                       rng.choice([4, 8, 16, 32]))
    if kind.startswith("experts"):
        tokens = _log_int(rng, 1, 2048) if kind == "experts_forward" else _log_int(rng, 128, 4096)
        if rng.random() < 0.7:
            return _experts(kind, tokens, rng.choice([1024, 1536, 2048]), rng.choice([256, 512, 768]), rng.choice([64, 128, 256]),
                            rng.randint(4, 8), Q4_K, Q4_K, rng.choice([8, 16]))
        return _experts(kind, min(tokens, 2048), rng.choice([2048, 4096]), rng.choice([1024, 2048]), rng.choice([128, 256]),
                        rng.choice([6, 8]), IQ2_XXS, rng.choice([IQ2_XXS, Q2_K]), rng.choice([8, 16]))
    if kind == "head_forward":
        return _head(kind, _log_int(rng, 1, 64), 256 * rng.randint(4, 16), rng.randint(32000, 151936), rng.choice([Q8_0, Q6_K]))
    return _head(kind, _log_int(rng, 128, 4096), 256 * rng.randint(4, 8), rng.randint(32000, 151936), rng.choice([Q8_0, Q6_K]),
                 rng.choice([256, 512, 1024]))


# ------------------------------------------------------------------------------------------------
# what a program holds before the call
def _package():
    return __graft_entry__.import_package()


def _bf16(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEVICE) * std).to(torch.bfloat16)


def _packed_rows(pkg, gen, rows, k, quant):
    """[rows, row bytes] of weights N(0, 0.02^2)."""
    if quant == IQ2_XXS:
        # the nearest-point fit is slow: 4096 rows are fitted, and the matrix takes rows of those in random order
        pool = pkg.gguf.quantize(torch.randn(min(rows, 4096), k, generator=gen, device=DEVICE) * 0.02, quant)
        return pool[torch.randint(0, pool.shape[0], (rows,), generator=gen, device=DEVICE)]
    if quant == Q2_K:
        # uniform levels and sub-block scales; d and dmin such that the weights are centred with a spread of about 0.02
        b = torch.randint(0, 256, (rows * (k // 256), 84), dtype=torch.uint8, generator=gen, device=DEVICE)
        d = 0.002 * (0.8 + 0.4 * torch.rand(b.shape[0], 1, generator=gen, device=DEVICE))
        half = torch.cat([d, 1.5 * d], dim=1).to(torch.float16).contiguous()
        b[:, 80:84] = half.view(torch.uint8).reshape(-1, 4)
        return b.reshape(rows, k // 256 * 84)
    step = max(1, (1 << 26) // k)  # slices of 64 M weights bound the fp32 copy
    return torch.cat([pkg.gguf.quantize(torch.randn(min(step, rows - lo), k, generator=gen, device=DEVICE) * 0.02, quant)
                      for lo in range(0, rows, step)])


def _prepare_linear(pkg, case, gen):
    k, n, r = case["in_features"], case["out_features"], case["rank"]
    weight = pkg.gguf.GGUFQuantizedTensor(_packed_rows(pkg, gen, n, k, case["quant"]), case["quant"], (n, k))
    layer = pkg.fast_lora.FastGGUFLoraLinear(pkg.fast_lora.GGUFLinear(k, n, weight), "default", r=r, lora_alpha=2 * r)
    with torch.no_grad():
        layer.lora_A["default"].weight.copy_(_bf16(gen, r, k, std=k ** -0.5))
        layer.lora_B["default"].weight.copy_(_bf16(gen, n, r, std=0.01))
    state = dict(layer=layer, x=_bf16(gen, case["tokens"], k))
    if case["kind"] == "linear_step":
        state["x"].requires_grad_(True)
        state["dy"] = _bf16(gen, case["tokens"], n)
    return state


def _prepare_experts(pkg, case, gen):
    e, h, i, r, tokens = case["experts"], case["hidden"], case["inter"], case["rank"], case["tokens"]

    def planes(n, k, quant):
        rows = _packed_rows(pkg, gen, e * n, k, quant)
        return pkg.gguf.GGUFQuantizedTensor(rows.reshape(e, n, -1), quant, (e, n, k))

    experts = pkg.fast_moe_lora.GGUFExperts(planes(i, h, case["quant"]), planes(i, h, case["quant"]), planes(h, i, case["down_quant"]))
    layer = pkg.fast_moe_lora.FastGGUFMoeLora(experts, r=r, lora_alpha=2 * r)
    with torch.no_grad():
        layer.lora_A["default"].weight.copy_(_bf16(gen, e, r, h, std=h ** -0.5))
        layer.lora_B["default"].weight.copy_(_bf16(gen, e, 2 * i, r, std=0.01))
        layer.lora_A_down["default"].weight.copy_(_bf16(gen, e, r, i, std=i ** -0.5))
        layer.lora_B_down["default"].weight.copy_(_bf16(gen, e, h, r, std=0.01))
    state = dict(layer=layer, x=_bf16(gen, tokens, h), top_k=case["top_k"])
    if case["kind"] == "experts_forward":
        state["router"] = _bf16(gen, e, h, std=h ** -0.5)
    else:
        top = torch.topk(torch.randn(tokens, e, generator=gen, device=DEVICE), case["top_k"], dim=-1)
        state["ids"] = top.indices
        state["weights"] = torch.softmax(top.values, dim=-1).requires_grad_(True)
        state["x"].requires_grad_(True)
        state["dy"] = _bf16(gen, tokens, h)
    return state


def _prepare_head(pkg, case, gen):
    h, v = case["hidden"], case["vocab"]
    payload = _packed_rows(pkg, gen, v, h, case["quant"])
    state = dict(x=_bf16(gen, case["tokens"], h))
    if case["kind"] == "head_forward":
        state["layer"] = pkg.fast_lora.GGUFLinear(h, v, pkg.gguf.GGUFQuantizedTensor(payload, case["quant"], (v, h)))
    else:
        labels = torch.randint(0, v, (case["tokens"],), generator=gen, device=DEVICE)
        labels[torch.rand(case["tokens"], generator=gen, device=DEVICE) < 0.05] = -100  # padding and prompt positions
        state.update(payload=payload, labels=labels, quant=case["quant"], vocab=v, chunk=case["chunk"])
        state["x"].requires_grad_(True)
    return state


def prepare(case, seed):
    pkg = _package()
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    maker = {"linear": _prepare_linear, "experts": _prepare_experts, "head": _prepare_head, "loss": _prepare_head}[case["kind"].split("_")[0]]
    return dict(maker(pkg, case, gen), kind=case["kind"])


# ------------------------------------------------------------------------------------------------
# one pass
def run(state):
    pkg = _package()
    kind, x = state["kind"], state["x"]
    if kind in ("linear_forward", "head_forward"):
        with torch.no_grad():
            return state["layer"](x)
    if kind == "experts_forward":
        with torch.no_grad():
            _, scores, ids = pkg.fast_moe_ranking.qwen_router_forward(state["router"], x, state["top_k"])
            return state["layer"](x, ids, scores)
    x.grad = None
    if kind == "loss_step":
        loss = pkg.gguf_liger_loss.packed_linear_cross_entropy(x, state["payload"], state["labels"], state["quant"], state["vocab"], state["chunk"])
        loss.backward()
        return dict(loss=loss.detach(), d_hidden=x.grad)
    layer, out = state["layer"], {}
    layer.zero_grad(set_to_none=True)
    if kind == "linear_step":
        y = layer(x)
    else:
        state["weights"].grad = None
        y = layer(x, state["ids"], state["weights"])
    y.backward(state["dy"])
    if kind == "experts_step":
        out["d_weights"] = state["weights"].grad
    out.update(y=y.detach(), d_hidden=x.grad)
    out.update({"d_" + name: p.grad for name, p in layer.named_parameters() if p.grad is not None})
    return out


# ------------------------------------------------------------------------------------------------
def _packed_bytes(n, k, quant):
    elems, nbytes = BLOCKS[quant]
    return n * (k // elems) * nbytes


def work(case):
    kind, t = case["kind"], case["tokens"]
    step = kind.endswith("_step")
    if kind.startswith("linear"):
        k, n, r = case["in_features"], case["out_features"], case["rank"]
        factors = 2 * r * (n + k)
        flops = 2 * t * n * k + 2 * t * r * (n + k)
        nbytes = _packed_bytes(n, k, case["quant"]) + factors + 2 * t * (k + n)
        if step:  # dX like the forward, dA and dB; reads dY and the factors, writes dX, dA, dB
            flops += 2 * t * n * k + 4 * t * r * (n + k)
            nbytes += 2 * t * (k + n) + factors
        return {"bytes": nbytes, "flops": flops}
    if kind.startswith("experts"):
        h, i, e, r, routes = case["hidden"], case["inter"], case["experts"], case["rank"], t * case["top_k"]
        active = e * (1 - (1 - case["top_k"] / e) ** t)  # experts that some token chose, in the mean
        plane = 2 * _packed_bytes(i, h, case["quant"]) + _packed_bytes(h, i, case["down_quant"])
        factors = 2 * r * ((h + 2 * i) + (i + h))
        gemm, lora = 2 * routes * 3 * h * i, 2 * routes * r * ((h + 2 * i) + (i + h))
        if step:  # (ids int64 and weights fp32 in, their gradient out; every expert's factor gradients are written)
            return {"bytes": active * (plane + factors) + e * factors + 2 * t * h * 4 + routes * 16, "flops": 2 * gemm + 3 * lora}
        return {"bytes": active * (plane + factors) + 2 * t * h * 2 + 2 * e * h, "flops": gemm + lora + 2 * t * e * h}
    h, v = case["hidden"], case["vocab"]
    weight = _packed_bytes(v, h, case["quant"])
    if step:
        return {"bytes": weight + 2 * t * h * 2 + 8 * t, "flops": 2 * 2 * t * v * h}
    return {"bytes": weight + 2 * t * (h + v), "flops": 2 * t * v * h}


def tolerance(case):
    # bf16 results of fp32 sums, with bf16 intermediates (x A^T, the expert activations, the logits) between
    return {"rel": 1e-2}
