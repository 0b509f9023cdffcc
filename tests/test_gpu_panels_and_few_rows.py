"""The dense launches over decoded panels, the products of a few rows, and the layers' native host calls, at the sizes
where they can go wrong: tile edges, split contractions, ragged rows and columns, the ends of each range."""

import contextlib
import ctypes

import numpy as np
import pytest
import torch

from helpers import ALL_TYPES, TYPE_NAMES, assert_close_bf16, bf16_randn, make_payload
from oracle import gguf_blocks as gb
from oracle import lora_matmul as ref
from oracle import routing as rref

pytestmark = pytest.mark.gpu


def _lora_case(seed, m, n, k, r, qt):
    gen = torch.Generator().manual_seed(seed)
    payload = make_payload(seed, qt, n, k, "random")
    return payload, bf16_randn(gen, m, k), bf16_randn(gen, r, k, std=k ** -0.5), bf16_randn(gen, n, r, std=0.02), bf16_randn(gen, m, n)


def _check_lora(pkg, dev, payload, qt, x, a, b, s, dy):
    """Against fp32 products on the device of the oracle's decoded weights (bf16 values: their products are exact in fp32)."""
    w, n = ref.weights_bf16(payload, qt).to(dev).float(), b.shape[0]
    xd, ad, bd = (t.to(dev).requires_grad_(True) for t in (x, a, b))
    y = pkg.fast_lora.lora_mmq(xd, torch.from_numpy(payload).to(dev), qt, n, ad, bd, s)
    y.backward(dy.to(dev))
    xf, af, bf, df = (t.to(dev).float() for t in (x, a, b, dy))
    xa, dyb = (xf @ af.T).bfloat16().float(), (df @ bf).bfloat16().float()
    assert_close_bf16(y, xf @ w.T + s * xa @ bf.T, "Y")
    assert_close_bf16(xd.grad, df @ w + s * dyb @ af, "dX")
    assert_close_bf16(ad.grad, s * dyb.T @ xf, "dA")
    assert_close_bf16(bd.grad, s * df.T @ xa, "dB")


@pytest.mark.parametrize("m,n,k,r", [
    (48, 64, 256, 16),      # the fewest rows
    (49, 65, 512, 5),       # one row and one column past a tile; a rank that is no multiple of eight; columns that no split takes
    (63, 511, 4096, 32),    # the widest rank of the shared launch
    (64, 512, 8192, 16),    # sixteen contraction splits
    (257, 520, 2048, 33),   # a rank of the separate launches
    (1500, 2052, 1024, 8),  # 128 x 128 tiles forward
    (3001, 5001, 256, 16),  # 256 x 256 tiles, ragged both ways; the shortest contraction
    (4096, 1028, 2048, 4),
    (1999, 4097, 2048, 16),  # ragged both ways
    (4003, 4100, 2048, 24),  # 128 x 256 tiles in the grad-input; a contraction that ends inside a step
])
@pytest.mark.parametrize("qt", [gb.Q8_0, gb.Q4_K, gb.IQ2_XXS], ids=lambda q: TYPE_NAMES[q])
def test_dense_lora_over_panels(pkg, dev, qt, m, n, k, r):
    payload, x, a, b, dy = _lora_case(7000 + m + n, m, n, k, r, qt)
    _check_lora(pkg, dev, payload, qt, x, a, b, 32.0 / r, dy)


@pytest.mark.parametrize("m,n,k,r", [
    (49, 72, 256, 8),       # fewer spans of 128 than waves, the only one partial; half of the padded rank
    (65, 136, 512, 12),     # a rank that is no multiple of eight; a second span of eight elements
    (130, 1544, 1792, 16),  # spans beyond the ones in flight: twelve whole and a partial one over four waves
    (100, 1096, 3072, 24),  # the same with two blocks of ranks, the second one half full
    (64, 2048, 3328, 32),
    # ranks whose rows of B are no whole pieces
    (50, 8, 256, 1),        # one piece in all
    (49, 1672, 256, 4),     # the spans in flight once over and a partial one of eight elements
    (97, 1416, 512, 7),     # rows at odd elements
    (65, 1544, 512, 20),    # two blocks of ranks
    (100, 1096, 512, 31),
])
def test_rank_sized_products_beside_the_decoding_pass(pkg, dev, m, n, k, r):
    payload, x, a, b, dy = _lora_case(7100 + n + k, m, n, k, r, gb.Q8_0)
    _check_lora(pkg, dev, payload, gb.Q8_0, x, a, b, 32.0 / r, dy)


@pytest.mark.parametrize("n,splits", [(1301, 1), (1304, 1), (1304, 3), (1304, 4)])  # an odd column count; forward splits of 7, 7, 6 steps, grad-input of 6, 6, 6, 3
@pytest.mark.parametrize("shape,rows", [(0, 517), (1, 515), (2, 131), (3, 389)])
def test_every_panel_tile_at_ragged_sizes(pkg, dev, shape, rows, n, splits):
    lib, k, qt = pkg._lib.load(), 1280, gb.Q4_K
    payload, x, a, b, dy = _lora_case(shape + n, rows, n, k, 24, qt)
    try:
        pkg._lib.check(lib.ggq_debug_force_dense_tile(shape, splits))
        got = [ctypes.c_int(), ctypes.c_int()]
        pkg._lib.check(lib.ggq_debug_dense_plan(0, rows, n, k, 1 << 40, *map(ctypes.byref, got)))
        assert [v.value for v in got] == [shape, splits if n % 4 == 0 else 1]
        _check_lora(pkg, dev, payload, qt, x, a, b, 1.5, dy)
    finally:
        pkg._lib.check(lib.ggq_debug_force_dense_tile(-1, 0))


def test_a_workspace_without_room_for_panels_keeps_the_tile_kernel(pkg, dev):
    # through the C ABI: what the calls needed before there were panels is still enough
    qt, m, n, k, r, s = gb.Q4_K, 100, 320, 512, 16, 2.0
    payload, x, a, b, dy = _lora_case(17, m, n, k, r, qt)
    w = ref.weights_bf16(payload, qt).to(dev).float()
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    p, xd, ad, bd, gd = (t.to(dev) for t in (torch.from_numpy(payload), x, a, b, dy))
    y, xa, dx, da, db = (torch.empty(*shape, dtype=torch.bfloat16, device=dev) for shape in ((m, n), (m, r), (m, k), (r, k), (n, r)))
    small = 8192 + m * r * 2
    assert small < lib.ggq_lora_workspace_bytes(m, 0, 1, n, k, 0)
    ws = torch.empty(small, dtype=torch.uint8, device=dev)
    xf, af, bf, df = (t.float() for t in (xd, ad, bd, gd))
    pkg._lib.check(lib.ggq_lora_mmq_forward(xd.data_ptr(), p.data_ptr(), qt, m, n, k, None, None, 0, 0.0, None, y.data_ptr(), ws.data_ptr(), 256, stream))
    assert_close_bf16(y, xf @ w.T, "plain Y")
    pkg._lib.check(lib.ggq_lora_mmq_forward(xd.data_ptr(), p.data_ptr(), qt, m, n, k, ad.data_ptr(), bd.data_ptr(), r, s, xa.data_ptr(), y.data_ptr(), ws.data_ptr(), 256, stream))
    assert_close_bf16(y, xf @ w.T + s * xa.float() @ bf.T, "Y")
    pkg._lib.check(lib.ggq_lora_mmq_backward(gd.data_ptr(), p.data_ptr(), qt, m, n, k, xd.data_ptr(), xa.data_ptr(), ad.data_ptr(), bd.data_ptr(), r, s, dx.data_ptr(),
                                             da.data_ptr(), db.data_ptr(), ws.data_ptr(), small, stream))
    dyb = (df @ bf).bfloat16().float()
    assert_close_bf16(dx, df @ w + s * dyb @ af, "dX")
    assert_close_bf16(da, s * dyb.T @ xf, "dA")
    assert_close_bf16(db, s * df.T @ xa.float(), "dB")
    with pytest.raises(RuntimeError, match="workspace too small"):
        pkg._lib.check(lib.ggq_lora_mmq_backward(gd.data_ptr(), p.data_ptr(), qt, m, n, k, xd.data_ptr(), xa.data_ptr(), ad.data_ptr(), bd.data_ptr(), r, s, dx.data_ptr(),
                                                 da.data_ptr(), db.data_ptr(), ws.data_ptr(), 256, stream))


def test_dense_matrix_in_slabs(pkg, dev):
    # more than 128 MB of decoded weights: forward in slabs of output columns (70000 x 1024 x 2 bytes)
    qt, m, n, k = gb.Q8_0, 50, 70001, 1024
    payload, x, *_ = _lora_case(88, m, n, k, 4, qt)
    y = pkg.fast_lora.mmq(x.to(dev), torch.from_numpy(payload).to(dev), qt, n)
    assert_close_bf16(y, x.to(dev).float() @ ref.weights_bf16(payload, qt).to(dev).float().T, "Y")


def test_dense_lora_in_slabs(pkg, dev):
    # both directions: 65536 of 70008 output columns forward, 768 of 1024 backward (decoded from a column offset); the LoRA
    # factors follow the slab, the rank-sized products ride in the first one's pass
    qt = gb.Q8_0
    payload, x, a, b, dy = _lora_case(89, 50, 70008, 1024, 16, qt)
    _check_lora(pkg, dev, payload, qt, x, a, b, 2.0, dy)


@pytest.mark.parametrize("m,k", [(33, 2560), (47, 2560), (17, 4352), (47, 4352), (1, 8448), (47, 8448)])
@pytest.mark.parametrize("qt", [gb.Q8_0, gb.Q4_K], ids=lambda q: TYPE_NAMES[q])
def test_rows_between_the_few_row_kernel_and_the_panels(pkg, dev, qt, m, k):
    payload, x, a, b, dy = _lora_case(m + k, m, 100, k, 8, qt)
    _check_lora(pkg, dev, payload, qt, x, a, b, 2.0, dy)


@pytest.mark.parametrize("m,n,k,r", [
    (1, 1, 256, 1), (1, 4099, 2048, 16), (16, 17, 512, 64), (17, 48, 2048, 24), (64, 5000, 2048, 8),  # two LDS buffers from 4097 columns
    (32, 100, 4096, 40), (16, 33, 8192, 16), (47, 31, 1024, 5),
])
@pytest.mark.parametrize("qt", ALL_TYPES, ids=[TYPE_NAMES[q] for q in ALL_TYPES])
def test_few_rows(pkg, dev, qt, m, n, k, r):
    payload, x, a, b, _ = _lora_case(9000 + m + n, m, n, k, r, qt)
    w = ref.weights_bf16(payload, qt).to(dev).float()
    p, xf, s = torch.from_numpy(payload).to(dev), x.to(dev).float(), 2.0
    y = pkg.fast_lora.lora_mmq(x.to(dev), p, qt, n, a.to(dev), b.to(dev), s)
    xa = (xf @ a.to(dev).float().T).bfloat16().float()
    assert_close_bf16(y, xf @ w.T + s * xa @ b.to(dev).float().T, "Y with LoRA")
    assert_close_bf16(pkg.fast_lora.mmq(x.to(dev), p, qt, n), xf @ w.T, "Y")


@pytest.mark.parametrize("k", [64, 192, 320])
def test_few_rows_of_a_contraction_that_ends_inside_a_span(pkg, dev, k):
    # 128-element spans; only the 32-element block format has such lengths
    payload, x, *_ = _lora_case(k, 5, 70, k, 4, gb.Q8_0)
    y = pkg.fast_lora.mmq(x.to(dev), torch.from_numpy(payload).to(dev), gb.Q8_0, 70)
    assert_close_bf16(y, x.to(dev).float() @ ref.weights_bf16(payload, gb.Q8_0).to(dev).float().T, "Y")


def test_a_broken_block_at_the_end_of_a_contraction_stays_in_its_row(pkg, dev):
    # k = 192 ends inside a span: the lanes past it read the last block again, against zeros.  An infinite scale there makes its
    # own row NaN, as the decoded weights themselves are, and no other
    payload, x, *_ = _lora_case(3, 5, 70, 192, 4, gb.Q8_0)
    payload[33, -34:-32] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    y = pkg.fast_lora.mmq(x.to(dev), torch.from_numpy(payload).to(dev), gb.Q8_0, 70)
    others = torch.arange(70) != 33
    assert not torch.isfinite(y[:, 33]).any()
    assert_close_bf16(y[:, others.to(dev)], x.float() @ ref.weights_bf16(payload, gb.Q8_0)[others].float().T, "the other rows")


def _expert_layer(pkg, dev, qt, qt_down, experts, hidden, inter, r, limit=None, seed=0):
    gen = torch.Generator().manual_seed(4000 + seed)
    planes = [np.stack([make_payload(seed + 31 * i + e, q, n, k, "random") for e in range(experts)])
              for i, (q, n, k) in enumerate([(qt, inter, hidden), (qt, inter, hidden), (qt_down, hidden, inter)])]
    packed = [pkg.gguf.GGUFQuantizedTensor(torch.from_numpy(p).to(dev), q, (experts, n, k))
              for p, (q, n, k) in zip(planes, [(qt, inter, hidden), (qt, inter, hidden), (qt_down, hidden, inter)])]
    base = pkg.fast_moe_lora.GGUFExperts(*packed)
    if limit:
        base.swiglu_limit = limit
    layer = pkg.fast_moe_lora.FastGGUFMoeLora(base, r=r, lora_alpha=2 * r)
    factors = {"lora_A": (experts, r, hidden), "lora_B": (experts, 2 * inter, r), "lora_A_down": (experts, r, inter), "lora_B_down": (experts, hidden, r)}
    with torch.no_grad():
        for name, shape in factors.items():
            getattr(layer, name)["default"].weight.copy_(bf16_randn(gen, *shape, std=0.02).to(dev))
    return layer, [ref.weights_bf16(p, q) for p, q in zip(planes, (qt, qt, qt_down))], gen


@pytest.mark.parametrize("tokens,top_k,hidden,inter,r,limit,ids", [
    (1, 8, 2048, 512, 16, None, torch.int64), (8, 8, 256, 256, 5, 0.25, torch.int32),   # 64 routes: past every limit of the path without a plan
    (4, 16, 512, 768, 64, None, torch.int64), (2, 16, 256, 512, 40, None, torch.int64), (3, 1, 4096, 256, 24, None, torch.int32),
    (1, 2, 256, 3584, 24, None, torch.int64),  # Q2_K, Q3_K: sixteen packed rows per wave leave no LDS for x
    (1, 8, 4096, 512, 16, None, torch.int64),  # more than 2048 elements of x: Q2_K, Q3_K two column sets per workgroup, the others one
    (1, 4, 3072, 1024, 40, None, torch.int64),  # and IQ2_XXS two, a rank padded to 48
])
@pytest.mark.parametrize("qt", ALL_TYPES, ids=[TYPE_NAMES[q] for q in ALL_TYPES])
def test_experts_of_a_few_routes(pkg, dev, qt, tokens, top_k, hidden, inter, r, limit, ids):
    experts = max(top_k, 4)
    layer, (wg, wu, wd), gen = _expert_layer(pkg, dev, qt, qt, experts, hidden, inter, r, limit)
    x = bf16_randn(gen, tokens, hidden)
    top = torch.stack([torch.randperm(experts, generator=gen)[:top_k] for _ in range(tokens)])
    weights = torch.softmax(torch.randn(tokens, top_k, generator=gen), -1)
    with torch.no_grad():
        got = layer(x.to(dev), top.to(dev, ids), weights.to(dev))
    _, perm, inv = rref.plan(top)
    active, offsets = rref.active_offsets(rref.expert_counts(top, experts))
    factors = [getattr(layer, name)["default"].weight.detach().cpu() for name in ("lora_A", "lora_B", "lora_A_down", "lora_B_down")]
    rows = ref.expert_layer(rref.gather_forward(x, perm, top_k), active, offsets, wg, wu, wd, *factors, 2.0, limit=limit)["out"]
    want = rref.combine_forward(ref.bf16_round(rows).to(torch.bfloat16), weights, inv)
    # bf16 roundings that a sum in another order may land on the other side of: x A^T, gate and up, the activation, a route's row
    assert_close_bf16(got, want, "experts", ulps=4)


@pytest.mark.parametrize("tokens,experts,hidden", [(1, 4, 8), (1, 256, 2048), (8, 100, 1000), (5, 8, 136)])
def test_router_logits_of_a_few_tokens(pkg, dev, tokens, experts, hidden):
    gen = torch.Generator().manual_seed(tokens + experts)
    x, w = bf16_randn(gen, tokens, hidden), bf16_randn(gen, experts, hidden, std=hidden ** -0.5)
    with torch.no_grad():
        logits, scores, ids = pkg.fast_moe_ranking.qwen_router_forward(w.to(dev), x.to(dev), 4)
    assert_close_bf16(logits, x.double() @ w.double().T, "logits")
    want, order = torch.sort(logits.float().cpu(), dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu(), order[:, :4])
    assert_close_bf16(scores, torch.softmax(want[:, :4].double(), -1), "scores")


# ------------------------------------------------------------------------------------------------
# What stands around a call: saved-tensor hooks, module hooks, tracing, forward mode.
def _small_linear(pkg, dev):
    payload, x, a, b, dy = _lora_case(5, 64, 96, 256, 8, gb.Q4_K)
    return torch.from_numpy(payload).to(dev), *(t.to(dev) for t in (x, a, b, dy))


def test_saved_tensor_hooks_reach_the_native_nodes(pkg, dev):
    p, x, a, b, dy = _small_linear(pkg, dev)

    def grads(hooks):
        xs = [t.clone().requires_grad_(True) for t in (x, a, b)]
        with hooks:
            y = pkg.fast_lora.lora_mmq(xs[0], p, gb.Q4_K, 96, xs[1], xs[2], 2.0)
        y.backward(dy)
        return [t.grad for t in xs]

    for got, want in zip(grads(torch.autograd.graph.save_on_cpu()), grads(contextlib.nullcontext())):
        assert torch.equal(got, want)


def test_module_hooks_of_the_expert_base_layer_run(pkg, dev):
    layer, _, gen = _expert_layer(pkg, dev, gb.Q4_K, gb.Q4_K, 4, 256, 256, 8)
    seen = []
    layer.base_layer.register_forward_hook(lambda module, args, out: seen.append(tuple(out.shape)))
    with torch.no_grad():
        layer(bf16_randn(gen, 3, 256).to(dev), torch.tensor([[0, 1], [2, 3], [1, 0]], device=dev), torch.full((3, 2), 0.5, device=dev))
    assert seen == [(3, 256)]


def test_two_dimensional_hidden_states_of_another_width_are_regrouped(pkg, dev):
    # [T, n * hidden] is n T tokens, as any other shape is
    layer, _, gen = _expert_layer(pkg, dev, gb.Q4_K, gb.Q4_K, 4, 256, 256, 8)
    x, router = bf16_randn(gen, 6, 256).to(dev), bf16_randn(gen, 8, 256).to(dev)
    ids, weights = torch.tensor([[0, 3]], device=dev).repeat(6, 1), torch.full((6, 2), 0.5, device=dev)
    with torch.no_grad():
        assert torch.equal(layer(x.reshape(3, 512), ids, weights), layer(x, ids, weights).reshape(3, 512))
        for got, want in zip(pkg.fast_moe_ranking.qwen_router_forward(router, x.reshape(3, 512), 2), pkg.fast_moe_ranking.qwen_router_forward(router, x, 2)):
            assert torch.equal(got, want)


def test_function_transforms_are_refused(pkg, dev):
    p, x, a, b, _ = _small_linear(pkg, dev)
    layer, _, gen = _expert_layer(pkg, dev, gb.Q4_K, gb.Q4_K, 4, 256, 256, 8)
    ids, weights = torch.tensor([[0, 3]], device=dev).repeat(3, 1), torch.full((3, 2), 0.5, device=dev)
    tokens = bf16_randn(gen, 3, 256).to(dev)
    three = torch.ones(3, device=dev)
    for call, operand in ((lambda t: pkg.fast_lora.lora_mmq(t, p, gb.Q4_K, 96, a, b, 2.0), x), (lambda t: layer(t, ids, weights), tokens)):
        for transformed in (lambda: torch.func.vmap(call)(operand.expand(2, *operand.shape)),
                            lambda: torch.func.grad(lambda t: call(t).float().sum())(operand),
                            # an operand that the transform does not wrap
                            lambda: torch.func.vmap(lambda s: call(operand).float().sum() * s)(three),
                            lambda: torch.func.grad(lambda s: (call(operand).float() * s).sum())(three[0])):
            with pytest.raises(RuntimeError):
                transformed()


@pytest.mark.parametrize("limit", [0.0, -1.0, float("nan")])
@pytest.mark.parametrize("tokens,needs_grad", [(2, False), (2, True), (40, False)])  # (the path without a plan, and with one)
def test_a_clamp_that_is_not_positive_is_refused(pkg, dev, tokens, needs_grad, limit):
    layer, _, gen = _expert_layer(pkg, dev, gb.Q4_K, gb.Q4_K, 4, 256, 256, 8)
    layer.base_layer.swiglu_limit = limit
    x = bf16_randn(gen, tokens, 256).to(dev).requires_grad_(needs_grad)
    ids, weights = torch.tensor([[0, 3]], device=dev).repeat(tokens, 1), torch.full((tokens, 2), 0.5, device=dev)
    with torch.set_grad_enabled(needs_grad), pytest.raises(ValueError, match="limit must be positive"):
        layer(x, ids, weights)


def test_a_traced_linear_computes_on_its_inputs(pkg, dev):
    p, x, a, b, _ = _small_linear(pkg, dev)

    def call(inp):
        return pkg.fast_lora.lora_mmq(inp, p, gb.Q4_K, 96, a, b, 2.0)

    with torch.no_grad():
        traced = torch.jit.trace(call, (x,), check_trace=False)
        other = x.flip(0).contiguous()
        assert torch.equal(traced(other), call(other)), "the trace holds the first call's result"


def test_forward_mode_is_refused(pkg, dev):
    import torch.autograd.forward_ad as fwad

    p, x, a, b, _ = _small_linear(pkg, dev)
    with fwad.dual_level(), torch.no_grad():
        dual = fwad.make_dual(x, torch.ones_like(x))
        with pytest.raises((RuntimeError, NotImplementedError)):
            pkg.fast_lora.lora_mmq(dual, p, gb.Q4_K, 96, a, b, 2.0)


# ------------------------------------------------------------------------------------------------
# Expert-sorted rows while an expert has a few: row tiles of sixteen, one to eight waves per contraction.
@pytest.mark.parametrize("n,k,r", [(40, 256, 5), (64, 512, 16), (264, 768, 40), (48, 2048, 16), (24, 4096, 64)])
@pytest.mark.parametrize("qt", ALL_TYPES, ids=[TYPE_NAMES[q] for q in ALL_TYPES])
def test_grouped_forward_of_a_few_rows_per_expert(pkg, dev, qt, n, k, r):
    sizes = [1, 0, 16, 17, 0, 40, 3, 0, 15, 2, 33, 0] if qt != gb.Q4_K else [1, 0, 0, 17, 0, 0, 3, 0] + [0] * 40
    experts, offsets = torch.arange(len(sizes)), torch.tensor(np.cumsum(sizes), dtype=torch.int32)
    rows, s = sum(sizes), 2.0
    gen = torch.Generator().manual_seed(n + k)
    planes = [np.stack([make_payload(seed + e % 12, qt, n, k, "random") for e in range(len(sizes))]) for seed in (300, 400)]
    x, a = bf16_randn(gen, rows, k), bf16_randn(gen, len(sizes), r, k, std=k ** -0.5)
    b = bf16_randn(gen, len(sizes), 2 * n, r, std=0.02)
    args = experts.to(dev), offsets.to(dev), qt, n
    with torch.no_grad():
        gate, up = pkg.fast_moe_lora.grouped_lora_mmq_pair(x.to(dev), *(torch.from_numpy(p).to(dev) for p in planes), *args, a.to(dev), b.to(dev), s)
        single = pkg.fast_moe_lora.grouped_mmq(x.to(dev), torch.from_numpy(planes[1]).to(dev), *args)
    w = [ref.weights_bf16(p, qt) for p in planes]
    want = ref.grouped_lora_linear(x, torch.cat(w, dim=1), experts, offsets, a, b, s)["y"]
    assert_close_bf16(gate, want[:, :n], "gate")
    assert_close_bf16(up, want[:, n:], "up")
    assert_close_bf16(single, ref.grouped_lora_linear(x, w[1], experts, offsets)["y"], "single")


@pytest.mark.parametrize("ids_type", [torch.int64, torch.int32])
@pytest.mark.parametrize("tokens,top_k,experts", [(1, 1, 1), (1, 8, 256), (128, 8, 256), (515, 8, 250), (997, 3, 1024), (1536, 8, 256), (1537, 8, 60)])
def test_plan_and_tables_in_one_launch(pkg, dev, tokens, top_k, experts, ids_type):
    # one chunk, several, the most that one launch takes (12 of 1024 routes), and one more (separate launches)
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator().manual_seed(tokens)
    ids = (torch.rand(tokens, top_k, generator=gen) ** 2 * experts).long().clamp_(max=experts - 1)  # (uneven groups)
    d_ids, routes = ids.to(dev, ids_type), tokens * top_k
    i64 = [torch.empty(n, dtype=torch.int64, device=dev) for n in (routes, routes, routes, experts)]
    i32 = [torch.empty(n, dtype=torch.int32, device=dev) for n in (experts, experts, experts, 2)]
    tables = [torch.zeros(lib.ggq_group_tables_bytes(routes, experts, experts), dtype=torch.uint8, device=dev) for _ in range(2)]
    ws = torch.empty(lib.ggq_route_plan_workspace_bytes(tokens, top_k, experts), dtype=torch.uint8, device=dev)
    sorted_ids, perm, inv, active = i64
    counts, ends, active_ends, status = i32
    pkg._lib.check(lib.ggq_route_plan_with_tables(d_ids.data_ptr(), ids_type == torch.int64, tokens, top_k, experts, sorted_ids.data_ptr(), perm.data_ptr(), inv.data_ptr(),
                                                  counts.data_ptr(), ends.data_ptr(), active.data_ptr(), active_ends.data_ptr(), status.data_ptr(), tables[0].data_ptr(),
                                                  tables[0].numel(), ws.data_ptr(), ws.numel(), stream))
    pkg._lib.check(lib.ggq_group_tables_build(torch.arange(experts, device=dev).data_ptr(), ends.data_ptr(), experts, experts, routes, tables[1].data_ptr(), tables[1].numel(), stream))
    for got, want in zip((sorted_ids, perm, inv), rref.plan(ids)):
        assert torch.equal(got.cpu(), want)
    want_counts = rref.expert_counts(ids, experts)
    assert torch.equal(counts.cpu(), want_counts) and torch.equal(ends.cpu(), torch.cumsum(want_counts.long(), 0).int())
    want_active, want_ends = rref.active_offsets(want_counts)
    assert status.tolist() == [want_active.numel(), 0]
    assert torch.equal(active[:want_active.numel()].cpu(), want_active) and torch.equal(active_ends[:want_active.numel()].cpu(), want_ends)
    assert torch.equal(*tables)


@pytest.mark.parametrize("tokens,top_k,experts,chosen", [(1536, 8, 256, 255), (1500, 8, 256, 0), (130, 8, 8, 3)])
def test_plan_of_routes_that_all_go_to_one_expert(pkg, dev, tokens, top_k, experts, chosen):
    # every count of the one launch lands on one LDS word, every lane of a wave holds the same id
    lib, stream, routes = pkg._lib.load(), torch.cuda.current_stream().cuda_stream, tokens * top_k
    ids = torch.full((tokens, top_k), chosen, dtype=torch.int64, device=dev)
    sorted_ids, perm, inv, active = (torch.empty(n, dtype=torch.int64, device=dev) for n in (routes, routes, routes, experts))
    counts, ends, active_ends, status = (torch.empty(n, dtype=torch.int32, device=dev) for n in (experts, experts, experts, 2))
    tables = [torch.zeros(lib.ggq_group_tables_bytes(routes, experts, experts), dtype=torch.uint8, device=dev) for _ in range(2)]
    ws = torch.empty(lib.ggq_route_plan_workspace_bytes(tokens, top_k, experts), dtype=torch.uint8, device=dev)
    pkg._lib.check(lib.ggq_route_plan_with_tables(ids.data_ptr(), 1, tokens, top_k, experts, sorted_ids.data_ptr(), perm.data_ptr(), inv.data_ptr(), counts.data_ptr(),
                                                  ends.data_ptr(), active.data_ptr(), active_ends.data_ptr(), status.data_ptr(), tables[0].data_ptr(), tables[0].numel(),
                                                  ws.data_ptr(), ws.numel(), stream))
    pkg._lib.check(lib.ggq_group_tables_build(torch.arange(experts, device=dev).data_ptr(), ends.data_ptr(), experts, experts, routes, tables[1].data_ptr(), tables[1].numel(), stream))
    every = torch.arange(routes, device=dev)
    assert torch.equal(perm, every) and torch.equal(inv, every) and bool((sorted_ids == chosen).all())
    assert counts.tolist() == [routes if e == chosen else 0 for e in range(experts)]
    assert ends.tolist() == [routes if e >= chosen else 0 for e in range(experts)]
    assert status.tolist() == [1, 0] and active[0] == chosen and active_ends[0] == routes
    assert torch.equal(*tables)


# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("rows", [1, 17, 64, 100])  # (few rows, and panels)
@pytest.mark.parametrize("qt,n_group,k", [(gb.Q8_0, 33, 64), (gb.Q8_0, 21, 320), (gb.Q6_K, 33, 256), (gb.Q6_K, 20, 256), (gb.IQ2_XXS, 7, 256), (gb.Q2_K, 5, 256), (gb.Q3_K, 13, 256)],
                         ids=lambda v: TYPE_NAMES.get(v, str(v)))
def test_fixed_groups_whose_packed_rows_start_anywhere(pkg, dev, qt, n_group, k, rows):
    # group g's rows start g * n_group * row_bytes into the payload: only a multiple of the block format's own alignment
    groups = 3
    payload = np.stack([make_payload(60 + g, qt, n_group, k, "random") for g in range(groups)])
    assert payload[0].size % 16
    gen = torch.Generator().manual_seed(n_group)
    x, dy = bf16_randn(gen, rows, groups, k), bf16_randn(gen, rows, groups, n_group)
    xd = x.to(dev).requires_grad_(True)
    y = pkg.fast_lora.fixed_grouped_mmq(xd, torch.from_numpy(payload).to(dev), qt)
    y.backward(dy.to(dev))
    w = ref.weights_bf16(payload, qt).float()
    assert_close_bf16(y, torch.einsum("rgk,gnk->rgn", x.float(), w), "Y")
    assert_close_bf16(xd.grad, torch.einsum("rgn,gnk->rgk", dy.float(), w), "dX")
    for g in range(groups):  # the same bits as the dense calls on copies of their own
        xg = x[:, g].contiguous().to(dev).requires_grad_(True)
        yg = pkg.fast_lora.mmq(xg, torch.from_numpy(payload[g]).to(dev), qt, n_group)
        yg.backward(dy[:, g].contiguous().to(dev))
        assert torch.equal(y[:, g], yg) and torch.equal(xd.grad[:, g], xg.grad)
