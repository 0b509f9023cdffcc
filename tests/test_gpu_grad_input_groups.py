"""Grad-input of expert groups of very different sizes in one call, on the kernels for groups of a few rows."""

import statistics

import pytest
import torch

from helpers import TYPE_NAMES, assert_close_bf16
from oracle import gguf_blocks as gb

pytestmark = pytest.mark.gpu

BLOCKS = {gb.Q4_K: 144, gb.IQ2_XXS: 66}


def _payload(dev, seed, qt, experts, n, k):
    """Arbitrary quants with block scales of about 1e-4 (and, for Q4_K, offsets of the same size), made on the device."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    blocks = torch.randint(0, 256, (experts * n * (k // 256), BLOCKS[qt]), dtype=torch.uint8, generator=gen, device=dev)
    scales = ((0.5 + torch.rand(blocks.shape[0], 2, generator=gen, device=dev)) * 1e-4).half().view(torch.uint8)
    fields = 4 if qt == gb.Q4_K else 2
    blocks[:, :fields] = scales[:, :fields]
    return blocks.reshape(experts, n, -1)


def _rows(dev, seed, rows, cols):
    return torch.randn(rows, cols, generator=torch.Generator(device=dev).manual_seed(seed), device=dev).bfloat16()


def _ends(dev, sizes):
    return torch.tensor(sizes, device=dev).cumsum(0).int()


def _microseconds(call, repeats=7, calls=10):
    times = []
    call()
    for _ in range(repeats):
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(calls):
            call()
        stop.record()
        stop.synchronize()
        times.append(start.elapsed_time(stop) * 1e3 / calls)
    return statistics.median(times)


@pytest.mark.parametrize("qt,n,k,even,skewed", [
    # one workgroup per compute unit in the even grouping; six groups of 192 rows must not each be one workgroup's chain of tiles
    (gb.Q4_K, 2048, 512, [5] * 256, [192] * 6 + [0, 1] * 64 + [0] * 122),
    (gb.Q4_K, 768, 1024, [16] * 256, [192] * 20 + [0, 2] * 64 + [0] * 108),
], ids=lambda v: TYPE_NAMES.get(v, str(v)) if isinstance(v, int) else f"max{max(v)}")
def test_skewed_groups_cost_little_more_than_even_ones(pkg, dev, qt, n, k, even, skewed):
    # measured 1.1 to 1.3 times the even grouping's time; with one workgroup per 192 rows it was 2.6 and 3.8 times
    assert len(even) == len(skewed) == 256 and abs(sum(even) - sum(skewed)) <= 0.05 * sum(even)
    w, ids = _payload(dev, 1, qt, 256, n, k), torch.arange(256, device=dev)
    times = []
    for sizes in (even, skewed):
        dy, ends = _rows(dev, 2, sum(sizes), n), _ends(dev, sizes)
        times.append(_microseconds(lambda: pkg.fast_moe_lora.grouped_mmq_grad_input(dy, w, ids, ends, qt, k)))
    assert times[1] <= 1.8 * times[0], f"even {times[0]:.1f} us, skewed {times[1]:.1f} us"


@pytest.mark.parametrize("sizes", [[96] * 42 + [0] * 214, [128] * 16 + [1] * 240], ids=["96_or_none", "128_or_1"])
def test_iq2xxs_groups_beyond_a_tile_cost_what_they_cost_on_the_tile_kernel(pkg, dev, sizes, force_grouped_shape):
    # measured (4096 rows of W) 1.03 and 0.8 times the tile kernel's time; with groups of more than 80 rows walked in two parts the first was 1.7 times
    qt, n, k = gb.IQ2_XXS, 2048, 2048
    w, ids = _payload(dev, 1, qt, 256, n, k), torch.arange(256, device=dev)
    dy, ends = _rows(dev, 2, sum(sizes), n), _ends(dev, sizes)
    times = []
    for shape in ("", "1"):
        force_grouped_shape(shape)
        times.append(_microseconds(lambda: pkg.fast_moe_lora.grouped_mmq_grad_input(dy, w, ids, ends, qt, k)))
    assert times[0] <= 1.3 * times[1], f"{times[0]:.1f} us, tile kernel {times[1]:.1f} us"


@pytest.mark.parametrize("rank", [0, 16, 32, 40, 64])
@pytest.mark.parametrize("sizes", [[49, 63, 64, 65, 0, 0, 0], [127, 128, 129, 1] + [0] * 7, [192, 193, 0, 48] + [0] * 12, [255, 0, 0, 0, 0, 0, 0, 16]])
def test_q4k_groups_beyond_a_tile_match_the_kernel_for_larger_groups(pkg, dev, sizes, rank):
    # the same rows with the empty groups left out average more rows than the rule takes: the eight-wave kernel, bit for bit
    qt, n, k, groups = gb.Q4_K, 256, 4096, 64
    ml = pkg.fast_moe_lora
    sizes = (sizes * groups)[:groups]
    active = [g for g, size in enumerate(sizes) if size]
    assert sum(sizes) <= 40 * groups and sum(sizes) > 40 * len(active)
    w = _payload(dev, 3, qt, groups, n, k)
    dy, x = _rows(dev, 4, sum(sizes), n), _rows(dev, 5, sum(sizes), k)
    a, b = _rows(dev, 6, groups * rank, k).view(groups, rank, k), _rows(dev, 7, groups * n, rank).view(groups, n, rank)
    got = []
    for ids in (list(range(groups)), active):
        e, o = torch.tensor(ids, device=dev), _ends(dev, [sizes[g] for g in ids])
        if rank:
            xd = x.clone().requires_grad_(True)
            ml.grouped_lora_mmq(xd, w, e, o, qt, n, a, b, 2.0).backward(dy)
            got.append(xd.grad)
        else:
            got.append(ml.grouped_mmq_grad_input(dy, w, e, o, qt, k))
    assert torch.isfinite(got[0]).all() and torch.equal(*got)


@pytest.mark.parametrize("rank", [0, 16, 40])
@pytest.mark.parametrize("pair", [False, True], ids=["one", "pair"])
def test_iq2xxs_groups_of_few_rows_match_the_tile_kernel(pkg, dev, pair, rank, force_grouped_shape):
    # the same products in the same order, the LoRA term ahead of them: bit for bit
    qt, n, k, groups = gb.IQ2_XXS, 384, 4096, 64
    ml = pkg.fast_moe_lora
    sizes = ([1, 15, 16, 17, 33, 48, 49, 64, 65, 80, 81, 96, 128, 0, 2, 129] * groups)[:groups]
    assert sum(sizes) <= 72 * groups
    ids, ends = torch.arange(groups, device=dev), _ends(dev, sizes)
    planes = [_payload(dev, 10 + i, qt, groups, n, k) for i in range(2 if pair else 1)]
    cotangents = [_rows(dev, 20 + i, sum(sizes), n) for i in range(len(planes))]
    x, nt = _rows(dev, 30, sum(sizes), k), n * len(planes)
    a, b = _rows(dev, 31, groups * rank, k).view(groups, rank, k), _rows(dev, 32, groups * nt, rank).view(groups, nt, rank)
    got = []
    for shape in ("", "1"):
        force_grouped_shape(shape)
        if rank:
            xd = x.clone().requires_grad_(True)
            if pair:
                out = ml.grouped_lora_mmq_pair(xd, *planes, ids, ends, qt, n, a, b, 2.0)
            else:
                out = (ml.grouped_lora_mmq(xd, planes[0], ids, ends, qt, n, a, b, 2.0),)
            torch.autograd.backward(out, cotangents)
            got.append(xd.grad)
        elif pair:
            xd = x.clone().requires_grad_(True)
            torch.autograd.backward(ml.grouped_mmq_pair(xd, *planes, ids, ends, qt, n), cotangents)
            got.append(xd.grad)
        else:
            got.append(ml.grouped_mmq_grad_input(cotangents[0], planes[0], ids, ends, qt, k))
    assert torch.isfinite(got[0]).all() and torch.equal(*got)


@pytest.mark.parametrize("rank", [0, 16])
def test_iq2xxs_workspace_without_room_for_the_small_tables_keeps_the_tile_kernel(pkg, dev, rank):
    # through the C ABI: what the call needed before there was a launch of its own for small groups is still enough
    qt, n, k, groups, s = gb.IQ2_XXS, 256, 4096, 64, 2.0
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    sizes = ([5, 33, 90, 1] * groups)[:groups]
    rows, w, ids, ends = sum(sizes), _payload(dev, 40, qt, groups, n, k), torch.arange(groups, device=dev), _ends(dev, sizes)
    dy, x = _rows(dev, 41, rows, n), _rows(dev, 42, rows, k)
    a, b = _rows(dev, 43, groups * rank, k), _rows(dev, 44, groups * n, rank)
    # tables of 16-byte entries (wide, tall, 64-row), the counts, the row ranges, dy . B, each a multiple of 256 bytes
    up = lambda v: -(-v // 256) * 256
    tall = min(rows // 256 + groups, rows // 129 + rows // 256 + 1)
    small = up(16 * groups) + up(16 * tall) + 256 + ((up(16 * (rows // 64 + groups)) + up(8 * groups) + up(rows * rank * 2)) if rank else 0)
    whole = lib.ggq_lora_workspace_bytes(rows, groups, groups, n, k, rank)
    got = []
    for size in (small, whole):
        ws, dx = torch.empty(size, dtype=torch.uint8, device=dev), torch.empty(rows, k, dtype=torch.bfloat16, device=dev)
        lora = (a.data_ptr(), b.data_ptr(), rank, s) if rank else (None, None, 0, 0.0)
        pkg._lib.check(lib.ggq_grouped_lora_mmq_backward(dy.data_ptr(), None, w.data_ptr(), None, ids.data_ptr(), ends.data_ptr(), groups, groups, qt, rows, n, k,
                                                         x.data_ptr(), x.data_ptr(), *lora, dx.data_ptr(), None, None, None, ws.data_ptr(), size, stream))
        got.append(dx)
    assert torch.equal(*got)
    with pytest.raises(RuntimeError, match="workspace too small"):
        pkg._lib.check(lib.ggq_grouped_lora_mmq_backward(dy.data_ptr(), None, w.data_ptr(), None, ids.data_ptr(), ends.data_ptr(), groups, groups, qt, rows, n, k,
                                                         x.data_ptr(), x.data_ptr(), *lora, dx.data_ptr(), None, None, None, ws.data_ptr(), small - 256, stream))


@pytest.mark.parametrize("tokens,experts,skew", [
    (500, 256, 0.0),     # Q4_K tiles of 64 rows, the caller's tables, a cotangent read through the routing permutation
    (700, 256, 0.25),    # and groups of several tiles among them
    (1601, 16, 0.0),     # factor gradients of a gathered matrix of more than 6 MB: units in the order of its column blocks
])
def test_backward_of_a_combined_output(pkg, dev, tokens, experts, skew):
    # against the same rows materialised with tables built by the call (bit for bit), and fp32 products of sampled experts
    qt, n, k, top_k, rank, s = gb.Q4_K, 2048, 512, 8, 16, 2.0
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=dev).manual_seed(60 + experts)
    scores = torch.rand(tokens, experts, generator=gen, device=dev)
    scores[:, 3:6] += skew
    idx, weights = scores.topk(top_k, dim=1).indices, torch.rand(tokens, top_k, generator=gen, device=dev)
    plan = pkg.fast_moe_routing.prepare_expert_routing(_rows(dev, 61, tokens, n), idx, weights, experts, gather=False)
    perm, ends, rows = plan.permutation, plan.expert_end_offsets, tokens * top_k
    w, ids = _payload(dev, 62, qt, experts, n, k), torch.arange(experts, device=dev)
    grad_out, x, xa = _rows(dev, 63, tokens, n), _rows(dev, 64, rows, k), _rows(dev, 65, rows, rank)
    a, b = (0.02 * _rows(dev, 66, experts * rank, k)).view(experts, rank, k), (0.02 * _rows(dev, 67, experts * n, rank)).view(experts, n, rank)
    tables = torch.empty(lib.ggq_group_tables_bytes(rows, experts, experts), dtype=torch.uint8, device=dev)
    pkg._lib.check(lib.ggq_group_tables_build(ids.data_ptr(), ends.data_ptr(), experts, experts, rows, tables.data_ptr(), tables.numel(), stream))
    ws = torch.empty(lib.ggq_lora_workspace_bytes(rows, experts, experts, n, k, rank), dtype=torch.uint8, device=dev)
    dx, dx_rows = (torch.empty(rows, k, dtype=torch.bfloat16, device=dev) for _ in range(2))
    da, db = torch.empty_like(a), torch.empty_like(b)
    pkg._lib.check(lib.ggq_grouped_lora_mmq_backward_routed_output(
        grad_out.data_ptr(), tokens, perm.data_ptr(), top_k, weights.data_ptr(), 0, w.data_ptr(), ids.data_ptr(), ends.data_ptr(), experts, experts, qt, rows, n, k,
        x.data_ptr(), xa.data_ptr(), a.data_ptr(), b.data_ptr(), rank, s, dx.data_ptr(), da.data_ptr(), db.data_ptr(), tables.data_ptr(), ws.data_ptr(), ws.numel(), stream))
    dy = grad_out[perm // top_k].contiguous()
    pkg._lib.check(lib.ggq_grouped_lora_mmq_backward(
        dy.data_ptr(), None, w.data_ptr(), None, ids.data_ptr(), ends.data_ptr(), experts, experts, qt, rows, n, k,
        x.data_ptr(), xa.data_ptr(), a.data_ptr(), b.data_ptr(), rank, s, dx_rows.data_ptr(), None, None, None, ws.data_ptr(), ws.numel(), stream))
    assert torch.equal(dx, dx_rows)
    bounds, route_weights = [0] + ends.tolist(), weights.reshape(-1)[perm].bfloat16().float()[:, None]  # (weights act at bf16 precision)
    for e in {0, 3, 7, experts - 1}:
        r = slice(bounds[e], bounds[e + 1])
        if r.start == r.stop:
            continue
        d, we = dy[r].float(), pkg.gguf.dequantize_gguf_tensor(pkg.gguf.GGUFQuantizedTensor(w[e : e + 1], qt, (1, n, k)), qt, torch.float32)[0].bfloat16().float()
        dyb = (d @ b[e].float()).bfloat16().float()
        assert_close_bf16(dx[r], (d @ we + s * dyb @ a[e].float()).double(), f"dX of expert {e}")
        # (dY . B may round to the neighbour, a bf16 step of each of its terms, and once more with its weight)
        assert_close_bf16(da[e], (s * (route_weights[r] * dyb).bfloat16().float().T @ x[r].float()).double(), f"dA of expert {e}", ulps=4)
        assert_close_bf16(db[e], (s * d.T @ (route_weights[r] * xa[r].float()).bfloat16().float()).double(), f"dB of expert {e}")


@pytest.mark.parametrize("tokens,k", [(1601, 2048), (801, 4096), (300, 512)])
def test_factor_gradients_of_tokens_read_in_place(pkg, dev, tokens, k):
    # the order of the units (column blocks outer beyond 6 MB) against the gathered copy's, bit for bit
    ml, mr = pkg.fast_moe_lora, pkg.fast_moe_routing
    qt, n, experts, top_k, rank = gb.Q4_K, 256, 24, 8, 16
    x, w = _rows(dev, 70, tokens, k), [_payload(dev, 71 + i, qt, experts, n, k) for i in range(2)]
    idx = torch.rand(tokens, experts, generator=torch.Generator(device=dev).manual_seed(73), device=dev).topk(top_k, dim=1).indices
    a, b = _rows(dev, 74, experts * rank, k).view(experts, rank, k), _rows(dev, 75, experts * 2 * n, rank).view(experts, 2 * n, rank)
    ids, dy = torch.arange(experts, device=dev), [_rows(dev, 76 + i, tokens * top_k, n) for i in range(2)]
    got = []
    for in_place in (True, False):
        plan = mr.prepare_expert_routing(x, idx, torch.full((tokens, top_k), 0.125, device=dev), experts, gather=not in_place)
        ad, bd = a.clone().requires_grad_(True), b.clone().requires_grad_(True)
        if in_place:
            out = ml._RoutedGroupedLoraProjection.apply(x, plan.permutation, plan.inverse_permutation, top_k, *w, ids, plan.expert_end_offsets, qt, n, ad, bd, 2.0)
        else:
            rows, ends = plan.selected_hidden_states, plan.expert_end_offsets
            out = ml._GroupedLoraProjection.apply(rows, *w, ids, ends, qt, n, ad, bd, 2.0)
        torch.autograd.backward(out, dy)
        got.append((ad.grad, bd.grad))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    bounds, e = [0] + ends.tolist(), 5
    r = slice(bounds[e], bounds[e + 1])
    d = torch.cat([t[r] for t in dy], dim=1).float()
    dyb, xa = (d @ b[e].float()).bfloat16().float(), (rows[r].float() @ a[e].float().T).bfloat16().float()
    assert_close_bf16(got[0][0][e], (2.0 * dyb.T @ rows[r].float()).double(), "dA")
    assert_close_bf16(got[0][1][e], (2.0 * d.T @ xa).double(), "dB")


@pytest.mark.parametrize("qt,n", [(gb.Q4_K, 256), (gb.IQ2_XXS, 256)], ids=lambda v: TYPE_NAMES.get(v, str(v)))
def test_an_output_at_any_address(pkg, dev, qt, n):
    # stores of a row that is not 16-byte aligned, element by element
    k, groups = 4096, 64
    lib, stream = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    sizes = ([1, 17, 48, 66, 0] * groups)[:groups]
    rows, w, ids, ends = sum(sizes), _payload(dev, 80, qt, groups, n, k), torch.arange(groups, device=dev), _ends(dev, sizes)
    assert rows <= 40 * groups
    dy, ws = _rows(dev, 81, rows, n), torch.empty(lib.ggq_lora_workspace_bytes(rows, groups, groups, n, k, 0), dtype=torch.uint8, device=dev)
    got = []
    for skip in (0, 1):
        buffer = torch.zeros(rows * k + 8, dtype=torch.bfloat16, device=dev)
        pkg._lib.check(lib.ggq_grouped_lora_mmq_backward(dy.data_ptr(), None, w.data_ptr(), None, ids.data_ptr(), ends.data_ptr(), groups, groups, qt, rows, n, k, None, None,
                                                         None, None, 0, 0.0, buffer.data_ptr() + 2 * skip, None, None, None, ws.data_ptr(), ws.numel(), stream))
        got.append(buffer[skip : skip + rows * k])
        assert not buffer[:skip].any() and not buffer[skip + rows * k :].any()
    assert torch.equal(*got) and got[0].any()


def test_iq2xxs_pair_of_skewed_groups_beside_tall_tiles(pkg, dev, force_grouped_shape):
    # groups of every table of one call: small, wide and tall, with a pair of matrices; bit for bit the tile kernel's results
    qt, n, k, groups, ml = gb.IQ2_XXS, 256, 4096, 64, pkg.fast_moe_lora
    sizes = ([300, 0, 0, 0, 81, 7, 131, 0, 512, 0, 0, 0, 0, 80, 0, 1] * groups)[:groups]
    assert sum(sizes) <= 72 * groups
    ids, ends = torch.arange(groups, device=dev), _ends(dev, sizes)
    planes, cotangents, x = [_payload(dev, 90 + i, qt, groups, n, k) for i in range(2)], [_rows(dev, 92 + i, sum(sizes), n) for i in range(2)], _rows(dev, 94, sum(sizes), k)
    got = []
    for shape in ("", "1"):
        force_grouped_shape(shape)
        xd = x.clone().requires_grad_(True)
        torch.autograd.backward(ml.grouped_mmq_pair(xd, *planes, ids, ends, qt, n), cotangents)
        got.append(xd.grad)
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
