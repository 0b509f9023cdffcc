"""Grad-input of expert groups of very different sizes in one call, on the kernels for groups of a few rows."""

import statistics

import pytest
import torch

from helpers import TYPE_NAMES
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


@pytest.mark.parametrize("rank", [0, 16, 40, 64])
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
