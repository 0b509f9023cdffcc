"""Registers of kernels whose launch counts on a number of workgroups per compute unit, as the compiler reports them.

A SIMD has 512 registers per lane: a kernel of up to 128 runs four waves on it, of up to 168 three, of up to 80 six."""
import pathlib
import re
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "transformers5-qwen3.5-recipe_amd" / "csrc"


def _compiled(source, directory):
    """{mangled kernel name: (registers, bytes of scratch per lane)} of a source file."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not pathlib.Path(hipcc).exists():
        pytest.skip("hipcc is not installed")
    cmd = [hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-c", "--cuda-device-only",
           "-Rpass-analysis=kernel-resource-usage", str(CSRC / source), "-o", str(directory / "out.o")]
    done = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert done.returncode == 0, done.stderr[-2000:]
    out = {}
    for block in done.stderr.split("Function Name: ")[1:]:
        vgprs, agprs, scratch = (int(re.search(key + r": (\d+)", block).group(1)) for key in (r" VGPRs", r" AGPRs", r"ScratchSize \[bytes/lane\]"))
        out[block.split()[0]] = (vgprs + agprs, scratch)
    return out


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    return _compiled("gemv.hip", tmp_path_factory.mktemp("registers"))


@pytest.fixture(scope="module")
def dense_resources(tmp_path_factory):
    return _compiled("dense_gemm.hip", tmp_path_factory.mktemp("registers"))


def _named(resources, pattern):
    found = {name: r for name, r in resources.items() if re.search(pattern, name)}
    assert found, pattern
    return found


def test_few_routes_gate_up_leaves_room_for_two_workgroups(resources):
    for name, (registers, scratch) in _named(resources, r"few_routes_gate_up_kernelILi\d+ELi\d+ELi\d+E").items():
        assert registers <= 128 and scratch == 0, (name, registers, scratch)


def test_one_row_block_products_leave_room_for_the_workgroups_the_launch_asks_for(resources):
    # gemv_kernel<type, 8 waves, 2 spans, 1 row block, no LoRA>: three workgroups of eight waves unless the rule names the type, else two
    rule = re.search(r"static bool many_small_workgroups\(.*", (CSRC / "gemv.hip").read_text()).group(0)
    ids = {"kQ8_0": 8, "kQ2_K": 10, "kQ3_K": 11, "kQ4_K": 12, "kQ5_K": 13, "kQ6_K": 14, "kIQ2_XXS": 16}
    for name, qt in ids.items():
        ((kernel, (registers, scratch)),) = _named(resources, rf"11gemv_kernelILi{qt}ELi8ELi2ELi1ELb0E").items()
        assert registers <= (128 if f"qt != {name}" in rule else 80) and scratch == 0, (kernel, registers, scratch)


def test_rank_sized_products_beside_the_decoding_pass_need_no_scratch(dense_resources):
    # decode_side_kernel<type, blocks of sixteen ranks>: its decoding workgroups pay for what the product's take
    kernels = _named(dense_resources, r"decode_side_kernelILi\d+ELi[12]E")
    assert len(kernels) == 14, sorted(kernels)
    for name, (registers, scratch) in kernels.items():
        assert registers <= (128 if re.search(r"ELi1E", name) else 168) and scratch == 0, (name, registers, scratch)
