"""The prefill GEMMs' and the prompt attention's hot instantiations must stay free of scratch (register spills): gemm4w_kernel keeps up to 256 accumulators and 217 other registers a lane at
one wave a SIMD, gemm8p_kernel sits at 251 of 256 VGPRs, and a few more live values in a
rarely taken branch once doubled the whole prefill (a runtime `skip X half 1` flag in the ragged loop -> 88 bytes of spills per lane -> ragged tiles
took two tile-times).  Kernels whose loads are counted by hand have a bound besides (csrc/wstream.h).  hipcc reports the numbers at compile time; these tests recompile the files (~2 min, no GPU
needed)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llava-plus-codebase_amd", "csrc")


def resources(source, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    r = subprocess.run([hipcc, "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-I.", "-I../../include",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-c", source, "-o", str(tmp_path / "g.o"),
                        "-Rpass-analysis=kernel-resource-usage"], cwd=CSRC, capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    blocks = re.split(r"Function Name: (\S+)", r.stderr)[1:]
    return {name: {k: int(v) for k, v in re.findall(r"remark:\s+(\w[^:\n]*): (\d+)", text)} for name, text in zip(blocks[::2], blocks[1::2])}


def scratch_sizes(source, tmp_path):
    return {k: v["ScratchSize [bytes/lane]"] for k, v in resources(source, tmp_path).items()}


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
@pytest.mark.parametrize("source,tiles", [("gemm4w_large_bf16.hip", 4), ("gemm4w_small_f16.hip", 6)])
def test_four_wave_tiles_have_no_scratch(tmp_path, source, tiles):
    """Each tile un-sliced, sliced and grouped, and its reductions of two and three slices."""
    usage = scratch_sizes(source, tmp_path)
    assert len([k for k in usage if "gemm4w" in k]) == 5 * tiles, sorted(usage)
    assert not {k: v for k, v in usage.items() if v}, usage


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
def test_hot_gemm8p_instantiations_have_no_scratch(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    r = subprocess.run([hipcc, "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-I.", "-I../../include",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-c", "gemm8p.hip", "-o", str(tmp_path / "g.o"),
                        "-Rpass-analysis=kernel-resource-usage"], cwd=CSRC, capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    usage = {}
    name = None
    for line in r.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m and name:
            usage[name] = int(m.group(1))
    # every instantiation of the ping-pong kernel: <T, SPLIT> = {bf16, f16} x {1 (q|k|v, gate|up), 2, 3 (o_proj, down_proj)}
    hot = [k for k in usage if "gemm8p_kernel" in k]
    assert len(hot) == 6, sorted(usage)
    bad = {k: usage[k] for k in hot if usage[k] != 0}
    assert not bad, bad


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
def test_prompt_attention_has_no_scratch(tmp_path):
    """flash_prefill2_kernel stands at two waves a SIMD; a reload from scratch waits for every tile that is on its way into LDS."""
    usage = {k: v for k, v in scratch_sizes("attention.hip", tmp_path).items() if "flash_" in k}
    assert len([k for k in usage if "flash_prefill2" in k]) == 12, sorted(usage)      # {bf16, f16} x {64, 128 / 64 rows, 128 / 128 rows} x {plain, windowed}
    assert not {k: v for k, v in usage.items() if v}, usage


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
@pytest.mark.parametrize("source,kernels,forms", [("gemm.hip", "gemv2_", 58), ("skinny.hip", "skinny_gemm_kernel", 36), ("decode_attn.hip", "decode_kv_attn_kernel", 8), ("delta.hip", "delta_decode_linear_kernel", 12),
                                                  ("moe.hip", "group_gemv_linear_kernel", 8)])
def test_hand_counted_loads_keep_their_registers(tmp_path, source, kernels, forms):
    """Past 256 registers the compiler moves destinations of loads on their way (csrc/wstream.h): fewer than that, none in scratch, and accumulators only where matrix instructions are."""
    usage = {k: v for k, v in resources(source, tmp_path).items() if kernels in k}
    assert len(usage) == forms, sorted(usage)
    assert not {k: v for k, v in usage.items() if v["VGPRs"] >= 256 or v["ScratchSize [bytes/lane]"] or (v["AGPRs"] and source != "skinny.hip")}, usage
