"""Registers of the kernels that are held to a number of wavefronts: a build that spills
them to memory is found here, without a GPU."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "graphiler_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="no hipcc")
def test_pair_attention_builds_spill_nothing(tmp_path):
    r = subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3",
                        "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                        "pair_attn.hip", "-o", str(tmp_path / "pair_attn.o")],
                       cwd=CSRC, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "failed to meet occupancy" not in r.stderr
    spills = [int(x) for x in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    waves = [int(x) for x in re.findall(r"Occupancy \[waves/SIMD\]: (\d+)", r.stderr)]
    assert len(spills) == len(waves) == 16
    assert not any(spills), spills
    assert min(waves) >= 4, waves


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="no hipcc")
def test_pair_tiles_builds_spill_nothing(tmp_path):
    r = subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3",
                        "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                        "pair_tiles.hip", "-o", str(tmp_path / "pair_tiles.o")],
                       cwd=CSRC, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "failed to meet occupancy" not in r.stderr
    spills = [int(x) for x in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    waves = [int(x) for x in re.findall(r"Occupancy \[waves/SIMD\]: (\d+)", r.stderr)]
    assert len(spills) == len(waves) == 21      # 16 of the pass, tiles, four of the matrices
    assert not any(spills), spills
    assert min(waves) >= 4, waves


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="no hipcc")
def test_opaque_row_stores_keep_four_wavefronts(tmp_path):
    """The aggregation's bf16 builds that exist for their registers: four wavefronts per SIMD."""
    r = subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3",
                        "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                        "gat.hip", "-o", str(tmp_path / "gat.o")],
                       cwd=CSRC, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    waves = re.findall(r"Function Name: \S*11runs_kernelINS_12_GLOBAL__N_114GatOpaqueStore"
                       r".*?Occupancy \[waves/SIMD\]: (\d+)", r.stderr, re.S)
    assert len(waves) == 3 and min(map(int, waves)) >= 4, waves


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="no hipcc")
@pytest.mark.parametrize("source,kernel,builds,waves", [
    ("gat_inputs", "17gat_inputs_kernelILi", 4, {"8": 3, None: 4}),
    ("typed_rows", "17typed_rows_kernelILi", 9, {"4": 3, "1": 5, None: 4}),
    ("linear", "22linear_few_rows_kernelILb[01]ELi[48]ELi", 12, {"4": 2, "2": 3, None: 4})])
def test_register_budgets(tmp_path, source, kernel, builds, waves):
    """The layer over its inputs (by heads), typed fp32 rows (by k steps) and the projection of few
    rows (by column blocks): no spills, the wavefronts per SIMD that their comments count on."""
    r = subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3",
                        "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "-c",
                        source + ".hip", "-o", str(tmp_path / "kernel.o")],
                       cwd=CSRC, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    found = re.findall(r"Function Name: \S*" + kernel + r"(\d+).*?Occupancy \[waves/SIMD\]: (\d+)"
                       r".*?VGPRs Spill: (\d+)", r.stderr, re.S)
    assert len(found) == builds, found
    for build, occupancy, spilled in found:
        assert int(occupancy) >= waves.get(build, waves[None]) and int(spilled) == 0, (build, occupancy, spilled)
