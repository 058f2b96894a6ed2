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
