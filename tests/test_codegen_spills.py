"""Registers of the ensemble's kernels and of the reductions that end a step (no GPU needed).

Compiled to assembly with the library's own flags; the kernels' metadata must show
no scratch and no spilled registers where an earlier form of the source had none.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rast-3dmhd_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None,
                                reason="hipcc not available")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(unit, demangled name without arguments): metadata}"""
    d = tmp_path_factory.mktemp("spills")
    cc = HIPCC if os.path.exists(HIPCC) else shutil.which("hipcc")
    units = ["r3d_hip", "r3d_ens"]
    jobs = [subprocess.Popen([cc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off",
                              "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                              "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                              "--cuda-device-only", "-S", "-o", str(d / (u + ".s")),
                              os.path.join(CSRC, u + ".hip")], stderr=subprocess.DEVNULL)
            for u in units]
    assert all(j.wait() == 0 for j in jobs)
    out = {}
    for u in units:
        text = (d / (u + ".s")).read_text()
        meta = text[text.index("amdhsa.kernels:"):]
        for block in meta.split("  - .agpr_count:")[1:]:
            name = re.search(r"\.name: +(\S+)", block).group(1)
            plain = subprocess.run(["c++filt", name], capture_output=True, text=True).stdout
            out[u, re.search(r"k_\w+(<[^(]*>)?", plain).group(0)] = {
                k: int(re.search(r"\." + k + r": +(\d+)", block).group(1))
                for k in ("vgpr_count", "vgpr_spill_count", "sgpr_spill_count",
                          "private_segment_fixed_size")}
    return out


@pytest.mark.parametrize("kernel", [("r3d_hip", "k_finish"), ("r3d_hip", "k_finish_redo"),
                                    ("r3d_hip", "k_dt_redo"), ("r3d_ens", "k_finish_ens"),
                                    ("r3d_ens", "k_dt_redo_ens")], ids=lambda k: k[1])
def test_reductions_do_not_spill(kernels, kernel):
    k = kernels[kernel]
    assert k["private_segment_fixed_size"] == 0 and k["vgpr_spill_count"] == 0, k
    assert k["sgpr_spill_count"] == 0, k


HYDRO = [(4, 64), (8, 64), (9, 64), (8, 32), (16, 32), (16, 16), (28, 16)]


@pytest.mark.parametrize("stage", [0, 1, 2])
@pytest.mark.parametrize("ty,tw", HYDRO)
def test_ensemble_stage_kernels(kernels, ty, tw, stage):
    """Three waves on a SIMD (168 VGPRs), and the members' scalars in scalar registers."""
    k = kernels["r3d_ens", f"k_stage_ens<{ty}, {stage}, false, {tw}>"]
    assert k["vgpr_count"] <= 168 and k["vgpr_spill_count"] == 0, k
    assert k["private_segment_fixed_size"] == 0 and k["sgpr_spill_count"] <= 16, k


@pytest.mark.parametrize("stage", [0, 1, 2])
def test_mhd_ensemble_stage_kernels(kernels, stage):
    k = kernels["r3d_ens", f"k_stage_ens<12, {stage}, true, 32>"]
    assert k["private_segment_fixed_size"] == 0 and k["vgpr_spill_count"] == 0, k


@pytest.mark.parametrize("ty,tw", HYDRO + [(12, 32)])
def test_persistent_ensemble_kernel(kernels, ty, tw):
    """One tile loop over three stages: a little scratch outside the z loops (at most
    what it took when it measured 5.4 ms a step of 64 members), no more."""
    k = kernels["r3d_ens", f"k_ens_run<{ty}, {'true' if ty == 12 else 'false'}, {tw}>"]
    assert k["private_segment_fixed_size"] <= 84, k
