"""The built gfx950 kernels and their register use, from the compiler's own
resource remarks.  CPU only (hipcc cross-compiles).

The tile passes of a coarse level have one form of the element each, the
constant-moduli mode form or the Gauss-point sums: a kernel that holds both
holds the registers of both, for every level.  The phase-field passes run four
waves per SIMD without a spill.  The bounds are the waves per SIMD that the
registers leave room for (512 per SIMD lane, given out in eights)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SOURCES = ["hpcr_kernels.hip", "hpcr_mixed.hip"]


def remarks(text):
    """{kernel symbol: (VGPRs with AGPRs, spilled VGPRs)}"""
    out = {}
    for part in text.split("Function Name: ")[1:]:
        num = {k: int(re.search(re.escape(k) + r": (\d+)", part)[1]) for k in ("VGPRs", "AGPRs", "VGPRs Spill")}
        out[part.split()[0]] = (num["VGPRs"] + num["AGPRs"], num["VGPRs Spill"])
    return out


def vgprs_of_waves(n):
    return 512 // n // 8 * 8


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    run = []
    for src in SOURCES:
        cmd = [HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
               "-packed-fp32-ops", "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c", "-o", os.devnull,
               "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "hpcrack_amd", "csrc", src)]
        run.append(subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True))
    out = {}
    for p in run:
        err = p.communicate()[1]
        assert p.returncode == 0, err[-2000:]
        out.update(remarks(err))
    return out


# symbol patterns of the coarse levels' tile passes, with the least waves per
# SIMD: FP64 FAS passes (operator, residual, pass A), FP32 and FP64
# preconditioner passes; mode form, Gauss-point sums
FAS = r"tile_kernelINS_6MechOpILi[012]ELb0ELb[01]E(Lb%dE)?EE"
PRE = r"tile_kernelINS_7MechOpPI%sLi\dELb0ELb[01]ELb0ELi\d(ELb%d)?EEE"
CASES = {
    "fas-modes": (FAS % 0, 3, 6),
    "fas-gauss": (r"tile_kernelINS_6MechOpILi[012]ELb0ELb[01]ELb1EEE", 2, 4),
    "f32-modes": (PRE % ("f", 1), 5, 16),
    "f32-gauss": (PRE % ("f", 0), 4, 16),
    "f64-modes": (PRE % ("d", 1), 3, 16),
    "f64-gauss": (PRE % ("d", 0), 2, 16),
}


@pytest.mark.parametrize("name", CASES)
def test_coarse_passes_hold_one_element_form(kernels, name):
    pattern, waves, count = CASES[name]
    found = {k: v for k, v in kernels.items() if re.search(pattern, k)}
    assert len(found) == count, sorted(found)
    for k, (v, spill) in found.items():
        assert v <= vgprs_of_waves(waves) and spill == 0, f"{k}: {v} registers, {spill} spilled"


def test_phase_field_passes_do_not_spill(kernels):
    found = {k: v for k, v in kernels.items() if re.search(r"tile_kernelINS_4PfOpI", k)}
    assert len(found) >= 4, sorted(found)
    for k, (v, spill) in found.items():
        assert v <= vgprs_of_waves(4) and spill == 0, f"{k}: {v} registers, {spill} spilled"


def test_passes_b_are_the_ones_that_run(kernels):
    """Inside a call a pass B applies no update or a whole group of four; only
    the phase field's calls may end on an iteration that keeps z (LAST false)."""
    last_of = {r"17mech_pcg_b_kernelILb[01]ELi(\d)ELb[01]ELb([01])E": {"0": "04", "1": "1234"},
               r"17open_pcg_b_kernelILi[13]ELi(\d)ELb([01])E": {"0": "04", "1": "1234"},
               r"15pf_pcg_b_kernelILi(\d)ELb([01])E": {"0": "01234", "1": "1234"}}
    for pattern, want in last_of.items():
        found = {m.groups() for m in (re.search(pattern, k) for k in kernels) if m}
        assert found == {(n, l) for l in want for n in want[l]}, (pattern, sorted(found))
