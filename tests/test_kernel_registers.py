"""Registers of kernels, from their descriptors in the built library.  FP32 sweeps
of the main path in launches without soft sources: no vector register of the H
sweeps in scratch memory; of the E sweeps none, 3 with a ragged z extent or with
a folded plane wave, 7 with both.  The TF/SF correction that evaluates the
incident field at every point: no scratch memory, and registers for three waves
a SIMD."""
import os
import re
import shutil
import subprocess

import pytest

from dtmaxwell4_amd import abi

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")) or not os.path.exists(abi.LIB_PATH):
        pytest.skip("needs the built library and ROCm's LLVM tools")
    d = str(tmp_path_factory.mktemp("code"))
    shutil.copy(abi.LIB_PATH, os.path.join(d, "lib.so"))
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True,
                   stdout=subprocess.DEVNULL)
    out = {}
    for name in os.listdir(d):
        if "gfx950" not in name:
            continue
        text = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", name], cwd=d, check=True,
                              stdout=subprocess.PIPE, text=True).stdout
        for k in text.split("- .agpr_count:")[1:]:
            out[re.search(r"\.name:\s+(\S+)", k).group(1)] = {
                f: int(re.search(rf"\.{f}:\s+(\d+)", k).group(1))
                for f in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size")}
    return out


def sweep(up, general, fold, soft=0):
    """FP32 k_sweep<up, 0, general, no split layer, fold, no zone, set below 4 GiB, soft>."""
    return f"k_sweepILi{up}ELi0ELb{general}ELb0ELb{fold}ELb0ELi0ELb{soft}E"


@pytest.mark.parametrize("up,general,fold,most", [
    (0, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0), (0, 1, 1, 0), (1, 0, 0, 0), (1, 1, 0, 3), (1, 0, 1, 3), (1, 1, 1, 7)])
def test_sweeps_without_soft_sources(kernels, up, general, fold, most):
    got = [k["vgpr_spill_count"] for name, k in kernels.items() if sweep(up, general, fold) in name]
    assert len(got) == 1 and got[0] <= most


@pytest.mark.parametrize("store", [0, 1])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_correction_with_the_incident_field(kernels, store, mode):
    got = [k for name, k in kernels.items() if f"6k_tfsfILi{store}ELi{mode}E" in name]
    assert len(got) == 1 and got[0]["private_segment_fixed_size"] == 0 and got[0]["vgpr_count"] <= 168
