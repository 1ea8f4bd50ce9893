"""Registers and scratch memory of the kernels as built, read from the library's own metadata: what
their launches rely on for the number of wavefronts that a SIMD holds.  Nothing is launched here."""
import os
import re
import shutil
import subprocess

import pytest

from lydion_amd import _lib

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
OBJDUMP, READELF = (os.path.join(LLVM, t) for t in ("llvm-objdump", "llvm-readelf"))

pytestmark = pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(READELF)),
                                reason="the toolchain's readers are not installed")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> (VGPRs with AGPRs, bytes of scratch per lane)"""
    d = tmp_path_factory.mktemp("code")
    shutil.copy(_lib.LIB_PATH, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    out = {}
    for f in d.glob("*gfx950"):
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for part in notes.split("- .agpr_count:")[1:]:
            def get(key, text=part):
                return re.search(rf"\.{key}:\s+(\S+)", text).group(1)
            if re.search(r"\.name:\s+_Z", part):
                name = re.search(r"\.name:\s+(_Z\S+)", part).group(1)
                out[name] = (int(get("vgpr_count")), int(get("private_segment_fixed_size")))
    assert out
    return out


def test_column_kernel_keeps_two_wavefronts_per_simd(kernels):
    """Its grid is sized for two blocks of four wavefronts on a CU, over all bins per lane."""
    cols = {k: v for k, v in kernels.items() if "k_columnI" in k}
    assert len(cols) >= 18
    for k, (vgprs, scratch) in cols.items():
        assert vgprs <= 256, (k, vgprs)
        # a few spilled registers at eight and nine bins per lane, next to none below
        wide = re.search(r"k_columnILi1ELi[89]", k)
        assert scratch <= (256 if wide else 72), (k, scratch)


def test_paired_step_keeps_five_wavefronts_per_simd(kernels):
    """Two cells per wavefront, no sheared gradients: tiles of four rows and fewer rely on 512 / 5
    registers, in units of eight."""
    pair = [v for k, v in kernels.items() if "k_stepILb0ELi1ELb1E" in k]
    assert pair and all(vgprs <= 96 and scratch == 0 for vgprs, scratch in pair), pair
