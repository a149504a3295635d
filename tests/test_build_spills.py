"""No stage kernel of the built library spills a vector register, the per-cell
checking kernels (VAH_FLUX_PER_CELL) excepted.  Trial forms of the FP64 3+1D role
kernel that spilled a few gave wrong values in some cells; the committed forms use
up to 255 of 256 registers, and the batch's 3+1D half stays free of spills through a
scheduler option of the Makefile only, so a small edit or another compiler can end
it.  Read from the code-object metadata of the library built here."""
import os
import re
import shutil
import subprocess

import pytest

from tests.test_build_isa import LIB, OBJDUMP

READELF = os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf")


def kernels(notes):
    """{mangled kernel name: {metadata key: value}} of one code object's notes."""
    out = {}
    for part in re.split(r"^  - (?=\.a)", notes, flags=re.M)[1:]:
        meta = dict(re.findall(r"^ {4}(\.\w+): +(\S+)$", part, flags=re.M))
        out[meta[".name"]] = meta
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="ROCm llvm-readelf not installed")
def test_stage_kernels_spill_no_vector_register(tmp_path):
    if not os.path.exists(LIB):
        pytest.skip("libvah.so not built")
    lib = tmp_path / "libvah.so"
    shutil.copy(LIB, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp_path)
    found = {}
    for obj in sorted(p for p in tmp_path.iterdir() if "amdgcn-amd-amdhsa" in p.name):
        notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
        found.update({n: m for n, m in kernels(notes).items() if re.match(r"_ZN3vah\d+(batch_)?stage_kernelI", n)})
    # one lattice: two tile shapes, a batch: three, in 2+1D and 3+1D; each for two stages
    # and two precisions
    assert len(found) == 4 * (4 + 6), sorted(found)
    for name, meta in found.items():
        assert int(meta[".vgpr_count"]) <= 256, (name, meta)
        assert int(meta[".vgpr_spill_count"]) == 0, (name, meta)
