"""Registers of the kNN lane search in the built library: every form keeps the
waves a SIMD that its launch bound names (512 registers: 128 a lane for four
waves, 168 for three). Read from the code object built here; skipped where the
objects or the compiler's tools are not there."""
import os
import re
import subprocess

import pytest

OBJ = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tgmm_amd", "_build",
                   "tgmm_kernels.o")
BIN = "/opt/rocm/llvm/bin/"
TOOLS = [BIN + t for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]

if not all(os.path.exists(p) for p in [OBJ] + TOOLS):
    pytest.skip("built objects or compiler tools not there", allow_module_level=True)


@pytest.fixture(scope="module")
def vgprs(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("co"))
    fat, co = d + "/fat", d + "/co"
    subprocess.run([TOOLS[0], "--dump-section", ".hip_fatbin=" + fat, OBJ, d + "/o"], check=True)
    subprocess.run([TOOLS[1], "--type=o", "--unbundle", "--input=" + fat, "--output=" + co,
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([TOOLS[2], "--notes", co], check=True, stdout=subprocess.PIPE,
                           text=True).stdout
    out, name = {}, None
    for line in notes.splitlines():
        m = re.match(r"\s+\.(symbol|vgpr_count):\s+(\S+)", line)
        if m and m[1] == "symbol":
            name = m[2]
        elif m:
            out[name] = int(m[2])
    return out


@pytest.mark.parametrize("km,most", [(5, 128), (8, 128), (16, 168)])
def test_lane_search_occupancy(vgprs, km, most):
    got = {k: v for k, v in vgprs.items() if re.search(r"5k_knnILi%dE" % km, k or "")}
    assert len(got) == 6, sorted(got)
    assert max(got.values()) <= most, got
