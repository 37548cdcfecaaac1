"""Registers of the built kernels that go to scratch memory, read from the metadata that the
compiler put into libmgpu.so.  The passes here are bound by memory, and a spill in one is
traffic of its own: each of these has had too many at a size that no benchmark ran."""
import os
import re
import subprocess

import pytest

import mgpicola as M

LLVM = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def spilled(tmp_path_factory):
    d = tmp_path_factory.mktemp("code")
    os.symlink(os.path.abspath(M.LIBMGPU), d / "lib.so")
    subprocess.run([LLVM + "llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    out = {}
    for f in sorted(os.listdir(d)):
        if "gfx950" not in f:
            continue
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(d / f)], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n  - ", notes)[1:]:
            m = re.search(r"\.symbol:\s+(\S+)\.kd", k)
            if m:
                out[m.group(1)] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", k).group(1))
    names = subprocess.run(["c++filt"], input="\n".join(out), check=True, capture_output=True, text=True).stdout.split("\n")
    return {n.replace("(anonymous namespace)::", "").replace("void ", "").split("(")[0]: v for n, v in zip(names, out.values())}


@pytest.mark.parametrize("kernel,most", [
    (r"k_fft_col<2048, 8, -?1, 2>", 6),  # the plain column passes of the largest mesh
    (r"k_col_fused<1536, 8, [12], 0, true>", 2),  # the force pairs of screened models
    (r"k_z_screen<512, [01]>", 0),  # the screening rows of the learned runs' coarse mesh
])
def test_spilled_registers(spilled, kernel, most):
    found = {k: v for k, v in spilled.items() if re.fullmatch(kernel, k)}
    assert len(found) >= 2
    assert max(found.values()) <= most, found
