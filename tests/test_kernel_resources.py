"""Registers of the built kernels, from the library's own code-object notes.

The FP64 kernels of the explicit path are sized to run without spilling: a cap
that makes one spill costs it a third of its speed or more.
"""

import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

LLVM = "/opt/rocm/llvm/bin"
TOOLS = ["llvm-objcopy", "clang-offload-bundler", "llvm-readelf"]


def kernel_spills(lib, tmp):
    """mangled name -> spilled vector registers, of every gfx950 kernel in the library"""
    fat = os.path.join(tmp, "fatbin")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", lib,
                    os.path.join(tmp, "copy.so")], check=True)
    data = open(fat, "rb").read()
    at = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)] + [len(data)]
    out = {}
    for i, (a, b) in enumerate(zip(at, at[1:])):
        bundle, obj = os.path.join(tmp, f"b{i}"), os.path.join(tmp, f"o{i}")
        with open(bundle, "wb") as f:
            f.write(data[a:b])
        subprocess.run([f"{LLVM}/clang-offload-bundler", "--type=o", "--unbundle", f"--input={bundle}",
                        f"--output={obj}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], check=True, capture_output=True,
                               text=True).stdout
        out.update((m.group(1), int(m.group(2))) for m in
                   re.finditer(r"\.name:\s+(_Z\S+).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S))
    return out


@pytest.fixture(scope="module")
def spills(tmp_path_factory):
    for t in TOOLS:
        if shutil.which(t, path=LLVM) is None:
            pytest.skip(f"{t} is not available")
    return kernel_spills(PKG.solver.LIB_PATH, str(tmp_path_factory.mktemp("notes")))


# mangled template arguments that make the kernel an FP64 one
@pytest.mark.parametrize("kernel,fp64", [("k_flux_fused", "dLi"), ("k_flux_small", "dLi"),
                                         ("k_qderiv_timestep", "dLi")])
def test_fp64_kernels_do_not_spill(spills, kernel, fp64):
    found = {n: v for n, v in spills.items() if kernel in n and fp64 in n.split(kernel)[1]}
    assert found
    assert not {n: v for n, v in found.items() if v}
