"""Registers of kernels whose occupancy a change of the sources can take away without a difference in any result, from the notes of
the built code objects, without a GPU.  A SIMD has 512 a lane: 256 are two waves, 64 eight."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vtpack_amd", "csrc")
LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.parametrize("source,kernel,most", [("grained_sample", r"router_kernel<unsigned short, 4, \d+, true>", 256),
                                                ("grained_sample", r"router_kernel<float, 4, \d+, true>", 168),
                                                ("grained_sample", r"router_kernel<float, 2, \d+, true>", 64)])
def test_registers(tmp_path, source, kernel, most):
    if shutil.which("hipcc") is None or not os.path.exists(f"{LLVM}/clang-offload-bundler"):
        pytest.skip("needs the compiler's tools")
    obj, bundle, code = os.path.join("build", source + ".o"), tmp_path / "bundle", tmp_path / "code"
    subprocess.run(["make", "-C", CSRC, obj], check=True, capture_output=True)
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", os.path.join(CSRC, obj), "/dev/null"], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}"], check=True)
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(code)], check=True, capture_output=True, text=True).stdout
    notes = subprocess.run(["c++filt"], input=notes, check=True, capture_output=True, text=True).stdout
    found = re.findall(r"\.name: +(.*)\n(?:.*\n)*?.*\.vgpr_count: +(\d+)", notes)
    counts = [int(n) for name, n in found if re.search(kernel, name)]
    assert len(counts) == 4 and max(counts) <= most
