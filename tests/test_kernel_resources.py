"""Registers of the built GEMM kernels, from the code object's own metadata.

A kernel whose registers do not suffice keeps the rest in private memory, which
the runtime then allocates for the whole device when the kernel is first
launched: the allocation-free entry point promises none, so no kernel of the
prefill GEMM may use any.  Needs no device."""
import os
import re
import subprocess

import pytest

from aihost_amd import build

LLVM = os.path.join(build.ROCM, "llvm", "bin")


def _private_bytes(src, tmp_path):
    """{kernel: bytes of private memory per lane} of one built source."""
    obj, fat, code = os.path.join(build.OBJ, src + ".o"), str(tmp_path / "fat"), str(tmp_path / "code.o")
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]
    if not all(os.path.exists(p) for p in [obj] + tools):
        pytest.skip("the built objects or the LLVM tools are not here")
    subprocess.run([tools[0], "--dump-section", ".hip_fatbin=" + fat, obj, os.devnull], check=True)
    subprocess.run([tools[1], "--type=o", "--unbundle", "--targets=hipv4-amdgcn-amd-amdhsa--" + build.ARCH,
                    "--input=" + fat, "--output=" + code], check=True)
    notes = subprocess.run([tools[2], "--notes", code], check=True, capture_output=True, text=True).stdout
    names = re.findall(r"^ +\.name: +(_Z\S+)$", notes, re.M)
    sizes = re.findall(r"^ +\.private_segment_fixed_size: +(\d+)$", notes, re.M)
    assert names and len(names) == len(sizes)
    return dict(zip(names, map(int, sizes)))


@pytest.mark.parametrize("src", ["aih_qgemm.hip", "aih_qmatvec_mfma.hip"])
def test_matrix_core_kernels_use_no_private_memory(src, tmp_path):
    used = {k: b for k, b in _private_bytes(src, tmp_path).items() if b}
    assert not used, used
