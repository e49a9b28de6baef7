"""What the compiler says of the product's kernels (the metadata in the code objects of libpto_amd.so)."""
import os
import re
import shutil
import subprocess

import pytest

from pto_amd import capi

LLVM = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")))), "llvm", "bin")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """[(symbol, bytes of scratch, spilled vector registers)] of every kernel of the library."""
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no LLVM tools in " + LLVM)
    d = str(tmp_path_factory.mktemp("code_objects"))
    shutil.copy(capi.LIB_PATH, os.path.join(d, "lib.so"))
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    found = []
    for name in os.listdir(d):
        if "gfx950" in name:
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", os.path.join(d, name)], check=True, capture_output=True, text=True).stdout
            for m in re.finditer(r"\.private_segment_fixed_size: (\d+)\s[\s\S]*?\.symbol:\s+(\S+)\.kd\s[\s\S]*?\.vgpr_spill_count: (\d+)", notes):
                found.append((m.group(2), int(m.group(1)), int(m.group(3))))
    return found


def test_no_kernel_spills(kernels):
    """No kernel keeps registers in scratch.  The GEMM and attention kernels read the LDS with waits that they place
    themselves: where such a read is assembly, the compiler would store its registers before they hold anything."""
    assert len(kernels) > 150 and any("GemmF16F32Ks" in k[0] for k in kernels)
    assert [k for k in kernels if k[1] or k[2]] == []
