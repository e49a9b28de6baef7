"""What the compiler says of the product's kernels (the metadata in the code objects of libpto_amd.so)."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

from pto_amd import capi

LLVM = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")))), "llvm", "bin")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """[(symbol, bytes of scratch, spilled vector registers, spilled scalar registers)] of every kernel of the library."""
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no LLVM tools in " + LLVM)
    d = str(tmp_path_factory.mktemp("code_objects"))
    shutil.copy(capi.LIB_PATH, os.path.join(d, "lib.so"))
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    found = []
    for name in os.listdir(d):
        if "gfx950" in name:
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", os.path.join(d, name)], check=True, capture_output=True, text=True).stdout
            for m in re.finditer(r"\.private_segment_fixed_size: (\d+)\s[\s\S]*?\.sgpr_spill_count: (\d+)\s[\s\S]*?\.symbol:\s+(\S+)\.kd\s[\s\S]*?\.vgpr_spill_count: (\d+)", notes):
                found.append((m.group(3), int(m.group(1)), int(m.group(4)), int(m.group(2))))
    return found


def test_no_kernel_spills(kernels):
    """No kernel keeps registers in scratch.  The GEMM and attention kernels read the LDS with waits that they place
    themselves: where such a read is assembly, the compiler would store its registers before they hold anything."""
    assert len(kernels) > 150 and any("GemmF16F32Ks" in k[0] for k in kernels)
    assert [k for k in kernels if k[1] or k[2]] == []


def test_no_kernel_keeps_scalars_in_vector_lanes(kernels):
    """Spilled scalar registers go to lanes of vector registers, two instructions each time (the selecting top-k kernels had 110 of them)."""
    assert [k for k in kernels if k[3]] == []


def test_write_through_stores_leave_their_registers_alone(tmp_path):
    """A store of 16 bytes reads its data registers up to two wait states after it (gfx940 and later).  The compiler, which does not
    look into assembly, may overwrite them in the very next instruction, so the assembly itself has to hold both."""
    build = importlib.util.module_from_spec(importlib.util.spec_from_file_location("pto_amd_build", os.path.join(os.path.dirname(capi.LIB_PATH), "build.py")))
    build.__spec__.loader.exec_module(build)
    source, listing = tmp_path / "stores.hip", tmp_path / "listing"
    source.write_text("""#include <pto/pto-inst.hpp>
#include "stores.hpp"
__global__ void Fours(float *p, Four v)
{
    for (int i = 0; i < 4; ++i, p += 1024, v *= 2.0f)
        StoreFour(p + 4 * threadIdx.x, v + (float)threadIdx.x, 1);
}
__global__ void Eights(_Float16 *p, Words4 v)
{
    for (int i = 0; i < 4; ++i, p += 1024, v *= 3u)
        StoreEight(p + 8 * threadIdx.x, v + threadIdx.x, true, 1);
}
""")
    r = subprocess.run([build.HIPCC] + build.FLAGS + ["--cuda-device-only", "-S", str(source), "-o", str(listing)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    code = [l.split(";")[0].split() for l in listing.read_text().split("\n")]
    code = [w for w in code if w and not w[0].startswith(".") and not w[0].endswith(":")]
    stores = [i for i, w in enumerate(code) if w[0] == "global_store_dwordx4" and "sc1" in w]
    assert len(stores) == 8
    for i in stores:
        waited = 0
        for w in code[i + 1:]:
            if w[0].startswith("v_") or waited >= 2:
                break
            waited += int(w[1]) + 1 if w[0] == "s_nop" else 1
        assert waited >= 2, code[i:i + 4]


def test_mx_tile_of_three_blocks_a_wave_is_refused(tmp_path):
    """The bf16 way out of the k-split MX kernels stores whole blocks of a wave, or half of its only one: a shape with three is a compile error
    (it would store a third of its columns, and at the wrong place)."""
    build = importlib.util.module_from_spec(importlib.util.spec_from_file_location("pto_amd_build", os.path.join(os.path.dirname(capi.LIB_PATH), "build.py")))
    build.__spec__.loader.exec_module(build)
    for bn, fine in ((128, True), (192, False)):
        source = tmp_path / ("shape%d.hip" % bn)
        source.write_text("""#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_mxks.hpp"
int Launch(void *c, const uint8_t *x) { return launch_gemm_mxks<0, 0, bfloat16_t, 64, %d, 3, 2>(nullptr, c, x, x, x, x, 64, 192, 512); }
""" % bn)
        r = subprocess.run([build.HIPCC] + build.FLAGS + ["--cuda-device-only", "-fsyntax-only", str(source)], capture_output=True, text=True)
        assert (r.returncode == 0) == fine and fine == ("half of the only one" not in r.stderr), r.stderr
