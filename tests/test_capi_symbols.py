"""The C-ABI library loads and exports every symbol that include/pto_amd.h declares (no GPU needed)."""
import os
import re

from pto_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "pto_amd.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(pto_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations parsed"
    lib = capi.load()
    for name in sorted(declared):
        assert hasattr(lib, name), name
    assert declared == set(capi.SYMBOLS), declared ^ set(capi.SYMBOLS)


def test_product_library_holds_no_test_entry_points():
    """Single-tile test programs and tuning hooks live in libpto_st.so (include/pto_amd_st.h) only."""
    import subprocess
    names = subprocess.run(["nm", "-D", "--defined-only", capi.LIB_PATH], capture_output=True, text=True, check=True).stdout
    exported = set(re.findall(r"\b(pto_[a-z0-9_]+)$", names, flags=re.M))
    assert exported == set(capi.SYMBOLS), exported ^ set(capi.SYMBOLS)


def test_test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "pto_amd_st.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(pto_[a-z0-9_]+)\s*\(", header))
    lib = capi.load_st()
    for name in sorted(declared):
        assert hasattr(lib, name), name
    assert declared == set(capi.ST_SYMBOLS), declared ^ set(capi.ST_SYMBOLS)


def test_argument_validation_needs_no_gpu():
    lib = capi.load()
    assert lib.pto_gemm_f16f32(0, 0, 0, 0, 128, 256, 64) == capi.ERR_BAD_ARG
    assert lib.pto_tcvt_f32_f16(0, 0, 0, 0, capi.CAST_RINT) == capi.OK          # empty input: nothing to do
    assert lib.pto_gather_rows(0, 0, 0, 0, 0, 0, 0, 2) == capi.OK
    assert lib.pto_version().startswith(b"pto-amd")


def test_gemm_choice_of_a_shape():
    """The shape that the fp16 product takes is the one of the shortest expected time, whatever is left out on the way to it; few tiles: 32 x 32 ones."""
    import ctypes
    import random
    lib, rng, times = capi.load_st(), random.Random(5), (ctypes.c_double * 17)()
    for _ in range(4000):
        m, n, k = (rng.randint(1, 24 if rng.random() < 0.7 else 80) * step for step in (128, 256, 32))
        if rng.random() < 0.5:  # any rows and columns from 192 and 128 on
            m, n, k = m + rng.randint(64, 191), n - 4 * rng.randint(0, 31), (k + 127) // 128 * 128
        units = rng.choice((64, 256, 304))
        shape = lib.pto_gemm_f16f32_choice(m, n, k, units, times)
        assert 0 <= shape < 17 and times[shape] == min(times), (m, n, k, units)
        assert shape == lib.pto_gemm_f16f32_choice(m, n, k, units, None)
    for m, n, k in ((512, 512, 512), (192, 128, 128), (256, 256, 6144)):
        assert lib.pto_gemm_f16f32_choice(m, n, k, 256, None) == 0
    assert lib.pto_gemm_f16f32_choice(191, 128, 128, 256, None) == capi.ERR_UNSUPPORTED


def test_mx_gemm_choice_of_a_shape():
    """As above: the shortest expected time of all variants, whatever is left out on the way to it."""
    import ctypes
    import random
    lib, rng, times = capi.load_st(), random.Random(7), (ctypes.c_double * 19)()
    seen = set()
    for _ in range(6000):
        top = rng.choice((1000, 6000, 12000))
        m, n, k = rng.randint(256, top), rng.randint(64, top // 4) * 4 + rng.choice((0, 0, 0, 1)), 1024 * rng.randint(1, 8)
        fmt, fp32, units = rng.choice((0, 4)), rng.randint(0, 1), rng.choice((64, 256, 304))
        variant = lib.pto_gemm_mx_choice(m, n, k, fmt, fp32, units, times)
        assert 0 <= variant < 19 and times[variant] == min(times) < float("inf"), (m, n, k, fmt, fp32, units)
        assert variant == lib.pto_gemm_mx_choice(m, n, k, fmt, fp32, units, None)
        seen.add((fmt, variant))
    assert seen >= {(fmt, variant) for fmt in (0, 4) for variant in (1, 5, 6, 7, 8, 10, 13, 14, 15, 16, 17, 18)}, seen
    assert lib.pto_gemm_mx_choice(255, 256, 1024, 0, 1, 256, None) == capi.ERR_UNSUPPORTED
