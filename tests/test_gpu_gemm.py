"""GPU parity of the PTO GEMM path (TLOAD -> TEXTRACT -> TMATMUL -> TSTORE) through the C ABI.

Bar: max |gpu - ref| <= 2e-3 * max|ref| against an fp32-accumulated reference (the oracle, which
restates the reference's CPU-simulation arithmetic); integer-valued inputs must match exactly."""
import numpy as np
import pytest
import torch

from pto_amd import capi, datagen

pytestmark = pytest.mark.gpu

TOL = 2e-3   # stated by the task: max relative error against an fp32-accumulated reference


def rel_err(got, want):
    return float(np.max(np.abs(got - want)) / np.max(np.abs(want)))


@pytest.mark.parametrize("m,n,k", [(128, 256, 32), (128, 256, 64), (128, 256, 96), (256, 512, 256), (384, 256, 1024),
                                   (4096, 4096, 256), (4096, 4352, 384), (4352, 4096, 128)])
def test_gemm_small_vs_oracle(oracle, m, n, k):
    from gpu_util import gemm
    a, b = datagen.gemm_inputs(m, n, k)
    got = gemm(a, b)
    want = oracle.gemm_f16f32(a, b, base_k=64)
    assert rel_err(got, want) <= TOL
    # element-wise relative error where the reference is not tiny
    big = np.abs(want) > 0.05 * np.max(np.abs(want))
    assert np.max(np.abs(got - want)[big] / np.abs(want)[big]) <= TOL


def test_gemm_every_dispatch_path_agrees_with_integer_reference():
    """4096 x 4096 selects the four-wave kernel with 256 x 256 tiles, 4096 x 4224 and 4224 x 4224 (rows not a multiple of
    256: the last tile row is moved back) the same kernel with 256 x 192 tiles, 3072 x 3072 its 192 x 192 tiles,
    1024 x 1024 its 192 x 128 tiles; a K extent that is no multiple of 128 (1024 x 1024 x 96) and fewer than 192 rows
    (128 x 512) the 128 x 256-block kernel: all exact on integer inputs."""
    from gpu_util import gemm
    for m, n, k in ((4096, 4096, 512), (4096, 4224, 512), (4224, 4224, 512), (3072, 3072, 512), (1024, 1024, 512),
                    (1024, 1024, 96), (128, 512, 256)):
        a, b = datagen.gemm_inputs_integer(m, n, k)
        got = gemm(a, b)
        rows = np.r_[0:64, m // 2:m // 2 + 64, m - 64:m]
        want = (a[rows].astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
        assert np.array_equal(got[rows], want), (m, n, k)
        colsum = b.astype(np.float64).sum(axis=0)
        assert np.array_equal(got.astype(np.float64).sum(axis=1), a.astype(np.float64) @ colsum)


def test_gemm_four_wave_tile_widths_exact():
    """Every tile shape of the four-wave kernel (tuning hook: 256 or 192 rows x 256 / 192 / 128 columns) on integer inputs, the whole
    matrix exactly, with K extents of whole groups of six K-steps (384, 768), of groups plus two or four steps (512, 640,
    1152 + 128) and of a tail alone (128, 256); one tile and several; and the shapes that the kernel refuses."""
    import torch
    from gpu_util import to_dev
    fn = capi.load_st().pto_gemm_f16f32_w4_variant
    for m, n, k in ((256, 768, 128), (512, 768, 256), (768, 1536, 384), (256, 768, 512), (1024, 768, 640), (512, 1536, 768),
                    (768, 768, 1280), (2560, 3072, 384)):
        a, b = datagen.gemm_inputs_integer(m, n, k)
        want = (a.astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
        ta, tb = to_dev(a), to_dev(b)
        for variant in range(6):
            tc = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
            capi.check(fn(0, tc.data_ptr(), ta.data_ptr(), tb.data_ptr(), m, n, k, variant), "four-wave GEMM shape %d" % variant)
            torch.cuda.synchronize()
            assert np.array_equal(tc.cpu().numpy(), want), (m, n, k, variant)
    p = ta.data_ptr()
    assert fn(0, p, p, p, 256, 768, 192, 0) == capi.ERR_UNSUPPORTED      # k not a multiple of 128
    assert fn(0, p, p, p, 192, 768, 256, 0) == capi.ERR_UNSUPPORTED      # fewer rows than a tile
    assert fn(0, p, p, p, 128, 768, 256, 4) == capi.ERR_UNSUPPORTED
    assert fn(0, p, p, p, 256, 160, 256, 1) == capi.ERR_UNSUPPORTED      # fewer columns than the width
    assert fn(0, p, p, p, 256, 770, 256, 1) == capi.ERR_UNSUPPORTED      # rows of C not a multiple of 16 bytes


@pytest.mark.parametrize("variant,bm,bn", [(0, 32, 64), (1, 64, 64), (2, 64, 96), (3, 128, 64), (4, 128, 96), (5, 128, 128), (6, 192, 128),
                                           (7, 256, 128), (8, 192, 192)])
def test_gemm_k_split_tile_shapes_exact(variant, bm, bn):
    """Every tile shape of the kernel that splits k over two groups of wavefronts, integer inputs, the whole matrix exactly:
    less than a tile, one tile, edges one row / four columns past a tile, several tile rows and columns; one K-step, an odd
    and an even number of them, a last half step (k % 64 == 32) alone and behind whole ones.  Nothing outside C is written."""
    import torch
    from gpu_util import to_dev
    fn = capi.load_st().pto_gemm_f16f32_ks_variant
    for m, n, k in ((1, 4, 32), (bm, bn, 64), (bm + 1, bn + 4, 96), (bm - 1, bn - 4, 128), (3 * bm + 5, 2 * bn + 12, 192), (2 * bm, 9 * bn, 352),
                    (9 * bm - 7, bn, 448)):
        a, b = datagen.gemm_inputs_integer(m, n, k)
        want = (a.astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
        ta, tb = to_dev(a), to_dev(b)
        guarded = torch.full((m * n + 512,), -1.0, dtype=torch.float32, device="cuda:0")
        capi.check(fn(0, guarded.data_ptr() + 1024, ta.data_ptr(), tb.data_ptr(), m, n, k, variant), "k-split GEMM shape %d" % variant)
        torch.cuda.synchronize()
        got = guarded.cpu().numpy()
        assert np.array_equal(got[256:256 + m * n].reshape(m, n), want), (m, n, k)
        assert (got[:256] == -1.0).all() and (got[256 + m * n:] == -1.0).all(), (m, n, k)


def test_gemm_k_split_element_alignment():
    """C one element past a 16-byte boundary, every shape of the k-split kernel and the entry point."""
    import torch
    from gpu_util import to_dev
    m, n, k = 256, 512, 96
    a, b = datagen.gemm_inputs_integer(m, n, k)
    want = (a.astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
    ta, tb = to_dev(a), to_dev(b)
    lib = capi.load_st()
    for variant in range(-1, 9):
        guarded = torch.full((m * n + 64,), -1.0, dtype=torch.float32, device="cuda:0")
        args = (0, guarded.data_ptr() + 4, ta.data_ptr(), tb.data_ptr(), m, n, k)
        capi.check(lib.pto_gemm_f16f32(*args) if variant < 0 else lib.pto_gemm_f16f32_ks_variant(*args, variant), "shape %d" % variant)
        torch.cuda.synchronize()
        got = guarded.cpu().numpy()
        assert np.array_equal(got[1:1 + m * n].reshape(m, n), want), variant
        assert got[0] == -1.0 and (got[1 + m * n:] == -1.0).all(), variant


def test_gemm_ragged_m_and_n_exact():
    """Extents that the tiles do not divide: the last tile row / column is moved back to end with the matrix.  Integer
    operands, every element exact: each width of the four-wave kernel on small shapes (one tile that is also the moved
    one, several, m or n alone ragged), then 6000 x 6100 x 6144 through the public entry point."""
    import torch
    from gpu_util import to_dev, stream
    fn = capi.load_st().pto_gemm_f16f32_w4_variant
    for m, n, k in ((300, 772, 256), (256, 260, 128), (1000, 1100, 384), (512, 1000, 640), (777, 768, 256)):
        a, b = datagen.gemm_inputs_integer(m, n, k)
        want = (a.astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
        ta, tb = to_dev(a), to_dev(b)
        for variant in range(6):
            tc = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
            capi.check(fn(0, tc.data_ptr(), ta.data_ptr(), tb.data_ptr(), m, n, k, variant), "four-wave GEMM shape %d" % variant)
            torch.cuda.synchronize()
            assert np.array_equal(tc.cpu().numpy(), want), (m, n, k, variant)
    lib = capi.load()
    for m, n, k in ((6000, 6100, 6144), (300, 772, 256)):   # the second: too small for the size rule, taken because nothing else fits
        a, b = datagen.gemm_inputs_integer(m, n, k)
        ta, tb = to_dev(a), to_dev(b)
        tc = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        capi.check(lib.pto_gemm_f16f32(stream(), tc.data_ptr(), ta.data_ptr(), tb.data_ptr(), m, n, k), "pto_gemm_f16f32")
        torch.cuda.synchronize()
        want = ta.view(torch.float16).double() @ tb.view(torch.float16).double().T
        assert torch.equal(tc.double(), want), (m, n, k)


def test_gemm_6144_every_element_exact():
    """The headline problem through the public entry point (it selects the four-wave kernel with 256 x 192 tiles) on integer operands in
    [1, 5): all 6144 x 6144 sums (at most 16 * 6144 < 2^24) are exact in fp32, so every element must equal the product
    taken in float64 by the BLAS behind torch (an independent code path)."""
    import torch
    from gpu_util import to_dev, stream
    lib = capi.load()
    m = n = k = 6144
    a, b = datagen.gemm_inputs_integer(m, n, k)
    ta, tb = to_dev(a), to_dev(b)
    tc = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
    capi.check(lib.pto_gemm_f16f32(stream(), tc.data_ptr(), ta.data_ptr(), tb.data_ptr(), m, n, k), "pto_gemm_f16f32")
    torch.cuda.synchronize()
    want = ta.view(torch.float16).double() @ tb.view(torch.float16).double().T
    assert torch.equal(tc.double(), want)
    # and the float64 product itself against int64 numpy on a band of rows
    rows = np.r_[0:8, 3000:3008, 6136:6144]
    assert np.array_equal(want[rows].cpu().numpy(), (a[rows].astype(np.int64) @ b.astype(np.int64).T).astype(np.float64))


def test_gemm_integer_inputs_exact(oracle):
    """Integer operands in [1,5): every partial sum is exact in fp32 whatever the summation order, so a
    wrong fragment layout, a dropped K step or a transposed operand cannot hide inside a tolerance."""
    from gpu_util import gemm
    a, b = datagen.gemm_inputs_integer(256, 512, 512)
    got = gemm(a, b)
    want = (a.astype(np.int64) @ b.astype(np.int64).T).astype(np.float32)
    assert np.array_equal(got, want)
    assert np.array_equal(got, oracle.gemm_f16f32(a, b, base_k=64))


def test_gemm_golden_fixture():
    """Committed output of the compiled reference on the seeded 128x512x128... the GPU tile is 128x256,
    so use the 128 x 64 x 256 fixture (one K step)."""
    import os
    from gpu_util import gemm
    G = np.load(os.path.join(os.path.dirname(__file__), "golden", "ref_vectors.npz"))
    a, b = datagen.gemm_inputs(128, 256, 64)
    assert rel_err(gemm(a, b), G["gemm_128x64x256_ks64"]) <= TOL


def test_gemm_1536_single_tile_config(oracle):
    """Config 1: C[1536,1536] = A x B, uniform[-1,1] fp16 from seed; oracle = one TMATMUL with K = 1536
    on a sample of rows (the full product takes the CPU path seconds), plus linearity over all rows."""
    from gpu_util import gemm
    a, b = datagen.gemm_inputs(1536, 1536, 1536)
    got = gemm(a, b)
    want = oracle.gemm_f16f32(a, b, base_k=1536, row0=640, row1=768)
    assert rel_err(got[640:768], want[640:768]) <= TOL
    want64 = a[:64].astype(np.float64) @ b.astype(np.float64).T
    assert rel_err(got[:64], want64) <= TOL


@pytest.mark.parametrize("size", [3072, 6144, 7680])
def test_gemm_full_size_properties(oracle, size):
    """Config 2 at full size.  Size-independent checks: a sampled set of rows against the oracle, and
    exactness on integer inputs through a checksum identity: sum_j C[i,j] = A[i,:] . (sum_j B[j,:])."""
    from gpu_util import gemm
    a, b = datagen.gemm_inputs(size, size, size)
    got = gemm(a, b)
    rows = [0, 127, 128, size // 2 + 5, size - 1]
    for r in rows:
        want = a[r].astype(np.float64) @ b.astype(np.float64).T
        assert np.max(np.abs(got[r] - want)) <= TOL * np.max(np.abs(want))
        big = np.abs(want) > 0.05 * np.max(np.abs(want))  # element by element where the reference is not tiny
        assert np.max(np.abs(got[r] - want)[big] / np.abs(want)[big]) <= TOL
    want = oracle.gemm_f16f32(a, b, base_k=64, row0=256, row1=264)
    assert rel_err(got[256:264], want[256:264]) <= TOL
    big = np.abs(want[256:264]) > 0.05 * np.max(np.abs(want[256:264]))
    assert np.max(np.abs(got[256:264] - want[256:264])[big] / np.abs(want[256:264])[big]) <= TOL
    ai, bi = datagen.gemm_inputs_integer(size, size, size)
    goti = gemm(ai, bi)
    colsum = bi.astype(np.float64).sum(axis=0)
    assert np.array_equal(goti.astype(np.float64).sum(axis=1), ai.astype(np.float64) @ colsum)
    assert np.array_equal(goti[size - 1], (ai[size - 1].astype(np.int64) @ bi.astype(np.int64).T).astype(np.float32))


def test_gemm_rejects_bad_shapes():
    import torch
    lib = capi.load()
    t = torch.zeros(16, device="cuda:0")
    p = t.data_ptr()
    assert lib.pto_gemm_f16f32(0, p, p, p, 100, 256, 64) == capi.ERR_UNSUPPORTED
    assert lib.pto_gemm_f16f32(0, p, p, p, 128, 256, 16) == capi.ERR_UNSUPPORTED
    assert lib.pto_gemm_f16f32(0, 0, p, p, 128, 256, 64) == capi.ERR_BAD_ARG
    assert lib.pto_gemm_f16f32(0, p, p, p, 0, 256, 64) == capi.ERR_BAD_ARG


@pytest.mark.parametrize("m,n,k,shift", [(256, 512, 256, 0), (256, 512, 256, 4), (256, 520, 256, 0), (256, 520, 256, 4), (250, 516, 256, 0), (1024, 3072, 128, 0),
                                         (1024, 3072, 128, 1), (1024, 3080, 128, 0), (6144, 4096, 128, 0), (6145, 4096, 128, 0)])
def test_gemm_results_past_the_l2(m, n, k, shift):
    """Whole and half 64-byte pieces of C, a C that begins `shift` elements past them, and both sides of the largest C that goes
    past the L2: whole numbers, exact; nothing outside C is written."""
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(m + n)
    a, b = (torch.randint(-4, 5, (r, k), generator=g, device="cuda:0").half() for r in (m, n))
    c = torch.full((m * n + 64,), 7.0, device="cuda:0")
    for _ in range(2):
        capi.check(lib.pto_gemm_f16f32(torch.cuda.current_stream().cuda_stream, c.data_ptr() + 4 * shift, a.data_ptr(), b.data_ptr(), m, n, k),
                   "pto_gemm_f16f32")
    want = a.float() @ b.float().t()
    assert torch.equal(c[shift:shift + m * n].view(m, n), want)
    assert (c[:shift] == 7.0).all() and (c[shift + m * n:] == 7.0).all()


@pytest.mark.parametrize("m,n,k", [(250, 520, 1280), (250, 520, 1408), (1000, 3000, 1280), (1000, 3000, 1408)])
def test_gemm_half_pieces_and_k(m, n, k):
    """Half 64-byte pieces of C on both sides of the longest k at which they go past the L2: whole numbers, exact."""
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(k)
    a, b = (torch.randint(-4, 5, (r, k), generator=g, device="cuda:0").half() for r in (m, n))
    c = torch.full((m * n + 64,), 7.0, device="cuda:0")
    capi.check(lib.pto_gemm_f16f32(torch.cuda.current_stream().cuda_stream, c.data_ptr(), a.data_ptr(), b.data_ptr(), m, n, k), "pto_gemm_f16f32")
    assert torch.equal(c[:m * n].view(m, n), a.float() @ b.float().t()) and (c[m * n:] == 7.0).all()


def test_gemm_32x32_tiles_exact():
    """The tile of one block a wave, as the other shapes are tested; then the entry point on both sides of a whole round of such tiles, k of one step and of more and
    fewer than the ring has stages."""
    test_gemm_k_split_tile_shapes_exact(9, 32, 32)
    lib = capi.load()
    for m, n, k in ((512, 512, 128), (513, 512, 128), (512, 516, 256), (192, 128, 384), (250, 260, 512), (192, 1364, 640), (128, 256, 32), (128, 2048, 96)):
        g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
        a, b = (torch.randint(-4, 5, (r, k), generator=g, device="cuda:0").half() for r in (m, n))
        c = torch.full((m * n + 64,), 7.0, device="cuda:0")
        capi.check(lib.pto_gemm_f16f32(torch.cuda.current_stream().cuda_stream, c.data_ptr(), a.data_ptr(), b.data_ptr(), m, n, k), "pto_gemm_f16f32")
        assert torch.equal(c[:m * n].view(m, n), a.float() @ b.float().t()) and (c[m * n:] == 7.0).all(), (m, n, k)
