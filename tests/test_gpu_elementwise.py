"""GPU parity of TCVT and the gathers through the C ABI: bit-exact against the oracle."""
import os

import numpy as np
import pytest
import torch

from pto_amd import capi, datagen

pytestmark = pytest.mark.gpu


def boundary_patterns():
    exps = np.arange(0, 256, dtype=np.uint32) << 23
    mants = np.array([0, 1, 0xfff, 0x1000, 0x1001, 0x1fff, 0x2000, 0x2001, 0x2fff, 0x3000, 0x3001, 0x7fe000, 0x7fefff,
                      0x7ff000, 0x7ff001, 0x7fffff, 0x400000, 0x3fffff, 0x400001, 0x200000, 0x600000, 0x100000,
                      0x080000, 0x7fc000, 0x7f8000, 0x7fff, 0x8000, 0x8001, 0x17fff, 0x18000, 0x18001], dtype=np.uint32)
    pos = (exps[:, None] | mants[None, :]).reshape(-1)
    return np.concatenate([pos, pos | np.uint32(0x80000000)])


def test_tcvt_f16_boundaries_and_strided_sweep(oracle):
    """Every exponent x mantissa pattern around the fp16 rounding boundaries (NaN payloads, +-inf,
    overflow at 65520, subnormal results, ties) and a 2^32 / 1021 strided sweep."""
    from gpu_util import tcvt
    bits = np.concatenate([boundary_patterns(), np.arange(0, 2**32, 1021, dtype=np.uint64).astype(np.uint32)])
    x = bits.view(np.float32)
    assert np.array_equal(tcvt(x, "f16"), oracle.tcvt_f32_f16(x))


def test_tcvt_bf16_boundaries_and_strided_sweep(oracle):
    from gpu_util import tcvt
    bits = np.concatenate([boundary_patterns(), np.arange(0, 2**32, 1021, dtype=np.uint64).astype(np.uint32)])
    x = bits.view(np.float32)
    got = tcvt(x, "bf16")
    assert np.array_equal(got, oracle.tcvt_f32_bf16(x))
    nan = np.isnan(x)
    want = torch.from_numpy(x.copy()).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
    assert np.array_equal(got[~nan], want[~nan])


def test_bf16_of_two_floats_is_the_closed_form():
    """The hardware conversion by which the MX GEMMs store bf16: the bits of the closed form (pinned above) for every float, ties, subnormals, the edge to
    infinity, infinities and NaNs among them, in either half of the pair."""
    out = torch.zeros(2, dtype=torch.int32, device="cuda:0")
    capi.check(capi.load_st().pto_st_bf16_pairs(torch.cuda.current_stream().cuda_stream, out.data_ptr()), "pto_st_bf16_pairs")
    wrong, one = out.cpu().numpy().view(np.uint32)
    assert wrong == 0, hex(one)


@pytest.mark.parametrize("n", [0, 1, 7, 8, 8191, 8192, 8193, 3 * 8192 + 5])
def test_tcvt_ragged_sizes(oracle, n):
    from gpu_util import tcvt
    x = datagen.tcvt_input(1, max(n, 8), inject=0.05).reshape(-1)[:n]
    assert np.array_equal(tcvt(x, "f16"), oracle.tcvt_f32_f16(x))
    assert np.array_equal(tcvt(x, "bf16"), oracle.tcvt_f32_bf16(x))


def test_tcvt_golden_fixture():
    from gpu_util import tcvt
    G = np.load(os.path.join(os.path.dirname(__file__), "golden", "ref_vectors.npz"))
    x = datagen.tcvt_input(64, 256, inject=0.05).reshape(-1)
    assert np.array_equal(tcvt(x, "f16"), G["tcvt_f32_f16_64x256"])


def test_tcvt_round_modes(oracle):
    """CAST_ROUND (ties away) against the oracle's ties-away conversion; directed modes against
    numpy's nextafter-based definition on finite inputs."""
    from gpu_util import tcvt
    bits = np.concatenate([boundary_patterns(), np.arange(0, 2**32, 65521, dtype=np.uint64).astype(np.uint32)])
    x = bits.view(np.float32)
    got = tcvt(x, "f16", capi.CAST_ROUND)
    want = np.array([oracle.lib().po_f32_to_f16_rna(int(b)) for b in bits[:20000]], dtype=np.uint16)
    assert np.array_equal(got[:20000], want)
    fin = np.isfinite(x) & (np.abs(x) < 65504)
    xf = x[fin].astype(np.float64)
    for mode, pred in ((capi.CAST_FLOOR, lambda h: h <= xf), (capi.CAST_CEIL, lambda h: h >= xf),
                       (capi.CAST_TRUNC, lambda h: np.abs(h) <= np.abs(xf))):
        h = tcvt(x, "f16", mode)[fin].view(np.float16).astype(np.float64)
        assert np.all(pred(h))
        assert np.all(np.abs(h - xf) <= np.maximum(np.abs(xf) * 2.0**-10, 2.0**-24))   # within one fp16 ulp


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 2048, 2051, 4096, 4101, 3 * 4096 + 1021])
def test_tcvt_streaming_and_tile_forms_agree(n):
    """Buffers aligned to 16 / 8 bytes take the streaming kernel, others the tile form: the same bits in every mode, whole
    pieces, their edges and the rest behind them; nothing written behind the last element."""
    from gpu_util import to_dev
    lib = capi.load()
    x = datagen.tcvt_input(1, n + 8, inject=0.05).reshape(-1)[:n]
    src = torch.zeros(n + 1, dtype=torch.float32, device="cuda:0")
    tx = to_dev(x)
    src[1:] = tx                                      # 4 bytes off: not aligned
    for fn, modes in ((lib.pto_tcvt_f32_f16, range(capi.CAST_RINT, capi.CAST_ODD + 1)), (lib.pto_tcvt_f32_bf16, (capi.CAST_RINT,))):
        for mode in modes:
            a, b = (torch.full((n + 16,), 0x5a5a, dtype=torch.int16, device="cuda:0") for _ in range(2))
            capi.check(fn(0, a.data_ptr(), tx.data_ptr(), n, mode), "aligned")
            capi.check(fn(0, b.data_ptr(), src.data_ptr() + 4, n, mode), "not aligned")
            torch.cuda.synchronize()
            assert torch.equal(a, b), (n, mode)
            assert (a[n:] == 0x5a5a).all() and (b[n:] == 0x5a5a).all(), (n, mode)


@pytest.mark.parametrize("n", [(1 << 24) - 1, 1 << 24, (1 << 24) + 2047, (1 << 24) + 2051])
def test_tcvt_f16_loads_per_lane(n):
    """Both sides of the size from which a lane has two loads in flight, whole and partial last pieces: the bits of the tile
    form, nothing written behind the last element."""
    lib = capi.load()
    memory = torch.empty(n + 1, device="cuda:0").normal_()
    memory[::1001] = float("nan")
    x = memory[1:].clone()
    a, b = (torch.full((n + 16,), 0x5a5a, dtype=torch.int16, device="cuda:0") for _ in range(2))
    capi.check(lib.pto_tcvt_f32_f16(0, a.data_ptr(), x.data_ptr(), n, capi.CAST_RINT), "aligned")
    capi.check(lib.pto_tcvt_f32_f16(0, b.data_ptr(), memory.data_ptr() + 4, n, capi.CAST_RINT), "tile form")
    torch.cuda.synchronize()
    assert torch.equal(a, b) and (a[n:] == 0x5a5a).all()


def test_tcvt_full_size_config(oracle):
    """Config 5 at full size 16384 x 8192 with 0.1% special values: compared in slabs against the oracle."""
    from gpu_util import to_dev, stream
    lib = capi.load()
    x = datagen.tcvt_input(16384, 8192)
    tx = to_dev(x.reshape(-1))
    for kind, fn, ofn in (("f16", lib.pto_tcvt_f32_f16, oracle.tcvt_f32_f16), ("bf16", lib.pto_tcvt_f32_bf16, oracle.tcvt_f32_bf16)):
        th = torch.zeros(x.size, dtype=torch.int16, device="cuda:0")
        capi.check(fn(stream(), th.data_ptr(), tx.data_ptr(), x.size, capi.CAST_RINT), kind)
        torch.cuda.synchronize()
        got = th.cpu().numpy().view(np.uint16).reshape(16384, 8192)
        for r0 in range(0, 16384, 2048):
            assert np.array_equal(got[r0:r0 + 2048], ofn(x[r0:r0 + 2048])), (kind, r0)


@pytest.mark.parametrize("rows,cols,nidx", [(64, 1024, 100), (16, 8, 1), (33, 264, 70), (128, 256, 32), (50, 2048, 31)])
def test_gather_rows_small(oracle, rows, cols, nidx):
    from gpu_util import gather_rows
    table, idx = datagen.gather_inputs(rows, cols, nidx)
    assert np.array_equal(gather_rows(table, idx), oracle.gather_rows(table, idx))
    t32 = np.random.default_rng(1).integers(0, 2**32, size=(rows, cols), dtype=np.uint64).astype(np.uint32)
    assert np.array_equal(gather_rows(t32, idx), oracle.gather_rows(t32, idx))


def test_gather_rows_out_of_range_indices_give_zero_rows(oracle):
    from gpu_util import gather_rows
    table, _ = datagen.gather_inputs(64, 512, 8)
    idx = np.array([0, 63, -1, 64, 5, 2**31 - 1, -2**31, 7], dtype=np.int32)
    got = gather_rows(table, idx)
    assert np.array_equal(got, oracle.gather_rows(table, idx))
    assert not got[2].any() and not got[3].any() and np.array_equal(got[4], table[5])


@pytest.mark.parametrize("rows,cols,nidx", [(3, 8, 1), (5, 24, 700), (700, 40, 131), (1024, 1024, 2048), (1500, 1032, 3001), (2048, 2048, 4096), (3000, 1024, 6001),
                                            (9000, 1024, 18001)])
def test_gather_rows_widths_and_slices(oracle, rows, cols, nidx):
    """Rows narrower than a wave's accesses and rows that no power of two divides; tables that are cut into 1, 2, 4 and 8
    slices (read twice or more, larger than 2 / 4 / 8 MiB) with a last workgroup that is partly full, both element sizes."""
    from gpu_util import gather_rows
    table, idx = datagen.gather_inputs(rows, cols, nidx)
    idx = idx.copy()
    idx[::17] = -1 - idx[::17]
    idx[5::31] = rows
    assert np.array_equal(gather_rows(table, idx), oracle.gather_rows(table, idx))
    t32 = np.random.default_rng(1).integers(0, 2**32, size=(rows, cols), dtype=np.uint64).astype(np.uint32)
    assert np.array_equal(gather_rows(t32, idx), oracle.gather_rows(t32, idx))


@pytest.mark.parametrize("rows,cols,nidx", [(600, 2848, 1201), (1972, 2848, 4001), (1100, 1920, 2300), (4096, 448, 9000), (2300, 864, 5001), (8192, 64, 17000),
                                            (700, 8000, 1401)])
def test_gather_rows_unequal_slices(oracle, rows, cols, nidx):
    """Rows of whole lines or half lines that the slices do not divide: a last slice with fewer chunks, two to eight slices."""
    from gpu_util import gather_rows
    table, idx = datagen.gather_inputs(rows, cols, nidx)
    idx = idx.copy()
    idx[::19] = -5
    idx[7::41] = rows + 3
    assert np.array_equal(gather_rows(table, idx), oracle.gather_rows(table, idx))
    t32 = np.random.default_rng(2).integers(0, 2**32, size=(rows, cols // 2), dtype=np.uint64).astype(np.uint32)
    assert np.array_equal(gather_rows(t32, idx), oracle.gather_rows(t32, idx))


@pytest.mark.parametrize("rows,cols,nidx", [(2048, 264, 16384), (4200, 328, 17001), (2000, 536, 8203), (1600, 584, 7333), (900, 1032, 4099), (900, 1048, 4101), (300, 4008, 1203),
                                            (77, 8184, 523)])
def test_gather_rows_in_pieces_of_the_output(oracle, rows, cols, nidx):
    """Rows of no whole number of 64 bytes, read four times and more: two to eight slices, with one, two or three chunks past a piece; widths on both sides of
    where the number of slices changes; indices outside the table; and into an output that begins in the middle of a piece, which stays whole."""
    from gpu_util import gather_rows
    for name, dtype, width in (("half", np.uint16, cols), ("float", np.uint32, cols - 8 * (cols > 264))):
        r = np.random.default_rng(cols)
        table = r.integers(0, np.iinfo(dtype).max, size=(rows, width), dtype=dtype)
        idx = r.integers(0, rows, size=nidx).astype(np.int32)
        idx[::17] = -1 - idx[::17]
        idx[5::31] = rows
        want = oracle.gather_rows(table, idx)
        assert np.array_equal(gather_rows(table, idx), want), name
        view = {2: np.int16, 4: np.int32}[table.itemsize]
        tt, ti = torch.from_numpy(table.view(view)).to("cuda:0"), torch.from_numpy(idx).to("cuda:0")
        for shift in (0, 32 // table.itemsize):
            out = torch.full((nidx * width + 128,), 77, dtype=tt.dtype, device="cuda:0")
            capi.check(capi.load().pto_gather_rows(torch.cuda.current_stream().cuda_stream, out.data_ptr() + shift * table.itemsize, tt.data_ptr(), ti.data_ptr(),
                                                   nidx, rows, width, table.itemsize), "pto_gather_rows")
            got = out.cpu().numpy()
            assert np.array_equal(got[shift:shift + nidx * width].view(dtype).reshape(nidx, width), want), (name, shift)
            assert (got[:shift] == 77).all() and (got[shift + nidx * width:] == 77).all()


@pytest.mark.parametrize("rows,cols,nidx", [(3850, 520, 61601), (2560, 760, 40961), (2530, 776, 40481), (1290, 1544, 20641), (1290, 1544, 20639), (2100, 1032, 14501), (2100, 1016, 14701), (1020, 1928, 7621),
                                            (1100, 2056, 7142), (600, 3592, 4101), (270, 8008, 1841)])
def test_gather_rows_in_pieces_of_large_tables(oracle, rows, cols, nidx):
    """Tables that no XCD's L2 holds, read sixteen times and more (two, four and eight slices of 24 chunks and more) or less (four of 32 and more, eight of 56 and more), widths on both
    sides of where the number of slices changes; indices outside the table; nothing around the output, which begins at a piece or in one."""
    r = np.random.default_rng(cols)
    table = r.integers(0, 1 << 16, size=(rows, cols), dtype=np.uint16)
    idx = r.integers(0, rows, size=nidx).astype(np.int32)
    idx[::17] = -1 - idx[::17]
    idx[5::31] = rows
    want = oracle.gather_rows(table, idx)
    tt, ti = torch.from_numpy(table.view(np.int16)).to("cuda:0"), torch.from_numpy(idx).to("cuda:0")
    for shift in (0, 32, 8):
        out = torch.full((nidx * cols + 128,), 77, dtype=tt.dtype, device="cuda:0")
        capi.check(capi.load().pto_gather_rows(torch.cuda.current_stream().cuda_stream, out.data_ptr() + shift * 2, tt.data_ptr(), ti.data_ptr(), nidx, rows, cols, 2),
                   "pto_gather_rows")
        got = out.cpu().numpy()
        assert np.array_equal(got[shift:shift + nidx * cols].view(np.uint16).reshape(nidx, cols), want), shift
        assert (got[:shift] == 77).all() and (got[shift + nidx * cols:] == 77).all()


@pytest.mark.parametrize("rows,cols,nidx", [(5, 24, 700), (1500, 1032, 3001), (3000, 1024, 6001)])
@pytest.mark.parametrize("dtype", [torch.int16, torch.int32])
def test_gather_rows_element_alignment(rows, cols, nidx, dtype):
    """Table and output one element past a 16-byte boundary, one and several slices: the rows, and nothing around the output."""
    top = torch.iinfo(dtype).max
    memory = torch.randint(-top, top, (rows * cols + 1,), dtype=dtype, device="cuda:0")
    ids = torch.randint(0, rows, (nidx,), dtype=torch.int32, device="cuda:0")
    out = torch.full((nidx * cols + 64,), 77, dtype=dtype, device="cuda:0")
    size = memory.element_size()
    capi.check(capi.load().pto_gather_rows(torch.cuda.current_stream().cuda_stream, out.data_ptr() + size, memory.data_ptr() + size, ids.data_ptr(),
                                           nidx, rows, cols, size), "pto_gather_rows")
    assert torch.equal(out[1:1 + nidx * cols].view(nidx, cols), memory[1:].view(rows, cols)[ids.long()])
    assert out[0] == 77 and (out[1 + nidx * cols:] == 77).all()


def test_gather_rows_full_size_config(oracle):
    """Config 5: 65536 int32 row indices over a 16384 x 1024 fp16 table: bit-exact copy."""
    from gpu_util import gather_rows
    table, idx = datagen.gather_inputs(16384, 1024, 65536)
    got = gather_rows(table, idx)
    assert np.array_equal(got, table[idx])
    assert np.array_equal(got[:4096], oracle.gather_rows(table, idx[:4096]))


def test_tgather_index_tile(oracle):
    """Index-form TGATHER on one tile pair (half 16x1024 -> 16x128 of the reference's tgather test),
    with out-of-range indices, against the oracle and the committed reference output."""
    from gpu_util import to_dev, stream
    lib = capi.load()
    rng = np.random.default_rng(9)
    src = rng.integers(0, 2**16, size=(16, 1024), dtype=np.uint16)
    idx = rng.integers(-50, 16 * 1024 + 50, size=(16, 128), dtype=np.int32)
    ts, ti = to_dev(src), to_dev(idx)
    td = torch.full((16, 128), -1, dtype=torch.int16, device="cuda:0")
    capi.check(lib.pto_tgather_index_f16_16x1024_16x128(stream(), td.data_ptr(), ts.data_ptr(), ti.data_ptr()), "tgather")
    torch.cuda.synchronize()
    got = td.cpu().numpy().view(np.uint16)
    o = oracle
    want = o.tgather_index(o.make_layout(16, 128), src.reshape(-1), o.make_layout(16, 1024), idx.reshape(-1),
                           o.make_layout(16, 128, elem_bytes=4), 16, 128).reshape(16, 128)
    assert np.array_equal(got, want)
    G = np.load(os.path.join(os.path.dirname(__file__), "golden", "ref_vectors.npz"))
    assert np.array_equal(got, G["tgather_index_f16_16x1024_16x128"])
