"""GPU parity of the row-wise top-k (kernels/manual/a2a3/topk) through the C ABI: bit-exact scores and indices against
the oracle (the TSORT32 / TMRGSORT comparator applied to the whole row)."""
import numpy as np
import pytest
import torch

from pto_amd import capi, datagen

pytestmark = pytest.mark.gpu


def topk_gpu(src, in_idx, valid_cols, topk):
    from gpu_util import to_dev, stream
    lib = capi.load()
    rows, ld = src.shape
    ts, ti = to_dev(src), to_dev(np.ascontiguousarray(in_idx, dtype=np.uint32))
    os_ = torch.full((rows, topk), float("nan"), dtype=torch.float32, device="cuda:0")
    oi = torch.full((rows, topk), -1, dtype=torch.int32, device="cuda:0")
    capi.check(lib.pto_topk_f32(stream(), os_.data_ptr(), oi.data_ptr(), ts.data_ptr(), ti.data_ptr(), rows, valid_cols, ld, topk),
               "pto_topk_f32")
    torch.cuda.synchronize()
    return os_.cpu().numpy(), oi.cpu().numpy().view(np.uint32)


def same(got, want):
    return np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32)) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("rows,valid_cols,ld,topk", [(7, 256, 256, 256), (5, 1000, 1024, 37), (3, 1024, 1280, 1000), (4, 777, 800, 777),
                                                     (2, 33, 64, 5), (3, 2048, 2048, 100), (2, 4096, 4096, 4096), (9, 1, 8, 1)])
def test_topk_small_vs_oracle(oracle, rows, valid_cols, ld, topk):
    src, idx = datagen.topk_inputs(rows, valid_cols, ld)
    assert same(topk_gpu(src, idx, valid_cols, topk), oracle.topk_f32(src, idx, valid_cols, topk))


def test_topk_ties_signed_zeros_infinities_and_arbitrary_indices(oracle):
    rows, cols = 6, 1024
    src, _ = datagen.topk_inputs(rows, cols, cols, distinct=7)           # many equal scores: the index decides
    src[0, ::5] = -0.0
    src[1, ::3] = np.inf
    src[2, 1::4] = -np.inf
    src[3] = 0.0
    src[3, ::2] = -0.0                                                   # -0 == +0: pure index order, bit patterns kept
    src[4] = 3.0
    r = np.random.Generator(np.random.Philox(key=11))
    idx = r.permutation(1 << 20)[:cols].astype(np.uint32)                # not monotonic: ties follow the index, not the column
    idx[0] = 0xFFFFFFFF
    for k in (1, 100, cols):
        assert same(topk_gpu(src, idx, cols, k), oracle.topk_f32(src, idx, cols, k))
    # indices that increase with the column
    for mono in (np.arange(cols, dtype=np.uint32), (np.arange(cols, dtype=np.uint32) * 3 + 7) ** 2):
        for k in (1, 100, cols):
            assert same(topk_gpu(src, mono, cols, k), oracle.topk_f32(src, mono, cols, k))
    # and with other row lengths (1, 2, 8 keys per thread; padded rows)
    for c in (200, 512, 1900):
        s2, _ = datagen.topk_inputs(4, c, c + 8, distinct=5)
        s2[1, ::9] = -0.0
        for mono in (np.arange(c, dtype=np.uint32), r.permutation(1 << 16)[:c].astype(np.uint32)):
            assert same(topk_gpu(s2, mono, c, c), oracle.topk_f32(s2, mono, c, c))


@pytest.mark.parametrize("cols", [1, 63, 64, 65, 128, 129, 250, 256, 257, 512, 513, 1000, 1024, 1025, 2048, 2049, 4095, 4096])
def test_topk_row_lengths_and_kept_lengths(oracle, cols):
    """Every number of keys per lane and waves per row at its smallest and largest rows, topk on both sides of every length that
    the merges stop at (keys per lane times powers of two), row counts that do not fill the last workgroup, many ties and
    signed zeros; consecutive indices, increasing ones, ones that start near 2^32, and any."""
    r = np.random.Generator(np.random.Philox(key=cols))
    keys = next(e for e in (2, 4, 8, 16) if cols <= 64 * e or e == 16)
    kept = sorted({k for b in range(9) for k in ((keys << b) - 1, keys << b, (keys << b) + 1) if 1 <= k <= cols} | {1, cols})
    for n, k in enumerate(kept):
        rows = 1 + n % 6
        src, idx = datagen.topk_inputs(rows, cols, cols + 8 * (n % 2), distinct=0 if n % 3 else 11)
        src[0, ::7] = -0.0
        assert same(topk_gpu(src, idx, cols, k), oracle.topk_f32(src, idx, cols, k)), (k, "consecutive")
        which = (idx * np.uint32(5) + np.uint32(3), np.uint32(0xFFFFFFFF) - idx[::-1], r.permutation(1 << 16)[:cols].astype(np.uint32))[n % 3]
        assert same(topk_gpu(src, which, cols, k), oracle.topk_f32(src, which, cols, k)), (k, n % 3)


@pytest.mark.parametrize("cols,k", [(500, 500), (500, 9), (1024, 1000), (1024, 70), (1900, 1900), (1900, 200)])
@pytest.mark.parametrize("rows", [1280, 1281, 2560, 2563])
def test_topk_waves_per_row(oracle, rows, cols, k):
    """Around 256 units times five and ten waves (1024 columns change from two waves per row to one behind 2560), and a last workgroup
    that is not full; consecutive and other increasing indices."""
    src, idx = datagen.topk_inputs(rows, cols, cols + 1, distinct=300)
    for ids in (idx, idx * np.uint32(3)):
        assert same(topk_gpu(src, ids, cols, k), oracle.topk_f32(src, ids, cols, k))


@pytest.mark.parametrize("rows", [1, 365, 366])
@pytest.mark.parametrize("cols", [60, 129, 256, 500, 1000, 2000, 4000])
def test_topk_whole_and_cut_sorts(oracle, rows, cols):
    """topk on both sides of 16 (256 columns in four waves) and of an eighth of the padded row (whole sorts), rows on both sides
    of where 256 columns change their waves; indices in order and in any order."""
    if rows * cols > 1 << 20:
        rows = rows // 366 * 128 + 1
    r = np.random.Generator(np.random.Philox(key=rows + cols))
    src, idx = datagen.topk_inputs(rows, cols, cols + 3, distinct=200)
    src[0, ::7] = -0.0
    eighth = max(64, 1 << (cols - 1).bit_length()) // 8
    for k in sorted({k for k in (16, 17, eighth, eighth + 1, cols) if k <= cols}):
        for ids in (idx, r.permutation(cols).astype(np.uint32)):
            assert same(topk_gpu(src, ids, cols, k), oracle.topk_f32(src, ids, cols, k)), k


@pytest.mark.parametrize("rows,cols", [(300, 60), (501, 128), (1000, 250), (130, 512), (800, 500), (500, 1000), (1001, 1024), (2700, 1000), (500, 1900), (1800, 2048),
                                       (150, 4096)])
def test_topk_index_vectors_in_any_order(oracle, rows, cols):
    """Many rows under a permutation, a descending vector, one with repeated values and one that holds both ends of the range and
    its middle (as signed and as unsigned numbers), every number of waves per row; few distinct scores, signed zeros."""
    r = np.random.Generator(np.random.Philox(key=rows))
    src, idx = datagen.topk_inputs(rows, cols, cols + 1, distinct=9)
    mixed = r.permutation(1 << 16)[:cols].astype(np.uint32)
    mixed[:5] = (0xFFFFFFFF, 0x80000000, 0, 0x7FFFFFFF, 0x80000001)
    for ids in (r.permutation(cols).astype(np.uint32), idx[::-1] + np.uint32(0xFFFF0000), mixed):
        src[::7, ::5], src[::7, 1::5] = -0.0, 0.0
        for k in (cols, max(1, cols // 9)):
            assert same(topk_gpu(src, ids, cols, k), oracle.topk_f32(src, ids, cols, k)), k
    src[src == 0] = 1.5                                                  # (equal pairs would differ in the zeros' signs alone)
    ids = (idx // np.uint32(3)).astype(np.uint32)[r.permutation(cols)]
    assert same(topk_gpu(src, ids, cols, cols), oracle.topk_f32(src, ids, cols, cols))


@pytest.mark.parametrize("rows,cols", [(4096, 60), (4097, 60), (4097, 120), (4096, 200), (4097, 200), (731, 500), (732, 500), (2048, 500),
                                       (2049, 500), (4097, 500), (853, 1000), (854, 1000), (1706, 1900), (1707, 1900)])
def test_topk_lane_moves(oracle, rows, cols):
    """Both sides of the row counts where the lower words' way between lanes and the waves per row of 512 columns change."""
    src, idx = datagen.topk_inputs(rows, cols, cols + 1, distinct=300)
    for k in (cols, 9):
        assert same(topk_gpu(src, idx, cols, k), oracle.topk_f32(src, idx, cols, k))


def test_topk_every_kind_of_score():
    """Infinities, denormals, NaNs of either sign and random bit patterns: ordered by bit pattern as the interface states
    (the float comparison of the oracle puts NaNs nowhere), equal ones by column, and their bits are kept."""
    r = np.random.Generator(np.random.Philox(key=5))
    for cols in (100, 1024, 3000):
        bits = r.integers(0, 2**32, size=(5, cols), dtype=np.uint64).astype(np.uint32)
        bits[1, ::3] = 0x7F800000
        bits[2, ::5] = 0x00000123
        bits[3, ::4] = 0xFFFFFFFF
        bits[3, 1::4] = 0x7FFFFFFF
        bits[4, ::2] = 0x80000000
        plain = np.where(bits == 0x80000000, 0, bits)
        order = np.where(plain & 0x80000000, ~plain, plain | 0x80000000).astype(np.int64)
        idx = np.arange(cols, dtype=np.uint32)
        want = np.argsort(-order, axis=1, kind="stable")
        for k in (cols, 17):
            got = topk_gpu(bits.view(np.float32), idx, cols, k)
            assert np.array_equal(got[1], want[:, :k]), (cols, k)
            assert np.array_equal(got[0].view(np.uint32), np.take_along_axis(bits, want[:, :k], axis=1)), (cols, k)


def test_topk_reference_config_4800x1024_top1000(oracle):
    """The reference kernel's case: 4800 rows of 1024 valid columns (row stride 1280), top 1000, its generator's data."""
    rows, cols, ld, k = 4800, 1024, 1280, 1000
    src, idx = datagen.topk_inputs(rows, cols, ld)
    got = topk_gpu(src, idx, cols, k)
    assert same(got, oracle.topk_f32(src, idx, cols, k))
    # properties that hold whatever the implementation: sorted, indices distinct and in range, scores = src at the indices
    s, i = got
    assert np.all(s[:, :-1] >= s[:, 1:]) and int(i.max()) < cols
    assert np.array_equal(np.take_along_axis(src[:, :cols], i.astype(np.int64), axis=1), s)
    assert all(np.unique(i[r]).size == k for r in (0, 2399, 4799))


def test_topk_rejects_bad_arguments():
    lib = capi.load()
    t = torch.zeros(16, device="cuda:0")
    p = t.data_ptr()
    assert lib.pto_topk_f32(0, p, p, p, p, 4, 8192, 8192, 4) == capi.ERR_UNSUPPORTED     # more than 4096 columns
    assert lib.pto_topk_f32(0, p, p, p, p, 4, 100, 64, 4) == capi.ERR_UNSUPPORTED        # row stride below the valid columns
    assert lib.pto_topk_f32(0, p, p, p, p, 4, 100, 128, 101) == capi.ERR_UNSUPPORTED     # k above the valid columns
    assert lib.pto_topk_f32(0, p, 0, p, p, 4, 100, 128, 10) == capi.ERR_BAD_ARG
    assert lib.pto_topk_f32(0, p, p, p, p, 0, 100, 128, 10) == capi.ERR_BAD_ARG


@pytest.mark.parametrize("rows,cols,topk", [(100, 128, 63), (100, 128, 64), (7, 130, 65), (9, 1024, 127), (33, 2048, 2047), (16384, 1024, 512), (16385, 1024, 512)])
def test_topk_results_past_the_l2(rows, cols, topk):
    """Both sides of the lines at which results are stored past the L2, rows that are no whole store instruction long: torch's stable sort."""
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(rows + topk)
    src = torch.randint(-1000, 1000, (rows, cols), generator=g, device="cuda:0").float()
    ids = torch.arange(cols, dtype=torch.int32, device="cuda:0")
    guard = torch.full((rows * topk + 64,), 7.0, device="cuda:0")
    index = torch.full((rows * topk + 64,), -7, dtype=torch.int32, device="cuda:0")
    capi.check(lib.pto_topk_f32(torch.cuda.current_stream().cuda_stream, guard.data_ptr(), index.data_ptr(), src.data_ptr(), ids.data_ptr(), rows, cols,
                                cols, topk), "pto_topk_f32")
    score, order = torch.sort(src, dim=1, descending=True, stable=True)
    assert torch.equal(guard[:rows * topk].view(rows, topk), score[:, :topk]) and torch.equal(index[:rows * topk].view(rows, topk), order[:, :topk].int())
    assert (guard[rows * topk:] == 7.0).all() and (index[rows * topk:] == -7).all()


@pytest.mark.parametrize("rows,cols", [(2561, 257), (2565, 512), (641, 513), (1026, 1024), (5, 1025), (5, 1100), (515, 1500), (9, 2048), (4, 2049), (7, 3248), (3, 4096)])
def test_topk_by_threshold(oracle, rows, cols):
    """topk of an eighth of the padded row and less, on both sides of the numbers of groups that the threshold is taken over (24, 48, 64) and of the
    lengths that the lists are sorted by (64, 128, 256, 512): continuous scores; all equal; two values; most of a row masked; zeros of both signs as
    the threshold; ascending and descending rows; the largest scores side by side, in one lane, in one wave."""
    r = np.random.Generator(np.random.Philox(key=cols))
    padded = max(512, 1 << (cols - 1).bit_length())
    src = r.standard_normal((rows, cols + 3)).astype(np.float32)
    kinds = 10
    for kind in range(kinds):
        row = src[kind % rows::kinds] if rows >= kinds else src[kind % rows:kind % rows + 1]
        if kind == 1:
            row[:] = 2.5
        elif kind == 2:
            row[:] = np.where(row > 0.3, np.float32(1.0), np.float32(-1.0))
        elif kind == 3:
            row[:] = np.where(np.arange(cols + 3) % 37 == 5, row, -np.inf)
        elif kind == 4:
            row[:] = np.where(np.arange(cols + 3) % 97 == 5, np.abs(row), np.where(row > 0, np.float32(0.0), np.float32(-0.0)))
        elif kind == 5:
            row[:] = np.arange(cols + 3, dtype=np.float32)
        elif kind == 6:
            row[:] = -np.arange(cols + 3, dtype=np.float32)
        elif kind == 7:
            row[:, 100:228] += 50.0
        elif kind == 8:
            row[:, 17::64] += 50.0
        elif kind == 9:
            row[:] = np.where(row > 1.0, np.float32(np.inf), np.round(row * 3.0))
    idx = np.arange(cols, dtype=np.uint32)
    few = [k for k in (1, 2, 23, 24, 25, 48, 49, 63, 64, 65, 97, 128, 160, 161, 255, 256, 320, 321) if k <= min(cols, padded // 8 + 1)]
    if rows * cols > 1 << 20:
        few = few[::3] + few[-1:]
    for n, k in enumerate(few):
        assert same(topk_gpu(src, idx, cols, k), oracle.topk_f32(src, idx, cols, k)), (k, "consecutive")
        if n % 3 == 0:
            ids = (idx * np.uint32(3) + np.uint32(5), np.uint32(0xFFFFFFFF) - idx)[n // 3 % 2]
            assert same(topk_gpu(src, ids, cols, k), oracle.topk_f32(src, ids, cols, k)), (k, "other indices")


@pytest.mark.parametrize("rows,cols,topk", [(740, 1024, 120), (2564, 512, 60)])
def test_topk_threshold_fails_next_to_a_long_list(oracle, rows, cols, topk):
    """Rows of one workgroup in turn: keys of the longest list, and so many in so few groups (every fourth block of 64 columns of a lane) that the
    row is sorted whole; a wave's list and its neighbour's sort do not share memory."""
    r = np.random.Generator(np.random.Philox(key=rows))
    src, idx = datagen.topk_inputs(rows, cols, cols)
    src[:] = r.standard_normal(src.shape)
    block, lane = np.arange(cols) // 64, np.arange(cols) % 64
    src[0::2, (block % 4 == 0)] += 100.0
    src[1::2, (block % 4 == 0) | (block % 4 == 1) | ((block % 4 == 2) & (lane < 6))] += 100.0
    assert same(topk_gpu(src, idx, cols, topk), oracle.topk_f32(src, idx, cols, topk))


@pytest.mark.parametrize("rows,cols,topks", [(515, 1025, (20, 228, 244, 256)), (515, 1100, (37, 228, 256)), (517, 2048, (100, 256)), (130, 2049, (33, 256, 320)),
                                             (130, 4096, (97, 320)), (900, 1024, (9, 60, 128)), (5200, 512, (16, 64)), (250, 1500, (128, 129)), (300, 1500, (160, 161))])
def test_topk_threshold_and_the_columns(oracle, rows, cols, topks):
    """Rows whose level changes along the columns, which the waves of a row share out among them, next to random ones in the same workgroup, and rows of
    which far more keys equal the threshold than are wanted, in all blocks of 64 columns: those with the lowest columns, behind the larger ones, and
    zeros of either sign among them."""
    r = np.random.Generator(np.random.Philox(key=cols))
    src, c = r.standard_normal((rows, cols)).astype(np.float32), np.arange(cols, dtype=np.float32)
    kinds = (src[0::7], src[1::7], src[2::7], src[3::7], src[4::7], src[5::7])
    kinds[0][:] = c
    kinds[1][:] += 8 * c / cols
    kinds[2][:, cols // 2:] = -np.inf
    kinds[3][:] = np.where(r.random(kinds[3].shape) < 0.98, -np.inf, kinds[3])
    kinds[4][:] = np.where(r.random(kinds[4].shape) < 0.02, np.abs(kinds[4]), np.where(r.random(kinds[4].shape) < 0.5, np.float32(0.0), np.float32(-0.0)))
    kinds[5][:] = np.round(kinds[5] * 4)
    idx = np.arange(cols, dtype=np.uint32)
    for k in topks:
        assert same(topk_gpu(src, idx, cols, k), oracle.topk_f32(src, idx, cols, k)), k


@pytest.mark.parametrize("rows,cols", [(750, 512), (803, 257), (9, 1024), (12, 513), (900, 1024), (860, 700), (2563, 1024), (2565, 600), (5, 2048), (14, 1025), (1710, 2048), (1711, 1100),
                                       (13, 4096), (14, 2049), (12, 3000)])
def test_topk_by_buckets(rows, cols):
    """Whole sorts (more than an eighth of the padded row), and an eighth where no threshold is taken, of every kind of row that buckets take, give up on at the look, after counting, or after a first exchange: even
    scores; equal ones in numbers around the fullest bucket's limits (16, 24, 48); ascending and descending; one far outlier; a cluster of distinct scores; infinities; NaNs of either
    sign; zeros of either sign; ranges too small and too large to spread; a part of the columns at another level.  NaNs, which the
    comparator leaves open, in the order of their bits as before."""
    r = np.random.Generator(np.random.Philox(key=rows + cols))
    src, c = r.standard_normal((rows, cols + 5)).astype(np.float32), np.arange(cols + 5, dtype=np.float32)
    kinds = 12 if rows < 100 else 18
    for kind in range(kinds):
        row = src[kind::kinds]
        if kind == 1:
            row[:] = r.integers(0, max(1, cols // 16), row.shape)
        elif kind == 2:
            row[:] = r.integers(0, max(1, cols // 40), row.shape)
        elif kind == 3:
            row[:] = c
        elif kind == 4:
            row[:] = np.where(c == cols // 3, np.float32(1e6), row)
        elif kind == 5:
            row[:, cols // 2:cols // 2 + 40] = 0.25 + row[:, cols // 2:cols // 2 + 40] * np.float32(1e-5)
        elif kind == 6:
            row[:] = np.where(c == cols - 1, np.float32(np.inf), np.where(c == 7, np.float32(-np.inf), row))
        elif kind == 7:
            row[:] = np.where(c == cols - 2, np.uint32(0xffc00001).view(np.float32), np.where(c == 70, np.float32(np.nan), row))
        elif kind == 8:
            row[:] = np.where(row < 0.0, np.float32(-0.0), np.where(row < 0.3, np.float32(0.0), row))
        elif kind == 9:
            row[:] *= np.float32(1e-33)
        elif kind == 10:
            row[:] *= np.float32(3e37)
        elif kind == 11:
            row[:] = np.where(c >= cols * 3 // 4, row + 100, row)
        elif kind == 12:
            row[:] = -c
        elif kind == 13:
            row[:] = np.exp(row * 4)
        elif kind == 14:
            row[:] = np.where(c >= cols // 2, -np.inf, row)
        elif kind == 15:
            row[:] = np.where(r.random(row.shape) < 0.98, np.float32(1.5), row)
        elif kind == 16:
            row[:] = np.float32(-2.0)
        elif kind == 17:
            row[:] = np.round(row * 64) / 64
    idx = np.arange(cols, dtype=np.uint32)
    eighth = (1 << (cols - 1).bit_length()) // 8
    bits = src[:, :cols].view(np.uint32)
    plain = np.where(bits == 0x80000000, np.uint32(0), bits)
    order = np.where(plain >> 31, ~plain, plain | np.uint32(0x80000000))
    for ids, k in ((idx, cols), (idx, max(321, eighth + 1) if cols > 321 else cols), (idx * np.uint32(3) + np.uint32(5), cols - 1), (np.uint32(0xFFFFFFFF) - idx, cols),
                   (idx, eighth), (idx * np.uint32(3) + np.uint32(5), eighth - 1), (np.uint32(0xFFFFFFFF) - idx, eighth)):
        at = np.lexsort((np.broadcast_to(ids, order.shape), ~order))[:, :k]
        assert same(topk_gpu(src, ids, cols, k), (np.take_along_axis(src, at, 1), ids[at])), (k, ids[:2])


@pytest.mark.parametrize("rows,cols", [(748, 512), (741, 300), (36, 1024), (37, 600), (888, 1000), (2592, 1024), (2571, 700), (40, 2048), (19, 1300), (1716, 1500), (38, 4096), (21, 2500)])
def test_topk_of_crowded_scores(rows, cols):
    """Rows around every limit of the sort by buckets: clusters of 14 to 60 distinct scores closer than a bucket (16, 24 and 48 are exchanged by neighbours), few
    distinct scores (whose equal ones stand in order), a part of the row equal with other scores among it, squares and others that crowd at an end of their range, bfloat16 scores."""
    r = np.random.Generator(np.random.Philox(key=7 * rows + cols))
    src = r.random((rows, cols), dtype=np.float32)
    normal = r.standard_normal((rows, cols)).astype(np.float32)
    for row in range(rows):
        kind = row % 20
        if kind < 10:
            n = (14, 15, 16, 17, 22, 23, 24, 25, 46, 60)[kind]
            src[row, r.permutation(cols)[:n]] = np.float32(0.5) + np.arange(n, dtype=np.float32) * np.float32(6e-8)
        elif kind < 14:
            src[row] = r.integers(0, (11, 30, 70, 190)[kind - 10], cols)
        elif kind < 17:
            src[row] = np.where(r.random(cols) < (0.05, 0.25, 0.6)[kind - 14], np.float32(0.3), normal[row])
        elif kind < 19:
            src[row] = normal[row] ** 2 if kind == 17 else 1 / (1 + np.exp(-6 * normal[row]))
        else:
            src[row] = (normal[row].view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    idx = np.arange(cols, dtype=np.uint32)
    for ids, k in ((idx, cols), (r.permutation(cols).astype(np.uint32), cols - cols // 3)):
        at = np.lexsort((np.broadcast_to(ids, src.shape), -src))[:, :k]
        assert same(topk_gpu(src, ids, cols, k), (np.take_along_axis(src, at, 1), ids[at])), k


@pytest.mark.parametrize("rows,cols", [(803, 257), (750, 512), (9, 1024), (12, 513), (900, 1024), (860, 700), (2563, 1024), (2565, 600), (5, 2048), (14, 1025), (1710, 2048), (1711, 1100),
                                       (7, 4096)])
def test_topk_any_index_order_by_buckets(rows, cols):
    """Indices in any order whose order is found by buckets (below 2^24), or not (one at 2^24, all of them far apart, crowded, all equal but a few): equal
    ones by column. Random scores, and every third row of few distinct ones with zeros of either sign, every fifth masked with infinities from the middle on."""
    r = np.random.Generator(np.random.Philox(key=3 * rows + cols))
    src, column = r.standard_normal((rows, cols)).astype(np.float32), np.arange(cols)
    src[1::3] = np.where(r.random(src[1::3].shape) < 0.5, np.float32(-1.0), np.float32(1.0)) * r.integers(0, 9, src[1::3].shape).astype(np.float32)
    src[4::5, cols // 2:] = -np.inf
    shuffled = r.permutation(cols)
    top = (1 << 24) - 1
    kinds = (shuffled, top - shuffled, np.where(shuffled == 3, top + 1, shuffled), shuffled * ((1 << 32) // cols - 1), r.integers(0, cols // 2, cols),
             np.where(shuffled < 5, shuffled, 77), np.where(shuffled == 0, top, shuffled % 40), 2 * shuffled + 1000 - 7 * (shuffled % 2))
    score = -(src + np.float32(0.0))
    for n, ids in enumerate(kinds):
        ids = ids.astype(np.uint32)
        k = cols if n % 2 else cols - cols // 4
        order = np.lexsort((np.broadcast_to(column, src.shape), np.broadcast_to(ids, src.shape), score))[:, :k]
        assert same(topk_gpu(src, ids, cols, k), (np.take_along_axis(src, order, 1), ids[order])), n
