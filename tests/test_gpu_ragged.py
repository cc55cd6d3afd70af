"""GPU tests of widths and alignments that do not fit a lane's vector: the
kernels read and write rows of B and C with 16-byte accesses at any 4-byte
boundary, the last vector of a row moved back to end with it."""
import numpy as np
import pytest

from conftest import items_per_wave, tile_csr, work_items
from test_gpu_parity import _block_csr, _Shifted, assert_within_tolerance

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def st(gpu):
    return gpu.Stream()


def _spmm(vs, fmt, B, C0, off, st, accumulate):
    """C0 + A*B or A*B with B and C `off` bytes past an aligned address."""
    dB, dC = _Shifted(vs, B, off, st), _Shifted(vs, C0, off, st)
    vs.run_vcsr_spmm_gpu_ex(fmt, dB, B.shape[1], 64, dC, st, timed=True, kernel=vs.KERNEL_TILE,
                            accumulate=accumulate)
    return dC.numpy()


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("O", [1, 15, 16, 17, 31, 33, 34, 63, 65, 66, 127, 259])
def test_mfma_tiles_any_width_are_bit_exact(gpu, orc, st, O, off):
    """Few 16-row MFMA tiles: lanes of 1 and 2 floats (4 take more tiles, below),
    bit for bit the oracle's FP32 loop; C += A*B on top of C0 = 2 stays within
    one rounding of it."""
    vs = gpu
    rng = np.random.default_rng(O)
    csr = _block_csr(vs, rng, 9, 16, 400, 6, 16, 0.9)
    fmt = vs.build_vcsr(csr, 16, 16, vs.LAYOUT_TC)
    fmt.set_tile_rows(16)
    fmt.upload(st)
    B = vs.gen_dense(O, 1, csr.N, O)
    C0 = np.full((csr.M, O), 2.0, np.float32)
    ref = orc.spmm_f32(csr.M, csr.row_ptr, csr.col, csr.val, B)
    got = _spmm(vs, fmt, B, C0, off, st, False)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    got = _spmm(vs, fmt, B, C0, off, st, True)
    assert np.array_equal(got, C0 + ref)


def _sixteen_rows(vs, rng, copies):
    """Seven 16-row tiles of 1 to 7 whole groups of 16 entries, one entry in ten
    absent, `copies` times below each other; and the seven alone."""
    rows, cols = [], []
    for t in range(7):
        c = np.sort(rng.choice(200, size=16 * (t + 1), replace=False))
        for i in range(16):
            keep = c[(rng.random(c.size) < 0.9) | (np.arange(c.size) % 16 == i)]
            rows.append(np.full(keep.size, 16 * t + i))
            cols.append(keep)
    rows, cols = np.concatenate(rows).astype(np.int32), np.concatenate(cols).astype(np.int32)
    one = vs.coo_to_csr(vs.Coo.from_arrays(112, 200, rows, cols,
                                           rng.standard_normal(rows.size).astype(np.float32)))
    return one, tile_csr(vs, one, copies)


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("tiles,O,vec", [
    (91, 8, 1), (602, 16, 1), (399, 18, 1), (602, 31, 2), (1099, 24, 2), (1099, 31, 2), (91, 47, 1),
    (91, 48, 2), (98, 257, 1), (98, 259, 1), (602, 33, 4), (602, 50, 4), (602, 64, 4), (1022, 61, 4),
    (602, 65, 2), (602, 72, 2), (384, 131, 2), (1099, 33, 4), (1099, 64, 4), (1099, 127, 4),
    (700, 101, 4), (700, 131, 2), (1099, 259, 4), (1099, 256, 4)])
def test_mfma_tiles_of_every_wave_count(gpu, orc, st, tiles, O, vec, off):
    """16-row MFMA tiles at lanes of 1, 2 and 4 floats, whole rows and odd ones,
    at up to 1,024 waves (two operand sets), up to 3,072 (loads ahead) and more
    (mixed), with pieces of an odd and an even number of blocks: bit for bit the
    oracle's FP32 loop, C += A*B and inf and NaN next to a row's moved-back end
    among them."""
    vs = gpu
    one, csr = _sixteen_rows(vs, np.random.default_rng(O), tiles // 7)
    fmt = vs.build_vcsr(csr, 16, 16, vs.LAYOUT_TC)
    fmt.set_tile_rows(16)
    fmt.upload(st)
    info = fmt.launch_info(O)
    assert info["tiles"] == tiles // 7 * 7 and info["split_rows"] == 0 and info["vec"] == vec
    B = vs.gen_dense(O, 1, csr.N, O)
    C0 = np.full((csr.M, O), 2.0, np.float32)
    ref = np.tile(orc.spmm_f32(one.M, one.row_ptr, one.col, one.val, B), (tiles // 7, 1))
    got = _spmm(vs, fmt, B, C0, off, st, False)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(_spmm(vs, fmt, B, C0, off, st, True), C0 + ref)
    B[3, O - 1], B[50, O - 2], B[199, 0] = np.inf, np.nan, -np.inf
    ref = np.tile(orc.spmm_f32(one.M, one.row_ptr, one.col, one.val, B), (tiles // 7, 1))
    got = _spmm(vs, fmt, B, C0, off, st, False)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])


def _mixed_blocks(vs, rng, h, N=1500):
    """Block rows of h equal-pattern rows: short and long ones, one cut into
    several pieces (600 columns), empty rows, a last block row cut short."""
    rows, cols, r = [], [], 0
    for n in [1, 5, 33, 64, 65, 97, 129, 600, 0, 7, 40, 63, 2, 90, 20, 20, 11]:
        c = np.sort(rng.choice(N, size=n, replace=False))
        for i in range(h):
            keep = c if i == 0 else c[rng.random(n) < 0.9]
            rows.append(np.full(keep.size, r + i))
            cols.append(keep)
        r += h
    rows, cols = np.concatenate(rows).astype(np.int32), np.concatenate(cols).astype(np.int32)
    vals = rng.standard_normal(rows.size).astype(np.float32)
    live = rows < r - 1 if h > 1 else rows < r
    return vs.coo_to_csr(vs.Coo.from_arrays(r - (h > 1), N, rows[live], cols[live], vals[live]))


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("O", [1, 3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 50, 64, 65, 127, 129, 255,
                               257])
@pytest.mark.parametrize("R", [2, 3, 4, 8])
def test_tall_tiles_any_width(gpu, orc, st, R, O, off):
    """Tiles of 2 to 8 rows at every width class and its edges, split tiles
    and their reduce among them: C = A*B and C += A*B against the oracle."""
    vs = gpu
    rng = np.random.default_rng(1000 * R + O)
    csr = _mixed_blocks(vs, rng, R)
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(R)
    fmt.upload(st)
    assert fmt.launch_info(O)["split_rows"] >= R - 1
    B = vs.gen_dense(O, 0, csr.N, O)
    C0 = rng.integers(-2, 3, size=(csr.M, O)).astype(np.float32)
    ref = orc.spmm_f64(csr.M, csr.row_ptr, csr.col, csr.val, B)
    assert_within_tolerance(_spmm(vs, fmt, B, C0, off, st, False), ref, csr.row_ptr, csr.val, B,
                            f"R{R} O{O}")
    got = _spmm(vs, fmt, B, C0, off, st, True)
    # One more rounding of values up to |C0| + |ref|.
    err = np.abs(got - (C0 + ref)) - 2.0 ** -23 * (np.abs(C0) + np.abs(ref))
    l1 = np.array([np.abs(csr.val[a:b]).sum() for a, b in zip(csr.row_ptr, csr.row_ptr[1:])])
    assert (err <= 1e-4 * l1[:, None] * np.abs(B).max()).all()


@pytest.mark.parametrize("copies", [40, 500])
@pytest.mark.parametrize("O", [128, 129, 200, 256, 259])
@pytest.mark.parametrize("R", [2, 3, 4])
def test_tall_tiles_accumulate_many(gpu, orc, st, R, O, copies):
    """C += A*B on fewer and on more tiles than 8 waves per SIMD: rows of C read
    ahead, and for 2 and 3 rows at O > 128 late; split tiles among them, one
    rounding from C0 + A*B, the same bits twice."""
    vs = gpu
    one = _mixed_blocks(vs, np.random.default_rng(R + O), R)
    csr = tile_csr(vs, one, copies)
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(R)
    fmt.upload(st)
    assert (fmt.launch_info(O)["tiles"] > 8192) == (copies == 500)
    B = vs.gen_dense(O, 0, csr.N, O)
    C0 = np.random.default_rng(O).integers(-2, 3, size=(csr.M, O)).astype(np.float32)
    ref = np.tile(orc.spmm_f64(one.M, one.row_ptr, one.col, one.val, B), (copies, 1))
    got = _spmm(vs, fmt, B, C0, 4, st, True)
    err = np.abs(got - (C0 + ref)) - 2.0 ** -23 * (np.abs(C0) + np.abs(ref))
    l1 = np.array([np.abs(one.val[a:b]).sum() for a, b in zip(one.row_ptr, one.row_ptr[1:])])
    assert (err <= 1e-4 * np.tile(l1, copies)[:, None] * np.abs(B).max()).all()
    assert np.array_equal(got, _spmm(vs, fmt, B, C0, 0, st, True))


@pytest.mark.parametrize("O", [5, 12, 30, 47, 100])
@pytest.mark.parametrize("R", [2, 3, 4, 8])
def test_tall_tiles_nonfinite_b(gpu, orc, st, R, O):
    """inf and NaN in B reach exactly the rows the oracle's loop reaches,
    also in the last, moved-back vector of a row and its neighbours."""
    vs = gpu
    rng = np.random.default_rng(R + O)
    csr = _mixed_blocks(vs, rng, R)
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(R)
    fmt.upload(st)
    B = vs.gen_dense(O, 0, csr.N, O)
    for r, c, x in [(3, O - 1, np.inf), (700, O - 2, np.nan), (701, 0, -np.inf), (1499, O - 1, np.nan)]:
        B[r, c] = x
    ref = orc.spmm_f32(csr.M, csr.row_ptr, csr.col, csr.val, B)
    got = _spmm(vs, fmt, B, np.zeros((csr.M, O), np.float32), 0, st, False)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref))
    fin = np.isfinite(ref)
    assert np.allclose(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


def _mixed_rows(vs, rng, long_row=True):
    """Row lengths around the edges of work items (16, 32, 64 entries), empty
    rows, runs of one-entry rows and a row cut into ten pieces."""
    lens = [0, 1, 2, 15, 16, 17, 31, 32, 33, 0, 0, 63, 64, 65, 1, 1, 1, 129] + [1] * 70 + \
        [3, 5, 7] * 30 + [40, 20] * 8 + ([600] if long_row else []) + [0] * 40 + [2]
    N = 1500
    rows = np.repeat(np.arange(len(lens)), lens).astype(np.int32)
    cols = np.concatenate([np.sort(rng.choice(N, size=n, replace=False)) for n in lens])
    return vs.coo_to_csr(vs.Coo.from_arrays(len(lens), N, rows, cols.astype(np.int32),
                                            rng.standard_normal(rows.size).astype(np.float32)))


_ROW_WIDTHS = [1, 3, 7, 8, 9, 16, 17, 30, 32, 33, 50, 64, 65, 127, 129, 255, 257]


@pytest.mark.parametrize("copies,O,off", [(c, O, off) for c in (1, 40) for O in _ROW_WIDTHS
                                          for off in (0, 4)] +
                         [(120, O, 0) for O in _ROW_WIDTHS if O < 33] +
                         [(600, O, 0) for O in _ROW_WIDTHS if O < 130])
def test_row_tiles_any_width(gpu, orc, st, copies, O, off):
    """Single-row tiles at every width class and its edges; 40, 120 and 600
    copies of the matrix below each other: waves of 1, 2 and 4 work items.
    C = A*B and C += A*B against the oracle, twice the same bits."""
    vs = gpu
    rng = np.random.default_rng(O)
    one = _mixed_rows(vs, rng)
    csr = tile_csr(vs, one, copies)
    *counts, piece = work_items(csr)
    assert piece == 64
    assert items_per_wave(*counts, O) == {1: 1, 40: 1, 120: 2, 600: 4}[copies] or O > 32
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(1)
    fmt.upload(st)
    B = vs.gen_dense(O, 0, csr.N, O)
    C0 = rng.integers(-2, 3, size=(csr.M, O)).astype(np.float32)
    ref = np.tile(orc.spmm_f64(one.M, one.row_ptr, one.col, one.val, B), (copies, 1))
    got = _spmm(vs, fmt, B, C0, off, st, False)
    assert_within_tolerance(got, ref, csr.row_ptr, csr.val, B, f"O{O}")
    assert np.array_equal(got, _spmm(vs, fmt, B, C0, off, st, False))
    got = _spmm(vs, fmt, B, C0, off, st, True)
    err = np.abs(got - (C0 + ref)) - 2.0 ** -23 * (np.abs(C0) + np.abs(ref))
    l1 = np.add.reduceat(np.append(np.abs(csr.val), 0), csr.row_ptr[:-1])
    l1[np.diff(csr.row_ptr) == 0] = 0
    assert (err <= 1e-4 * l1[:, None] * np.abs(B).max()).all()


# Rows of one piece each: 17 to 64 entries (mean 35 or 20), 65 to 128, or short
# ones and one of 100 that makes the largest piece 128.
_ONE_PIECE = {"mid": [17, 20, 33, 64, 40, 31, 25, 48], "short": [17, 19, 20, 24, 22, 18],
              "long": [65, 128, 100, 77], "some": [17, 18, 100, 19, 17, 20, 18, 17]}


@pytest.mark.parametrize("kind,copies,O,merge", [
    ("mid", 1, 1, 1), ("mid", 1, 12, 1), ("mid", 1, 31, 1), ("mid", 1, 50, 1), ("mid", 1, 101, 1),
    ("mid", 1, 257, 1), ("long", 1, 8, 1), ("long", 1, 13, 1), ("long", 1, 64, 1),
    ("long", 1, 128, 1), ("short", 1000, 20, 0), ("short", 1000, 32, 1), ("mid", 2100, 8, 4),
    ("mid", 2100, 12, 0), ("mid", 2100, 17, 0), ("mid", 2100, 31, 0), ("mid", 2100, 32, 4),
    ("mid", 2100, 50, 2), ("short", 1, 33, 0), ("short", 40, 63, 0), ("short", 40, 60, 1),
    ("short", 5400, 47, 0), ("some", 1, 47, 0), ("some", 30, 21, 0), ("some", 30, 63, 0),
    ("long", 3, 31, 0), ("short", 5500, 30, 4), ("short", 5500, 47, 2), ("long", 4200, 7, 4), ("long", 4200, 15, 0),
    ("long", 4200, 33, 2), ("short", 5500, 12, 4), ("short", 5500, 15, 4), ("short", 8300, 100, 2),
    ("short", 11000, 130, 2)])
def test_row_tiles_of_one_piece(gpu, orc, st, kind, copies, O, merge):
    """Single-row tiles where every work item is one row: a wave of one item
    (its streams' sums meet in a butterfly), and waves of several (pieces cut
    between streams), C = A*B and C += A*B.  merge 0: one float a lane, one item a
    wave at any size (33 to 63 columns: C = A*B only)."""
    vs = gpu
    rng = np.random.default_rng(copies + O)
    lens = _ONE_PIECE[kind]
    N = 700
    rows = np.repeat(np.arange(len(lens)), lens).astype(np.int32)
    cols = np.concatenate([np.sort(rng.choice(N, size=n, replace=False)) for n in lens])
    one = vs.coo_to_csr(vs.Coo.from_arrays(len(lens), N, rows, cols.astype(np.int32),
                                           rng.standard_normal(rows.size).astype(np.float32)))
    csr = tile_csr(vs, one, copies)
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(1)
    fmt.upload(st)
    info = fmt.launch_info(O)
    assert info["split_rows"] == 0
    assert items_per_wave(csr.M, csr.M, csr.nnz, O) == max(merge, 1)
    if not merge:
        assert info["vec"] == 1
    B = vs.gen_dense(O, 0, N, O)
    ref = np.tile(orc.spmm_f64(one.M, one.row_ptr, one.col, one.val, B), (copies, 1))
    C0 = np.ones((csr.M, O), np.float32)
    for accumulate in (False, True):
        got = _spmm(vs, fmt, B, C0, 4 * accumulate, st, accumulate)
        assert_within_tolerance(got - C0 if accumulate else got, ref, csr.row_ptr, csr.val, B,
                                f"{kind} O{O}")


@pytest.mark.parametrize("O", [5, 8, 12, 30, 47, 100])
def test_row_tiles_nonfinite_b(gpu, orc, st, O):
    """inf and NaN in B reach exactly the rows the oracle's loop reaches."""
    vs = gpu
    rng = np.random.default_rng(O)
    csr = _mixed_rows(vs, rng)
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(1)
    fmt.upload(st)
    B = vs.gen_dense(O, 0, csr.N, O)
    for r, c, x in [(0, 0, np.nan), (3, O - 1, np.inf), (700, O - 2, np.nan), (701, 0, -np.inf)]:
        B[r, c] = x
    ref = orc.spmm_f32(csr.M, csr.row_ptr, csr.col, csr.val, B)
    got = _spmm(vs, fmt, B, np.zeros((csr.M, O), np.float32), 0, st, False)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref))
    fin = np.isfinite(ref)
    assert np.allclose(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("O", [1, 8, 9, 16, 17, 31, 33, 50, 64, 65, 100, 128, 130, 257, 300])
def test_csr_wave_long_rows_are_bit_exact(gpu, orc, st, O, off):
    """The plain-CSR kernel on rows around its long-row limit (128 entries)
    and around whole turns of it, empty rows and columns outside [0, N)
    (which contribute nothing): bit for bit the oracle's FP32 loop."""
    vs = gpu
    rng = np.random.default_rng(O)
    N = 2000
    lens = [0, 1, 127, 128, 129, 136, 0, 159, 160, 161, 1700, 3] + [5] * 40 + [257, 300, 1] * 9
    rows = np.repeat(np.arange(len(lens)), lens)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, N, rows.size).astype(np.int32)
    val = rng.standard_normal(rows.size).astype(np.float32)
    B = vs.gen_dense(O, 0, N, O)
    ref = orc.spmm_f32(len(lens), rp, col, val, B)

    def run(rp, col, val):
        d = [vs.DeviceArray.from_numpy(x, st) for x in (rp, col, val)]
        dB = _Shifted(vs, B, off, st)
        dC = _Shifted(vs, np.full((len(lens), O), 5.0, np.float32), off, st)
        vs.run_csr_wave_spmm_gpu(len(lens), N, *d, dB, O, dC, st, timed=True)
        return dC.numpy()

    assert np.array_equal(run(rp, col, val).view(np.uint32), ref.view(np.uint32))
    bad = rng.random(rows.size) < 0.1
    outside = np.where(bad, np.where(rng.random(rows.size) < 0.5, -1, N), col).astype(np.int32)
    keep = ~bad
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=len(lens)))])
    ref = orc.spmm_f32(len(lens), rp2.astype(np.int32), col[keep], val[keep], B)
    assert np.array_equal(run(rp, outside, val).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("O", [1, 3, 7, 8, 9, 13, 16, 17, 20, 32, 33, 47, 64, 65, 127, 128, 129, 200,
                               256, 257, 516])
def test_csr_wave_short_rows_are_bit_exact(gpu, orc, st, O, off):
    """The plain-CSR kernel where no row is long (no barrier in a block):
    lengths around the blocks of 8 loads and the 32 and 64 entries staged at
    a time, matrices that end inside a wave and a block, a single row, and
    inf and NaN in the columns next to those that idle lanes read again."""
    vs = gpu
    rng = np.random.default_rng(7 * O)
    N = 300
    base = [0, 1, 7, 8, 9, 0, 15, 16, 17, 31, 32, 33, 5, 63, 64, 65, 100, 127, 128, 2]
    for M in (1, 3, 17, 33, 61, 100):
        lens = [base[(3 * i + M) % len(base)] for i in range(M)]
        rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        col = rng.integers(0, N, rp[-1]).astype(np.int32)
        val = rng.standard_normal(rp[-1]).astype(np.float32)
        B = vs.gen_dense(O, 0, N, O)
        if M == 61:
            B[3, O - 1], B[100, 0], B[299, O // 2] = np.inf, np.nan, -np.inf
        d = [vs.DeviceArray.from_numpy(x if x.size else np.zeros(1, x.dtype), st)
             for x in (rp, col, val)]
        dB = _Shifted(vs, B, off, st)
        dC = _Shifted(vs, np.full((M, O), 5.0, np.float32), off, st)
        vs.run_csr_wave_spmm_gpu(M, N, *d, dB, O, dC, st, timed=True)
        got, ref = dC.numpy(), orc.spmm_f32(M, rp, col, val, B)
        nan = np.isnan(ref)
        assert np.array_equal(np.isnan(got), nan), M
        assert np.array_equal(got.view(np.uint32)[~nan], ref.view(np.uint32)[~nan]), M


@pytest.mark.parametrize("copies,O", [(2, 8), (2, 16), (2, 31), (2, 50), (2, 128), (2, 257),
                                      (900, 8), (900, 12), (900, 32), (900, 64), (1800, 8)])
def test_row_tiles_of_up_to_128_entries_stay_whole(gpu, orc, st, copies, O):
    """Where rows of 65 to 128 entries hold much of the matrix they are one
    piece each (only the 129- and 300-entry rows are split), also with 2 and
    4 work items per wave."""
    vs = gpu
    rng = np.random.default_rng(O)
    lens = [64, 65, 128, 1, 127, 0, 100, 129, 66, 30, 300, 97]
    N = 1200
    rp1 = np.concatenate([[0], np.cumsum(lens)])
    col = np.concatenate([np.sort(rng.choice(N, size=n, replace=False)) for n in lens])
    val = rng.standard_normal(col.size).astype(np.float32)
    rp = np.concatenate([[0]] + [rp1[1:] + i * col.size for i in range(copies)]).astype(np.int32)
    csr = vs.Csr.from_arrays(len(lens) * copies, N, rp, np.tile(col, copies).astype(np.int32),
                             np.tile(val, copies))
    fmt = vs.build_vcsr(csr, 4, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(1)
    fmt.upload(st)
    assert fmt.launch_info(O)["split_rows"] == 2 * copies
    B = vs.gen_dense(O, 0, N, O)
    ref = np.tile(orc.spmm_f64(len(lens), rp1.astype(np.int32), col.astype(np.int32), val, B),
                  (copies, 1))
    C0 = np.ones((csr.M, O), np.float32)
    for accumulate in (False, True):
        got = _spmm(vs, fmt, B, C0, 0, st, accumulate)
        assert_within_tolerance(got - C0 if accumulate else got, ref, csr.row_ptr, csr.val, B,
                                f"O{O}")


# B of 2 GiB and a little more, addressed with 64 bits; rows of any width O.
_BIG_FLOATS = (1 << 29) + 4096


@pytest.fixture(scope="module")
def big_b(gpu, st):
    vs = gpu
    host = vs.gen_dense(77, 0, _BIG_FLOATS // 1024, 1024).reshape(-1)
    return host, vs.DeviceArray.from_numpy(host, st)


class _Rows:
    """The big buffer as N x O."""

    def __init__(self, big, N, O):
        self.host = big[0][:N * O].reshape(N, O)
        self.ptr, self.shape, self.nbytes, self.dtype = big[1].ptr, (N, O), N * O * 4, np.float32


def _far(csr_cols, N):
    """Columns of a 1500-column matrix, the upper half moved to the end of N."""
    return np.where(csr_cols < 750, csr_cols, csr_cols + (N - 1500)).astype(np.int32)


@pytest.mark.parametrize("O", [50, 257, 1024])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 8, 16])
def test_tiles_on_b_of_2gb_or_more(gpu, orc, st, big_b, R, O):
    """Every tile height with B of 2 GiB (64-bit addresses; at O = 257 a last
    slice of one column): the first and last B rows, split tiles, placeholders
    and padding, which read B row 0 there; C = A*B and C += A*B, and inf and NaN
    in B row 0 reach only the rows that hold column 0."""
    vs = gpu
    N = (1 << 29) // O + 2
    rng = np.random.default_rng(R + O)
    one = _mixed_blocks(vs, rng, R) if R > 1 else _mixed_rows(vs, rng)
    col = one.col.copy()
    col[one.row_ptr[7]] = 0  # a row that holds column 0, and one with the last
    one = vs.Csr.from_arrays(one.M, 1500, one.row_ptr, col, one.val)
    csr = vs.Csr.from_arrays(one.M, N, one.row_ptr, _far(one.col, N), one.val)
    fmt = vs.build_vcsr(csr, 64, 64, vs.LAYOUT_S)
    fmt.set_tile_rows(R)
    fmt.upload(st)
    B = _Rows(big_b, N, O)
    assert B.nbytes >= 1 << 31
    small = np.concatenate([B.host[:750], B.host[N - 750:]])
    C0 = rng.integers(-2, 3, size=(csr.M, O)).astype(np.float32)

    def run(accumulate):
        dC = _Shifted(vs, C0, 4, st)
        vs.run_vcsr_spmm_gpu_ex(fmt, B, O, 64, dC, st, timed=True, kernel=vs.KERNEL_TILE,
                                accumulate=accumulate)
        return dC.numpy()

    ref = orc.spmm_f64(one.M, one.row_ptr, one.col, one.val, small)
    assert_within_tolerance(run(False), ref, one.row_ptr, one.val, small, f"R{R} O{O}")
    err = np.abs(run(True) - (C0 + ref)) - 2.0 ** -23 * (np.abs(C0) + np.abs(ref))
    l1 = np.array([np.abs(one.val[a:b]).sum() for a, b in zip(one.row_ptr, one.row_ptr[1:])])
    assert (err <= 1e-4 * l1[:, None] * np.abs(small).max()).all()

    row0, odd = B.host[0].copy(), np.full(O, np.inf, np.float32)
    odd[O // 2], odd[0] = np.nan, -np.inf
    lib = vs.load_library()
    try:
        assert lib.vcsr_memcpy_h2d(B.ptr, odd.ctypes.data, odd.nbytes, st.h) == 0
        st.sync()
        small[0] = odd
        got = run(False)
    finally:
        assert lib.vcsr_memcpy_h2d(B.ptr, row0.ctypes.data, row0.nbytes, st.h) == 0
        st.sync()
    ref = orc.spmm_f32(one.M, one.row_ptr, one.col, one.val, small)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.isinf(ref).any()
    fin = np.isfinite(ref)
    assert np.allclose(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("O", [7, 16, 30, 47, 100, 130, 1024])
def test_csr_wave_on_b_of_2gb_or_more_is_bit_exact(gpu, orc, st, big_b, O):
    """The plain-CSR kernel with B of 2 GiB (64-bit addresses) in each of its
    shapes: long rows taken by turns, short and empty rows, columns outside
    [0, N), the first and last rows of B: bit for bit the oracle's FP32 loop."""
    vs = gpu
    rng = np.random.default_rng(O)
    N = (1 << 29) // O + 2
    lens = [0, 1, 127, 128, 129, 0, 160, 1700, 3] + [5] * 40 + [257, 1] * 5
    rows = np.repeat(np.arange(len(lens)), lens)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    near = rng.integers(0, 1500, rows.size).astype(np.int32)
    near[1:3] = 0, 1499
    val = rng.standard_normal(rows.size).astype(np.float32)
    bad = rng.random(rows.size) < 0.1
    far = np.where(bad, np.where(rng.random(rows.size) < 0.5, -1, N), _far(near, N)).astype(np.int32)
    B = _Rows(big_b, N, O)
    small = np.concatenate([B.host[:750], B.host[N - 750:]])
    d = [vs.DeviceArray.from_numpy(x, st) for x in (rp, far, val)]
    dC = _Shifted(vs, np.full((len(lens), O), 5.0, np.float32), 4, st)
    vs.run_csr_wave_spmm_gpu(len(lens), N, *d, B, O, dC, st, timed=True)
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[~bad], minlength=len(lens)))])
    ref = orc.spmm_f32(len(lens), rp2.astype(np.int32), near[~bad], val[~bad], small)
    assert np.array_equal(dC.numpy().view(np.uint32), ref.view(np.uint32))
