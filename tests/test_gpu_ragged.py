"""GPU tests of widths and alignments that do not fit a lane's vector: the
kernels read and write rows of B and C with 16-byte accesses at any 4-byte
boundary, the last vector of a row moved back to end with it."""
import numpy as np
import pytest

from test_gpu_parity import _block_csr, _Shifted

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
    """16-row MFMA tiles: lanes of 1, 2 and 4 floats with a moved-back last
    vector, bit for bit the oracle's FP32 loop; C += A*B on top of C0 = 2
    stays within one rounding of it."""
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
