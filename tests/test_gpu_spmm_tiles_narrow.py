"""CSR x dense on row tiles with FP32 operands of 17 to 64 columns (FP32 and BF16
values), each case with the tile kernel it is for: windows x columns per lane of
one wave.  test_spmm_forms.py checks that the cases reach those kernels."""
import numpy as np
import pytest

from test_gpu_spmm_tiles import check

pytestmark = pytest.mark.gpu

# (precision, k, kernel): 64 or more non-zeros per row take the tiles from k = 17 on
CASES = [(prec, k, (1, 2 if k <= 32 else 4)) for prec in ("f32", "bf16") for k in (17, 18, 31, 32, 33, 34, 63, 64)]


def wide_band(m=60000, band=110, per=72, seed=7):
    """Rows of 72 non-zeros in a band of 110 columns: 430,000 listed columns."""
    rng = np.random.default_rng(seed)
    lo = np.minimum(np.maximum(np.arange(m) - band // 2, 0), m - band)
    skip = rng.integers(0, band - per + 1, (m, 1))
    ci = lo[:, None] + skip + np.arange(per)[None, :]
    rp = (per * np.arange(m + 1)).astype(np.int32)
    return rp, ci.ravel().astype(np.int32), rng.standard_normal(m * per)


@pytest.mark.parametrize("prec,k,kernel", CASES)
def test_fp32_windows(pls, orc, prec, k, kernel):
    rp, ci, v = wide_band()
    bad = [(100, k - 1, np.inf), (20000, 0, np.nan), (20001, 16, -np.inf)]
    check(pls, orc, rp, ci, v, 60000, k, prec, 0.5 if k % 2 else 0.0, bad=bad)
