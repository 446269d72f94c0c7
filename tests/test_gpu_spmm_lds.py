"""CSR x dense products on row blocks staged in LDS: rows of every length around
the steps of 8, 4, 2 and 1, lists of both sizes, consecutive and clustered blocks,
every column chunk width, long rows, infinite and NaN values of B."""
import numpy as np
import pytest

from test_gpu_spmm_tiles import check, shared_rows

pytestmark = pytest.mark.gpu


def stepped_rows(m, band, longest, seed):
    """Banded rows of 0, 1, ..., `longest` non-zeros in turn."""
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(m):
        lo = min(max(0, i - band // 2), m - band)
        rows.append(np.sort(lo + rng.choice(band, i % (longest + 1), replace=False)))
    rp = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    return rp, np.concatenate(rows).astype(np.int32), rng.standard_normal(int(rp[-1]))


@pytest.mark.parametrize("k,beta", [(8, 0.0), (8, 0.5), (13, 0.5), (33, 0.0)])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("band,longest", [(40, 18), (100, 37), (200, 90)])
def test_stepped_rows(pls, orc, band, longest, rows, prec, k, beta):
    rp, ci, v = stepped_rows(1501, band, longest, band)
    check(pls, orc, rp, ci, v, 1501, k, prec, beta, rows=rows)


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
def test_long_empty_and_repeated(pls, orc, prec):
    rp, ci, v = shared_rows(np.random.default_rng(3))
    bad = [(30, 2, np.inf), (411, 5, np.nan), (700, 7, -np.inf)]
    check(pls, orc, rp, ci, v, 1000, 8, prec, 0.5, bad=bad)
