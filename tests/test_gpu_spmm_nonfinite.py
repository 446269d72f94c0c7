"""Infinite and NaN values of B in the matrix-core products, which multiply more
than the stored entries: every element equals the entry-by-entry product, and
few or many such values cost little."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_spmm_tiles import shared_rows

pytestmark = pytest.mark.gpu

BAD = ["entry", "row", "nan column", "inf column", "signs", "all"]


def spoil(Bh, what):
    n, k = Bh.shape
    if what == "entry":
        Bh[n // 2, k // 2] = np.inf
        Bh[n // 3, k - 1] = np.nan
        Bh[n // 4, 0] = -np.inf
    elif what == "row":
        Bh[n // 2] = np.inf
    elif what == "nan column":
        Bh[:, k - 1] = np.nan
    elif what == "inf column":
        Bh[:, k // 2] = np.inf
    elif what == "signs":
        Bh[:, k // 2] = np.where(np.arange(n) % 2, np.inf, -np.inf)
    elif what == "all":
        Bh[:] = np.where(Bh > 0.9, np.nan, np.inf)


def compare(got, M, Bh, old, beta, prec):
    """got against 0.75 M B + beta old, M the stored entries in FP64."""
    with np.errstate(invalid="ignore"):
        ref = 0.75 * (M @ Bh) + (beta * old if beta else 0.0)
    fin = np.isfinite(Bh)
    mag = 0.75 * (abs(M) @ np.where(fin, abs(Bh), 0.0)) + abs(beta * old if beta else 0.0)
    assert (np.isnan(got) == np.isnan(ref)).all()
    inf = np.isinf(ref)
    assert (got[inf] == ref[inf]).all()
    ok = np.isfinite(ref)
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    lim = (np.diff(M.indptr)[:, None] + 6) * u * mag + 1e-300  # rounding bound of a sum in any order
    assert (np.abs(got[ok] - ref[ok]) <= lim[ok]).all()


def run(pls, A, m, n, k, prec, beta, M, what):
    import torch

    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    rng = np.random.default_rng(k)
    Bh = rng.uniform(-1, 1, (n, k)).astype(hdt)
    spoil(Bh, what)
    old = rng.uniform(-1, 1, (m, k)).astype(hdt)
    B, C = torch.from_numpy(Bh).cuda(), torch.from_numpy(old.copy() if beta else np.full_like(old, np.nan)).cuda()
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k, 0.75, beta)
    torch.cuda.synchronize()
    compare(C.double().cpu().numpy(), M, Bh.astype(np.float64), old.astype(np.float64), beta, prec)


def stored(pls, A, v, prec):
    import torch

    if prec == "bf16":
        A.set_precision(pls.VALUES_BF16)
        return torch.from_numpy(v.astype(np.float32)).to(torch.bfloat16).double().numpy()
    return v.astype(np.float64 if prec == "f64" else np.float32).astype(np.float64)


@pytest.mark.parametrize("what", BAD)
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("k,beta", [(65, 0.5), (128, 0.0), (161, 0.5)])
def test_row_tiles(pls, k, beta, prec, what):
    rp, ci, v = shared_rows(np.random.default_rng(11))
    v[::50] = 0.0  # a stored zero of a CSR matrix does multiply
    m, n = len(rp) - 1, 1000
    A = pls.SpMat.csr(m, n, rp, ci, v.astype(np.float64 if prec == "f64" else np.float32))
    # (entries stored twice stay two entries)
    M = sp.csr_matrix((stored(pls, A, v, prec), ci, rp), shape=(m, n))
    run(pls, A, m, n, k, prec, beta, M, what)


@pytest.mark.parametrize("what", BAD)
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("b", [4, 8])
@pytest.mark.parametrize("per,k,beta", [(2, 7, 0.5), (2, 33, 0.0), (20, 3, 0.0), (20, 12, 0.5), (20, 40, 0.5), (20, 130, 0.0)])
@pytest.mark.parametrize("layout", ["rows", "columns"])
def test_blocks(pls, gen, layout, per, k, beta, b, prec, what):
    mb = 60
    rp, ci, v = gen.block_random(mb, b, per, 30, 5)
    v = v.copy()
    v[::3] = 0.0  # a stored zero of a block adds nothing
    lay = pls.ROW_MAJOR if layout == "rows" else pls.COL_MAJOR
    A = pls.SpMat.bsr(lay, mb * b, mb * b, b, rp, ci, v.astype(np.float64 if prec == "f64" else np.float32))
    s = stored(pls, A, v, prec).reshape(-1, b, b)
    if layout == "columns":
        s = s.transpose(0, 2, 1)
    M = sp.csr_matrix(sp.bsr_matrix((s, ci, rp), shape=(mb * b, mb * b)))
    M.eliminate_zeros()
    run(pls, A, mb * b, mb * b, k, prec, beta, M, what)


@pytest.mark.parametrize("kind", ["tiles", "blocks"])
def test_a_column_of_nan_costs_little(pls, gen, kind):
    """Each product against itself on a finite B: recomputing every element of
    the waves that hold a NaN took 12 (tiles) and 45 (blocks) times as long."""
    import torch

    if kind == "tiles":
        rp, ci, v = gen.stencil27(64)
        m, k = 64 ** 3, 32
        A = pls.SpMat.csr(m, m, rp, ci, v)
    else:
        rp, ci, v = gen.block_stencil(20, 20, 20, 8, 3)
        m, k = 64000, 8
        A = pls.SpMat.bsr(pls.ROW_MAJOR, m, m, 8, rp, ci, v)
    B = torch.rand((m, k), dtype=torch.float64, device="cuda")
    C = torch.empty_like(B)

    def us():
        best = float("inf")
        for _ in range(6):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(10):
                A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]))
        return best

    us()
    finite = us()
    B[:, k // 2] = float("nan")
    assert us() < 4 * finite
