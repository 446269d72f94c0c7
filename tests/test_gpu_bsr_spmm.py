"""BSR x dense on the matrix cores: block rows around the block steps of a wave
(4, 8, 16 and 64 blocks), every window width and remainder of k, odd leading
dimensions and pointers with element alignment only, both block layouts; and
stored zeros against infinite and NaN values of B."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# blocks per block row: long rows (lane groups share one), short ones (a group each)
COUNTS = {"long": [0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 27, 33, 63, 64, 65, 130] * 2,
          "short": [0, 1, 2, 3, 4, 5, 0, 1, 1, 70, 2] + [1, 3] * 13}
NB = 140


def operand(rng, b, layout, pls, rows="long"):
    counts = np.array(COUNTS[rows])
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(NB, int(c), replace=False)) for c in counts]).astype(np.int32)
    blocks = rng.standard_normal((len(ci), b, b))
    blocks[rng.random(blocks.shape) < 0.05] = 0.0  # stored zeros
    stored = blocks if layout == pls.ROW_MAJOR else blocks.transpose(0, 2, 1)
    return counts, rp, ci, blocks, np.ascontiguousarray(stored).reshape(-1)


def dense_of(b, rp, ci, blocks):
    D = np.zeros(((len(rp) - 1) * b, NB * b))
    for r in range(len(rp) - 1):
        for p in range(rp[r], rp[r + 1]):
            D[r * b:(r + 1) * b, ci[p] * b:(ci[p] + 1) * b] = blocks[p]
    return D


@pytest.mark.parametrize("layout", ["row", "col"])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("b", [4, 8])
@pytest.mark.parametrize("rows", ["long", "short"])
def test_bsr_spmm_tiles(pls, rows, b, prec, layout):
    import torch

    rng = np.random.default_rng(b)
    lay = pls.ROW_MAJOR if layout == "row" else pls.COL_MAJOR
    counts, rp, ci, blocks, stored = operand(rng, b, lay, pls, rows)
    m, n = len(counts) * b, NB * b
    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    D = dense_of(b, rp, ci, blocks.astype(hdt).astype(np.float64))
    if prec == "bf16":
        D = torch.from_numpy(D.astype(np.float32)).to(torch.bfloat16).double().numpy()
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    terms = np.repeat(counts * b, b)[:, None] + 6
    for k in (1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 128, 129, 200, 257):
        beta = 0.5 if k % 2 else 0.0
        A = pls.SpMat.bsr(lay, m, n, b, rp, ci, stored.astype(hdt))
        if prec == "bf16":
            A.set_precision(pls.VALUES_BF16)
        ldb, ldc, off = k + 3, k + 1, 1
        Bh = rng.uniform(-1, 1, (n, k)).astype(hdt)
        Ch = rng.uniform(-1, 1, (m, k)).astype(hdt)
        if beta == 0.0:
            Ch[::5] = np.nan  # never read
        B = torch.full((n * ldb + off,), float("nan"), dtype=tdt, device="cuda")
        B[off:].view(n, ldb)[:, :k] = torch.from_numpy(Bh).cuda()
        C = torch.full((m * ldc + off,), 7.0, dtype=tdt, device="cuda")
        Cv = C[off:].view(m, ldc)
        Cv[:, :k] = torch.from_numpy(Ch).cuda()
        es = B.element_size()
        A.spmm_async(k, B.data_ptr() + off * es, ldb, C.data_ptr() + off * es, ldc, 0.75, beta)
        torch.cuda.synchronize()
        assert bool((Cv[:, k:] == 7.0).all()) and float(C[0]) == 7.0
        old = Ch.astype(np.float64) if beta else 0.0
        ref = 0.75 * (D @ Bh.astype(np.float64)) + beta * old
        mag = 0.75 * (np.abs(D) @ np.abs(Bh).astype(np.float64)) + beta * np.abs(old)
        err = np.abs(Cv[:, :k].double().cpu().numpy() - ref)
        # rounding bound of a sum of the row's terms in any order, here and in the reference
        assert np.all(err <= terms * (u + 2.0 ** -53) * mag), k


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("b", [4, 8])
@pytest.mark.parametrize("rows", ["long", "short"])
def test_bsr_spmm_stored_zero_against_nonfinite(pls, rows, b, prec, bad):
    """0 (stored) * Inf or NaN adds nothing; a non-zero value passes it on."""
    import torch

    rng = np.random.default_rng(3)
    hdt = np.float64 if prec == "f64" else np.float32
    counts, rp, ci, blocks, stored = operand(rng, b, pls.ROW_MAJOR, pls, rows)
    D = dense_of(b, rp, ci, blocks.astype(hdt).astype(np.float64))
    m, n, k = D.shape[0], NB * b, 33
    Bh = rng.uniform(-1, 1, (n, k)).astype(hdt)
    hit = [(3, 5), (17, 0), (40, 32), (41, 32)]
    for r, c in hit:
        Bh[r, c] = bad
    A = pls.SpMat.bsr(pls.ROW_MAJOR, m, n, b, rp, ci, stored.astype(hdt))
    B = torch.from_numpy(Bh).cuda()
    C = torch.zeros((m, k), dtype=B.dtype, device="cuda")
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
    torch.cuda.synchronize()
    with np.errstate(invalid="ignore"):
        terms = np.where(D[:, :, None] != 0.0, D[:, :, None] * Bh.astype(np.float64)[None], 0.0)
        ref = terms.sum(axis=1)
        mag = np.abs(terms).sum(axis=1)
    got = C.double().cpu().numpy()
    fine = np.isfinite(ref)
    assert not fine.all() and np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)])
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    got, ref = np.where(fine, got, 0.0), np.where(fine, ref, 0.0)
    lim = (np.repeat(counts * b, b)[:, None] + 6) * (u + 2.0 ** -53) * mag
    assert np.all(np.abs(got - ref)[fine] <= lim[fine])
