"""CSR x dense products that gather B rows directly (scattered columns, k < 8):
row lengths around the whole-workgroup limit (512) and the lane-group steps, all
window widths, odd leading dimensions and pointers with element alignment only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M, N = 700, 40000
LENGTHS = [0, 1, 2, 3, 5, 8, 15, 16, 17, 31, 33, 64, 65, 200, 511, 512, 513, 514, 1027, 3000]


def operand(rng):
    lens = np.array([LENGTHS[i % len(LENGTHS)] if i % 3 == 0 else i % 23 for i in range(M)])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(N, int(l), replace=False)) for l in lens]).astype(np.int32)
    return rp, ci, rng.standard_normal(int(rp[-1])), lens


@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 33, 64, 65, 100, 128, 129, 257, 300])
def test_spmm_gather(pls, orc, k, prec, beta):
    import torch

    rng = np.random.default_rng(k)
    rp, ci, v, lens = operand(rng)
    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    A = pls.SpMat.csr(M, N, rp, ci, v.astype(hdt))
    stored = v.astype(hdt).astype(np.float64)
    if prec == "bf16":
        A.set_precision(pls.VALUES_BF16)
        stored = torch.from_numpy(v.astype(np.float32)).to(torch.bfloat16).double().numpy()
    ldb, ldc, off = k + 3, k + 1, 1  # odd strides, pointers one element off
    Bh = rng.uniform(-1, 1, (N, k)).astype(hdt)
    Ch = rng.uniform(-1, 1, (M, k)).astype(hdt)
    if beta == 0.0:
        Ch[::7] = np.nan  # never read
    B = torch.full((N * ldb + off,), float("nan"), dtype=tdt, device="cuda")
    B[off:].view(N, ldb)[:, :k] = torch.from_numpy(Bh).cuda()
    C = torch.full((M * ldc + off,), 7.0, dtype=tdt, device="cuda")
    Cv = C[off:].view(M, ldc)
    Cv[:, :k] = torch.from_numpy(Ch).cuda()
    es = B.element_size()
    A.spmm_async(k, B.data_ptr() + off * es, ldb, C.data_ptr() + off * es, ldc, 0.75, beta)
    torch.cuda.synchronize()
    if k >= 8:
        assert A.spmm_info()["blocks_state"] == -1  # the gather kernel ran
    assert bool((Cv[:, k:] == 7.0).all()) and float(C[0]) == 7.0  # nothing past column k
    ref = orc.spmm(M, k, rp, ci, stored, Bh.astype(np.float64), 0.75, beta,
                   Ch.astype(np.float64) if beta else None)
    # rounding bound of a sum of len + 3 terms in any order
    mag = orc.spmm(M, k, rp, ci, np.abs(stored), np.abs(Bh).astype(np.float64), 0.75, beta,
                   np.abs(Ch).astype(np.float64) if beta else None)
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    err = np.abs(Cv[:, :k].double().cpu().numpy() - ref)
    assert np.all(err <= (lens[:, None] + 6) * u * mag + 1e-300)


@pytest.mark.parametrize("k", [3, 33])
def test_spmm_gather_infinities_stay_in_their_rows(pls, orc, k):
    """An infinite B row reaches exactly the rows that reference it."""
    import torch

    rng = np.random.default_rng(5)
    rp, ci, v, _ = operand(rng)
    Bh = rng.uniform(-1, 1, (N, k))
    hit = int(ci[100])
    Bh[hit] = np.inf
    A = pls.SpMat.csr(M, N, rp, ci, v)
    B = torch.from_numpy(Bh).cuda()
    C = torch.zeros((M, k), dtype=torch.float64, device="cuda")
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
    torch.cuda.synchronize()
    rows = np.repeat(np.arange(M), np.diff(rp))[ci == hit]
    bad = ~np.isfinite(C.cpu().numpy()).all(axis=1)
    assert set(np.nonzero(bad)[0]) == set(rows.tolist())
