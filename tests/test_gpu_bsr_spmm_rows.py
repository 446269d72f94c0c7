"""BSR x dense with a lane group per block row: the lines of the rule (mean blocks
per row and number of block rows) from both sides, every window of few columns.
test_spmm_forms.py checks which kernel each case takes."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

# (block rows, block size, blocks per row, precision, own lanes per block row)
CASES = [(49152, 4, 12, "f64", True), (49151, 4, 12, "f64", False), (16384, 4, 9, "f64", True), (16383, 4, 9, "f64", False),
         (16383, 4, 4, "f64", True), (16384, 4, 12, "f32", True), (16383, 4, 12, "f32", False), (16384, 4, 13, "bf16", False),
         (4096, 8, 5, "f64", True), (4095, 8, 5, "f64", False), (4095, 8, 3, "f64", True), (16384, 8, 11, "f32", True),
         (16383, 8, 11, "bf16", False), (4096, 8, 7, "bf16", True)]


@pytest.mark.parametrize("mb,b,per,prec,own", CASES)
def test_lines_of_the_rule(pls, gen, mb, b, per, prec, own):
    import torch

    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    rp, ci, v = gen.block_random(mb, b, per, 300, 5)
    n = mb * b
    s = v.astype(hdt).astype(np.float64)
    for layout in (pls.ROW_MAJOR, pls.COL_MAJOR):
        A = pls.SpMat.bsr(layout, n, n, b, rp, ci, v.astype(hdt))
        if prec == "bf16":
            A.set_precision(pls.VALUES_BF16)
            s = torch.from_numpy(v.astype(np.float32)).to(torch.bfloat16).double().numpy()
        blocks = s.reshape(-1, b, b)
        if layout == pls.COL_MAJOR:
            blocks = blocks.transpose(0, 2, 1)
        M = sp.bsr_matrix((blocks, ci, rp), shape=(n, n))
        absM = sp.bsr_matrix((abs(blocks), ci, rp), shape=(n, n))
        lens = np.repeat(np.diff(rp) * b, b)[:, None]
        for k, beta in ((1, 0.0), (3, 0.5), (4, 0.0), (6, 0.5), (8, 0.0), (11, 0.5), (16, 0.0), (19, 0.5)):
            rng = np.random.default_rng(k)
            Bh, old = (rng.uniform(-1, 1, (n, k)).astype(hdt) for _ in range(2))
            B, C = torch.from_numpy(Bh).cuda(), torch.from_numpy(old.copy() if beta else np.full_like(old, np.nan)).cuda()
            A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k, 0.75, beta)
            torch.cuda.synchronize()
            Bd, od = Bh.astype(np.float64), old.astype(np.float64)
            ref = 0.75 * (M @ Bd) + beta * od
            mag = 0.75 * (absM @ abs(Bd)) + beta * abs(od)
            u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
            assert (np.abs(C.double().cpu().numpy() - ref) <= (lens + 6) * u * mag + 1e-300).all()
