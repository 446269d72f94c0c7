"""Subnormal values in the matrix-core products: operands and results below the
normal range keep their bits (one rounding of the smallest subnormal per entry)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("which", ["A", "B", "product"])
@pytest.mark.parametrize("kind,k", [("csr", 8), ("csr", 64), ("csr", 128), ("bsr4", 7), ("bsr4", 32), ("bsr8", 8), ("bsr8", 64)])
def test_subnormals(pls, gen, kind, k, which, prec):
    import torch

    hdt, tdt, e, tiny, u = ((np.float64, torch.float64, -1060, 2.0 ** -1074, 2.0 ** -53) if prec == "f64" else
                            (np.float32, torch.float32, -140, 2.0 ** -149, 2.0 ** -24))
    rng = np.random.default_rng(k)
    sa, sb = {"A": (e, 0), "B": (0, e), "product": (e // 2, e - e // 2)}[which]
    if kind == "csr":
        rp, ci, v = gen.stencil27(12)
        m, b = 12 ** 3, 1
    else:
        b = int(kind[-1])
        rp, ci, v = gen.block_stencil(5, 5, 5, b, 3)
        m = 125 * b
    v = (np.ldexp(rng.uniform(0.5, 1.5, len(v)) * np.sign(v), sa)).astype(hdt)
    Bh = np.ldexp(rng.uniform(-1, 1, (m, k)), sb).astype(hdt)
    if b == 1:
        A = pls.SpMat.csr(m, m, rp, ci, v)
        M = sp.csr_matrix((v.astype(np.longdouble), ci, rp), shape=(m, m))
    else:
        A = pls.SpMat.bsr(pls.ROW_MAJOR, m, m, b, rp, ci, v)
        M = sp.bsr_matrix((v.astype(np.float64).reshape(-1, b, b), ci, rp), shape=(m, m)).tocsr().astype(np.longdouble)
    B, C = torch.from_numpy(Bh).cuda(), torch.zeros((m, k), dtype=tdt, device="cuda")
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
    torch.cuda.synchronize()
    ref = M @ Bh.astype(np.longdouble)
    mag = abs(M) @ abs(Bh.astype(np.longdouble))
    lim = (np.diff(M.indptr)[:, None] + 6) * (u * mag + tiny)
    assert (np.abs(C.cpu().numpy().astype(np.longdouble) - ref) <= lim).all()
    assert (np.abs(ref) > lim).mean() > 0.5  # a flush to zero would be seen
