"""CSR x dense on two streams: a product that builds a device form of the row
blocks on one stream, the next of the same width at once on another."""
import numpy as np
import pytest

from test_gpu_spmm_tiles import shared_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("warm,k", [(0, 128), (0, 8), (8, 128), (128, 8)])
def test_form_built_on_one_stream_used_on_another(pls, orc, gen, warm, k, rows):
    import torch

    rng = np.random.default_rng(3)
    rp, ci, v = gen.stencil27(40)
    m = 40 ** 3
    v = v * rng.uniform(0.5, 1.5, len(v))
    Bh = rng.uniform(-1, 1, (m, k))
    B = torch.from_numpy(Bh).cuda()
    W = torch.zeros((m, max(warm, 1)), dtype=torch.float64, device="cuda")
    C1, C2 = (torch.zeros((m, k), dtype=torch.float64, device="cuda") for _ in range(2))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    A = pls.SpMat.csr(m, m, rp, ci, v)
    A.set_spmm_rows(rows)
    prev = torch.cuda.current_stream()
    torch.cuda.synchronize()
    try:
        if warm:
            A.spmm_async(warm, W.data_ptr(), warm, W.data_ptr(), warm)
            torch.cuda.synchronize()
        pls.set_stream(s1.cuda_stream)
        A.spmm_async(k, B.data_ptr(), k, C1.data_ptr(), k)
        pls.set_stream(s2.cuda_stream)
        A.spmm_async(k, B.data_ptr(), k, C2.data_ptr(), k)
        torch.cuda.synchronize()
    finally:
        pls.set_stream(prev.cuda_stream)
    ref = orc.spmm(m, k, rp, ci, v, Bh)
    lim = 40 * 2.0 ** -53 * orc.spmm(m, k, rp, ci, np.abs(v), np.abs(Bh))  # rounding bound, any order
    for C in (C1, C2):
        assert (np.abs(C.cpu().numpy() - ref) <= lim).all()


def test_updates_reach_a_form_used_on_another_stream(pls, orc, gen):
    """Values updated with the library on one stream, the products on another."""
    import torch

    rng = np.random.default_rng(4)
    rp, ci, v = gen.stencil27(20)
    m, k = 20 ** 3, 72
    A = pls.SpMat.csr(m, m, rp, ci, v.copy())
    Bh = rng.uniform(-1, 1, (m, k))
    B = torch.from_numpy(Bh).cuda()
    C = torch.zeros((m, k), dtype=torch.float64, device="cuda")
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    prev = torch.cuda.current_stream()
    torch.cuda.synchronize()
    try:
        for s, t in ((s1, s2), (s2, s1)):
            pls.set_stream(s.cuda_stream)
            A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
            torch.cuda.synchronize()
            pick = rng.choice(len(v), 500, replace=False)
            v[pick] = rng.standard_normal(500)
            A.update(np.searchsorted(rp, pick, side="right") - 1, ci[pick], v[pick])
            pls.set_stream(t.cuda_stream)
            A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
            torch.cuda.synchronize()
            lim = 40 * 2.0 ** -53 * orc.spmm(m, k, rp, ci, np.abs(v), np.abs(Bh))
            assert (np.abs(C.cpu().numpy() - orc.spmm(m, k, rp, ci, v, Bh)) <= lim).all()
    finally:
        pls.set_stream(prev.cuda_stream)
