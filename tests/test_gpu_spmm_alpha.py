"""alpha in CSR x dense: multiplied into the stored values, whatever kernel the
number of columns takes, so that products whose unscaled sums leave the range of
the type stay finite, at every width alike."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", [1, 5, 8, 16, 33, 64, 65, 128, 161])
def test_alpha_before_the_sum(pls, orc, gen, k, prec):
    import torch

    hdt, tdt, big = (np.float64, torch.float64, 1e200) if prec == "f64" else (np.float32, torch.float32, 1e25)
    rng = np.random.default_rng(k)
    rp, ci, v = gen.stencil27(16)
    m = 16 ** 3
    v = (v * rng.uniform(0.5, 1.5, len(v))).astype(hdt)
    Bh = rng.uniform(-1, 1, (m, k)).astype(hdt)
    # powers of two: exact scalings of the whole product
    sa = hdt(2.0 ** np.floor(np.log2(big)))
    A = pls.SpMat.csr(m, m, rp, ci, v * sa)
    B = torch.from_numpy(Bh * sa).cuda()
    C = torch.zeros((m, k), dtype=tdt, device="cuda")
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k, float(1 / sa))
    torch.cuda.synchronize()
    got = C.cpu().numpy().astype(np.float64) / float(sa)
    ref = orc.spmm(m, k, rp, ci, v.astype(np.float64), Bh.astype(np.float64))
    mag = orc.spmm(m, k, rp, ci, abs(v).astype(np.float64), abs(Bh).astype(np.float64))
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    assert (np.abs(got - ref) <= (np.diff(rp)[:, None] + 6) * u * mag).all()
