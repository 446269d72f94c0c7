"""The batch kernel's persistent loop (more tiles than workgroups: the next tile
loaded while the current one is computed) and its SELL-C-sigma tiles beside and
after the CSR tiles.  test_spmm_forms.py checks which launches the cases make."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def problems(gen, kind):
    """Uneven problems with every k, few or many tiles; "thin": many short rows, k = 1."""
    out = []
    rng = np.random.default_rng(9)
    for p, k in enumerate([1, 1, 1, 1, 4] if kind == "thin" else [1, 4, 1, 16, 2, 1, 8, 1]):
        m = {"few": 300, "many": 36000, "thin": 140000 if k == 1 else 300}[kind] + 101 * p
        out.append((m, *gen.banded(m, *((8, 1, 3) if kind == "thin" else (64, 5, 40)), p + 1), k))
    # an empty row, a row longer than a staged tile, tiles of single-entry rows
    # and of exactly 2048 entries from odd positions
    lens = np.r_[0, 3001, np.ones(1501, int), 1, np.full(64, 32), 0, 2047, 1, 5]
    for k in (1, 4):
        m = len(lens)
        rp = np.r_[0, np.cumsum(lens)].astype(np.int32)
        out.append((m, rp, rng.integers(0, m, rp[-1]).astype(np.int32), rng.standard_normal(rp[-1]), k))
    return out


# (problems, tile_nnz, SELL C, SELL sigma)
CASES = [("few", 2048, 0, 0), ("few", 2048, 32, 256), ("few", 2048, 64, 0), ("many", 256, 0, 0), ("many", 64, 32, 0),
         ("many", 64, 64, 1024), ("many", 512, 32, 256), ("many", 100000, 64, 64), ("thin", 64, 64, 0)]


@pytest.mark.parametrize("prec,beta", [("f64", 0.0), ("f64", 0.5), ("f32", 0.5), ("bf16", 0.0)])
@pytest.mark.parametrize("kind,tile,C,sigma", CASES)
def test_batch_loop(pls, orc, gen, kind, tile, C, sigma, prec, beta):
    import torch

    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    probs = problems(gen, kind)
    mats = [pls.SpMat.csr(m, m, rp, ci, v.astype(hdt)) for m, rp, ci, v, _ in probs]
    B = pls.Batch(mats, [p[4] for p in probs], pls.VALUES_BF16 if prec == "bf16" else pls.VALUES_NATIVE)
    B.set_shape(tile, [2, 2, 2, 8, 8], [1, 1, 2, 1, 2])
    if C:
        B.set_sell(C, sigma)
    rng = np.random.default_rng(tile + C)
    Xh = [rng.uniform(-1, 1, (p[0], p[4])).astype(hdt) for p in probs]
    Yh = [rng.uniform(-1, 1, (p[0], p[4])).astype(hdt) for p in probs]
    X = [torch.from_numpy(x).cuda() for x in Xh]
    Y = [torch.full((p[0], p[4]), float("nan"), dtype=tdt, device="cuda") for p in probs]
    B.set_operands([x.data_ptr() for x in X], [y.data_ptr() for y in Y])
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    for _ in range(3):  # the first launch captures, the others replay
        for y, h in zip(Y, Yh):
            y.copy_(torch.from_numpy(h)) if beta else y.fill_(float("nan"))
        B.exec(0.75, beta)
        torch.cuda.synchronize()
        for (m, rp, ci, v, k), x, h, y in zip(probs, Xh, Yh, Y):
            s = v.astype(hdt).astype(np.float64)
            if prec == "bf16":
                s = torch.from_numpy(v.astype(np.float32)).to(torch.bfloat16).double().numpy()
            x, old = x.astype(np.float64), h.astype(np.float64) if beta else None
            ref = orc.spmm(m, k, rp, ci, s, x, 0.75, beta, old)
            mag = orc.spmm(m, k, rp, ci, abs(s), abs(x), 0.75, beta, None if old is None else abs(old))
            lim = (np.diff(rp)[:, None] + 6) * u * mag + 1e-300  # rounding bound of a sum in any order
            assert (np.abs(y.double().cpu().numpy() - ref) <= lim).all()
