"""CSR x dense products on row tiles (k > 16, at least 10 non-zeros per row, rows
that share columns): runs of 1 to 32 rows, empty rows, columns stored twice, rows
too long for a list, every window width, odd leading dimensions and pointers with
element alignment only; infinite and NaN values of B, value updates, TRANS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shared_rows(rng, m=900, n=1000):
    """Bands of ~20 non-zeros with empty rows, duplicates and rows of 300 and 1500."""
    rows = []
    for i in range(m):
        lo = min(max(0, i - 25), n - 50)
        cols = np.sort(rng.choice(np.arange(lo, lo + 50), int(rng.integers(12, 30)), replace=False))
        if i % 97 == 5:
            cols = np.sort(rng.choice(n, 300, replace=False))
        if i % 401 == 7:
            cols = np.sort(rng.integers(0, 60, 1500))
        if 400 <= i < 460:
            cols = np.array([], np.int64)
        if i % 19 == 0 and len(cols):
            cols = np.sort(np.concatenate([cols, cols[:1], cols[:1]]))
        rows.append(cols)
    rp = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    return rp, np.concatenate(rows).astype(np.int32), rng.standard_normal(int(rp[-1]))


def check(pls, orc, rp, ci, v, n, k, prec, beta, rows=0, bad=()):
    import torch

    rng = np.random.default_rng(k)
    m = len(rp) - 1
    hdt, tdt = (np.float64, torch.float64) if prec == "f64" else (np.float32, torch.float32)
    A = pls.SpMat.csr(m, n, rp, ci, v.astype(hdt))
    A.set_spmm_rows(rows) if rows else None
    stored = v.astype(hdt).astype(np.float64)
    if prec == "bf16":
        A.set_precision(pls.VALUES_BF16)
        stored = torch.from_numpy(v.astype(np.float32)).to(torch.bfloat16).double().numpy()
    ldb, ldc, off = k + 3, k + 1, 1
    Bh = rng.uniform(-1, 1, (n, k)).astype(hdt)
    for r, c, x in bad:
        Bh[r, c] = x
    Ch = rng.uniform(-1, 1, (m, k)).astype(hdt)
    if beta == 0.0:
        Ch[::7] = np.nan  # never read
    B = torch.full((n * ldb + off,), float("nan"), dtype=tdt, device="cuda")
    B[off:].view(n, ldb)[:, :k] = torch.from_numpy(Bh).cuda()
    C = torch.full((m * ldc + off,), 7.0, dtype=tdt, device="cuda")
    Cv = C[off:].view(m, ldc)
    Cv[:, :k] = torch.from_numpy(Ch).cuda()
    es = B.element_size()
    A.spmm_async(k, B.data_ptr() + off * es, ldb, C.data_ptr() + off * es, ldc, 0.75, beta)
    torch.cuda.synchronize()
    assert A.spmm_info()["blocks_state"] == 1
    assert bool((Cv[:, k:] == 7.0).all()) and float(C[0]) == 7.0  # nothing past column k
    got = Cv[:, :k].double().cpu().numpy()
    B64 = Bh.astype(np.float64)
    hit = np.zeros(m, bool)  # rows that reference a non-finite value
    for r, c, x in bad:
        mine = np.repeat(np.arange(m), np.diff(rp))[ci == r]
        hit[mine] = True
        assert not np.isfinite(got[mine, c]).any()
        B64[r, c] = 0.0
    old = Ch.astype(np.float64) if beta else None
    ref = orc.spmm(m, k, rp, ci, stored, B64, 0.75, beta, old)
    mag = orc.spmm(m, k, rp, ci, np.abs(stored), np.abs(B64), 0.75, beta, None if old is None else np.abs(old))
    u = 2.0 ** -53 if prec == "f64" else 2.0 ** -24
    lim = (np.diff(rp)[:, None] + 6) * u * mag + 1e-300  # rounding bound of a sum in any order
    ok = np.abs(got - ref) <= lim
    cols = [c for _, c, _ in bad]
    ok[np.ix_(hit, cols)] = True
    assert ok.all()


@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("k", [65, 96, 100, 127, 128, 129, 200, 257])
def test_tiles_uneven_rows(pls, orc, k, prec, beta):
    rp, ci, v = shared_rows(np.random.default_rng(1))
    check(pls, orc, rp, ci, v, 1000, k, prec, beta)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_tiles_consecutive_and_clustered(pls, orc, gen, rows, prec):
    rp, ci, v = gen.stencil27(14)
    v = v * np.random.default_rng(2).uniform(0.5, 1.5, len(v))
    check(pls, orc, rp, ci, v, 14 ** 3, 70, prec, 0.5, rows)
    brp, bci, bv = gen.block_stencil(5, 4, 4, 8, 3)
    rp, ci, v = gen.bsr_to_csr_rowmajor(brp, bci, bv, 8)  # lists of 256
    check(pls, orc, rp, ci, v, 640, 70, prec, 0.0, rows)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", [17, 24, 31, 32, 33, 63, 64])
def test_tiles_narrow_windows(pls, orc, gen, k, prec):
    rp, ci, v = gen.stencil27(40)
    v = v * np.random.default_rng(4).uniform(0.5, 1.5, len(v))
    check(pls, orc, rp, ci, v, 40 ** 3, k, prec, 0.0)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_tiles_nonfinite_values_stay_in_their_rows(pls, orc, prec, bad):
    """A tile multiplies columns that only some of its rows have."""
    rp, ci, v = shared_rows(np.random.default_rng(6))
    hits = [(int(ci[50]), 3, bad), (int(ci[9000]), 64, bad)]
    check(pls, orc, rp, ci, v, 1000, 66, prec, 0.0, bad=hits)


def test_tiles_updates_both_forms_and_trans(pls, orc, gen):
    """Value updates reach the tiles and the LDS blocks of one handle, and a
    TRANS product runs on tiles of the transpose."""
    import torch

    rng = np.random.default_rng(8)
    rp, ci, v = gen.stencil27(16)
    m = 16 ** 3
    v = v * rng.uniform(0.5, 1.5, len(v))
    A = pls.SpMat.csr(m, m, rp, ci, v)

    def product(k):
        Bv = rng.uniform(-1, 1, (m, k))
        B, C = torch.from_numpy(Bv).cuda(), torch.zeros((m, k), dtype=torch.float64, device="cuda")
        A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
        torch.cuda.synchronize()
        ref = orc.spmm(m, k, rp, ci, v, Bv)
        assert np.linalg.norm(C.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)

    for k in (80, 8):
        product(k)
    pick = rng.choice(len(v), 200, replace=False)
    r = np.searchsorted(rp, pick, side="right") - 1
    v[pick] = rng.standard_normal(200)
    A.update(r, ci[pick], v[pick])
    for k in (80, 8):
        product(k)
    k = 72
    Bv = rng.uniform(-1, 1, (m, k))
    Bo = pls.SpMat.dense(pls.ROW_MAJOR, m, k, k, Bv.reshape(-1))
    Co = pls.SpMat.null(m, k)
    T = pls.SpMat.csr(m, m, rp, ci, v)
    pls.spmm_exec(pls.TRANS, pls.NOTRANS, 1.0, T, Bo, 0.0, Co)
    D = np.zeros((m, k))
    np.add.at(D, ci, v[:, None] * np.repeat(Bv, np.diff(rp), axis=0))
    assert np.linalg.norm(Co.export_dense() - D) <= 1e-12 * np.linalg.norm(D)


@pytest.mark.parametrize("warm,k", [(16, 128), (128, 16)])
def test_first_use_of_a_form_inside_a_capture(pls, orc, warm, k):
    """A plan warmed with one width is captured with a width of the other form."""
    import torch

    rng = np.random.default_rng(5)
    rp, ci, v = shared_rows(rng)
    m, n = len(rp) - 1, 1000
    A = pls.SpMat.csr(m, n, rp, ci, v)
    Bh = rng.uniform(-1, 1, (n, max(k, warm)))
    B = torch.from_numpy(Bh[:, :k].copy()).cuda()
    Bw = torch.from_numpy(Bh[:, :warm].copy()).cuda()
    C, Cw = (torch.zeros((m, w), dtype=torch.float64, device="cuda") for w in (k, warm))
    prev = torch.cuda.current_stream()
    try:
        A.spmm_async(warm, Bw.data_ptr(), warm, Cw.data_ptr(), warm)
        torch.cuda.synchronize()
        side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            pls.set_stream(side.cuda_stream)
            A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)
    finally:
        pls.set_stream(prev.cuda_stream)
    mag = orc.spmm(m, k, rp, ci, np.abs(v), np.abs(Bh[:, :k]), 1.0, 0.0, None)
    for scale in (1.0, -2.0, 0.5):  # exact scalings: eager work between the replays
        B.copy_(torch.from_numpy(Bh[:, :k] * scale))
        C.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = C.cpu().numpy().copy()
        ref = orc.spmm(m, k, rp, ci, v, Bh[:, :k] * scale, 1.0, 0.0, None)
        lim = (np.diff(rp)[:, None] + 6) * 2.0 ** -53 * abs(scale) * mag + 1e-300
        assert (np.abs(got - ref) <= lim).all()
    A.spmm_async(k, B.data_ptr(), k, C.data_ptr(), k)  # outside: the form is built
    torch.cuda.synchronize()
    assert (np.abs(C.cpu().numpy() - ref) <= lim).all()


@pytest.mark.parametrize("k", [65, 96, 97, 161])
def test_narrow_window_for_the_rest(pls, orc, k):
    """Enough listed columns (320000) for a second launch: rests of 1, 32 and 33."""
    rng = np.random.default_rng(8)
    m, per = 100000, 20
    lo = np.minimum(np.maximum(np.arange(m) - 50, 0), m - 100)
    ci = (lo[:, None] + 5 * np.arange(per)[None, :] + rng.integers(0, 5, (m, per))).astype(np.int32)
    rp = (per * np.arange(m + 1)).astype(np.int32)
    bad = [(1000, k - 1, np.inf), (2000, 64, np.nan), (3000, 63, np.inf)]
    check(pls, orc, rp, ci.ravel(), rng.standard_normal(m * per), m, k, "f64", 0.5, bad=bad)
