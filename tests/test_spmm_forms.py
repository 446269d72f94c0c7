"""The device forms of a plan's SpMM row blocks (staged blocks, row tiles): when
they are built, what orders them, and which one a product runs on, from the HIP
calls of the library on a runtime without a device (hip_stub.cpp)."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent

PRELUDE = """
import ctypes, sys
sys.modules["torch"] = None  # one HIP runtime: the stub
sys.path[:0] = [{pkg!r}, {here!r}]
stub = ctypes.CDLL(None)
stub.stub_log.restype = ctypes.c_char_p
stub.stub_live.restype = ctypes.c_size_t
stub.stub_limit.argtypes = [ctypes.c_size_t]
stub.stub_host_limit.argtypes = [ctypes.c_size_t]
stub.stub_capture.argtypes = [ctypes.c_void_p]
import numpy as np
import plsparse as P
from test_gpu_spmm_tiles import shared_rows
rp, ci, v = shared_rows(np.random.default_rng(1))
m, n = len(rp) - 1, 1000
A = P.SpMat.csr(m, n, rp, ci, v)
buf = np.zeros(1 << 20)
S1, S2 = 0x11, 0x22

def product(k, stream=S1, h=None):
    '''The HIP calls of one product, as tuples of words.'''
    P.set_stream(stream)
    stub.stub_clear()
    (h or A).spmm_async(k, buf.ctypes.data, k, buf.ctypes.data, k)
    return [tuple(x.split()) for x in stub.stub_log().decode().splitlines()]

def kernels(calls):
    return [c[1] for c in calls if c[0] == "launch"]

def form(calls):
    return [f for f in ("k_spmm_tile", "k_spmm_lds", "k_spmm_gather") if any(f in x for x in kernels(calls))][0]
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = tmp_path_factory.mktemp("hip") / "libhipstub.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", str(HERE / "hip_stub.cpp"), "-o", str(out)], check=True)
    return out


@pytest.fixture
def run(stub):
    def go(body):
        env = dict(os.environ)
        env["LD_PRELOAD"] = ":".join(x for x in (str(stub), env.get("LD_PRELOAD", "")) if x)
        code = PRELUDE.format(pkg=str(HERE.parent / "perf-libs-sparse_amd"), here=str(HERE)) + body
        r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


@pytest.mark.parametrize("warm,k", [(0, 128), (0, 8), (16, 128), (128, 16)])
def test_values_are_written_before_a_form_is_used(run, warm, k):
    """The gather of a form's values is waited for on its stream, whichever
    stream the products before and after it run on."""
    run(f"""
A.set_spmm_rows(2)  # clustered: both forms copy values
if {warm}:
    product({warm})
calls = product({k}, S1)
at = [i for i, c in enumerate(calls) if c[0] == "launch" and "k_gather_vals" in c[1]]
assert at, calls
end = [i for i, c in enumerate(calls) if c[0] == "launch" and "k_spmm" in c[1]][0]
for i in at:
    assert ("sync", calls[i][2]) in calls[i:end], calls
later = product({k}, S2)
assert not any("k_gather_vals" in f for f in kernels(later)) and form(later) == form(calls)
""")


def test_threads_share_a_plan(run):
    """Products of both widths from several threads on one warmed handle: each
    form is built once, and every product runs on the form of its width."""
    run("""
import threading
product(8)
stub.stub_clear()
P.set_stream(S1)
def work(k):
    for _ in range(50):
        A.spmm_async(k, buf.ctypes.data, k, buf.ctypes.data, k)
ts = [threading.Thread(target=work, args=(k,)) for k in (128, 16, 128, 16)]
[t.start() for t in ts], [t.join() for t in ts]
ran = kernels([tuple(x.split()) for x in stub.stub_log().decode().splitlines()])
assert sum("k_spmm_tile" in f for f in ran) == 100 and sum("k_spmm_lds" in f for f in ran) == 100
assert sum("k_gather_vals" in f for f in ran) == 1  # the tiles' values
""")


@pytest.mark.parametrize("warm,k,kernel", [(16, 128, "k_spmm_tile"), (128, 16, "k_spmm_lds"), (128, 8, "k_spmm_lds")])
def test_captured_product_runs_on_the_form_of_its_width(run, warm, k, kernel):
    """A plan warmed with one width, captured with one of the other form: the
    form is built beside the capture, with no call that a capture forbids and
    nothing but the product's kernels on the captured stream."""
    run(f"""
product({warm})
stub.stub_capture(S1)
calls = product({k}, S1)
stub.stub_capture(None)
assert form(calls) == {kernel!r}, calls
assert not [c for c in calls if c[0] == "unsafe"], calls
assert all("k_spmm" in c[1] for c in calls if c[0] == "launch" and c[2] == str(S1)), calls
assert form(product({k}, S1)) == {kernel!r}
""")


@pytest.mark.parametrize("warm,k,kernel", [(16, 128, "k_spmm_lds"), (128, 16, "k_spmm_tile")])
def test_no_room_for_a_second_form(run, warm, k, kernel):
    """The form that is there serves a product whose own form does not fit, and
    the build is not tried again by every product after it."""
    run(f"""
product({warm})
held = stub.stub_live()
stub.stub_limit(held + 1000)
calls = product({k})
assert ("nomem",) in calls and form(calls) == {kernel!r}, calls
assert stub.stub_live() == held  # nothing of the failed build is kept
assert ("nomem",) not in product({k}) and form(product({warm})) == {kernel!r}
stub.stub_limit(1 << 40)
A.set_spmm_rows(1)  # a new cut tries again
assert form(product({warm})) == {kernel!r} and form(product({k})) != {kernel!r}
""")


def test_no_room_for_the_first_form_is_an_error(run):
    run("""
product(4)
stub.stub_limit(stub.stub_live() + 1000)
for k in (16, 128):
    try:
        product(k)
    except P.PerflibsError:
        continue
    raise AssertionError(k)
stub.stub_limit(1 << 40)
assert form(product(128)) == "k_spmm_tile"
""")


def test_the_cut_is_given_back_when_both_forms_exist(run):
    run("""
from plsparse import workloads as W
class Info(ctypes.Structure):
    _fields_ = [(f, ctypes.c_size_t) for f in "arena ordblks smblks hblks hblkhd usmblks fsmblks uordblks fordblks keepcost".split()]
libc = ctypes.CDLL(None)
libc.mallinfo2.restype = Info
def host():  # heap in use, without the stub's device memory
    i = libc.mallinfo2()
    return i.uordblks + i.hblkhd - stub.stub_live()
rp, ci, v = W.stencil27(60)
T = P.SpMat.csr(60 ** 3, 60 ** 3, rp, ci, v, flags=P.CREATE_NOCOPY)
product(4, h=T)
before = host()
product(16, h=T)
assert host() - before > len(v)  # the cut: a byte per non-zero and the lists
product(128, h=T)
assert host() - before < len(v) // 4
assert form(product(16, h=T)) == "k_spmm_lds" and form(product(128, h=T)) == "k_spmm_tile"
T.set_spmm_rows(1)  # and cut again from the handle's arrays
assert form(product(16, h=T)) == "k_spmm_lds" and form(product(128, h=T)) == "k_spmm_tile"
""")


def test_the_narrow_tile_cases_reach_their_kernels(run):
    run("""
from test_gpu_spmm_tiles_narrow import CASES, wide_band
rp, ci, v = wide_band()
m = len(rp) - 1
H = {}
for prec, k, (nw, vw) in CASES:
    if prec not in H:
        H[prec] = P.SpMat.csr(m, m, rp, ci, v.astype(np.float32))
        if prec == "bf16":
            H[prec].set_precision(P.VALUES_BF16)
    ran = kernels(product(k, h=H[prec]))
    want = f"k_spmm_tileILi{nw}ELi{vw}E{'tf' if prec == 'bf16' else 'ff'}"
    assert any(want in f for f in ran), (prec, k, ran, H[prec].spmm_info())
""")


def test_sell_tiles_of_a_batch_beside_or_after_the_csr_tiles(run):
    """Few SELL tiles share the CSR tiles' launch; many get their own after it."""
    run("""
from plsparse import workloads as W
from test_gpu_batch_loop import CASES, problems
seen = set()
for kind, tile, C, sigma in CASES:
    probs = problems(W, kind)
    mats = [P.SpMat.csr(p[0], p[0], p[1], p[2], p[3]) for p in probs]
    B = P.Batch(mats, [p[4] for p in probs])
    B.set_shape(tile, [2, 2, 2, 8, 8], [1, 1, 2, 1, 2])
    if C:
        B.set_sell(C, sigma)
    ptr = [buf.ctypes.data] * len(probs)
    B.set_operands(ptr, ptr)
    stub.stub_clear()
    B.exec(0.75, 0.5)
    ran = [(c[1], int(c[3])) for c in (x.split() for x in stub.stub_log().decode().splitlines()) if c[0] == "launch"]
    resident, tiles = 256 * 4, B.info()["ntiles"]
    if C == 0:
        loop = tiles > 1.5 * resident
        assert len(ran) == 1 and f"k_batchILi0ELb{int(loop)}" in ran[0][0], ran
        assert ran[0][1] == (resident if loop else tiles), ran
    elif len(ran) == 1:  # beside
        assert f"k_batchILi{C}E" in ran[0][0], ran
    else:
        assert "k_batchILi0E" in ran[0][0] and f"k_batch_sellILi{C}E" in ran[1][0] and ran[1][1] > 3 * resident, ran
    seen.add((C, len(ran), tiles > resident))
assert {(32, 1, False), (32, 2, True), (64, 1, True), (64, 2, True), (0, 1, True)} <= seen, seen
""")


def test_block_row_lengths_choose_the_block_kernel(run):
    run("""
from plsparse import workloads as W
from test_gpu_bsr_spmm_rows import CASES
for mb, b, per, prec, own in CASES:
    rp, ci, v = W.block_random(mb, b, per, 300, 5)
    H = P.SpMat.bsr(P.ROW_MAJOR, mb * b, mb * b, b, rp, ci, v.astype(np.float64 if prec == "f64" else np.float32),
                    flags=P.CREATE_NOCOPY)
    if prec == "bf16":
        H.set_precision(P.VALUES_BF16)
    for k, window in ((3, "ELi1"), (8, "ELi2")):
        f = kernels(product(k, h=H))[-1]
        kl = "" if prec == "f64" else f"ELi{b // 4}"
        assert f"Li{b}ELi1ELi1{kl}{window}ELb{int(own)}E" in f, (mb, b, per, prec, k, f)
    H.destroy()
""")


@pytest.mark.parametrize("warm,k,kernel", [(16, 128, "k_spmm_lds"), (128, 16, "k_spmm_tile")])
def test_no_host_memory_for_a_second_form(run, warm, k, kernel):
    """An allocation that fails while a form is built, on a thread of the build
    too, does not end the program."""
    run(f"""
from plsparse import workloads as W
rp, ci, v = W.stencil27(40)
T = P.SpMat.csr(40 ** 3, 40 ** 3, rp, ci, v, flags=P.CREATE_NOCOPY)
T.set_spmm_rows(2)
product({warm}, h=T)
stub.stub_host_limit(100000)
assert form(product({k}, h=T)) == {kernel!r}
stub.stub_host_limit(1 << 60)
assert form(product({k}, h=T)) == {kernel!r} and form(product({warm}, h=T)) == {kernel!r}
""")
