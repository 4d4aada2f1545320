"""Batches of different sizes on one handle: the captured PCG step of one batch
must not serve another whose launches differ, also where both have the same
kernel width (3 and 4 signals, or 5 to 8).  Every right-hand side against its
own single FP64 solve, with the band and the Fourier preconditioner, through
madam_solve_batch, madam_iterate_batch and the request loop's resident scans."""
import numpy as np
import pytest

from tests import madam_cases as mc
from tests.test_gpu_batch import offset_free, signals_for, single
from tests.test_gpu_parity import rel_rms, ring
from tests.test_gpu_serve import signal, submit

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _torch_gpu_first():
    try:
        import torch
        if torch.cuda.is_available():
            torch.cuda.init()
    except ImportError:
        pass
    yield


def handle(case):
    import libmadam_amd
    a = mc.call_args(mc.copy_case(case))
    m = libmadam_amd.Madam(0)
    m.configure(*a[:4], *a[7:], case["nnz"])
    m.set_pointing(a[4], a[5])
    return m


def check(case, res, ones, precision):
    """FP64 solves to 1e-10; mixed ones, both converged to cglimit 1e-20, to
    1e-6 less the null-space offset (the bars of the fixed-size batches)."""
    for r, s1 in zip(res, ones):
        good = s1["mask"] > 0
        if precision == 0:
            errs = rel_rms(r["map"], s1["map"]), rel_rms(r["aa"], s1["aa"])
        else:
            (a, m), (a1, m1) = offset_free(r["aa"], r["map"], good), offset_free(s1["aa"], s1["map"], good)
            errs = rel_rms(m, m1), rel_rms(a, a1)
        assert max(errs) <= (1e-10 if precision == 0 else 1e-6), errs


@pytest.mark.parametrize("precision,extra", [(0, {}), (1, {}), (1, dict(use_fprecond=True, iter_max=40))])
def test_batch_sizes_on_one_handle(precision, extra, monkeypatch):
    """Bit for bit what a handle of its own gives (the pixel-side cut is pinned:
    the autotuned one can differ between handles)."""
    monkeypatch.setenv("MADAM_BS_PIECE", "256")
    case = ring(prior=True, nsamp=30000, nperiod=2, extra={**dict(cglimit=1e-20, iter_max=2000), **extra})
    sig = signals_for(case, 8)
    ones = [single(case, s) for s in sig]
    m = handle(case)
    for nrhs in (3, 4, 3, 6, 8, 5, 7, 2, 1, 3):
        got = []
        for h in (m, handle(case)):
            h.solve_batch(sig[:nrhs], precision=precision)
            got.append([h.batch_result(k) for k in range(nrhs)])
            h.iterate_batch(3)
            if h is not m:
                h.close()
        for k, (r, fresh) in enumerate(zip(*got)):
            assert (r["info"]["steps"], r["info"]["passes"]) == (fresh["info"]["steps"], fresh["info"]["passes"])
            for name in ("map", "binmap", "aa", "yba"):
                assert np.array_equal(r[name], fresh[name]), (nrhs, k, name)
        if not extra:   # (the Fourier preconditioner cannot move segment offsets: its solves stop at iter_max)
            check(case, got[0], ones, precision)
    m.close()


def test_batch_after_another_preconditioner():
    """A single solve between two batches rebuilds the preconditioner (another
    kernel variant), whose tables the captured step refers to."""
    case = ring(prior=True, nsamp=30000, nperiod=2, extra=dict(cglimit=1e-20, iter_max=2000))
    sig = signals_for(case, 3)
    ones = [single(case, s) for s in sig]
    m = handle(case)
    m.solve_batch(sig, precision=1)
    m.set_kernel_variant(64)
    m.solve(sig[0].reshape(-1).copy())
    m.solve_batch(sig, precision=1)
    check(case, [m.batch_result(k) for k in range(3)], ones, 1)
    m.close()


def test_resident_scan_with_growing_groups():
    """Groups of three and then four jobs on one resident scan."""
    import libmadam_amd
    tight = dict(cglimit=1e-20, iter_max=2000)
    case = ring(nside=8, ndet=4, nsamp=20000, prior=True, nperiod=2, seed=1, extra=tight)
    slow = ring(nside=16, ndet=4, nsamp=400000, prior=True, nperiod=2, seed=2, extra=tight)
    sigs = [signal(case, s) for s in range(7)]
    blocker = signal(slow, 9)
    srv = libmadam_amd.Server(0, hbm_budget=16e9, max_inflight=1)
    try:
        out = []
        for group in (range(3), range(3, 7)):
            # the only worker is busy with jobs of their own while the group arrives
            first = [submit(srv, slow, 0, blocker, 0) for _ in range(6)]
            ids = [submit(srv, case, 7, sigs[k], 1) for k in group]
            for j in first + ids:
                srv.wait(j)
            out += [srv.result(j) for j in ids]
    finally:
        srv.close()
    assert [r["batch"] for r in out] == [3] * 3 + [4] * 4
    assert [bool(r["resident"]) for r in out] == [False] * 3 + [True] * 4
    for k, r in enumerate(out):
        s1 = single(case, sigs[k])
        (a, mp), (a1, m1) = (offset_free(x["aa"], x["map"], s1["mask"] > 0) for x in (r, s1))
        assert rel_rms(mp, m1) <= 1e-6 and rel_rms(a, a1) <= 1e-6, k
