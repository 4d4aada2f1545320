"""The request loop's memory estimate against what a job holds on the device
while it runs: run records at 1.6 and 2.4 samples per run, one-pass band tables of
a flagged scan with short baselines, a group of jobs that is binned together."""
import threading

import numpy as np
import pytest

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


FS, SIGMA, NDET, NSAMP = 100.0, 2e-4, 4, 2 ** 22


def scan(nside, spin, flags):
    import torch
    import libmadam_amd
    pix = torch.empty(NDET, NSAMP, dtype=torch.int32, device="cuda")
    w = torch.empty(NDET, NSAMP, 3, dtype=torch.float32, device="cuda")
    s = dict(fsample=FS, spin_period=spin, prec_period=360 * 3600.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)
    torch.cuda.synchronize()
    libmadam_amd.expand_pointing_device(s, [dict(psi_turns=0.125 * d) for d in range(NDET)], nside, 0, NSAMP, pix, w)
    if flags:
        pix[torch.rand(NDET, NSAMP, device="cuda") < 0.02] = -1
    torch.cuda.synchronize()
    return pix, w


def submit(srv, pix, w, tod, nside, base, prior, precision, key):
    freqs = np.logspace(-5, np.log10(FS / 2), 100)
    psd = SIGMA ** 2 / FS * (1.0 + (freqs / 0.05) ** -1.5)
    pars = dict(base_first=base, fsample=FS, nside_map=nside, nside_cross=nside, kfilter=prior, info=0, iter_max=20)
    return srv.submit(pars, np.full(NDET, SIGMA ** -2), np.arange(NSAMP) / FS, pix, w, tod, np.zeros(1, np.int64),
                      np.ones(NDET, np.int64), np.zeros(NDET), freqs, np.tile(psd, NDET), nnz=3, scan_key=key,
                      precision=precision, on_device=True)


@pytest.mark.parametrize("nside,spin,base,prior,precision,flags,njobs", [
    (256, 60.0, 1.0, False, 0, False, 1), (512, 60.0, 1.0, True, 1, False, 1), (512, 90.0, 1.0, False, 1, False, 1),
    (512, 60.0, 0.25, True, 1, True, 1), (256, 60.0, 0.04, True, 1, True, 1), (512, 60.0, 0.25, True, 1, True, 4)])
def test_a_job_stays_within_its_estimate(nside, spin, base, prior, precision, flags, njobs):
    import torch
    import libmadam_amd
    pix, w = scan(nside, spin, flags)
    tod = torch.randn(NDET, NSAMP, device="cuda", dtype=torch.float64 if precision == 0 else torch.float32)
    torch.cuda.synchronize()
    for again in range(2):                      # the first job of a process has the runtime's own allocations
        srv = libmadam_amd.Server(0, hbm_budget=200e9, max_inflight=1)
        free = least = torch.cuda.mem_get_info()[0]
        done = threading.Event()

        def watch():
            nonlocal least
            while not done.wait(0.0005):
                least = min(least, torch.cuda.mem_get_info()[0])

        th = threading.Thread(target=watch)
        th.start()
        try:
            ids = [submit(srv, pix, w, tod, nside, base, prior, precision, njobs > 1) for _ in range(njobs)]
            for j in ids:
                srv.wait(j)
        finally:
            done.set()
            th.join()
            st = srv.stats()
            srv.close()
    assert st["done"] == njobs
    print("used %.0f MB, estimated %.0f MB" % ((free - least) / 1e6, st["peak_bytes"] / 1e6))
    assert free - least <= st["peak_bytes"]


def test_a_job_that_fits_only_without_its_tables_is_accepted():
    """The tables' share of the estimate never refuses a job."""
    import torch
    import libmadam_amd
    pix, w = scan(256, 60.0, False)
    tod = torch.randn(NDET, NSAMP, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    srv = libmadam_amd.Server(0, hbm_budget=200e9, max_inflight=1)
    srv.wait(submit(srv, pix, w, tod, 256, 1.0, False, 0, 0))
    est = srv.stats()["peak_bytes"]
    srv.close()
    tables = NDET * NSAMP * 22
    srv = libmadam_amd.Server(0, hbm_budget=est - 0.5 * tables, max_inflight=1)
    srv.wait(submit(srv, pix, w, tod, 256, 1.0, False, 0, 0))
    assert srv.stats()["peak_bytes"] == est - 0.5 * tables
    srv.close()
    srv = libmadam_amd.Server(0, hbm_budget=est - 1.5 * tables, max_inflight=1)
    with pytest.raises(Exception, match="budget"):
        submit(srv, pix, w, tod, 256, 1.0, False, 0, 0)
    srv.close()
