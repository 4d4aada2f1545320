"""PCG steps queued ahead of the host: a solve stops at the step whose residual
meets the limit, and the steps queued behind it change nothing.  Baseline
counts on both sides of the dot products' one-launch limit (128 blocks of 2048
baselines), with a diagonal preconditioner (fused residual update) and a band
one, and less than one block."""
import numpy as np
import pytest

import oracle
from tests import madam_cases as mc

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


@pytest.mark.parametrize("nbase,prior", [(301, False), (65536, False), (65537, False), (65536, True), (70001, True)])
def test_solve_stops_where_it_meets_the_limit(nbase, prior):
    import libmadam_amd
    ndet, nside, per = 4, 8, 4
    nsamp = nbase * per
    scan = dict(fsample=50.0, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=per / 50.0, prior=prior, seed=nbase,
                     pointing=pointing, extra_pars=dict(cglimit=1e-8))
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_pointing(c["pixels"], c["pixweights"])
    m.solve(c["signal"])
    assert m.sizes()["nbase"] == nbase
    niter, rr = int(m.stats()["niter"]), m.rr_history()
    assert len(rr) == niter and rr[-1] < 1e-8 and (niter <= 4 or rr[-2] >= 1e-8)
    aa = m.baselines()["aa"]
    # the same number of steps without exit tests
    m.iterate(niter, restart=True)
    assert np.array_equal(m.baselines()["aa"], aa)
    # FP64 residual of the solution against the recurrence's
    b = m.baselines()["yba"].reshape(-1)
    res = b - m.apply(2, aa)
    assert abs(res @ res / (b @ b) - rr[-1]) <= 1e-6 * rr[-1] + 1e-20
    m.close()
