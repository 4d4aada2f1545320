"""The noise prior's convolution at every column and row length with a kernel
of its own (128 to 512, 256 to 1024), and one below them.  FP64: the result
against the oracle's convolution with the GPU's own filter, to FFT rounding.
FP32: inside a mixed-precision solve, which converges to the FP64 solution with
any inner operator that is near enough, in more passes the further off it is.  So
the FP32 operator is pinned by a solve whose limit, 1e-5 of the right-hand
side, has to be met by the FP64 residual after one inner solve: it differs from
the inner residual by what the operators differ by, 2e-6 with FP32 transforms
and 7e-7 with FP64 ones in the same FP32 operator (MADAM_FFT32=0).
"""
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


# columns x rows: 128 x 128, 128 x 256, 256 x 256, 256 x 512, 512 x 512, 512 x 1024
@pytest.mark.parametrize("log2nof", [15, 16, 17, 18, 19, 20])
def test_convolution_lengths(log2nof, monkeypatch):
    import libmadam_amd
    nside, fs, ndet, nof = 8, 50.0, 4, 2 ** log2nof
    nbase = int(0.27 * nof) | 1    # just over a quarter: the next smaller filter would not do
    nsamp = 10 * nbase
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=0.2, prior=True, seed=log2nof, pointing=pointing,
                     nnz=1)
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_pointing(c["pixels"], c["pixweights"])
    m.solve(c["signal"].copy())
    aa, st = m.baselines()["aa"], m.stats()
    assert st["nof"] == nof and st["nseg"] == ndet
    x = np.random.default_rng(log2nof).standard_normal(ndet * nbase)
    y = m.apply(0, x).reshape(ndet, nbase)
    for d in range(ndet):
        ref = oracle.convolve(m.filter(0), x.reshape(ndet, nbase)[d], nof)
        assert np.linalg.norm(y[d] - ref) <= 1e-13 * np.linalg.norm(ref)
    m.solve_batch(np.stack([c["signal"].reshape(ndet, nsamp)] * 2), precision=1)
    for r in range(2):
        a = m.batch_result(r)["aa"]
        assert np.linalg.norm((a - a.mean()) - (aa - aa.mean())) <= 1e-4 * np.linalg.norm(aa)
    c["pars"]["cglimit"] = 1e-10
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_pointing(c["pixels"], c["pixweights"])
    steps = {}
    for fft32 in ("1", "0"):
        monkeypatch.setenv("MADAM_FFT32", fft32)
        m.solve_batch(np.stack([c["signal"].reshape(ndet, nsamp)] * 2), precision=1)
        for r in range(2):
            info = m.batch_result(r)["info"]
            assert info["passes"] == 1 and info["rr_final"] < 1e-10
            steps[fft32, r] = info["pcg_steps"]
    for r in range(2):
        assert abs(steps["1", r] - steps["0", r]) <= 1
    m.close()
