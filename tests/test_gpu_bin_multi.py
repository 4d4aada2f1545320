"""Several signals binned and cleaned in one pass over the pixels: each map as
its own single solve makes it.  Group sizes 4 and 8 with ragged last groups,
short pixels and ones long enough for a block of their own, FP64 and FP32
samples, temperature and polarised, solve pixels coarser than the map's,
signals on the device and on the host."""
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


@pytest.mark.parametrize("nrhs,nside,nnz,f32,ncross,device", [
    (3, 8, 3, False, 0, True), (5, 2, 3, False, 0, True), (6, 8, 1, True, 4, True), (9, 2, 1, False, 0, True),
    (10, 8, 3, True, 4, True), (4, 8, 3, False, 0, False)])
def test_batch_maps_match_single_solves(nrhs, nside, nnz, f32, ncross, device):
    import torch
    import libmadam_amd
    ndet, nsamp = 4, 40010      # 3333 samples per pixel at Nside 2: past the 2048 of one wave
    scan = dict(fsample=50.0, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, nnz=nnz, base_first=1.0, prior=True, seed=nrhs,
                     pointing=pointing, extra_pars=dict(nside_cross=ncross or nside))
    c["pixels"][::97] = -1
    rng = np.random.default_rng(nrhs)
    sig = np.stack([c["signal"] + 1e-4 * rng.standard_normal(c["signal"].size) for _ in range(nrhs)])
    sig = sig.reshape(nrhs, ndet, nsamp).astype(np.float32 if f32 else np.float64)
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_pointing(c["pixels"], c["pixweights"])
    batch = torch.from_numpy(sig).cuda() if device else sig
    torch.cuda.synchronize()
    m.solve_batch(batch, precision=0, on_device=device)
    got = [m.batch_result(r) for r in range(nrhs)]
    for r in range(nrhs):
        m.solve(sig[r].astype(np.float64).reshape(-1))
        one, aa = m.maps(), m.baselines()["aa"]
        # binning: FP64 sums of the same products in another order; the maps carry the solve's rounding too
        assert np.linalg.norm(got[r]["binmap"] - one["binmap"]) <= 1e-12 * np.linalg.norm(one["binmap"]), r
        assert np.linalg.norm(got[r]["map"] - one["map"]) <= 1e-9 * np.linalg.norm(one["map"]), r
        assert np.linalg.norm(got[r]["aa"] - aa) <= 1e-9 * np.linalg.norm(aa), r
    m.close()
