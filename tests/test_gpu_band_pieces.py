"""The band factor made in pieces, where flags keep it from repeating, against
the serial chain (kernel variant + 16): the same bits, and so the same
preconditioner, offsets and step count.  Segments around the 8192 rows from
which pieces are used, ragged last pieces, long stretches without data; bands of
20 baselines, over which a piece's start is remembered for longer than its
warm-up, so that pieces are factored again; and wider ones, which keep the
serial chain.
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


@pytest.mark.parametrize("nper,nperiod,gap", [(8192, 1, 0), (8193, 2, 0), (9217, 1, 2500), (20011, 1, 0),
                                              (20480, 2, 7000)])
def test_pieces_match_serial_chain(nper, nperiod, gap):
    import libmadam_amd
    nside, fs, ndet = 8, 50.0, 2
    nsamp = nper * nperiod * 10
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.25 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=0.2, prior=True, nperiod=nperiod, seed=nper,
                     pointing=pointing, nnz=1)
    rng = np.random.default_rng(1)
    pix = c["pixels"].reshape(ndet, -1)
    pix[:, rng.random(nsamp) < 0.1] = -1
    base = np.arange(nsamp) // 10 - 3 * nper // 10
    pix[:, (base >= 0) & (base < gap) & (base % 251 != 250)] = -1
    z = {}
    for variant in (0, 16):
        m = libmadam_amd.Madam(0)
        args = mc.call_args(c)
        m.configure(*args[:4], *args[7:], c["nnz"])
        m.set_kernel_variant(variant)
        m.set_pointing(c["pixels"].copy(), c["pixweights"])
        m.solve(c["signal"].copy())
        st = m.stats()
        assert st["precond_kind"] == 3 and st["band_rows_factored"] == ndet * nper * nperiod
        x = np.random.default_rng(5).standard_normal(ndet * m.sizes()["nbase"])
        z[variant] = m.apply(1, x), m.baselines()["aa"], st["niter"]
        m.close()
    np.testing.assert_array_equal(z[0][0], z[16][0])
    np.testing.assert_array_equal(z[0][1], z[16][1])
    assert z[0][2] == z[16][2]


def test_pieces_that_are_factored_again():
    """20 baselines under low knees, with a long stretch without data: some of the pieces' first windows differ
    from the serial chain's in their last bits.  30 baselines: no pieces."""
    import libmadam_amd
    nside, fs, ndet, nper = 8, 50.0, 2, 9217
    nsamp = nper * 10
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.25 * d), nside, 0, n)

    again = 0
    for knee, width in ((0.02, 20), (0.005, 20), (0.002, 20), (0.0005, 20), (0.02, 30)):
        c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=0.2, prior=True, seed=nper,
                         pointing=pointing, nnz=1,
                         extra_pars=dict(iter_max=2, precond_width_min=width, precond_width_max=width))
        white = c["psdvals"][c["psdfreqs"].size - 1]
        c["psdvals"] = np.tile(white * (1.0 + (c["psdfreqs"] / knee) ** -1.5), ndet)
        pix = c["pixels"].reshape(ndet, -1)
        pix[:, np.random.default_rng(1).random(nsamp) < 0.1] = -1
        base = np.arange(nsamp) // 10 - 3 * nper // 10
        pix[:, (base >= 0) & (base < 2500) & (base % 251 != 250)] = -1
        z = {}
        for variant in (0, 16):
            m = libmadam_amd.Madam(0)
            args = mc.call_args(c)
            m.configure(*args[:4], *args[7:], c["nnz"])
            m.set_kernel_variant(variant)
            m.set_pointing(c["pixels"].copy(), c["pixweights"])
            m.solve(c["signal"].copy())
            st = m.stats()
            assert st["precond_kind"] == 3 and st["nband"] == width and st["ncg"] == 0
            z[variant] = m.apply(1, np.random.default_rng(5).standard_normal(ndet * nper)), st["band_rows_factored"]
            m.close()
        np.testing.assert_array_equal(z[0][0], z[16][0])
        assert z[16][1] == ndet * nper
        if width == 20:
            assert z[0][1] >= ndet * nper
            again += z[0][1] - ndet * nper
        else:
            assert z[0][1] <= ndet * nper
    assert again > 0
