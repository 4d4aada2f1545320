"""The one-pass band solve against the chained one (kernel variant + 64 keeps
the carry chains): the same preconditioner applied to random vectors, on
segment lengths around its block (48 chunks of 64 rows), chunk and halo sizes,
with and without flags (repeating and non-repeating factors)."""
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


# baselines per period: less than a chunk, chunk edges, the halo's eight
# chunks, the block's 48 chunks, one over, several blocks with a ragged end
@pytest.mark.parametrize("nper,nperiod,flags", [(40, 2, False), (64, 1, False), (65, 3, True), (512, 2, False),
                                                (513, 1, True), (3072, 1, False), (3073, 2, True), (3584, 1, False),
                                                (20011, 1, False), (20011, 1, True)])
def test_direct_matches_chains(nper, nperiod, flags):
    import libmadam_amd
    nside, fs, ndet = 8, 50.0, 2
    nsamp = nper * nperiod * 10
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.25 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=0.2, prior=True, nperiod=nperiod, seed=nper,
                     pointing=pointing, nnz=1)
    if flags:
        rng = np.random.default_rng(1)
        c["pixels"].reshape(ndet, -1)[:, np.repeat(rng.random(nsamp // 10) < 0.2, 10)] = -1
    z = {}
    for variant in (0, 64):
        m = libmadam_amd.Madam(0)
        args = mc.call_args(c)
        m.configure(*args[:4], *args[7:], c["nnz"])
        m.set_kernel_variant(variant)
        m.set_pointing(c["pixels"].copy(), c["pixweights"])
        m.solve(c["signal"].copy())
        st = m.stats()
        assert st["precond_kind"] == 3 and st["nband"] == 10 and st["ncg"] == 0
        sz = m.sizes()
        x = np.random.default_rng(5).standard_normal(sz["ndet"] * sz["nbase"])
        x[: x.size // 3] *= 1e6        # a loud stretch beside a quiet one
        z[variant] = m.apply(1, x)
        z[variant, "aa"], z[variant, "niter"] = m.baselines()["aa"], st["niter"]
        m.close()
    # two orders of the same FP64 sums; the carries left out are below 2^-64 of the largest state
    assert np.linalg.norm(z[0] - z[64]) <= 1e-13 * np.linalg.norm(z[64])
    quiet = slice(x.size // 2, None)   # far enough from the loud stretch for its carries to have decayed
    assert np.linalg.norm(z[0][quiet] - z[64][quiet]) <= 1e-13 * np.linalg.norm(z[64][quiet])
    assert z[0, "niter"] == z[64, "niter"]


def test_direct_batch_and_mixed():
    """Several right-hand sides at once, FP64 and FP32 vectors: each as its own solve."""
    import libmadam_amd
    nside, fs, ndet, nsamp, R = 8, 50.0, 4, 40010, 3
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=0.2, prior=True, seed=11, pointing=pointing)
    rng = np.random.default_rng(2)
    sig = np.stack([c["signal"] + 1e-4 * rng.standard_normal(c["signal"].size) for _ in range(R)])
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_pointing(c["pixels"], c["pixweights"])
    one = []
    for r in range(R):
        m.solve(sig[r].copy())
        one.append(m.baselines()["aa"])
    for precision, tol in ((0, 1e-10), (1, 1e-4)):
        m.solve_batch(sig.reshape(R, ndet, nsamp), precision=precision)
        for r in range(R):
            a = m.batch_result(r)["aa"]
            assert np.linalg.norm((a - a.mean()) - (one[r] - one[r].mean())) <= tol * np.linalg.norm(one[r])
    m.close()


def test_tables_only_where_they_are_read():
    """The products of the one-pass solve (3.9 KB per 64 flagged rows) are held where it is used: not with the
    chains forced, nor where a low knee makes the carries decay too slowly, whose results are then the chains'."""
    import torch
    import libmadam_amd
    nside, fs, ndet, nper = 8, 50.0, 2, 300000
    scan = dict(fsample=fs, spin_period=2.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.25 * d), nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nper * 4, nside=nside, base_first=0.08, prior=True, seed=3, pointing=pointing,
                     nnz=1, extra_pars=dict(iter_max=5))
    c["pixels"][np.random.default_rng(1).random(c["pixels"].size) < 0.1] = -1
    white = c["psdvals"][-1]
    used, z = {}, {}
    for again in range(2):                      # the first time round the runtime allocates for itself
        for knee in (0.1, 0.002):
            c["psdvals"] = np.tile(white * (1.0 + (c["psdfreqs"] / knee) ** -1.5), ndet)
            for variant in (0, 64):
                m = libmadam_amd.Madam(0)
                args = mc.call_args(c)
                m.configure(*args[:4], *args[7:], c["nnz"])
                m.set_kernel_variant(variant)
                m.set_pointing(c["pixels"].copy(), c["pixweights"])
                free = torch.cuda.mem_get_info()[0]
                m.solve(c["signal"].copy())
                used[knee, variant] = free - torch.cuda.mem_get_info()[0]
                assert m.stats()["precond_kind"] == 3 and m.stats()["nband"] == 10 and m.stats()["ncg"] == 0
                z[knee, variant] = m.apply(1, np.random.default_rng(5).standard_normal(ndet * nper))
                m.close()
    tables = 2 * 8 * 3 * 81 * (ndet * nper // 64)
    assert used[0.1, 0] - used[0.1, 64] >= 0.9 * tables
    assert used[0.002, 0] - used[0.1, 64] <= 0.1 * tables
    assert not np.array_equal(z[0.1, 0], z[0.1, 64])
    np.testing.assert_array_equal(z[0.002, 0], z[0.002, 64])
