"""Run records of the one-right-hand-side projections: the destriping operator
from run records against the same operator in numpy from the samples, on scans
with long runs, where the run path is taken."""
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


def scan_case(ndet, nsamp, nside, base, nnz, flags, ncross, distinct):
    scan = dict(fsample=50.0, spin_period=20.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        det = dict(psi_turns=0.125 * (d % 4), open_offset_turns=0.004 * d if distinct else 0.0)
        return oracle.expand_pointing(scan, det, nside, 0, n)

    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=base, nnz=nnz, seed=ndet + nsamp,
                     pointing=pointing, extra_pars=dict(nside_cross=ncross or nside))
    if flags:
        rng = np.random.default_rng(3)
        c["pixels"][rng.random(c["pixels"].size) < 0.05] = -1
        c["pixels"].reshape(ndet, nsamp)[:, nsamp // 2:nsamp // 2 + 130] = -1
    return c


# detectors 1, 2, 3 and a ragged last group of 4; baselines of a few runs and
# longer than an LDS tile; block and tile remainders; flagged samples and
# whole flagged baselines; cross pixels coarser than map pixels
@pytest.mark.parametrize("ndet,nsamp,nside,base,nnz,flags,ncross,distinct", [
    (1, 4001, 4, 0.5, 1, False, 0, False),
    (2, 1279, 4, 0.5, 1, True, 0, False),
    (3, 4096, 4, 1.0, 3, True, 0, True),
    (4, 6001, 4, 0.1, 3, False, 0, False),
    (5, 9999, 8, 0.5, 3, True, 4, False),
    (9, 20000, 8, 40.0, 3, False, 0, True),
    (4, 260001, 8, 0.1, 3, True, 0, False),
])
def test_operator_from_runs(ndet, nsamp, nside, base, nnz, flags, ncross, distinct):
    import libmadam_amd
    c = scan_case(ndet, nsamp, nside, base, nnz, flags, ncross, distinct)
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_kernel_variant(128)
    m.set_pointing(c["pixels"], c["pixweights"])
    m.solve(c["signal"])
    st, nb = m.stats(), m.sizes()["nbase"]
    assert 0 < st["run_records"] < 0.5 * st["nactive"]
    x = np.random.default_rng(7).standard_normal(ndet * nb)
    got = m.apply(2, x)
    m.close()
    # F^T W (F x - P m), m = (P^T W P)^-1 P^T W F x on the well-conditioned pixels
    ok = c["pixels"].reshape(-1) >= 0
    q = c["pixels"].reshape(-1)[ok] // (nside // (ncross or nside)) ** 2
    b = (np.arange(nsamp) // round(base * 50.0) + np.arange(ndet)[:, None] * nb).reshape(-1)[ok]
    w = c["pixweights"].reshape(-1, nnz)[ok].astype(np.float64)
    dw = c["weights"][0]
    npix = 12 * (ncross or nside) ** 2
    cc = np.zeros((npix, nnz, nnz))
    for i in range(nnz):
        for j in range(nnz):
            cc[:, i, j] = dw * np.bincount(q, w[:, i] * w[:, j], npix)
    ev = np.linalg.eigvalsh(cc)
    good = (ev[:, -1] > 0) & (ev[:, 0] > 1e-3 * ev[:, -1])
    inv = np.zeros_like(cc)
    inv[good] = np.linalg.inv(cc[good])
    v = dw * x[b]
    mp = np.einsum("qij,qj->qi", inv, np.stack([np.bincount(q, w[:, j] * v, npix) for j in range(nnz)], -1))
    use = good[q]
    ref = np.bincount(b[use], v[use] - dw * np.einsum("sj,sj->s", w[use], mp[q[use]]), ndet * nb)
    # FP64 sums of at most 1e5 terms, the pixel matrices' condition below 1e3
    size = np.bincount(b[use], np.abs(v[use]), ndet * nb)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(size)


def test_mixed_solve_from_runs():
    """The FP32 run records inside the refinement: the solution meets the limit on the residual of the FP64
    operator (applied here from FP64 runs), with the rounding of that residual, 1e-15 of its terms, on top."""
    import libmadam_amd
    c = scan_case(4, 60000, 16, 0.5, 3, True, 0, False)
    c["pars"]["cglimit"] = 1e-20
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_kernel_variant(128)
    m.set_pointing(c["pixels"], c["pixweights"])
    m.solve_batch(c["signal"].reshape(1, 4, -1).astype(np.float64), precision=1)
    r = m.batch_result(0)
    assert m.stats()["run_records"] > 0
    m.solve(c["signal"])
    res = r["yba"].reshape(-1) - m.apply(2, r["aa"])
    m.close()
    assert np.linalg.norm(res) <= 1.01e-10 * np.linalg.norm(r["yba"])


@pytest.mark.parametrize("nnz", [3, 1])
def test_runs_that_only_fp32_reads(nnz):
    """Between 1.3 and 2 samples per run the FP64 operator reads samples and a mixed solve's FP32 operator
    runs: the records hold FP32 sums alone (12 bytes a run and side, not 28), each precision reports what it
    reads, and the solution meets the limit on the FP64 residual in as many steps as from samples."""
    import torch
    import libmadam_amd
    scan = dict(fsample=100.0, spin_period=7.5, prec_period=4000.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)
    m, steps = None, {}
    for nsamp in (2 ** 20, 2 ** 16 - 1):     # the shorter scan is below the 2^18 samples from which runs are used
        c = mc.ring_case(ndet=4, nsamp=nsamp, nside=64, base_first=1.0, nnz=nnz, seed=nnz, fsample=100.0,
                         pointing=lambda d, n: oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), 64, 0, n),
                         extra_pars=dict(cglimit=1e-14))
        for variant in ((0,) if nsamp > 2 ** 18 else (0, 128)):
            m = libmadam_amd.Madam(0)
            args = mc.call_args(c)
            m.configure(*args[:4], *args[7:], c["nnz"])
            m.set_kernel_variant(variant)
            m.set_pointing(c["pixels"], c["pixweights"])
            m.solve(c["signal"].copy())
            assert m.stats()["run_records"] == 0
            free = torch.cuda.mem_get_info()[0]
            m.solve_batch(c["signal"].reshape(1, 4, -1), precision=1)
            r = m.batch_result(0)
            used = free - torch.cuda.mem_get_info()[0]
            runs = r["info"]["run_records"]
            assert m.stats()["run_records"] == 0
            if nsamp < 2 ** 18 and variant == 0:
                assert runs == 0
            else:
                assert 1.3 <= m.stats()["nactive"] / runs < 2.0
            if nsamp > 2 ** 18:
                # both sides' records and segment tables, and the batch's own vectors and maps (under 40 MB)
                assert used <= 30 * runs + 40e6
            res = r["yba"].reshape(-1) - m.apply(2, r["aa"])
            assert np.linalg.norm(res) <= 1.01e-7 * np.linalg.norm(r["yba"])
            steps[nsamp, variant] = r["info"]["pcg_steps"]
            m.close()
    assert abs(steps[2 ** 16 - 1, 0] - steps[2 ** 16 - 1, 128]) <= 0.1 * steps[2 ** 16 - 1, 0] + 2


def operator(c, ndet, nsamp, nside, ncross, per, nnz, x):
    """F^T W (F x - P m), m = (P^T W P)^-1 P^T W F x on the well-conditioned pixels, and the size of its terms."""
    ok = c["pixels"].reshape(-1) >= 0
    q = c["pixels"].reshape(-1)[ok] // (nside // ncross) ** 2
    nb = x.size // ndet
    b = (np.arange(nsamp) // per + np.arange(ndet)[:, None] * nb).reshape(-1)[ok]
    w = c["pixweights"].reshape(-1, nnz)[ok].astype(np.float64)
    dw = c["weights"][0]
    npix = 12 * ncross ** 2
    cc = np.zeros((npix, nnz, nnz))
    for i in range(nnz):
        for j in range(nnz):
            cc[:, i, j] = dw * np.bincount(q, w[:, i] * w[:, j], npix)
    ev = np.linalg.eigvalsh(cc)
    good = (ev[:, -1] > 0) & (ev[:, 0] > 1e-3 * ev[:, -1])
    inv = np.zeros_like(cc)
    inv[good] = np.linalg.inv(cc[good])
    v = dw * x[b]
    mp = np.einsum("qij,qj->qi", inv, np.stack([np.bincount(q, w[:, j] * v, npix) for j in range(nnz)], -1))
    use = good[q]
    ref = np.bincount(b[use], v[use] - dw * np.einsum("sj,sj->s", w[use], mp[q[use]]), x.size)
    return ref, np.bincount(b[use], np.abs(v[use]), x.size)


# the sides decide for themselves: long runs on cross pixels that hold 64 map pixels of one sample each (baseline
# side only), runs between the two lines (pixel side only), temperature (both), and a solve that wants neither
@pytest.mark.parametrize("nside,ncross,spin,per,nnz,base_runs,pixel_runs", [
    (32, 4, 4.0, 50, 3, True, False), (8, 8, 2.47, 50, 3, False, True), (32, 4, 4.0, 50, 1, True, True),
    (32, 16, 4.3, 5, 3, False, False)])
def test_sides_use_runs_where_they_pay(nside, ncross, spin, per, nnz, base_runs, pixel_runs):
    import libmadam_amd
    ndet, nsamp = 3, 20003
    scan = dict(fsample=50.0, spin_period=spin, prec_period=4000.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)
    c = mc.ring_case(ndet=ndet, nsamp=nsamp, nside=nside, base_first=per / 50.0, nnz=nnz, seed=nside,
                     pointing=lambda d, n: oracle.expand_pointing(scan, dict(psi_turns=0.125 * d), nside, 0, n),
                     extra_pars=dict(nside_cross=ncross))
    # samples per run, of time-ordered cross pixels and of map pixels (whose entries may meet again later)
    pix = c["pixels"].reshape(ndet, nsamp)[0]

    def length(p):
        return nsamp / (1 + np.sum((p[1:] != p[:-1]) | (np.arange(1, nsamp) % per == 0)))
    cross, fine = length(pix // (nside // ncross) ** 2), length(pix)
    print("samples per run: cross %.2f, map %.2f" % (cross, fine))
    if nnz == 3:
        assert (cross >= 2.3) == base_runs and (cross >= 2.05 or not pixel_runs) and (fine >= 1.8) == pixel_runs
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_kernel_variant(128)
    m.set_pointing(c["pixels"], c["pixweights"])
    m.solve(c["signal"].copy())
    x = np.random.default_rng(7).standard_normal(ndet * m.sizes()["nbase"])
    got = m.apply(2, x)
    assert (m.stats()["run_records"] > 0) == base_runs
    ref, size = operator(c, ndet, nsamp, nside, ncross, per, nnz, x)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(size)
    # the mixed solve, whose sides have lines of their own
    m.solve_batch(c["signal"].reshape(1, ndet, -1).copy(), precision=1)
    r = m.batch_result(0)
    res = r["yba"].reshape(-1) - m.apply(2, r["aa"])
    assert np.linalg.norm(res) <= 1.01e-6 * np.linalg.norm(r["yba"])
    m.close()
