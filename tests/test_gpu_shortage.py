"""Device memory that runs short: a set-up or solve does without the tables that
only save time (run records, the one-pass band solve's products, the factor in
pieces, signals side by side) before it fails.  Every allocation of a call is
made to fail once, from the host (madam_fail_allocations); the results are those
of an undisturbed handle to the rounding of the other path."""
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


@pytest.fixture(autouse=True)
def _allocations_work_again():
    import libmadam_amd
    yield
    libmadam_amd.lib().madam_fail_allocations(-1, 0)


NDET, NBASE = 2, 9001       # segments over the 8192 rows from which a flagged factor is made in pieces


def case():
    scan = dict(fsample=50.0, spin_period=20.0, prec_period=400.0, opening_turns=85.0 / 360.0, lon0_turns=0.0)

    def pointing(d, n):
        return oracle.expand_pointing(scan, dict(psi_turns=0.25 * d), 4, 0, n)

    c = mc.ring_case(ndet=NDET, nsamp=NBASE * 4, nside=4, base_first=0.08, prior=True, seed=3, pointing=pointing,
                     extra_pars=dict(cglimit=1e-16))
    c["pixels"][np.random.default_rng(1).random(c["pixels"].size) < 0.1] = -1
    return c


def handle(c):
    import libmadam_amd
    m = libmadam_amd.Madam(0)
    args = mc.call_args(c)
    m.configure(*args[:4], *args[7:], c["nnz"])
    m.set_kernel_variant(128)
    return m


def point(m, c):
    m.set_pointing(c["pixels"].copy(), c["pixweights"])


def solver(c, kind):
    """(call, results): one right-hand side in FP64, one mixed, or four in FP64 from device memory"""
    import torch
    if kind == "fp64":
        return lambda m: m.solve(c["signal"].copy()), lambda m: [m.baselines()["aa"], m.maps()["map"]]
    n = 1 if kind == "mixed" else 4
    sig = np.stack([c["signal"] * (1 + r) for r in range(n)]).reshape(n, NDET, -1)
    dev = torch.from_numpy(sig).cuda()
    torch.cuda.synchronize()

    def results(m):
        return [m.batch_result(n - 1)["aa"], m.batch_result(n - 1)["map"]]
    return lambda m: m.solve_batch(dev, precision=int(kind == "mixed"), on_device=True), results


def close(got, want, kind):
    for a, b in zip(got, want):
        if kind == "mixed":     # two converged inner solves, less the null-space offset
            a, b = a - a.mean(axis=0), b - b.mean(axis=0)
        assert np.linalg.norm(a - b) <= (1e-5 if kind == "mixed" else 1e-9) * np.linalg.norm(b)


@pytest.mark.parametrize("kind", ["fp64", "mixed", "batch"])
def test_each_allocation_of_a_solve_fails_once(kind):
    import libmadam_amd
    fail = libmadam_amd.lib().madam_fail_allocations
    c = case()
    solve, results = solver(c, kind)
    m = handle(c)
    point(m, c)
    fail(-1, 0)
    solve(m)
    total, want = fail(-1, 0), results(m)
    assert m.stats()["precond_kind"] == 3 and m.stats()["ncg"] == 0 and m.stats()["run_records"] > 0
    m.close()
    without = 0
    for k in range(total):
        m = handle(c)
        point(m, c)
        fail(k, 1)
        solve(m)
        assert fail(-1, 0) > k
        close(results(m), want, kind)
        without += m.stats()["run_records"] == 0
        solve(m)                # and with memory again
        close(results(m), want, kind)
        m.close()
    assert 0 < without


@pytest.mark.parametrize("nside", [4, 64])       # one copy, and the pieces
def test_products_without_device_memory(nside):
    import libmadam_amd
    fail = libmadam_amd.lib().madam_fail_allocations
    c = case()
    c["pars"].update(nside_map=nside, nside_cross=4)
    m = handle(c)
    point(m, c)
    m.solve(c["signal"].copy())
    want = {**m.maps(), **m.baselines()}
    fail(0, 10 ** 6)
    got = {**m.maps(), **m.baselines()}
    fail(-1, 0)
    for name in want:
        np.testing.assert_array_equal(got[name], want[name])
    m.close()


def test_each_allocation_of_the_pointing_fails_once():
    """on a handle that holds the tables of a solve on the pointing before"""
    import libmadam_amd
    fail = libmadam_amd.lib().madam_fail_allocations
    c = case()
    solve, results = solver(c, "fp64")
    m = handle(c)
    point(m, c)
    solve(m)
    want = results(m)
    fail(-1, 0)
    point(m, c)
    total = fail(-1, 0)
    for k in range(total):
        fail(k, 1)
        point(m, c)
        fail(-1, 0)
        solve(m)
        close(results(m), want, "fp64")
    m.close()


@pytest.mark.parametrize("kind", ["fp64", "mixed", "batch"])
def test_no_memory_at_all_is_an_error(kind):
    import libmadam_amd
    fail = libmadam_amd.lib().madam_fail_allocations
    c = case()
    solve, results = solver(c, kind)
    m = handle(c)
    point(m, c)
    solve(m)
    want = results(m)
    m.close()
    m = handle(c)
    for k in (0, 5, 10):
        fail(k, 10 ** 6)
        with pytest.raises(libmadam_amd.MadamError, match="memory"):
            point(m, c)
        fail(-1, 0)
    m.close()
    for k in (0, 10, 30, 50):
        m = handle(c)
        point(m, c)
        fail(k, 10 ** 6)
        with pytest.raises(libmadam_amd.MadamError, match="memory"):
            solve(m)
        fail(-1, 0)
        solve(m)
        close(results(m), want, kind)
        point(m, c)
        solve(m)
        close(results(m), want, kind)
        m.close()
