"""Results are handed out only where they are there: after a batched solve that
failed, and on a handle whose configuration has changed (or was refused half
way), the products of an earlier solve are refused, not read with the new sizes."""
import numpy as np
import pytest

from tests import madam_cases as mc
from tests.test_gpu_batch import signals_for
from tests.test_gpu_parity import ring

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


def configure(m, case):
    a = mc.call_args(mc.copy_case(case))
    m.configure(*a[:4], *a[7:], case["nnz"])
    return a


def refused(m, nrhs):
    import libmadam_amd
    for call in [lambda: m.iterate_batch(1)] + [lambda k=k: m.batch_result(k) for k in range(nrhs)]:
        with pytest.raises(libmadam_amd.MadamError, match="batch"):
            call()


def test_results_of_a_failed_batch_are_refused():
    """A PSD with non-positive values: the batch fails when it builds the noise
    filter, after its right-hand sides are known."""
    import libmadam_amd
    case = ring(prior=True, nsamp=20000)
    sig = signals_for(case, 3)
    bad = mc.copy_case(case)
    bad["psdvals"] = np.where(np.tile(bad["psdfreqs"] < 1.0, 4), -bad["psdvals"], bad["psdvals"])
    m = libmadam_amd.Madam(0)
    a = configure(m, bad)
    m.set_pointing(a[4], a[5])
    with pytest.raises(libmadam_amd.MadamError, match="PSD"):
        m.solve_batch(sig, precision=0)
    refused(m, 3)
    # the same handle with a proper one
    a = configure(m, case)
    m.set_pointing(a[4], a[5])
    m.solve_batch(sig, precision=0)
    assert np.linalg.norm(m.batch_result(2)["aa"]) > 0
    m.close()


@pytest.mark.parametrize("accepted", [True, False])
def test_results_of_another_configuration_are_refused(accepted):
    import libmadam_amd
    case = ring(prior=True, nsamp=20000)
    large = ring(prior=True, nside=32, nsamp=40000)
    m = libmadam_amd.Madam(0)
    a = configure(m, case)
    m.set_pointing(a[4], a[5])
    m.solve(case["signal"].copy())
    m.solve_batch(signals_for(case, 3), precision=1)
    if accepted:
        configure(m, large)
    else:
        large["npsd"] = np.zeros_like(large["npsd"])   # a prior without PSDs: refused after the sizes are set
        with pytest.raises(libmadam_amd.MadamError, match="PSD"):
            configure(m, large)
    refused(m, 3)
    for call in (m.maps, m.baselines, lambda: m.iterate(1)):
        with pytest.raises(libmadam_amd.MadamError):
            call()
    m.close()


def test_products_after_an_error_of_the_callers():
    """A refused runtime call of the caller's own (a device that is not there)
    leaves an error behind; reading products must not take it for its own."""
    import ctypes
    import libmadam_amd
    case = ring(prior=False, nside=64, nsamp=20000)   # maps of 10 MB: the threaded path, the baselines the small one
    m = libmadam_amd.Madam(0)
    a = configure(m, case)
    m.set_pointing(a[4], a[5])
    m.solve(case["signal"].copy())
    want = m.maps(), m.baselines()
    hip = ctypes.CDLL(libmadam_amd.lib()._name)   # the runtime that the library is linked with
    for k, call in enumerate((m.maps, m.baselines)):
        assert hip.hipSetDevice(9999) != 0
        got = call()
        for name in got:
            assert np.array_equal(got[name], want[k][name]), name
    m.close()
