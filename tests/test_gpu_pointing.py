"""Pointing expansion where detectors share a boresight or a spin offset, in
groups of every size, and with 32- and 64-bit pixel arithmetic: bit for bit the
CPU expansion of each detector by itself."""
import numpy as np
import pytest

import oracle

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


HORNS = [dict(psi_turns=(0.0, 0.125, 0.25, 0.375)[j % 4], open_offset_turns=(j // 4) * 0.1 / 360.0)
         for j in range(17)]
MIXED = [dict(psi_turns=0.07 * j, open_offset_turns=0.001 * (j // 2), spin_offset_turns=0.0003 * (j // 3))
         for j in range(9)]


# one detector per thread, groups of 2, 4 and 8 (with a ragged last one), the
# smallest Nside, the last one of the 32-bit arithmetic and the first past it
@pytest.mark.parametrize("dets,n,nside", [(HORNS[:1], 1, 1), (HORNS[:8], 70001, 2), (HORNS[:8], 140001, 64),
                                          (HORNS, 262145, 1024), (MIXED, 524289, 8192), (MIXED[:3], 600000, 16384),
                                          (HORNS[:5], 600001, 256)])
def test_expansion_of_shared_boresights(dets, n, nside):
    import libmadam_amd
    scan = dict(fsample=100.0, spin_period=60.0, prec_period=360 * 3600.0, opening_turns=85 / 360, lon0_turns=0.01)
    gp, gw = libmadam_amd.expand_pointing(scan, dets, nside, 777, n)
    for d in sorted({0, len(dets) // 2, len(dets) - 1}):
        op, ow = oracle.expand_pointing(scan, dets[d], nside, 777, n)
        assert np.array_equal(gp[d], op), (d, np.sum(gp[d] != op))
        assert np.array_equal(gw[d].view(np.uint32), ow.view(np.uint32)), d
