"""NonLocalPP at the edges of what the calls accept: spline tables whose padding holds NaN."""
import dataclasses

import numpy as np
import pytest

from miniqmc_amd import nlpp, qmcx
from test_gpu_sm_update import orbital_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("n", [3, 33, 64, 100, 192, 257])
def test_padding_does_not_enter(n, precision):
    """The columns past norb belong to no orbital: their values do not reach a ratio."""
    base = orbital_system(n)
    npad = base.npad + 16   # whole 16-byte groups of padding too
    ratios = []
    for fill in (0.0, np.nan):
        points = base.coefs.reshape(-1, base.npad)
        coefs = np.full((len(points), npad), fill, dtype=np.float32)
        coefs[:, :n] = points[:, :n]
        sysd = dataclasses.replace(base, npad=npad, coefs=coefs.reshape(-1))
        dev = qmcx.System(sysd, precisions=(precision,))
        wb = qmcx.WalkerBatch(dev, 2, delay_rank=1, precision=precision)
        wb.set_positions(np.random.default_rng(n).random((2, 2 * n, 3)) @ sysd.lattice)
        wb.evaluate_log()
        spheres = nlpp.NonLocalPP(sysd, rmax=2.4, seed=n).randomize_walkers(2)
        r, pairs = wb.nlpp_evaluate(2.4, spheres, max_pairs=4)
        assert pairs.sum() > 0
        ratios.append(r)
    assert np.isfinite(ratios[0]).all()
    np.testing.assert_array_equal(ratios[0], ratios[1])
