"""flex_* moves whose caller accepts a proposal with a NaN ratio: the kernel rejects it, so the delayed rows
that count towards a flush are the kernel's, and the walker goes on as if the caller had rejected."""
import numpy as np
import pytest

from miniqmc_amd import qmcx, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("delay", [1, 2, 3, 8])
def test_nan_walker(delay, precision):
    sysd = systems.make_system("nio8-cubic")
    dev = qmcx.System(sysd, precisions=(precision,))
    W, rng = 4, np.random.default_rng(delay)
    R = systems.initial_positions(sysd, W)
    a, b = (qmcx.WalkerBatch(dev, W, delay_rank=delay, precision=precision) for _ in range(2))
    for x in (a, b):
        x.set_positions(R)
        x.evaluate_log()
    # walker 2 has a NaN displacement at some moves, of both determinants, before and after it has pending rows
    electrons = list(range(12)) + list(range(48, 60)) + [12, 13, 60]
    nans = {0, 3, 4, 11, 48, 50, 57, 60}
    for iel in electrons:
        displ = 0.3 * rng.standard_normal((W, 3))
        accept = (rng.random(W) < 0.8).astype(np.int32)
        accept[2] = 1
        bad, rejected = displ.copy(), accept.copy()
        if iel in nans:
            bad[2] = np.nan
            rejected[2] = 0
        ra, rb = a.flex_ratio_grad(iel, bad), b.flex_ratio_grad(iel, displ)
        for p, q in zip(ra, rb):
            np.testing.assert_array_equal(p[[0, 1, 3]], q[[0, 1, 3]])
            if iel not in nans:
                np.testing.assert_array_equal(p[2], q[2])
        assert np.isnan(ra[0][2]) == (iel in nans)
        a.flex_accept_restore(iel, accept)
        b.flex_accept_restore(iel, rejected)
    np.testing.assert_array_equal(a.positions(), b.positions())
    np.testing.assert_array_equal(a.accepts(), b.accepts())
    for w in range(W):
        for det in range(2):
            np.testing.assert_array_equal(a.inverse(w, det), b.inverse(w, det))


def test_accept_without_a_proposal():
    """Electron -1, the value that stands for no proposal, is an error before the first ratio_grad and after
    an accept."""
    sysd = systems.make_system("nio8-cubic")
    dev = qmcx.System(sysd, precisions=(qmcx.FP64,))
    wb = qmcx.WalkerBatch(dev, 2, delay_rank=2, precision=qmcx.FP64)
    R = systems.initial_positions(sysd, 2)
    wb.set_positions(R)
    wb.evaluate_log()
    yes = np.ones(2, dtype=np.int32)
    with pytest.raises(qmcx.QmcxError):
        wb.flex_accept_restore(-1, yes)
    wb.flex_ratio_grad(3, np.full((2, 3), 0.1))
    wb.flex_accept_restore(3, yes)
    after = wb.positions()
    for iel in (-1, 3):
        with pytest.raises(qmcx.QmcxError):
            wb.flex_accept_restore(iel, yes)
    np.testing.assert_array_equal(wb.positions(), after)
