"""The proposal that flex_ratio_grad keeps for flex_accept_restore is evaluated again when the system's
functors or spline table, or the batch's state, changed in between."""
import numpy as np
import pytest

from miniqmc_amd import qmcx, systems

pytestmark = pytest.mark.gpu


def set_j1(dev, rng):
    for s in range(2):
        f = systems.random_functor(rng, 8, 2.5, -0.25)
        assert qmcx.load().qmcx_system_set_j1(dev.h, s, f.nparams, f.rcut, f.cusp, np.ascontiguousarray(f.params)) == 0


def set_spline(dev):
    d = dev.desc
    coefs = systems.spline_coefficients(d.ng, d.norb, d.npad, 77)
    assert qmcx.load().qmcx_system_set_spline(dev.h, np.array(d.ng, dtype=np.int32), d.norb, d.npad, coefs.reshape(-1),
                                              np.ascontiguousarray(d.spo_lattice).reshape(-1), 3) == 0


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("change", ["j1, evaluate_log", "j1, another batch's evaluate_log", "j1 before the ratio",
                                    "spline", "spline, evaluate_log"])
def test_proposal_follows_the_tables(change, precision):
    """Batch `again` gets a setting (as it is) after the changes, which makes it evaluate the proposal again."""
    results = []
    for again in (False, True):
        dev = qmcx.System(systems.make_system("nio8-cubic"))
        wb, other = (qmcx.WalkerBatch(dev, 2, delay_rank=2, precision=precision) for _ in range(2))
        R = systems.initial_positions(dev.desc, 2)
        for x in (wb, other):
            x.set_positions(R)
            x.evaluate_log()
        if change == "j1 before the ratio":
            set_j1(dev, np.random.default_rng(5))
        wb.flex_ratio_grad(7, np.full((2, 3), 0.2))
        if change == "j1 before the ratio":   # uploaded by the other batch only now
            other.evaluate_log()
        if change.startswith("j1,"):
            set_j1(dev, np.random.default_rng(5))
        if change.startswith("spline"):
            set_spline(dev)
        if change.endswith("another batch's evaluate_log"):
            other.evaluate_log()
        elif change.endswith("evaluate_log"):
            wb.evaluate_log()
        if again:
            wb.set_flush(0)
        wb.flex_accept_restore(7, np.ones(2, dtype=np.int32))
        log = wb.flex_evaluate_gl()
        results.append((log, *wb.gl(), wb.inverse(0, 0), wb.inverse(1, 0)))
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
