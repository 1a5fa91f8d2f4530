"""evaluateLog of a batch large enough for the electrons to be ordered by place against the same walkers
in batches too small for it: the same SPO rows, so the same log|Psi|, G, L and inverses bit for bit."""
import numpy as np
import pytest

from miniqmc_amd import qmcx, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,fp64_rows", [(qmcx.FP64, False), (qmcx.FP32, False), (qmcx.FP32, True)])
@pytest.mark.parametrize("name,walkers,part", [("nio8-cubic", 91, 13), ("nio16", 55, 11), ("nio32", 45, 15)])
def test_same_as_small_batches(name, walkers, part, precision, fp64_rows):
    sysd = systems.make_system(name)
    dev = qmcx.System(sysd, precisions=(precision,))
    R = systems.initial_positions(sysd, walkers)

    def evaluate(r):
        wb = qmcx.WalkerBatch(dev, len(r), delay_rank=1, precision=precision)
        wb.set_fp64_rows(fp64_rows)
        wb.set_positions(r)
        log = wb.evaluate_log()
        G, L, _ = wb.gl()
        return log, G, L, wb.inverse(len(r) - 1, 1)

    whole = evaluate(R)
    for o in range(0, walkers, part):
        small = evaluate(R[o:o + part])
        for a, b in zip(whole[:3], small[:3]):
            np.testing.assert_array_equal(a[o:o + part], b)
    np.testing.assert_array_equal(whole[3], small[3])
