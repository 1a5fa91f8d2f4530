"""Sherman-Morrison update of the inverse by one accepted move, at orbital counts around the row
layouts of the update kernel (rows of 16, 32 and 64 lanes, remainders, rows that are not whole
16-byte vectors), against the same update in numpy."""
import numpy as np
import pytest

from miniqmc_amd import qmcx, systems

pytestmark = pytest.mark.gpu


def orbital_system(n, ng=(10, 11, 12)):
    """2n electrons and n orbitals in a skewed cell, with two ions and short Jastrows."""
    rng = np.random.default_rng(n)
    a = 6.0
    lattice = np.array([[a, 0.3, 0.0], [0.2, a, 0.1], [0.0, 0.4, a]])
    ion_pos = np.array([[0.1, 0.2, 0.3], [0.6, 0.5, 0.7]]) @ lattice
    npad = (n + 15) // 16 * 16
    f = [systems.random_functor(rng, 8, 2.9, c) for c in (-0.25, -0.25, 0.0, 0.0)]
    return systems.System(f"n{n}", lattice, ion_pos, np.array([0, 1], dtype=np.int32), 2, n, n, ng, n, npad,
                          lattice.copy(), systems.spline_coefficients(ng, n, npad, n), f[:2], f[2:])


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("n", [7, 8, 30, 50, 64, 96, 100, 132, 192, 200, 260, 384, 388, 512])
def test_one_accept(n, precision):
    sysd = orbital_system(n)
    dev = qmcx.System(sysd, precisions=(precision,))
    W, accept = 3, np.array([1, 0, 1], dtype=np.int32)
    wb = qmcx.WalkerBatch(dev, W, delay_rank=1, precision=precision)
    rng = np.random.default_rng(n + 1)
    R = rng.random((W, 2 * n, 3)) @ sysd.lattice
    wb.set_positions(R)
    wb.evaluate_log()
    eps = 2.0 ** -53 if precision == qmcx.FP64 else 2.0 ** -24
    for iel in (0, n + n // 2, 2 * n - 1):
        det, row = divmod(iel, n)
        before = [wb.inverse(w, det) for w in range(W)]
        displ = 0.5 * rng.standard_normal((W, 3))
        wb.flex_ratio_grad(iel, displ)
        wb.flex_accept_restore(iel, accept)
        psi = dev.spline_vgh(wb.positions()[:, iel], precision)[:, 0]
        for w in range(W):
            after = wb.inverse(w, det)
            if not accept[w]:
                np.testing.assert_array_equal(after, before[w])
                continue
            b = before[w]
            ratio = b[row] @ psi[w]
            t = b @ psi[w]
            t[row] -= 1
            t /= ratio
            expect = b - t[:, None] * b[row]
            # rounding of the stored result and of t, and of the orbital row (a 64-term sum of
            # coefficients in [-1, 1] with weights that sum to one) in t and in the ratio
            dt = 64 * eps * (np.abs(b).sum(1) + np.abs(t) * np.abs(b[row]).sum()) / abs(ratio)
            tol = 4 * eps * (np.abs(b) + np.abs(t)[:, None] * np.abs(b[row])) + dt[:, None] * np.abs(b[row])
            assert (np.abs(after - expect) <= tol).all(), (n, iel, w, (np.abs(after - expect) / tol).max())
