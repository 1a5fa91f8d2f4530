"""NonLocalPP ratios at orbital counts around the lane layouts of the ratio kernel (16, 32 and 64 lanes
per knot, one to twelve 16-byte orbital groups per lane, rows that are not whole vectors), against the
virtual-move ratios of the same batch at the same points."""
import numpy as np
import pytest

from miniqmc_amd import nlpp, qmcx
from test_gpu_sm_update import orbital_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("n", [3, 16, 33, 64, 100, 129, 192, 200, 257, 400, 512])
def test_ratios(n, precision):
    sysd = orbital_system(n)
    dev = qmcx.System(sysd, precisions=(precision,))
    rng = np.random.default_rng(n)
    W, rmax = 2, 2.4
    wb = qmcx.WalkerBatch(dev, W, delay_rank=1, precision=precision)
    R = rng.random((W, 2 * n, 3)) @ sysd.lattice
    wb.set_positions(R)
    wb.evaluate_log()
    spheres = nlpp.NonLocalPP(sysd, rmax=rmax, seed=n).randomize_walkers(W)
    ratios, pairs = wb.nlpp_evaluate(rmax, spheres, max_pairs=4)
    assert (ratios[np.arange(4) >= pairs[..., None]] == 0).all()   # unlisted slots stay as they were
    eps = 2.0 ** -53 if precision == qmcx.FP64 else 2.0 ** -24
    inv = [[wb.inverse(w, d) for d in range(2)] for w in range(W)]
    electrons = np.unique(rng.integers(0, 2 * n, 6))
    for e in electrons:
        near, pts = [], np.broadcast_to(R[:, e, None], (W, 48, 3)).copy()
        for w in range(W):
            disp, dist = nlpp.electron_ion_displacements(sysd.lattice, sysd.ion_pos, R[w, e])
            c = np.nonzero(dist < rmax)[0]
            near.append(c)
            assert pairs[w, e] == len(c)
            if len(c):
                pts[w, :12 * len(c)] = np.concatenate([dist[i] * spheres[w] + disp[i] + R[w, e] for i in c])
        ref = wb.flex_evaluate_ratios(int(e), pts)
        det, row = divmod(int(e), n)
        for w in range(W):
            m = 12 * len(near[w])
            if m == 0:
                continue
            psi = dev.spline_vgh(pts[w, :m], precision)[:, 0]
            terms = np.abs(psi * inv[w][det][row])
            jastrow = np.abs(ref[w, :m] / (psi @ inv[w][det][row]))
            # sums of the value row (64 terms per orbital, the points' own rounding) and over the
            # orbitals, and the exponents' sums over 2n electrons
            tol = (256 + 2 * n) * eps * terms.sum(1) * jastrow + 64 * eps * np.abs(ref[w, :m])
            got = ratios[w, e, :len(near[w])].reshape(-1)
            assert (np.abs(got - ref[w, :m]) <= tol).all(), (n, e, (np.abs(got - ref[w, :m]) / tol).max())
