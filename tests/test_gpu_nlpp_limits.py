"""NonLocalPP at the edges of what the calls accept: spline tables whose padding holds NaN, and
more ions than fit a workgroup's LDS beside the walker."""
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


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("nions", [6400, 9000])
def test_many_ions(nions, precision):
    """Against the virtual-move ratios at the same points."""
    rng = np.random.default_rng(nions)
    n, a, W, rmax = 24, 40.0, 2, 1.3
    base = orbital_system(n)
    lattice = np.diag([a, a, a])
    species = (np.arange(nions) >= nions // 2).astype(np.int32)
    sysd = dataclasses.replace(base, lattice=lattice, spo_lattice=lattice.copy(), ion_pos=rng.random((nions, 3)) * a,
                               ion_species=species)
    dev = qmcx.System(sysd, precisions=(precision,))
    wb = qmcx.WalkerBatch(dev, W, delay_rank=1, precision=precision)
    R = rng.random((W, 2 * n, 3)) * a
    wb.set_positions(R)
    wb.evaluate_log()
    spheres = nlpp.NonLocalPP(sysd, rmax=rmax, seed=3).randomize_walkers(W)
    ratios, pairs = wb.nlpp_evaluate(rmax, spheres, max_pairs=12)
    assert pairs.sum() > 0
    eps = 2.0 ** -53 if precision == qmcx.FP64 else 2.0 ** -24
    for e in range(0, 2 * n, 5):
        for w in range(W):
            disp, dist = nlpp.electron_ion_displacements(lattice, sysd.ion_pos, R[w, e])
            c = np.nonzero(dist < rmax)[0]
            assert pairs[w, e] == len(c)
            if len(c) == 0:
                continue
            pts = np.broadcast_to(R[:, e, None], (W, 12 * len(c), 3)).copy()
            pts[w] = np.concatenate([dist[i] * spheres[w] + disp[i] + R[w, e] for i in c])
            ref = wb.flex_evaluate_ratios(e, pts)[w]
            inv = wb.inverse(w, e // n)[e % n]
            psi = dev.spline_vgh(pts[w], precision)[:, 0]
            # value rows (64 terms an orbital, the points' own rounding times 10 cells of a/10), the sum over
            # the orbitals, and the exponents' sums over the ions in reach and 2n electrons
            terms = (np.abs(psi) + 1) * np.abs(inv)
            jastrow = np.abs(ref / (psi @ inv))
            tol = (256 + 2 * n) * eps * terms.sum(1) * jastrow + 256 * eps * np.abs(ref)
            got = ratios[w, e, :len(c)].reshape(-1)
            assert (np.abs(got - ref) <= tol).all(), (e, w, (np.abs(got - ref) / tol).max())
