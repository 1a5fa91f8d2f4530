"""Shapes that the prepared systems do not have, on the paths that are chosen by size: SPO rows ordered by
place (orbital counts that are not whole 16-byte vectors, a skewed cell, the largest orbital count of the path),
the flush inside the move kernel (tile counts below those its forms hold), virtual ratios at the sizes where the
pinned block grows and where the call leaves it, and NonLocalPP's knots ordered by place and not."""
import dataclasses

import numpy as np
import pytest

from miniqmc_amd import nlpp, qmcx, systems
from test_gpu_sm_update import orbital_system

pytestmark = pytest.mark.gpu


def fine_grid_system(n, ng):
    """orbital_system with a spline table of the given grid."""
    base = orbital_system(n)
    return dataclasses.replace(base, ng=ng, coefs=systems.spline_coefficients(ng, n, base.npad, n))


@pytest.mark.parametrize("precision,n,walkers,ng", [
    (qmcx.FP32, 161, 30, None), (qmcx.FP32, 250, 18, None), (qmcx.FP32, 384, 12, None), (qmcx.FP32, 97, 50, (28, 29, 30)),
    (qmcx.FP64, 83, 60, None), (qmcx.FP64, 129, 40, None), (qmcx.FP64, 512, 9, None), (qmcx.FP64, 50, 110, (32, 30, 31))])
def test_ordered_rows(precision, n, walkers, ng):
    """A batch whose electrons are ordered against the same walkers in batches of fewer than 8192 electrons."""
    sysd = orbital_system(n) if ng is None else fine_grid_system(n, ng)
    dev = qmcx.System(sysd, precisions=(precision,))
    R = np.random.default_rng(n).random((walkers, 2 * n, 3)) @ sysd.lattice
    # the call's own rule: 8192 electrons or more whose 64-point stencils cover the grid four times, and rows
    # of 40 groups of 16 bytes (24 with a table past 8 MB)
    row = sysd.npad * (4 if precision == qmcx.FP32 else 8)
    assert walkers * 2 * n >= 8192 and 64 * walkers * 2 * n >= 4 * np.prod(sysd.ng)
    assert row >= 40 * 16 or (row >= 24 * 16 and np.prod(np.array(sysd.ng) + 3) * row > 8e6)
    part = 8191 // (2 * n)

    def evaluate(r):
        wb = qmcx.WalkerBatch(dev, len(r), delay_rank=1, precision=precision)
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


@pytest.mark.parametrize("n,delay", [(n, d) for n in (16, 48, 80, 112, 160, 176, 208, 304, 368)
                                     for d in (8, 16, 32) if d <= n])
def test_flush_tiles(n, delay):
    """A sweep whose flushes take the U rows from LDS, in forms that hold 6, 12 or 24 tiles of 16 orbitals,
    against one whose flushes read them from HBM tile by tile: the same sums in the same order."""
    sysd = orbital_system(n)
    dev = qmcx.System(sysd, precisions=(qmcx.FP32,))
    W = 2
    R = np.random.default_rng(n).random((W, 2 * n, 3)) @ sysd.lattice
    out = []
    for kind in (0, 2):
        wb = qmcx.WalkerBatch(dev, W, delay_rank=delay, precision=qmcx.FP32)
        wb.set_flush(kind)
        wb.set_positions(R)
        wb.evaluate_log()
        wb.run(1, 3, 0.05, qmcx.ACCEPT_REFERENCE)
        out.append((wb.positions(), *[wb.inverse(w, d) for w in range(W) for d in range(2)]))
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("walkers,points", [(1, 2047), (1, 2049), (1, 16384), (1, 16385), (7, 300), (7, 2340),
                                            (7, 2341), (64, 256), (64, 257), (64, 1024), (64, 1025)])
def test_virtual_ratio_sizes(walkers, points):
    """A call's ratios are those of its points in small calls, whatever the sizes before it."""
    sysd = orbital_system(33)
    dev = qmcx.System(sysd, precisions=(qmcx.FP64,))
    rng = np.random.default_rng(points)
    wb = qmcx.WalkerBatch(dev, walkers, delay_rank=1, precision=qmcx.FP64)
    wb.set_positions(rng.random((walkers, 66, 3)) @ sysd.lattice)
    wb.evaluate_log()
    pts = rng.random((walkers, points, 3)) @ sysd.lattice
    whole = wb.flex_evaluate_ratios(5, pts)
    part = max(1, 2000 // walkers)
    for o in range(0, points, part):
        np.testing.assert_array_equal(whole[:, o:o + part], wb.flex_evaluate_ratios(5, pts[:, o:o + part]))


@pytest.mark.parametrize("precision", [qmcx.FP64, qmcx.FP32])
@pytest.mark.parametrize("n,ng", [(33, (60, 61, 59)), (100, (40, 41, 42))])
def test_nlpp_order(n, ng, precision):
    """NonLocalPP of walkers enough for their knots to be ordered by grid cell, in a table past 24 MB, against
    the same walkers one at a time, whose knots are not: the same ratios."""
    sysd = fine_grid_system(n, ng)
    dev = qmcx.System(sysd, precisions=(precision,))
    row = sysd.npad * (4 if precision == qmcx.FP32 else 8)
    assert np.prod(np.array(ng) + 3) * row > 24e6
    rmax = 1.1
    per_walker = 2 * 4 * np.pi / 3 * rmax**3 / abs(np.linalg.det(sysd.lattice)) * 2 * n * 12 * 64 * row
    walkers = int(512e6 / per_walker) + 1
    assert per_walker < 256e6 < walkers * per_walker   # the call's own rule
    R = np.random.default_rng(n).random((walkers, 2 * n, 3)) @ sysd.lattice
    spheres = nlpp.NonLocalPP(sysd, rmax=rmax, seed=n).randomize_walkers(walkers)

    def evaluate(lo, hi):
        wb = qmcx.WalkerBatch(dev, hi - lo, delay_rank=1, precision=precision)
        wb.set_positions(R[lo:hi])
        wb.evaluate_log()
        return wb.nlpp_evaluate(rmax, spheres[lo:hi], max_pairs=4)

    ratios, pairs = evaluate(0, walkers)
    assert pairs.sum() > 0
    for w in range(0, walkers, max(1, walkers // 12)):
        one, count = evaluate(w, w + 1)
        np.testing.assert_array_equal(count[0], pairs[w])
        np.testing.assert_array_equal(one[0], ratios[w])
