"""The FP64 Gauss-Jordan inversion at orders around its tiles (16), sub-panels (16), panels (32 up to
n = 512, 16 past it) and largest order, against numpy."""
import numpy as np
import pytest

from miniqmc_amd import qmcx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 81, 97, 200, 385, 511, 512, 513, 529, 1024])
def test_orders(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((2, n, n))
    if n > 2:
        a[1] = a[1][::-1] * np.exp(rng.uniform(-3, 3, (n, 1)))   # rows of different sizes, many exchanges
    psiM, logdet, phase = qmcx.invert_transpose(a)
    for m in range(2):
        x = psiM[m].T
        # backward-stable elimination with partial pivoting: |A X - I| <= c n eps |A| |X|
        bound = 8 * n * 2.0 ** -53 * np.linalg.norm(a[m], 2) * np.linalg.norm(x, 2)
        assert np.linalg.norm(a[m] @ x - np.eye(n), 2) <= bound + 1e-15
        sign, ld = np.linalg.slogdet(a[m])
        assert abs(logdet[m] - ld) <= 8 * n * 2.0 ** -53 * (np.linalg.cond(a[m]) + abs(ld)) + 1e-14
        assert (phase[m] == 0.0) == (sign > 0)


def test_permutations_and_signs():
    """Signed permutation matrices: the inverse and the sign are exact."""
    rng = np.random.default_rng(3)
    for n in (5, 33, 130):
        a = np.zeros((4, n, n))
        for m in range(4):
            a[m, np.arange(n), rng.permutation(n)] = rng.choice([-1.0, 1.0], n)
        psiM, logdet, phase = qmcx.invert_transpose(a)
        np.testing.assert_array_equal(psiM, a)   # (A^-1)^T = A
        np.testing.assert_array_equal(logdet, 0.0)
        np.testing.assert_array_equal(phase == 0.0, np.linalg.det(a) > 0)
