"""Columns whose squares underflow: two diagonal blocks of a symmetric matrix that
couple so weakly that every element of a column to be reduced lies below 1e-154.
A reflector formed from subnormal squares is not orthogonal, which spoils the
eigenpairs of a whole block (kSquareMin in reflector.hpp).

matrix_root gives A^-1/2 through all eigenpairs; R A R = I to the backward error of
an n-dimensional orthogonal reduction, bounded by 10 n eps cond(A): the couplings
themselves are far below rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _two_blocks(n, coupling, head):
    """An SPD matrix whose leading block is `head` ("diagonal": its columns are the
    couplings alone; "dense": they reach that size at the block's end only)."""
    rng = np.random.default_rng(7 * n)
    B = rng.normal(size=(n, n))
    A = B @ B.T / n + np.eye(n)
    h = n // 2 + 3
    if head == "diagonal":
        h = min(h, 40)
        A[:h, :h] = np.diag(rng.uniform(1.0, 3.0, size=h))
    A[:h, h:] *= coupling
    A[h:, :h] *= coupling
    return A


def _check(engine, A):
    n = A.shape[0]
    w = np.linalg.eigvalsh(A)
    tol = 10 * max(n, 8) * np.finfo(float).eps * w[-1] / w[0]
    R = engine.matrix_root(A)
    assert np.abs(R - R.T).max() < tol
    assert np.abs(R @ A @ R - np.eye(n)).max() < tol


# (dense heads shrink by up to 1e-16 from a column to the next, so their couplings
# cover what lands between 1e-163 and 1e-154 either way)
@pytest.mark.parametrize("head,exponents", [("diagonal", range(152, 165)), ("dense", range(138, 182))])
@pytest.mark.parametrize("n", [19, 60, 131])
def test_weakly_coupled_blocks(engine, n, head, exponents):
    for x in exponents:
        _check(engine, _two_blocks(n, 10.0 ** -x, head))


@pytest.mark.parametrize("n", [300, 600, 1100, 2100])
def test_weakly_coupled_blocks_of_every_route(engine, n):
    """Every register class of the panels and of the chase, the windows in memory,
    and the one-stage reduction above 2048 rows."""
    for x in (156, 159, 161):
        _check(engine, _two_blocks(n, 10.0 ** -x, "diagonal"))


@pytest.mark.parametrize("shift", [-400, -100, -40, -12, 12, 400])
@pytest.mark.parametrize("n", [2, 12, 17, 60, 300, 1100, 2100])
def test_scaled_matrices(engine, n, shift):
    """A power of two in front of a matrix comes out as its root, exactly but for the
    rounding of a reduction: no test in the solver compares with 1."""
    rng = np.random.default_rng(3 * n)
    B = rng.normal(size=(n, n))
    A = B @ B.T / n + np.eye(n)
    w = np.linalg.eigvalsh(A)
    tol = 10 * max(n, 8) * np.finfo(float).eps * w[-1] / w[0]
    R = np.ldexp(engine.matrix_root(np.ldexp(A, shift)), shift // 2)
    assert np.abs(R @ A @ R - np.eye(n)).max() < tol
