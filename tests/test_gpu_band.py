"""The two-stage tridiagonalisation (dense to band to tridiagonal) behind the
dense eigensolver, at the sizes where its pieces change: one and two rows, the
band width and its neighbours, the first panels, and both sides of every size
class of the panel and bulge-chasing kernels.  Inputs: a general matrix, and
ones whose columns need no reflector at all (diagonal, tridiagonal, a matrix that
is a band already), where every tau is zero.

matrix_root gives A^-1/2 through all eigenpairs; R A R = I to the backward
error of an n-dimensional orthogonal reduction, bounded by 10 n eps cond(A)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 15, 16, 17, 18, 19, 33, 34, 65, 66, 129, 130, 145, 257, 258, 273, 513, 514, 529,
         1025, 1026, 1041, 1100]


def _matrix(n, kind):
    rng = np.random.default_rng(1000 + n)
    if kind == "dense":
        B = rng.normal(size=(n, n))
        return B @ B.T / n + np.eye(n)
    A = np.diag(rng.uniform(1.0, 3.0, size=n))
    if kind == "tridiagonal" and n > 1:
        off = rng.uniform(-0.4, 0.4, size=n - 1)
        A += np.diag(off, 1) + np.diag(off, -1)
    if kind == "band":
        for k in range(1, min(17, n)):
            off = rng.uniform(-0.02, 0.02, size=n - k)
            A += np.diag(off, k) + np.diag(off, -k)
    return A


def _check(engine, A):
    n = A.shape[0]
    w = np.linalg.eigvalsh(A)
    tol = 10 * max(n, 8) * np.finfo(float).eps * w[-1] / w[0]
    R = engine.matrix_root(A)
    assert np.abs(R - R.T).max() < tol
    assert np.abs(R @ A @ R - np.eye(n)).max() < tol


@pytest.mark.parametrize("n", SIZES)
def test_general_matrix(engine, n):
    _check(engine, _matrix(n, "dense"))


@pytest.mark.parametrize("kind", ["diagonal", "tridiagonal", "band"])
@pytest.mark.parametrize("n", [2, 17, 40, 130, 300, 1040])
def test_matrices_without_reflectors(engine, n, kind):
    _check(engine, _matrix(n, kind))


@pytest.mark.parametrize("cols", [1, 2, 3])
def test_build_through_every_size_class(engine, cols):
    """A chain whose submatrices fall into several size classes at once, against
    the oracle."""
    from conftest import small_system
    from oracle import ptb_oracle as O
    mol, H, S = small_system("alkane", 14)
    ref = O.sm_stupid_simple(mol.ndim, mol.nel, H, S, mol.n, mol.xyz, mol.aoat, cols, 2)
    P = np.full_like(H, np.nan)
    rep = engine.sm_stupid_simple(mol.ndim, mol.nel, H, S, P, mol.n, mol.xyz, mol.aoat, cols, 2)
    assert np.abs(P - ref.P).max() < 1e-8
    assert rep["mu"] == ref.mu and rep["muiter"] == ref.muiter


@pytest.mark.parametrize("n", [1472, 2047, 2048])
def test_windows_in_memory(engine, n):
    """Above 1025 rows part of the chase's windows live in memory: the first
    sizes with two and three of them per wavefront, and the largest."""
    _check(engine, _matrix(n, "dense"))


def test_more_submatrices_than_compute_units(engine):
    """Single-column submatrices of 27 waters (621 of several size classes, a
    launch per class) against the oracle."""
    from conftest import small_system
    from oracle import ptb_oracle as O
    mol, H, S = small_system("water", (3, 3, 3), 4)
    ref = O.sm_stupid_simple(mol.ndim, mol.nel, H, S, mol.n, mol.xyz, mol.aoat, 1, 2)
    P = np.full_like(H, np.nan)
    rep = engine.sm_stupid_simple(mol.ndim, mol.nel, H, S, P, mol.n, mol.xyz, mol.aoat, 1, 2)
    assert np.abs(P - ref.P).max() < 1e-8
    assert rep["mu"] == ref.mu and rep["muiter"] == ref.muiter


@pytest.mark.parametrize("m", [3, 18, 19, 34, 66, 83, 98, 530])
def test_sweep_groups_of_every_remainder(engine, m):
    """One to five sweep groups and more (a pass of four wavefronts full, cut short,
    followed by another), last column pieces of several widths: solve2's
    eigenvectors are S-orthonormal and solve the pencil."""
    rng = np.random.default_rng(10 * m)
    A = _matrix(m, "dense")
    B = rng.normal(size=(m, m))
    S = np.eye(m) + 0.05 * (B + B.T) / np.sqrt(m)
    iu = np.tril_indices(m)
    P, e, focc, U, fail = engine.solve2(1, m, 2, 0, 300.0, A[iu].copy(), S[iu].copy())
    assert not fail
    tol = 100 * max(m, 8) * np.finfo(float).eps
    assert np.abs(U.T @ S @ U - np.eye(m)).max() < tol
    assert np.abs(A @ U - (S @ U) * e).max() < tol * np.abs(e).max()


def test_chase_routes_agree(engine):
    """The same submatrices in a batch of up to one per CU, of a few times as many
    (shared workgroups) and of more (a launch per size class): each batch's
    densities are those of the molecules built alone."""
    import torch
    from conftest import small_system
    mols = [small_system("water", (2, 2, 2), s) for s in range(3)] + [small_system("alkane", 6), small_system("alkane", 20)]

    def item(mol, H, S):
        dH, dS = torch.from_numpy(H).cuda(), torch.from_numpy(S).cuda()
        return (mol.ndim, mol.nel, dH, dS, torch.zeros_like(dH), mol.n, mol.xyz, mol.aoat)

    alone = []
    for m in mols:
        it = item(*m)
        engine.sm_stupid_simple_dev(*it, 2, 2)
        torch.cuda.synchronize()
        alone.append(it[4])
    for copies in (3, 10):
        items = [item(*m) for _ in range(copies) for m in mols]
        torch.cuda.synchronize()
        engine.sm_stupid_simple_batch(items, 2, 2, device=True)
        torch.cuda.synchronize()
        for k, it in enumerate(items):
            assert torch.equal(it[4], alone[k % len(mols)])
