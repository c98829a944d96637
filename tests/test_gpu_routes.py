"""One submatrix, several routes: which kernels reduce and bisect it depends on what
else is in its batch.  Every route must give what the molecule gives alone."""
import numpy as np
import pytest

from conftest import small_system

pytestmark = pytest.mark.gpu


def _item(ndim, nel, H, S, n, xyz, aoat):
    import torch
    dH, dS = torch.from_numpy(H).cuda(), torch.from_numpy(S).cuda()
    return (ndim, nel, dH, dS, torch.zeros_like(dH), n, xyz, aoat)


def _mol(kind, size, seed=0, filt=1e-4):
    mol, H, S = small_system(kind, size, seed, filt=filt)
    return _item(mol.ndim, mol.nel, H, S, mol.n, mol.xyz, mol.aoat)


def _blocks(sizes, hub=0):
    """A synthetic molecule of diagonal blocks, every orbital its own atom; `hub`
    more orbitals couple to the first one only."""
    n = sum(sizes) + hub
    rng = np.random.default_rng(n)
    H, S = np.zeros((n, n)), np.eye(n)
    at = 0
    for m in sizes:
        i = slice(at, at + m)
        S[i, i] += 0.2 / m * (1.0 - np.eye(m))
        H[i, i] = np.triu(rng.uniform(0.0, 0.4 / np.sqrt(m), size=(m, m)))
        at += m
    if hub:
        S[0, at:] = 0.01
    np.fill_diagonal(H, -np.linspace(0.2, 1.2, n))
    iu = np.triu_indices(n)
    Hp, Sp = (np.zeros(n * (n + 1) // 2) for _ in range(2))
    Hp[iu[0] + iu[1] * (iu[1] + 1) // 2] = H[iu]
    Sp[iu[0] + iu[1] * (iu[1] + 1) // 2] = S[iu]
    return n, 2 * (n // 4), Hp, Sp, n, np.zeros((n, 3)), np.arange(1, n + 1)


def _alone(engine, item, cols):
    import torch
    it = item[:4] + (torch.zeros_like(item[4]),) + item[5:]
    rep = engine.sm_stupid_simple_dev(*it, cols, 2)
    torch.cuda.synchronize()
    return it[4], rep


def _batch(engine, items, cols):
    import torch
    items = [it[:4] + (torch.zeros_like(it[4]),) + it[5:] for it in items]
    reps = engine.sm_stupid_simple_batch(items, cols, 2, device=True)
    torch.cuda.synchronize()
    return [it[4] for it in items], reps


def test_batches_above_2048_rows(engine):
    """Two blocks of more than 2048 rows in one call take the batched one-stage
    reduction (a lone one takes the multi-workgroup kernels), beside a small block on
    the band route.  The large densities agree to the engine's bar against the oracle
    (backward errors of two reductions, n eps cond(S) / gap, are about 3e-9), the
    small one bit for bit."""
    import torch
    items = [_mol("water", (6, 4, 4), 1, 1e-5), _mol("alkane", 95, 0, 1e-5), _mol("alkane", 12, 0, 1e-5)]
    alone = [_alone(engine, it, 3) for it in items]
    assert [a[1]["max_m"] > 2048 for a in alone] == [True, True, False]
    assert all(a[1]["not_spd"] == 0 for a in alone)
    P, reps = _batch(engine, items, 3)
    for k in range(3):
        assert reps[k]["not_spd"] == 0 and torch.isfinite(P[k]).all()
        assert (P[k] - alone[k][0]).abs().max().item() < 1e-8
    assert torch.equal(P[2], alone[2][0])
    # one large block beside a small one: the lone route for it, the same bits
    P, reps = _batch(engine, [items[0], items[2]], 3)
    assert torch.equal(P[0], alone[0][0]) and torch.equal(P[1], alone[2][0])


def test_every_size_class_of_the_chase(engine):
    """A batch of more than two workgroups per CU (a launch per size class) with
    submatrices in every class, one above 1025 rows (windows in memory) among them,
    against the molecules built alone (one launch)."""
    import torch
    mols = [_mol("water", (4, 4, 4), s) for s in range(3)] + [_mol("water", (2, 2, 2), s) for s in range(3)]
    mols += [_mol("water", (1, 1, 1), s) for s in range(4)] + [_mol("water", (2, 1, 1), s) for s in range(4)]
    mols += [_item(*_blocks([40, 60], hub=1000)), _item(*_blocks([100]))]
    alone = [_alone(engine, it, 2)[0] for it in mols]
    P, reps = _batch(engine, mols, 2)
    m, _, _ = engine.sm_spectra(sum(r["nsm"] for r in reps), sum(r["sum_m"] for r in reps))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    edges = [0, 65, 129, 257, 513, 1025, 2048]
    counts = [int(((m > a) & (m <= b)).sum()) for a, b in zip(edges, edges[1:])]
    assert min(counts) > 0
    # (workgroups of at most 1025 rows: 8, 4 and 2 small submatrices share one)
    assert counts[0] // 8 + counts[1] // 4 + counts[2] // 2 + counts[3] + counts[4] > 2 * cus
    for k in range(len(mols)):
        assert torch.equal(P[k], alone[k])


def test_bisection_at_the_limit_of_one_workgroup(engine):
    """4096 states are bisected by one workgroup, 4097 by the general kernels, and a
    batch takes the general ones for both: mu and passes as the oracle's, the same
    density in the batch."""
    import torch
    from oracle import ptb_oracle as O
    items, alone = [], []
    for sizes in ([64], [64, 1], [63]):
        args = _blocks(sizes)
        n, nel, H, S, na, xyz, aoat = args
        it = _item(*args)
        P, rep = _alone(engine, it, 1)
        assert rep["sum_m"] == sum(k * k for k in sizes)
        ref = O.sm_stupid_simple(n, nel, H, S, na, xyz, aoat, 1, 2)
        assert rep["mu"] == ref.mu and rep["muiter"] == ref.muiter
        assert np.abs(P.cpu().numpy() - ref.P).max() < 1e-8
        items.append(it)
        alone.append((P, rep))
    P, reps = _batch(engine, items, 1)
    for k, (Pk, rep) in enumerate(alone):
        assert torch.equal(P[k], Pk)
        assert (reps[k]["mu"], reps[k]["muiter"]) == (rep["mu"], rep["muiter"])
