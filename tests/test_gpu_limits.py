"""Limits of a launch's threads and of a product's offsets."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _packed(ndim, blocks, hub):
    """Packed (H, S) of `blocks` equal diagonal blocks of 24 rows (every column of a
    block has the block's rows), or (hub) of one column that couples to all."""
    rng = np.random.default_rng(ndim)
    H, S = np.zeros((ndim, ndim)), np.eye(ndim)
    if hub:
        S[0, 1:] = 0.01
        H[0, 1:] = 0.02 * rng.uniform(size=ndim - 1)
    else:
        for b in range(blocks):
            i = slice(24 * b, 24 * b + 24)
            S[i, i] += 0.01 * (1.0 - np.eye(24))
            H[i, i] = np.triu(0.05 * rng.uniform(size=(24, 24)))
    np.fill_diagonal(H, -np.linspace(0.2, 1.2, ndim))
    iu = np.triu_indices(ndim)
    at = iu[0] + iu[1] * (iu[1] + 1) // 2
    out = []
    for M in (H, S):
        p = np.zeros(ndim * (ndim + 1) // 2)
        p[at] = M[iu]
        out.append(p)
    return out


def test_more_submatrices_than_one_launch_of_the_largest(engine):
    """118 320 submatrices of 24 rows beside one of 2048: with the units of the
    largest for each, a launch over all of them would need more than 2^32 threads.
    The densities are those of the molecules built alone."""
    import torch
    small = [torch.from_numpy(x).cuda() for x in _packed(2040, 85, False)]
    large = [torch.from_numpy(x).cuda() for x in _packed(2048, 0, True)]

    def item(n, H, S):
        return (n, 2 * (n // 4), H, S, torch.zeros_like(H), 1, np.zeros((1, 3)), np.ones(n, dtype=np.int64))

    alone = [item(2040, *small), item(2048, *large)]
    for it in alone:
        rep = engine.sm_stupid_simple_dev(*it, 1, 2)
        assert rep["not_spd"] == 0
    assert rep["max_m"] == 2048
    items = [item(2040, *small) for _ in range(58)] + [item(2048, *large)]
    reps = engine.sm_stupid_simple_batch(items, 1, 2, device=True)
    torch.cuda.synchronize()
    assert sum(r["nsm"] for r in reps) == 58 * 2040 + 2048
    for it in items[:-1]:
        assert torch.equal(it[4], alone[0][4])
    assert torch.equal(items[-1][4], alone[1][4])


@pytest.mark.parametrize("edge", [0, 64, 128])
@pytest.mark.parametrize("ld", [(1 << 22) - 1, 1 << 22, (1 << 22) + 5])
@pytest.mark.parametrize("order", ["nn", "tn", "nt", "tt"])
def test_products_with_long_strides(engine, order, ld, edge):
    """Leading dimensions on both sides of 2^22, up to which a product forms its byte
    offsets once.  Error per element at most k eps |A| |B|."""
    import torch
    m, n, k = 130, 131, 70
    ta, tb = order[0] == "t", order[1] == "t"
    g = torch.Generator(device="cuda").manual_seed(ld)

    def stored(rows, cols):  # column-major, columns `ld` apart
        x = torch.empty((cols - 1) * ld + rows, device="cuda", dtype=torch.float64).as_strided((cols, rows), (ld, 1))
        return x.copy_(torch.randn((cols, rows), generator=g, device="cuda", dtype=torch.float64))

    A, B = stored(k, m) if ta else stored(m, k), stored(n, k) if tb else stored(k, n)
    C = torch.empty((n, m), device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    one = [np.array([v], dtype=np.int64) for v in (m, n, k, ld, ld, m)]
    ptr = [np.array([t.data_ptr()], dtype=np.uint64) for t in (A, B, C)]
    at = lambda x: x.ctypes.data
    saved = engine.get_tuning("gemm_tile")
    engine.set_tuning("gemm_tile", edge)
    try:
        engine._check(engine.lib.ptbgpu_gemm_batch_dev(
            engine.ctx, 0, int(ta), int(tb), 1, at(one[0]), at(one[1]), at(one[2]), at(ptr[0]), at(one[3]),
            at(ptr[1]), at(one[4]), at(ptr[2]), at(one[5]), 1.0, 0.0))
    finally:
        engine.set_tuning("gemm_tile", saved)
    a, b = (A if ta else A.t()).contiguous(), (B if tb else B.t()).contiguous()
    assert ((C.t() - a @ b).abs() <= k * np.finfo(float).eps * (a.abs() @ b.abs())).all()
