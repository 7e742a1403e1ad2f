"""Block FSAI rows of every pattern size class against the numpy restatement of the factor
(fsai_oracle): a ball of tets around one hub vertex, numbered last, whose block row has all
the n rim vertices below it.  Sizes at the edges of the classes (10 and 24 blocks), of the
64 lanes that hold a row's 3 k matrix rows, and of the 64 candidates ranked per pass.

Bar: the factor entry by entry within 1e-9, relative with a floor of 1e-6 of the block row's
largest entry, as for the whole scenes in test_gpu_solve: the rows' condition numbers
(below 1e6 here) times 1e-16, with a margin of ten."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ball(n):
    from scipy.spatial import ConvexHull
    from cipc import scenes
    k = np.arange(n) + 0.5
    phi, z = np.pi * (1 + 5 ** 0.5) * k, 1 - 2 * k / n
    rim = np.stack([np.cos(phi) * np.sqrt(1 - z * z), z, np.sin(phi) * np.sqrt(1 - z * z)], axis=1) * 0.5
    x = np.concatenate([rim, np.zeros((1, 3))])
    tets = np.concatenate([ConvexHull(rim).simplices, np.full((2 * n - 4, 1), n)], axis=1)
    d = x[tets[:, 1:]] - x[tets[:, :1]]
    flip = np.linalg.det(d) < 0
    tets[flip, 0], tets[flip, 1] = tets[flip, 1].copy(), tets[flip, 0].copy()
    s = scenes.finalize(f"ball{n}", x, tets, scenes.Material())
    rng = np.random.default_rng(n)
    s.x = s.x + rng.uniform(-0.02, 0.02, s.x.shape)     # strained: blocks of different norms
    return s


@pytest.mark.parametrize("n", [4, 9, 10, 20, 21, 22, 23, 24, 64, 65, 130])
def test_factor_rows(n):
    import scipy.sparse as sp
    import fsai_oracle as F
    from cipc import gpu
    g = gpu.GpuContext(_ball(n))
    try:
        g.active_set()
        r = g.assemble(1.0)
        m = len(r["outer"]) - 1
        L = sp.csc_matrix((r["val"], r["inner"], r["outer"]), shape=(m, m))
        B = sp.bsr_matrix((L + L.T - sp.diags(L.diagonal())).tocsr(), blocksize=(3, 3))
        B.sort_indices()
        assert np.count_nonzero(B.indices[B.indptr[n]:] <= n) == n + 1
        want = F.block_fsai(B.indptr, B.indices, np.asarray(B.data)).tocsr()
        g.solve(precision=0, rel_tol=1e-6, preconditioner=1)
        got = g.solve_factor().tocsr()
        # the matrix's block pattern, rows in order: every lower entry found at its row
        assert np.array_equal(got.indptr, B.tocsr().indptr) and np.array_equal(got.indices, B.tocsr().indices)
        assert np.count_nonzero(got[3 * n].toarray()) > 0
        D = (got - want).tocoo()
        top = np.asarray(abs(want).max(axis=1).todense()).ravel().reshape(-1, 3).max(axis=1).repeat(3)
        ref = np.asarray(want[D.row, D.col]).ravel()
        err = float((np.abs(D.data) / np.maximum(np.abs(ref), 1e-6 * top[D.row])).max(initial=0.0))
        assert err <= 1e-9, err
    finally:
        g.close()
