"""The conjugate-gradient kernels at the edges of their launch shapes: 32 block rows per
work-group (one row short, full, one over), the smallest systems, and a system of more than
65,536 block rows, whose partial sums a launch of their own adds up, alone and in a batch.

Bar: the true relative residual, in FP64 on the host with the exported matrix, at most 1.5e-6
for a target of 1e-6 (the FP64 form stops on its recursive residual), as in test_gpu_solve."""
import numpy as np
import pytest

from test_gpu_fsai_rows import _ball

pytestmark = pytest.mark.gpu


def _residual(g, r, precision, preconditioner):
    import scipy.sparse as sp
    n = len(r["outer"]) - 1
    L = sp.csc_matrix((r["val"], r["inner"], r["outer"]), shape=(n, n))
    A = L + L.T - sp.diags(L.diagonal())
    p, st = g.solve(precision=precision, preconditioner=preconditioner, max_iter=20000)
    assert st["iterations"] > 0 and st["rel_residual"] <= 1e-6
    return np.linalg.norm(r["rhs"] - A @ p.reshape(-1)) / np.linalg.norm(r["rhs"])


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("preconditioner", [0, 1])
@pytest.mark.parametrize("vertices", [5, 31, 32, 33, 65])
def test_small_systems(vertices, preconditioner, precision):
    from cipc import gpu
    g = gpu.GpuContext(_ball(vertices - 1))
    try:
        g.active_set()
        assert _residual(g, g.assemble(1.0), precision, preconditioner) <= 1.5e-6
    finally:
        g.close()


@pytest.fixture(scope="module")
def large():
    from cipc import gpu, scenes
    s = scenes.stacked_cubes(3, 28, 0.1, 1e-3, seed=6, velocity_scale=0.5)
    assert s.V > 65536
    xt, _ = scenes.newton_probe_state(s)
    kappa = scenes.suggest_kappa(s.hhat, s.bbox_diag2, s.mean_mass)
    g = gpu.GpuContext(s, xtilde=xt)
    g.set_state(V_prev=s.x - s.velocities * s.material.dt)
    g.active_set()
    g.friction_update(kappa)
    yield g, g.assemble(kappa)
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("preconditioner", [0, 1])
def test_sums_of_many_work_groups(large, preconditioner, precision):
    assert _residual(*large, precision, preconditioner) <= 1.5e-6


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("preconditioner", [0, 1])
def test_sums_of_many_work_groups_in_a_batch(batch, preconditioner, precision):
    """A scene past the work-groups' own sums between two small ones: the partial sums and results
    of each scene at its place.  Bit for bit what each gives alone (the sums' order follows from the
    scene's size only), the small ones with sums of their own there."""
    b, singles = batch
    p, st = b.solve(precision=precision, preconditioner=preconditioner, max_iter=20000)
    for k, g in enumerate(singles):
        q, sq = g.solve(precision=precision, preconditioner=preconditioner, max_iter=20000)
        assert st[k]["iterations"] == sq["iterations"] > 0, k
        assert np.array_equal(p[b.voff[k]:b.voff[k + 1]], q), k


@pytest.fixture(scope="module")
def batch():
    from cipc import gpu, scenes
    sc = [scenes.stacked_cubes(c, n, 0.1, 1e-3, seed=k, velocity_scale=0.5) for k, (c, n) in enumerate(((2, 4), (3, 28), (1, 5)))]
    assert sc[1].V > 65536
    for s in sc:
        s.hhat, s.fhat, s.dtol = sc[1].hhat, sc[1].fhat, sc[1].dtol
    xt = [scenes.newton_probe_state(s)[0] for s in sc]
    kappa = np.array([scenes.suggest_kappa(s.hhat, s.bbox_diag2, s.mean_mass) for s in sc])
    b = gpu.BatchContext(sc, xtildes=xt)
    singles = [gpu.GpuContext(s, xtilde=x) for s, x in zip(sc, xt)]
    b.active_set()
    b.assemble(kappa)
    for g, k in zip(singles, kappa):
        g.active_set()
        g.assemble(k)
    yield b, singles
    b.close()
    for g in singles:
        g.close()
