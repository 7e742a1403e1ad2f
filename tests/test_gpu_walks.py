"""The tree walks by groups of lanes where they can go wrong: queries that overlap most of a
tree (far more hits than a query's buffer holds, so that the compaction walks again, and the
deepest stacks), trees of a few leaves, fewer queries than a wavefront takes, and every group
size.

A large tetrahedron spans a fine cube: the boxes of its long edges meet thousands of the
cube's edges and faces, the cube's own queries a handful.  The active set and the step bound are minima and sets over pairs,
which no order changes: bit-exact against the oracle (CollisionBroadPhase.cpp:765-1059,
ContactMechanics.cpp:3754-3867), the intersection test (IPCSolver.cpp:476-542) equal to it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SETS = ("self_set", "ee_set", "ee_ie", "ccd_set", "env_set")
KEYS = ("alpha", "ground", "partial", "cfl", "full")


def _spanned(cells, gap):
    """A cube of cells^3 and a tetrahedron across it, gap (in cube edges) above its top face, or
    through it for a negative gap."""
    from cipc import scenes
    x, tets = scenes.lattice(cells, 1.0)
    x = (x - x.min(axis=0)) / cells
    x = x + np.array([0.0, scenes.GROUND_Y + 0.05, 0.0])
    top = x[:, 1].max()
    big = np.array([[-0.2, top + gap, -0.2], [1.2, top + gap, 1.2], [1.2, top + gap + 0.01, -0.2], [-0.2, top + gap - 1.01, -0.2]])
    if np.linalg.det(big[1:] - big[0]) < 0:
        big[[1, 2]] = big[[2, 1]]
    s = scenes.finalize("spanned", np.concatenate([x, big]), np.concatenate([tets, [np.arange(4) + len(x)]]), scenes.Material())
    return s


def _only(count):
    from cipc import scenes
    x = np.array([[0.0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    x = np.concatenate([x + np.array([0.0, scenes.GROUND_Y + 0.1 + 1.05 * k, 0.0]) for k in range(count)])
    return scenes.finalize("few", x, np.arange(4 * count).reshape(-1, 4), scenes.Material())


@pytest.mark.parametrize("case", ["spanned", "few1", "few2"])
def test_group_walks(oracle_lib, case):
    from cipc import gpu, scenes
    s = _spanned(24, 2e-3) if case == "spanned" else _only(int(case[-1]))
    xt, p = scenes.newton_probe_state(s)
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        ao, bo, io = o.active_set(), o.step_bound(p), o.is_intersected()
        for choice in range(5):
            for kernel in (0, 1, 3, 4):
                g.set_tune(kernel, choice)
            ag = g.active_set()
            for k in SETS:
                assert np.array_equal(ag[k], ao[k]), (choice, k)
            bg = g.step_bound(p)
            for k in KEYS:
                assert bg[k] == bo[k], (choice, k, bg[k], bo[k])
            assert g.is_intersected() == io, choice
    finally:
        g.close()
        o.close()


def test_crossing_the_whole_tree(oracle_lib):
    from cipc import gpu
    s = _spanned(24, -0.25)
    xt = s.inertial_target()
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        g.active_set()
        o.active_set()
        assert o.is_intersected() and g.is_intersected()
    finally:
        g.close()
        o.close()
