"""The tree walks by groups of lanes where they can go wrong: queries with more hits than their
buffer holds (64), so that the compaction walks again, trees of one leaf and of a few, fewer
queries than a wavefront takes, walks that run out of stack and go over the exact boxes
instead, and every group size.

Scenes: a fine cube under large slanted tetrahedra whose vertices come first, so that each long edge
is asked for the cube's later edges (it meets hundreds to thousands) and each of the cube's vertices
lies in the boxes of more than 64 large faces.  The active set and the step bound are minima and
sets over pairs, which no order changes: bit-exact against the oracle
(CollisionBroadPhase.cpp:765-1059, ContactMechanics.cpp:3754-3867), the intersection test
(IPCSolver.cpp:476-542) equal to it.

Boxes alone (eval_walk): hits against numpy's box test, with the library's stacks and with stacks
too small for the walk.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SETS = ("self_set", "ee_set", "ee_ie", "ccd_set", "env_set")
KEYS = ("alpha", "ground", "partial", "cfl", "full")
BUFFER = 64                # hits of a query that the first walk keeps


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


def _under_slants(cells, count):
    """count tetrahedra, each with a face in a plane x + y + z = const past the far corner of a
    unit cube of cells^3 (the first 1e-3 from it) and boxes that hold the whole cube, then the cube."""
    from cipc import scenes
    y0 = scenes.GROUND_Y + 0.6
    parts = []
    for k in range(count):
        h = 3.0 + 2e-3 + 0.03 * k
        big = np.array([[h, 0.5, -0.5], [-0.5, h, 0.5], [0.5, -0.5, h], [h, h, h]])
        parts.append(big if np.linalg.det(big[1:] - big[0]) > 0 else big[[0, 2, 1, 3]])
    x, tets = scenes.lattice(cells, 1.0)
    x = np.concatenate(parts + [(x - x.min(axis=0)) / cells]) + np.array([0.0, y0, 0.0])
    return scenes.finalize("slants", x, np.concatenate([np.arange(4 * count).reshape(-1, 4), tets + 4 * count]), scenes.Material())


def _only(count):
    from cipc import scenes
    x = np.array([[0.0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    x = np.concatenate([x + np.array([0.0, scenes.GROUND_Y + 0.1 + 1.05 * k, 0.0]) for k in range(count)])
    return scenes.finalize("few", x, np.arange(4 * count).reshape(-1, 4), scenes.Material())


def _triangle():
    """A cloth of one triangle: a face tree of one leaf."""
    from cipc import scenes
    x = np.array([[0.0, 0, 0], [0, 0, 1], [1, 0, 0]]) + np.array([0.0, scenes.GROUND_Y + 1e-3, 0.0])
    return scenes.finalize("triangle", x, np.zeros((0, 4)), scenes.Material(), triangles=np.arange(3).reshape(1, 3))


def _hits(s):
    """Faces near each surface vertex, later edges near each surface edge, by their boxes."""
    gap, x = np.sqrt(s.hhat), s.x
    f, e, p = x[s.faces[:, :3]], x[s.surf_edges], x[s.surf_verts]
    flo, fhi, elo, ehi = f.min(axis=1), f.max(axis=1), e.min(axis=1), e.max(axis=1)
    points = np.array([np.count_nonzero(np.all((flo - q <= gap) & (q - fhi <= gap), axis=1)) for q in p])
    edges = np.array([np.count_nonzero(np.all((elo[k + 1:] - ehi[k] <= gap) & (elo[k] - ehi[k + 1:] <= gap), axis=1))
                      for k in range(len(e))])
    return points, edges


@pytest.mark.parametrize("case", ["slants", "spanned", "few1", "few2", "triangle"])
def test_group_walks(oracle_lib, case):
    from cipc import gpu, scenes
    s = {"slants": lambda: _under_slants(16, 24), "spanned": lambda: _spanned(24, 2e-3), "triangle": _triangle,
         "few1": lambda: _only(1), "few2": lambda: _only(2)}[case]()
    if case == "slants":
        points, edges = _hits(s)
        assert np.count_nonzero(points > BUFFER) > 500 and np.count_nonzero(edges > BUFFER) > 50
        assert points.min() <= BUFFER and edges.min() <= BUFFER      # beside queries that fit
    if case == "triangle":
        assert len(s.faces) == 1
    xt, p = scenes.newton_probe_state(s)
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        ao, bo = o.active_set(), o.step_bound(p)
        if case == "slants":
            assert len(ao["self_set"]) > 0
        for choice in range(5):
            for kernel in (0, 1, 3, 4):
                g.set_tune(kernel, choice)
            ag = g.active_set()
            for k in SETS:
                assert np.array_equal(ag[k], ao[k]), (choice, k)
            bg = g.step_bound(p)
            for k in KEYS:
                assert bg[k] == bo[k], (choice, k, bg[k], bo[k])
        assert g.is_intersected() == o.is_intersected()
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


@pytest.mark.parametrize("n", [60, 66, 92, 132])
@pytest.mark.parametrize("dip", [1e-2, -1e-2])
def test_intersection_group_sizes(oracle_lib, n, dip):
    """A flat cloth of n^2 quads and a tetrahedron beside or through it: surfaces of 11,000, 13,000, 26,000
    and 52,000 edges, whose intersection walks have 32, 16, 8 and 4 lanes a query."""
    from cipc import gpu, scenes
    xc, tris = scenes.cloth_grid(n, 1.0)
    xc = xc + np.array([0.0, scenes.GROUND_Y + 0.5, 0.0])
    at = np.array([0.31, scenes.GROUND_Y + 0.5, -0.22])
    tet = at + np.array([[0.0, dip, 0.0], [0.02, 0.1, 0.0], [0.0, 0.1, 0.02], [0.0, 0.12, 0.0]])
    if np.linalg.det(tet[1:] - tet[0]) < 0:
        tet[[1, 2]] = tet[[2, 1]]
    s = scenes.finalize("dip", np.concatenate([tet, xc]), np.arange(4).reshape(1, 4), scenes.Material(), triangles=tris + 4)
    lanes = 0
    while lanes < 3 and len(s.surf_edges) << (lanes + 1) <= 3 << 15:
        lanes += 1
    assert lanes == {60: 3, 66: 2, 92: 1, 132: 0}[n], len(s.surf_edges)
    xt = s.inertial_target()
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        g.active_set()
        o.active_set()
        assert o.is_intersected() == (dip < 0)
        assert g.is_intersected() == (dip < 0)
    finally:
        g.close()
        o.close()


def _boxes(n, seed):
    """n small boxes in the unit cube, some in one place, some flat, and a few that span it."""
    rng = np.random.default_rng(seed)
    lo = rng.uniform(0, 1, (n, 3))
    lo[n // 2:n // 2 + n // 8] = 0.5
    size = rng.uniform(0, 0.1, (n, 3)) * rng.integers(0, 2, (n, 3))
    lo[::97], size[::97] = -0.1, 1.2
    return np.concatenate([lo, lo + size], axis=1)


def _near(q, b, gap):
    return np.all((b[:, :3] - q[3:] <= gap) & (q[:3] - b[:, 3:] <= gap), axis=1)


# the library's stacks; stacks that some queries outrun; stacks of one record a step
@pytest.mark.parametrize("depth", [64, 5, 1])
@pytest.mark.parametrize("bits", range(5))
@pytest.mark.parametrize("n", [1, 2, 3, 5, 700])
def test_boxes(n, bits, depth):
    from cipc import gpu
    boxes = _boxes(n, n)
    rng = np.random.default_rng(bits)
    lo = rng.uniform(-0.2, 1.2, (67, 3))
    queries = np.concatenate([lo, lo + rng.uniform(0, 0.3, (67, 3)) ** 2], axis=1)
    queries[::5] = [-1, -1, -1, 2, 2, 2]        # everything
    queries[1::5] = [3, 3, 3, 4, 4, 4]          # nothing
    gap = 0.01
    for q, h in zip(queries, gpu.eval_walk(boxes, queries, gap, bits, depth)):
        got = np.zeros(n, int)
        np.add.at(got, h, 1)
        assert got.max() <= 1                   # a walk that starts again counts from nothing
        assert np.all(got >= _near(q, boxes, gap))
        assert np.all(got <= _near(q, boxes, gap + 1e-6))   # float boxes: at most a few 2^-24 wider
    met = np.zeros((n, n), bool)
    for k, h in enumerate(gpu.eval_walk(boxes, None, 0.0, bits, depth, max_hits=4 * n)):
        met[k, h] = True
    want = np.array([_near(q, boxes, 0.0) for q in boxes])
    np.fill_diagonal(want, False)
    assert not np.any(met & met.T)              # from one side only
    assert np.array_equal(met | met.T, want)
