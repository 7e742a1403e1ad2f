"""The contact records' buckets and the merged columns at the sizes where their paths part.  A
bucket's records are placed by rank, 128, 256 or 512 of them at a time, in LDS if there are at most
512 and in global memory past that; their values are summed 128 at a time, runs of equal rows
going on from one part into the next.  And columns without a contact record, and columns of more merged
blocks than csr_fill has lanes.

A block of tiny cells, smaller than the contact distance, sits beside a large cube: every one
of its surface pairs is in contact, so its vertices collect up to 2,529 block records and 881
gradient records each.  The seeds are those whose buckets have the sizes on both sides of
each edge (counted from the oracle's contacts).  The CSR pattern and the counts are the oracle's
exactly; values at the bars of parity_util (sums in record order on both sides).  A second assembly of
the same state must repeat the first bit for bit: it starts from the counts the first cleared.
"""
import numpy as np
import pytest

from parity_util import csr_entry_err, vec3_entry_err

pytestmark = pytest.mark.gpu


def _tiny_beside_large(cells, seed):
    from cipc import scenes
    x, tets = scenes.lattice(2, 1.0)
    x = x / 2.0 + np.array([0.0, scenes.GROUND_Y + 0.05 - x[:, 1].min() / 2.0, 0.0])
    d = 1e-3 * np.linalg.norm(x.max(axis=0) - x.min(axis=0))   # about the contact distance
    y, small = scenes.lattice(cells, 1.0)
    rng = np.random.default_rng(seed)
    y = (y + rng.uniform(-0.1, 0.1, y.shape) - y.min(axis=0)) / cells * (0.5 * d)
    y = y + np.array([x[:, 0].max() + 0.3 * d, x[:, 1].mean(), x[:, 2].mean()])
    return scenes.finalize(f"tiny{cells}", np.concatenate([x, y]), np.concatenate([tets, small + len(x)]), scenes.Material())


def _records(s, sets):
    """Block records of each column and gradient records of each vertex, every vertex free."""
    blocks, gradients = np.zeros(s.V, int), np.zeros(s.V, int)
    contacts = [[c[0] if c[0] >= 0 else -c[0] - 1] + [v for v in c[1:] if v >= 0] for c in sets["self_set"]]
    contacts += [list(c) if c[3] >= 0 else [*s.surf_edges[e[0]], *s.surf_edges[e[1]]] for c, e in zip(sets["ee_set"], sets["ee_ie"])]
    for v in contacts:
        gradients[v] += 1
        for a in range(len(v)):
            for b in range(a + 1):
                blocks[min(v[a], v[b])] += 1
    return blocks, gradients


# (cells, seed), sizes of block buckets and of gradient buckets among its
@pytest.mark.parametrize("cells,seed,of_blocks,of_gradients", [
    (1, 3, (128, 129, 257), ()), (1, 5, (), ()), (2, 5, (), ()), (2, 6, (256,), (128, 129, 257)), (4, 6, (512, 513), (384, 385)),
    (3, 34, (385, 1024), (256,)), (3, 18, (1025,), ()), (3, 7, (), (513,))])
def test_long_columns(oracle_lib, cells, seed, of_blocks, of_gradients):
    from cipc import gpu, scenes
    s = _tiny_beside_large(cells, seed)
    xt = s.inertial_target()
    kappa = scenes.suggest_kappa(s.hhat, s.bbox_diag2, s.mean_mass)
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        ag, ao = g.active_set(), o.active_set()
        for k in ("self_set", "ee_set"):
            assert np.array_equal(ag[k], ao[k]), k
        blocks, gradients = _records(s, ao)
        assert set(of_blocks) <= set(blocks) and set(of_gradients) <= set(gradients) and 0 in blocks
        assert cells < 3 or blocks.max() > 1024
        rg, ro = g.assemble(kappa), o.assemble(kappa)
        contacts = len(ao["self_set"]) + len(ao["ee_set"])
        print(cells, "contacts", contacts, "nnz", len(ro["val"]))
        assert contacts > 100 * cells ** 3
        assert rg["collisions"] == ro["collisions"]
        assert np.array_equal(rg["outer"], ro["outer"]) and np.array_equal(rg["inner"], ro["inner"])
        assert csr_entry_err(ro["outer"], ro["inner"], rg["val"], ro["val"], scale=ro["val_scale"]) < 1e-10
        assert vec3_entry_err(rg["grad"], ro["grad"], scale=ro["grad_scale"]) < 1e-10
        again = g.assemble(kappa)
        for k in ("outer", "inner", "val", "grad"):
            assert np.array_equal(again[k], rg[k]), k
    finally:
        g.close()
        o.close()
