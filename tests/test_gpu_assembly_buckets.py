"""The contact records' buckets and the merged columns at the sizes where their paths part: a
block column with no contact record, a few, more than 64 (one register network), more than 512
(the LDS network; longer ones by rank), and columns of more merged blocks than csr_fill has lanes.

A block of tiny cells, smaller than the contact distance, sits beside a large cube: every one
of its surface pairs is in contact, so each of its vertices collects hundreds of block records
with 1^3 cells and thousands with 2^3.  The CSR pattern and the counts are the oracle's exactly;
values at the bars of parity_util (sums in record order on both sides).  A second assembly of
the same state must repeat the first bit for bit: it starts from the counts the first cleared.
"""
import numpy as np
import pytest

from parity_util import csr_entry_err, vec3_entry_err

pytestmark = pytest.mark.gpu


def _tiny_beside_large(cells):
    from cipc import scenes
    x, tets = scenes.lattice(2, 1.0)
    x = x / 2.0 + np.array([0.0, scenes.GROUND_Y + 0.05 - x[:, 1].min() / 2.0, 0.0])
    d = 1e-3 * np.linalg.norm(x.max(axis=0) - x.min(axis=0))   # about the contact distance
    y, small = scenes.lattice(cells, 1.0)
    rng = np.random.default_rng(5)
    y = (y + rng.uniform(-0.1, 0.1, y.shape) - y.min(axis=0)) / cells * (0.5 * d)
    y = y + np.array([x[:, 0].max() + 0.3 * d, x[:, 1].mean(), x[:, 2].mean()])
    return scenes.finalize(f"tiny{cells}", np.concatenate([x, y]), np.concatenate([tets, small + len(x)]), scenes.Material())


@pytest.mark.parametrize("cells", [1, 2])
def test_long_columns(oracle_lib, cells):
    from cipc import gpu, scenes
    s = _tiny_beside_large(cells)
    xt = s.inertial_target()
    kappa = scenes.suggest_kappa(s.hhat, s.bbox_diag2, s.mean_mass)
    g = gpu.GpuContext(s, xtilde=xt)
    o = oracle_lib.OracleMesh(s, xtilde=xt)
    try:
        ag, ao = g.active_set(), o.active_set()
        for k in ("self_set", "ee_set"):
            assert np.array_equal(ag[k], ao[k]), k
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
