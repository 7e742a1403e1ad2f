"""The placement of the active set's hits when they fill more blocks than a work-group adds up
itself (2,048 blocks of 1,024 hits): a folded 384^2 cloth, whose 13 million hits take a launch for
the blocks' starts, against the oracle's sets entry by entry (CollisionBroadPhase.cpp:765-1059).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_blocks_past_the_own_counts(oracle_lib):
    from cipc import gpu, scenes
    s = scenes.cloth_on_sphere(n=384, sphere_cells=4, fold=192)
    g = gpu.GpuContext(s, xtilde=s.inertial_target())
    o = oracle_lib.OracleMesh(s, xtilde=s.inertial_target())
    try:
        ao = o.active_set()
        assert len(ao["ccd_set"]) > 2 * 2048 * 1024      # hits, without the incident pairs
        for again in range(2):                           # the first builds with its capacities growing
            ag = g.active_set()
            for k in ("self_set", "ee_set", "ee_ie", "ccd_set", "env_set"):
                assert np.array_equal(ag[k], ao[k]), (again, k)
    finally:
        g.close()
        o.close()
