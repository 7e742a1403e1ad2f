"""The general projection of 12 x 12 blocks by 16 lanes, four blocks a wavefront: group tails,
blocks that stay as they are (already PSD, zero) beside blocks that change, repeated and zero
eigenvalues, and scales far from one, against numpy's eigendecomposition.

The blocks are translation-invariant (the form of every contact and hinge Hessian): B^T R B with
the orthonormal basis B of the complement of the translations.  Bound: the Jacobi sweeps and
the two changes of basis are orthogonal transforms of 12 x 12 blocks, each rounding by a few
dozen units in the last place of the block's norm: 64 * 12 * 2^-53 = 8.5e-14 of it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = 64 * 12 * 2.0 ** -53


def _blocks(count, seed):
    rng = np.random.default_rng(seed)
    one = np.ones((4, 1)) / 2.0
    q = np.linalg.qr(np.concatenate([one, rng.standard_normal((4, 3))], axis=1))[0][:, 1:]
    B = np.kron(q.T, np.eye(3))
    out = []
    for i in range(count):
        z = np.linalg.qr(rng.standard_normal((9, 9)))[0]
        w = rng.standard_normal(9) * 10.0 ** rng.uniform(-6, 6)
        kind = i % 6
        if kind == 1:
            w = np.abs(w)
        elif kind == 2:
            w[:] = 0.0
        elif kind == 3:
            w = np.repeat([-2.0, 1.0, 0.0], 3)
        elif kind == 4:
            w *= 10.0 ** rng.choice([-40, 40])
        elif kind == 5:
            w[1:] = 0.0
        H = B.T @ (z * w) @ z.T @ B
        out.append(0.5 * (H + H.T))
    return np.array(out)


@pytest.mark.parametrize("count", [1, 3, 4, 5, 66])
def test_rows_of_blocks(count):
    from cipc import gpu
    H = _blocks(count, seed=count)
    P = gpu.eval_contact_pd(H)
    for i in range(count):
        norm = np.linalg.norm(H[i], 2)
        w, z = np.linalg.eigh(H[i])
        want = (z * np.maximum(w, 0.0)) @ z.T
        assert np.abs(P[i] - want).max() <= BOUND * norm, (i, np.abs(P[i] - want).max() / max(norm, 1e-300))
        if i % 6 == 2:
            assert np.array_equal(P[i], H[i])
