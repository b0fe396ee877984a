"""Eigenpairs of symmetric 3 x 3 matrices over scales, coincident and zero
entries: residual and orthonormality, both bounded by a few roundings per
rotation of at most five sweeps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e-250, 1e-9, 1.0, 1e200])
@pytest.mark.parametrize("iso", [0.0, 1 / 3])
def test_eig3_residual(gpu_ctx, scale, iso):
    from specfab_amd import specfabpy as sf
    sf.init(4)
    rng = np.random.default_rng(5)
    M = rng.standard_normal((517, 3, 3))
    M = (M + M.transpose(0, 2, 1)) / 2
    M[::7, 0, 1] = M[::7, 1, 0] = 0.0
    M[::11, 0, 0] = M[::11, 1, 1]
    M[5], M[6], M[8] = 0.0, np.eye(3), [[0, -1, 0], [-1, 0, 0], [0, 0, 2]]
    if iso:
        M = iso * np.eye(3) + 1e-9 * M
    ei, lam = sf.eigframe_arr(M * scale, "ij")
    lam = lam / scale
    assert (np.diff(lam, axis=1) <= 0).all()
    res = np.einsum("pij,pkj->pki", M, ei) - lam[:, :, None] * ei
    big = np.maximum(np.abs(M).max((1, 2)), 1e-300)
    assert (np.abs(res).max((1, 2)) <= 30 * 2.2e-16 * big).all()
    assert np.abs(np.einsum("pki,pmi->pkm", ei, ei) - np.eye(3)).max() <= 30 * 2.2e-16
