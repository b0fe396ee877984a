"""The n' = 3 Sachs factors take the isotropic denominators of an orthonormal
frame from the Cartesian axes and those of given states 64 at a time; frames
given per parcel form their own.  The three forms against each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 63, 64, 65, 129])
def test_denominators_agree(gpu_ctx, P):
    import torch
    from specfab_amd import workloads as W
    from specfab_amd.batch import FabricBatch
    b = FabricBatch(8, nlm=W.perturbed_isotropic(np.random.default_rng(P), P, 8, sigma=0.05))
    Eg = (1.0, 10.0)
    for alpha in (0.0, 0.1):
        E, _, ei = b.Eij(Eij_grain=Eg, alpha=alpha, n_grain=3, frame="eig")
        Ex = b.Eij(Eij_grain=Eg, alpha=alpha, n_grain=3, frame="xyz")
        Eg_ei = b.Eij(Eij_grain=Eg, alpha=alpha, n_grain=3, frames=ei)
        Eg_xyz = b.Eij(Eij_grain=Eg, alpha=alpha, n_grain=3, frames=torch.eye(3, dtype=torch.float64).repeat(P, 1, 1).cuda())
        # a few thousand operations, and a frame orthonormal to rounding
        assert (E / Eg_ei - 1).abs().max() < 1e-12 and (Ex / Eg_xyz - 1).abs().max() < 1e-12
    # 70 states of which the last six are a Cartesian frame's
    I = np.eye(3)
    vw = [(0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1)]
    v, w = np.array([I[i] for i, _ in vw]), np.array([I[j] for _, j in vw])
    tau = np.array([I / 3 - np.outer(a, c) if i == j else np.outer(a, c) + np.outer(c, a)
                    for (i, j), a, c in zip(vw, v, w)])
    rep = lambda m: np.concatenate([m[np.arange(64) % 6], m])
    Ev = b.Evw(rep(v), rep(w), rep(tau), Eij_grain=Eg, alpha=0.0, n_grain=3)
    Ex = b.Eij(Eij_grain=Eg, alpha=0.0, n_grain=3, frame="xyz")
    assert (Ev[:, 64:] / Ex - 1).abs().max() < 1e-12
    assert (Ev[:, :64] / Ex[:, [i % 6 for i in range(64)]] - 1).abs().max() < 1e-12
    assert int(b.status.abs().sum()) == 0
