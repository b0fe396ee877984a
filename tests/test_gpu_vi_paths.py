"""Elastic velocities on both Reuss paths (the symmetric elimination, and the
pivoted solve of compliances that are not positive definite), at the edges of
the parcel blocks and of the ranges of the (block, direction) order, against
the oracle's acoustic tensor and complex Cardano roots."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LAME = np.array([7.15e9, 3.455e9, 5.88e9 / 7.15e9, 3.06e9 / 3.455e9, 15.24e9 / 14.06e9])


@pytest.mark.parametrize("P,nd", [(1, 1), (127, 3), (128, 7), (129, 9)])
@pytest.mark.parametrize("scale", [0.3, 30.0])
def test_reuss_paths(gpu_ctx, oracle, P, nd, scale):
    """scale 0.3: near-isotropic distributions; 30: coefficients far outside
    any distribution, so that many compliances are indefinite"""
    from specfab_amd import workloads as W
    from specfab_amd.batch import FabricBatch
    rng = np.random.default_rng(P)
    nlm = W.perturbed_isotropic(rng, P, 4, sigma=0.02 * scale)
    th, ph = np.arccos(rng.uniform(-1, 1, nd)), rng.uniform(0, 2 * np.pi, nd)
    fb = FabricBatch(4, nlm=nlm)
    for alpha in (0.0, 0.5, 1.0):
        v = fb.Vi_elastic(alpha, LAME, 917.0, th, ph).cpu().numpy()
        ref = np.stack([oracle.Vi_elastic_tranisotropic(n[:15], alpha, LAME, 917.0, th, ph).T for n in nlm])
        s = np.sort(ref ** -2.0, axis=2)
        gap = np.diff(s, axis=2).min(axis=2) / s.max(axis=2)
        # a root moves by the cubic's rounding (tens of operations) over its
        # distance to the next, at coincident ones by the square root of it;
        # the determinant in the cubic carries the tensor's rounding times its
        # condition, the ratio of the squared velocities
        cond = s.max(axis=2) / s.min(axis=2)
        tol = 200 * 2.2e-16 * cond * (1 + 1 / np.maximum(gap, 1.5e-8))
        err = np.abs(v - ref).max(axis=2) / ref.max(axis=2)
        assert (err < tol).all(), (alpha, (err / tol).max())
