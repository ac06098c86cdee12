"""Analytic pair integrals (ana_eval) on both sides of their ranges: nested
heads whose layers lie from far below to well above the distance where a wave
takes the short polynomials (2.5 edge lengths), block by block against the
oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def om():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openmeeg_amd
    return openmeeg_amd


@pytest.mark.parametrize("freqs,radii", [((2, 2, 2), (0.98, 0.99, 1.0)), ((2, 2, 2), (0.2, 0.5, 1.0)),
                                         ((4, 4, 4), (0.3, 0.65, 1.0)), ((5, 3, 2), (0.05, 0.9, 0.97)),
                                         ((6, 6, 6), (0.87, 0.92, 1.0))])
def test_headmat_near_and_far_layers(om, freqs, radii):
    from openmeeg_amd import spheres as S
    from oracle import oracle as O
    meshes = [S.nested_sphere_meshes(f, (r,))[0] for f, r in zip(freqs, radii)]
    cond = (1.0, 0.0125, 1.0)
    g = om.make_nested_geometry(meshes, cond)
    og = O.nested_geometry(meshes, cond)
    ref = O.unpack(O.head_mat(og), og.size)
    got = O.unpack(om.HeadMat(g).data(), og.size)
    # two FP64 evaluations of sums whose terms cancel to about edge/distance
    # of their size (below 1/40 here), some tens of roundings each, over the
    # largest entry of each row and column pair
    scale = np.sqrt(np.abs(ref).max(1)[:, None] * np.abs(ref).max(0)[None, :])
    assert np.abs(got - ref).max() > 0 or og.size == 0
    assert (np.abs(got - ref) / scale).max() < 40 * 50 * np.finfo(float).eps
