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
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) / scale).max() < 40 * 50 * np.finfo(float).eps
    # the S and D blocks of two different meshes, where the entries are weak
    # and the short polynomials run, at their own size.  S: a positive
    # integrand whose sum the oracle and the kernel round some tens of times.
    # D (the oracle's form): each logarithm is rounded to eps where it is
    # worth l / R, and the sum over the edges cancels to (l / R)^2 of its
    # terms, l the smallest edge of the triangles the hat functions live on
    # and R the largest distance.
    tens = 50 * np.finfo(float).eps
    for a in range(len(meshes)):
        for b in (a - 1, a + 1):
            if not 0 <= b < len(meshes) or g.mesh_info(a)["current_barrier"]:
                continue
            A, B = g.mesh_info(a), g.mesh_info(b)
            (Pa, Ta), (Pb, Tb) = meshes[a], meshes[b]
            assert A["ntris"] == len(Ta) and B["ntris"] == len(Tb)
            edge = min(np.linalg.norm(Pb[Tb[:, i]] - Pb[Tb[:, i - 1]], axis=1).min() for i in range(3))
            ratio = np.linalg.norm(Pa[:, None] - Pb[None], axis=2).max() / edge
            rows = slice(A["tri_first"], A["tri_first"] + A["ntris"])
            blocks = [(slice(B["vert_first"], B["vert_end"]), ratio ** 3)]
            if not B["current_barrier"]:
                blocks.append((slice(B["tri_first"], B["tri_first"] + B["ntris"]), 1.0))
            for cols, growth in blocks:
                err = np.abs(got[rows, cols] - ref[rows, cols]).max() / np.abs(ref[rows, cols]).max()
                print("meshes %d, %d: %.2e of the bound" % (a, b, err / (tens * growth)), flush=True)
                assert err < tens * growth
