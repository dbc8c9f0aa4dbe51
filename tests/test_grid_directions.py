"""The grid's directions and angles, evaluated on whole columns, carry the bits
of one scalar evaluation per direction: the tracer's rules switch at angles
that lie on the grid, where a unit in the last place chooses another rule."""
import numpy as np
import pytest

from anacor_public_amd import gridding as G


@pytest.mark.parametrize("n_theta,n_phi", [(1, 1), (2, 2), (8, 4), (36, 24), (37, 23), (120, 60),
                                           (144, 60), (360, 18)])
def test_directions_match_scalar_evaluation(n_theta, n_phi):
    vecs, angles = G.grid_directions(n_theta, n_phi)
    theta, phi = np.meshgrid(np.linspace(-180, 180, n_theta, endpoint=False),
                             np.linspace(-90, 90, n_phi, endpoint=False))
    data = np.stack((theta.ravel(), phi.ravel()), axis=-1) / 180 * np.pi
    assert vecs.shape == (len(data), 3) and angles.shape == (len(data), 2)
    for i, (t, p) in enumerate(data):
        v = G.myframe_2_dials(G.thetaphi_2_myframe(t, p))
        np.testing.assert_array_equal(vecs[i].view(np.uint64), v.view(np.uint64))
        a = np.array(G.dials_2_thetaphi(v))
        np.testing.assert_array_equal(angles[i].view(np.uint64), a.view(np.uint64))
