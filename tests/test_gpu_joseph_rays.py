"""The per-ray forward projector's batches of four slices: rays of fewer middle samples than
a batch, of a batch and one more, rays grazing the faces (whose samples keep the index
clamp), all dominant axes and both directions, against the float oracle.  The bar is the
projector's: relative L2 <= 1e-5."""
import numpy as np
import pytest

from helpers import hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu


def _rows(n, tilt, inplane=0.):
    return np.array([[700., 1100., 3. + i * 360. / n, 2. * (-1) ** i, 1.5, tilt, inplane, 0.4, 0.2] for i in range(n)])


CASES = {
    "two_slices": ((2, 2, 2), (30., 30., 30.), (19, 17), (7., 7.), _rows(9, 1.)),
    "three_slices": ((3, 5, 3), (25., 20., 25.), (23, 21), (7., 7.), _rows(9, -2.)),
    "five_to_seven": ((7, 6, 5), (15., 15., 15.), (31, 33), (5., 5.), _rows(11, 1.5, 2.)),
    "eight_to_eleven": ((8, 11, 10), (10., 10., 10.), (33, 31), (5., 5.), _rows(12, 0.7)),
    "odd": ((37, 31, 45), (3., 3., 3.), (67, 53), (3., 3.), _rows(10, 1.2, -0.8)),
    "y_dominant": ((24, 41, 27), (4., 4., 4.), (50, 45), (4., 4.), _rows(6, 62.)),
    "y_diagonal": ((32, 33, 32), (4., 4., 4.), (47, 49), (4., 4.), _rows(8, 45.)),
    "grazing": ((33, 33, 33), (3., 3., 3.), (129, 9), (1.6, 12.), _rows(4, 1e-3)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_rays_match_the_oracle(oracle, hip, name):
    vsize, vsp, (nu, nv), (du, dv), rows = CASES[name]
    n = len(rows)
    vorig = tuple(-(k - 1) * s / 2. + 0.3 for k, s in zip(vsize, vsp))
    sorig = (-(nu - 1) * du / 2., -(nv - 1) * dv / 2., 0.)
    rng = np.random.default_rng(41)
    vol = rng.random(vsize[::-1]).astype(np.float32)
    p0 = rng.normal(size=(n, nv, nu)).astype(np.float32)
    f = hip.HipForwardProjectionImageFilter()
    f.SetInput(0, to_device(hip, p0, sorig, (du, dv, 1.)))
    f.SetInput(1, to_device(hip, vol, vorig, vsp))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    out = f.GetOutput().numpy()
    ref = oracle.joseph(rows, oracle.image((nu, nv, n), sorig, (du, dv, 1.)), p0, oracle.image(vsize, vorig, vsp), vol)
    assert np.linalg.norm(ref - p0) > 0.
    assert rel_l2(out - p0, ref - p0) <= 1e-5
