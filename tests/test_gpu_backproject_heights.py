"""Voxel and FDK backprojection by blocks of 2, 4, 8 (small volumes) and 16 heights (from 2560
blocks of 16^3), at their edges, with footprints inside the detector, across its border
and outside it, against the float oracle with the backprojector's bar of 1e-5 relative L2."""
import numpy as np
import pytest

from helpers import hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu

SMALL = [(40, ny, 33) for ny in (1, 7, 8, 9, 16, 23, 24, 25, 47)]
# 6, 7 and 5 blocks of 16 heights by 21 x 21 columns of them; 8 blocks of 8 by 11 x 11
LARGE = [(330, 95, 335), (330, 97, 335), (330, 80, 335), (170, 59, 171), (170, 61, 171)]


def _run(oracle, hip, vsize, fdk, stack, tilt=0.):
    n, (nu, nv) = 5, (64, 46)
    rows = np.array([[600., 1000., 5. + 73. * i, 3. * (-1) ** i, 2. - i, tilt, -0.5 * tilt, 1., -2.] for i in range(n)])
    vsp = tuple(110. / max(vsize) for _ in range(3))
    vorig = tuple(-(k - 1) * s / 2. for k, s in zip(vsize, vsp))
    vsp, vorig = (vsp[0], 90. / vsize[1], vsp[2]), (vorig[0], -(vsize[1] - 1) * 45. / vsize[1], vorig[2])
    ssp, sorig = (2.6, 2.9, 1.), (-63 * 1.3, -45 * 1.45, 0.)
    rng = np.random.default_rng(51)
    v0 = rng.normal(size=vsize[::-1]).astype(np.float32)
    p = stack(rng, (n, nv, nu)).astype(np.float32)
    ref = oracle.backproject(rows, oracle.image(vsize, vorig, vsp), v0, oracle.image((nu, nv, n), sorig, ssp), p,
                             fdk=fdk)
    f = hip.HipFDKBackProjectionImageFilter() if fdk else hip.HipBackProjectionImageFilter()
    f.SetInput(0, to_device(hip, v0, vorig, vsp))
    f.SetInput(1, to_device(hip, p, sorig, ssp))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    assert np.linalg.norm(ref - v0) > 0.
    return f.GetOutput().numpy() - v0, ref - v0


@pytest.mark.parametrize("fdk", [False, True])
@pytest.mark.parametrize("vsize", SMALL)
def test_heights(oracle, hip, vsize, fdk):
    out, ref = _run(oracle, hip, vsize, fdk, lambda rng, shape: rng.normal(size=shape))
    assert rel_l2(out, ref) <= 1e-5


# tilted views take blocks from 655360 voxels: one voxel row under and at it, then 4, 8, 16 heights
@pytest.mark.parametrize("fdk", [False, True])
@pytest.mark.parametrize("vsize,tilt", [(v, 0.) for v in LARGE] +
                         [(v, 3.) for v in ((80, 63, 130), (80, 64, 128), (90, 83, 89), (170, 85, 171), (330, 95, 335))])
def test_heights_of_large_volumes(oracle, hip, vsize, tilt, fdk):
    """A value per view, so a voxel is off by rounding alone (1e-5 of the largest) unless it
    lies within one unit of u's or v's last place (8e-6 of 0.1 pixel a voxel) of the border:
    about 1.4e5 voxels a view lie on it, so some 50; 500 are allowed."""
    out, ref = _run(oracle, hip, vsize, fdk,
                    lambda rng, shape: np.broadcast_to(rng.uniform(0.5, 1.5, (shape[0], 1, 1)), shape), tilt)
    assert np.sum(np.abs(out - ref) > 1e-5 * np.abs(ref).max()) <= 500
