"""The matched backprojector's outer layers, 64 heights of a column a wavefront: heights
around 64, volumes that are all shell, detector row counts around the 16 x 16 blocks of the
per-ray pass, rays entering through every face, against the float oracle (relative L2 <= 1e-5,
the backprojector's bar)."""
import numpy as np
import pytest

from helpers import circular_rows, hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vsize,nu,nv", [((5, 63, 5), 21, 70), ((6, 64, 5), 17, 16), ((5, 65, 9), 33, 81),
                                         ((13, 129, 7), 31, 97), ((20, 5, 21), 45, 15), ((33, 62, 30), 49, 64)])
def test_outer_layers(oracle, hip, vsize, nu, nv):
    rows = circular_rows(7, 600., 1000., start=3.)
    n, sp = len(rows), 100. / max(vsize)
    ssp = (230. / nu, 230. / nv, 1.)
    # rows at most two voxels apart at the detector's scale, as the gather asks
    ssp = (min(ssp[0], 3. * sp), min(ssp[1], 2.4 * sp), 1.)
    vorig = tuple(-(k - 1) * sp / 2. for k in vsize)
    sorig = (-(nu - 1) * ssp[0] / 2., -(nv - 1) * ssp[1] / 2., 0.)
    rng = np.random.default_rng(61)
    v0 = rng.normal(size=vsize[::-1]).astype(np.float32)
    p = rng.normal(size=(n, nv, nu)).astype(np.float32)
    ref = oracle.joseph_back(rows, oracle.image(vsize, vorig, (sp,) * 3), v0, oracle.image((nu, nv, n), sorig, ssp), p)
    f = hip.HipJosephBackProjectionImageFilter()
    f.SetInput(0, to_device(hip, v0, vorig, (sp,) * 3))
    f.SetInput(1, to_device(hip, p, sorig, ssp))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    assert np.linalg.norm(ref - v0) > 0.
    assert rel_l2(f.GetOutput().numpy() - v0, ref - v0) <= 1e-5
