"""Rays along y through volumes whose z planes have 2^24 voxels and more, so that the in-slice
offsets of their taps need more than 24 bits: both Joseph projectors against the float oracle."""
import numpy as np
import pytest

from helpers import hip_geometry, to_device

pytestmark = pytest.mark.gpu

SIZE, SP = (4096, 4097, 3), 0.1
VORIG = tuple(-(k - 1) * SP / 2. for k in SIZE)
# the source above the volume: out-of-plane angle 90 degrees
ROWS = np.array([[5000., 6000., 3. * i, 0.02, 0.03, 90., 0., 0., 0.] for i in range(2)])


# pixels of a voxel, and so large that the backprojector's ray tiles exceed their window
@pytest.mark.parametrize("dsp", [(0.11, 0.07), (0.9, 0.07)])
def test_wide_slices(oracle, hip, dsp):
    nu, nv, n = 20, 9, len(ROWS)
    sorig, ssp = (-(nu - 1) * dsp[0] / 2., -(nv - 1) * dsp[1] / 2., 0.), dsp + (1.,)
    rng = np.random.default_rng(101)
    vol = rng.random(SIZE[::-1], dtype=np.float32) + np.arange(SIZE[2], dtype=np.float32)[:, None, None]
    p = rng.random((n, nv, nu), dtype=np.float32)
    ov, os_ = oracle.image(SIZE, VORIG, (SP,) * 3), oracle.image((nu, nv, n), sorig, ssp)
    g = hip_geometry(hip, ROWS)
    f = hip.HipForwardProjectionImageFilter()
    f.SetInput(0, to_device(hip, np.zeros_like(p), sorig, ssp))
    f.SetInput(1, to_device(hip, vol, VORIG, (SP,) * 3))
    f.SetGeometry(g)
    f.Update()
    ref = oracle.joseph(ROWS, os_, np.zeros_like(p), ov, vol)
    assert np.sum(ref > 100.) > 20  # rays that cross the volume
    # two FP32 sums of up to 4097 positive samples
    assert np.all(np.abs(f.GetOutput().numpy() - ref) <= 2 * 4100 * 2. ** -24 * ref.max())
    b = hip.HipJosephBackProjectionImageFilter()
    b.SetInput(0, hip.ConstantImageSource(SIZE, (SP,) * 3, VORIG, 0.))
    b.SetInput(1, to_device(hip, p, sorig, ssp))
    b.SetGeometry(g)
    b.Update()
    out = b.GetOutput().numpy()
    ref = oracle.joseph_back(ROWS, ov, np.zeros(SIZE[::-1], np.float32), os_, p)
    # a voxel's few contributions, each rounded a few times (weights, products, sums)
    assert np.abs(out - ref).max() <= 64 * 2. ** -24 * ref.max()
