"""Rays that run along a face of the volume: an odd, centred detector over a volume that begins
or ends in the plane of the source, along y (the central row of every view) or along x (the
central column of the views at 0 and 180 degrees).  RTK's box excludes its last plane and, by
the sign of a zero, its first, so those rays miss; on the other views rounding decides.  Sizes
are dyadic, so that at 0 degrees every position is exact."""
import numpy as np
import pytest

from helpers import hip_geometry, to_device

pytestmark = pytest.mark.gpu

N, SP, ND, DSP = 32, 4., 65, 2.75
HALF, SORIG = -(N - 1) * SP / 2., (-(ND - 1) * DSP / 2.,) * 2 + (0.,)
FACES = {"y_last": (HALF, -(N - 1) * SP, HALF), "y_first": (HALF, 0., HALF),
         "x_last": (-(N - 1) * SP, HALF, HALF), "x_first": (0., HALF, HALF),
         "edge": (0., -(N - 1) * SP, HALF)}


def _rows(angles):
    return np.array([[1000., 1300., a, 0., 0., 0., 0., 0., 0.] for a in angles])


def _project(hip, rows, vol, vorig, p0, count=False):
    f = hip.HipForwardProjectionImageFilter()
    f.SetInput(0, to_device(hip, p0, SORIG, (DSP, DSP, 1.)))
    f.SetInput(1, to_device(hip, vol, vorig, (SP,) * 3))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update(count_samples=True) if count else f.Update()
    return f.GetOutput().numpy()


@pytest.mark.parametrize("name", list(FACES))
def test_forward_along_faces(oracle, hip, name):
    """Elementwise: a missed or added ray is off by a whole line integral (about 64), FP32 sums
    of at most 45 samples of up to 5.7 by less than 1e-3."""
    rng = np.random.default_rng(81)
    vol = rng.random((N,) * 3).astype(np.float32)
    rows = _rows((0.,))
    p0 = rng.normal(size=(1, ND, ND)).astype(np.float32)
    out = _project(hip, rows, vol, FACES[name], p0)
    ref = oracle.joseph(rows, oracle.image((ND, ND, 1), SORIG, (DSP, DSP, 1.)), p0,
                        oracle.image((N,) * 3, FACES[name], (SP,) * 3), vol)
    assert np.abs(ref - p0).max() > 10.
    assert np.abs(out - ref).max() <= 1e-3
    # the rays that rounding decides are those of the per-ray projector
    rows = _rows((0., 20., 90., 135., 180., 270.))
    p0 = rng.normal(size=(len(rows), ND, ND)).astype(np.float32)
    out = _project(hip, rows, vol, FACES[name], p0)
    assert np.abs(out - _project(hip, rows, vol, FACES[name], p0, count=True)).max() <= 1e-3


@pytest.mark.parametrize("name", list(FACES))
def test_pair_is_a_transpose_along_faces(hip, name):
    """<FP v, p> = <v, BP p> with p on the rows and columns beside the source's plane."""
    rng = np.random.default_rng(82)
    rows = _rows((0., 20., 90., 180.))
    vol = rng.random((N,) * 3).astype(np.float32)
    p = np.zeros((len(rows), ND, ND), np.float32)
    mid = ND // 2
    p[:, mid - 1:mid + 2] = rng.random((len(rows), 3, ND))
    p[:, :, mid - 1:mid + 2] = rng.random((len(rows), ND, 3))
    fwd = _project(hip, rows, vol, FACES[name], np.zeros_like(p))
    f = hip.HipJosephBackProjectionImageFilter()
    f.SetInput(0, to_device(hip, np.zeros_like(vol), FACES[name], (SP,) * 3))
    f.SetInput(1, to_device(hip, p, SORIG, (DSP, DSP, 1.)))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    a = np.sum(fwd.astype(np.float64) * p)
    b = np.sum(vol.astype(np.float64) * f.GetOutput().numpy())
    assert a > 0. and abs(a - b) <= 1e-5 * a
