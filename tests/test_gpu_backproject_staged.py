"""Voxel and FDK backprojection from staged detector rectangles, at sizes that take blocks of 2
(untilted only), 4, 8 and 16 heights, of stacks that differ from pixel to pixel: tilted views
(from 655360 voxels), untilted views among them, views whose columns are horizontal, footprints
inside the detector, across its border and larger than the stage, rows of a multiple of four
pixels and others, every storage type, against the oracle in 64 bits."""
import numpy as np
import pytest
import torch

from helpers import hip_geometry, to_device

pytestmark = pytest.mark.gpu


def _rows(n, tilt=(3., -2.), off=0.):
    return np.array([[700., 1100., 11. + i * 360. / n, off, -off, tilt[0] * (-1) ** i, tilt[1], 2., -1.]
                     for i in range(n)])


MIXED = np.concatenate([_rows(2), _rows(2, tilt=(0., 0.)), _rows(1, tilt=(0., 90.)), _rows(2, tilt=(-4., 1.))])
UNTILTED = _rows(5, tilt=(0., 0.), off=3.)

# volume, voxel mm, detector, pixel mm, rows
CASES = {
    "tilted_4": ((80, 65, 130), (2., 2.1, 1.25), (64, 47), (4.2, 4.5), _rows(5)),
    "tilted_4_odd": ((81, 66, 127), (2., 2.1, 1.25), (61, 50), (4.4, 4.4), _rows(5)),
    "tilted_4_inside": ((80, 65, 130), (1., 1., 1.), (96, 93), (4., 4.), _rows(5)),
    "tilted_8": ((170, 85, 171), (1., 2., 1.), (64, 60), (4.2, 4.4), _rows(5, off=5.)),
    "tilted_8_odd": ((165, 90, 175), (1., 2., 1.), (63, 60), (4.2, 4.4), _rows(5)),
    "tilted_16": ((330, 95, 335), (0.5, 1.7, 0.5), (100, 90), (2.9, 2.9), _rows(5)),
    "steep_4": ((80, 65, 130), (2., 2.1, 1.25), (60, 62), (4.5, 4.5), _rows(4, tilt=(25., 40.))),
    "steep_16": ((330, 95, 335), (0.5, 1.7, 0.5), (101, 90), (2.9, 2.9), _rows(4, tilt=(25., 40.))),
    "mixed_4": ((80, 65, 130), (2., 2.1, 1.25), (64, 60), (4.2, 4.2), MIXED),
    "mixed_8_odd": ((170, 85, 171), (1., 2., 1.), (67, 60), (4.2, 4.4), MIXED),
    "beyond_the_stage_4": ((80, 70, 120), (2., 2., 1.4), (300, 280), (0.9, 0.95), _rows(5)),
    "beyond_the_stage_8": ((170, 85, 171), (1., 2., 1.), (301, 260), (0.9, 0.6), _rows(5)),
    "untilted_2": ((40, 33, 41), (4., 4., 4.), (64, 47), (4.2, 4.5), UNTILTED),
    "untilted_4": ((120, 75, 125), (1.3, 2.1, 1.3), (64, 47), (4.2, 4.5), UNTILTED),
    "untilted_4_odd": ((122, 73, 119), (1.3, 2.1, 1.3), (61, 50), (4.4, 4.4), UNTILTED),
    "untilted_8": ((170, 85, 171), (1., 2., 1.), (64, 60), (4.2, 4.4), UNTILTED),
    "untilted_16": ((330, 95, 335), (0.5, 1.7, 0.5), (100, 90), (2.9, 2.9), UNTILTED),
    "untilted_beyond_the_stage_4": ((120, 75, 125), (1.3, 2.1, 1.3), (302, 280), (0.9, 0.6), UNTILTED),
}
HEIGHTS = {"2": (0, 512), "4": (512, 1024), "8": (1024, 2560), "16": (2560, 1 << 30)}


def test_cases_take_the_heights_they_name(hip):
    """16 heights from 2560 blocks of them, 8 from 1024 blocks, 4 from 512."""
    for name, (vsize, *_) in CASES.items():
        columns = -(-vsize[0] // 16) * -(-vsize[2] // 16)
        groups = {h: columns * -(-vsize[1] // h) for h in (4, 8, 16)}
        heights = 16 if groups[16] >= 2560 else 8 if groups[8] >= 1024 else 4 if groups[4] >= 512 else 2
        assert str(heights) in name.split("_"), name
        assert "untilted" in name or (np.prod(vsize) >= 655360 and heights >= 4), name


def _near_border(oracle, rows, ov, os_, shape, detector, margin):
    """Voxels that some view sees within `margin` pixels of a line where either border rule
    ends (-1/2, 0, n - 1 and n - 1/2): rounding decides whether they count."""
    z, y, x = np.ogrid[tuple(slice(n) for n in shape)]
    near = np.zeros(shape, bool)
    for m in oracle.bp_matrices(rows, ov, os_, transpose=False):
        w, *uv = (m[r, 0] * x + m[r, 1] * y + m[r, 2] * z + m[r, 3] for r in (2, 0, 1))
        for c, n in zip(uv, detector):
            c = c / w
            for line in (-0.5, 0., n - 1., n - 0.5):
                near |= np.abs(c - line) < margin
    return near


@pytest.mark.parametrize("fdk", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_staged_backprojection(oracle, hip, name, fdk):
    """Elementwise, away from the border lines.  u and v are quotients of sums of four FP32 products
    each, of magnitudes up to twice the detector: 8 roundings each of numerator and w.  A pixel value
    in [0, 1], which changes by at most 1 a pixel along each axis, is then off by twice that a view
    (weights up to 1.5 in FDK); a wrong tap is off by about 1/3."""
    vsize, vsp, (nu, nv), (du, dv), rows = CASES[name]
    n = len(rows)
    vorig = tuple(-(k - 1) * s / 2. for k, s in zip(vsize, vsp))
    sorig, ssp = (-(nu - 1) * du / 2., -(nv - 1) * dv / 2., 0.), (du, dv, 1.)
    ov, os_ = oracle.image(vsize, vorig, vsp), oracle.image((nu, nv, n), sorig, ssp)
    rng = np.random.default_rng(121)
    v0 = rng.random(vsize[::-1], dtype=np.float32)
    p = rng.integers(0, 65, size=(n, nv, nu)) / 64.  # exact in every storage type
    ref = oracle.backproject(rows, ov, v0.astype(np.float64), os_, p, fdk=fdk)
    coord = 8 * 2. ** -24 * 2 * 2 * max(nu, nv)
    tol = 1.5 * n * (2 * coord + 1e-6)
    near = _near_border(oracle, rows, ov, os_, vsize[::-1], (nu, nv), coord)
    assert near.mean() < 0.02 and np.mean(ref - v0 > 0.2) > 0.2
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        f = hip.HipFDKBackProjectionImageFilter() if fdk else hip.HipBackProjectionImageFilter()
        f.SetInput(0, to_device(hip, v0, vorig, vsp))
        f.SetInput(1, to_device(hip, p, sorig, ssp, dtype=dtype))
        f.SetGeometry(hip_geometry(hip, rows))
        f.Update()
        err = np.where(near, 0., np.abs(f.GetOutput().numpy() - ref))
        assert err.max() <= tol, f"{dtype}: {err.max():.3g} > {tol:.3g}, {np.sum(err > tol)} voxels"
