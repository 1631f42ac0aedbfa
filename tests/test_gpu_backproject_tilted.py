"""Voxel and FDK backprojection of tilted geometries (per-voxel perspective, ITK's border
rule) at the edges of the staged kernel's 16^3 blocks and 64 x 48 detector tiles, against the
float oracle with the backprojector's bar of 1e-5 relative L2."""
import numpy as np
import pytest
import torch

from helpers import hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu


def _rows(n, tilt=(3., -2.), sid=700., sdd=1100., off=0.):
    return np.array([[sid, sdd, 11. + i * 360. / n, off, -off, tilt[0] * (-1) ** i, tilt[1], 2., -1.]
                     for i in range(n)])


# volume, voxel mm, detector, pixel mm, rows
CASES = {
    "block_remainders": ((17, 15, 33), (4., 4., 4.), (64, 60), (4., 4.), _rows(9)),
    "odd_detector": ((40, 36, 32), (3., 3., 3.), (61, 47), (4.4, 4.4), _rows(7)),
    "detector_inside_the_shadow": ((48, 50, 52), (4., 4., 4.), (40, 36), (5., 5.), _rows(8, off=6.)),
    "one_voxel_one_row": ((1, 1, 1), (2., 2., 2.), (9, 2), (3., 3.), _rows(4)),
    "steep_tilts": ((30, 31, 29), (4., 4., 4.), (96, 96), (3.5, 3.5), _rows(6, tilt=(25., 40.))),
    # untilted views among tilted ones keep their own border rule
    "mixed_views": ((33, 30, 31), (4., 4., 4.), (52, 50), (5., 5.),
                    np.concatenate([_rows(3), _rows(3, tilt=(0., 0.))])),
}


@pytest.mark.parametrize("fdk", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_tilted_backprojection(oracle, hip, name, fdk):
    vsize, vsp, (nu, nv), (du, dv), rows = CASES[name]
    n = len(rows)
    vorig = tuple(-(k - 1) * s / 2. for k, s in zip(vsize, vsp))
    sorig = (-(nu - 1) * du / 2., -(nv - 1) * dv / 2., 0.)
    rng = np.random.default_rng(41)
    v0 = rng.normal(size=vsize[::-1]).astype(np.float32)
    # values that FP16 holds exactly, so every storage type backprojects the same stack
    p = (rng.integers(-64, 65, size=(n, nv, nu)) / 16.).astype(np.float32)
    ref = oracle.backproject(rows, oracle.image(vsize, vorig, vsp), v0,
                             oracle.image((nu, nv, n), sorig, (du, dv, 1.)), p, fdk=fdk)
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        f = hip.HipFDKBackProjectionImageFilter() if fdk else hip.HipBackProjectionImageFilter()
        f.SetInput(0, to_device(hip, v0, vorig, vsp))
        f.SetInput(1, to_device(hip, p, sorig, (du, dv, 1.), dtype=dtype))
        f.SetGeometry(hip_geometry(hip, rows))
        f.Update()
        e = rel_l2(f.GetOutput().numpy() - v0, ref - v0)
        assert e <= (1e-5 if np.abs(ref - v0).max() > 1e-3 else 1e-3), f"{name} {dtype}: {e:.3g}"


@pytest.mark.parametrize("nu", [300, 301])
def test_footprints_beyond_the_tile(hip, nu):
    """Blocks whose footprint does not fit the stage: a volume that every view covers, from
    a stack of ones, is the number of views exactly (a + f (1 - 1) = 1 for any weight)."""
    rows = _rows(5)
    f = hip.HipBackProjectionImageFilter()
    f.SetInput(0, hip.ConstantImageSource((32, 32, 32), (2.5, 2.5, 2.5), (-38.75,) * 3, 0.))
    f.SetInput(1, hip.ConstantImageSource((nu, nu, 5), (0.8, 0.8, 1.), (-(nu - 1) * 0.4,) * 2 + (0.,), 1.))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    assert np.array_equal(f.GetOutput().numpy(), np.full((32, 32, 32), 5., np.float32))
