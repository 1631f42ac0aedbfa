"""Every shape of the column forward projector (columns a workgroup, rows a lane, 64-height runs)
at its edges: row counts just below, at and above its bands, groups of rows that miss the
volume, volumes shorter and taller than a run, columns on a diagonal.  The library's choice is
asserted, so no case falls back to another kernel unnoticed."""
import ctypes

import numpy as np
import pytest

from helpers import hip_geometry, rel_l2, to_device

SID, SDD = 1000., 1500.


def _rows(n, start=3., step=None, off=0.):
    return np.array([[SID, SDD, start + i * (step or 360. / n), off * (-1) ** i, 0.6 * off, 0., 0., 0.4 * off, 0.]
                     for i in range(n)])


# name: shape, volume, voxel mm, columns, rows, pixel rows in voxels at the isocenter, views
CASES = {
    "rows_below_64": ((4, 1, 1), (33, 40, 30), (3., 3., 3.), 40, 63, 0.55, _rows(8, off=4.)),
    "rows_64": ((4, 1, 1), (30, 37, 33), (3., 2.5, 3.), 37, 64, 0.60, _rows(8)),
    "rows_above_64": ((4, 1, 1), (33, 40, 30), (3., 3., 3.), 38, 65, 0.50, _rows(8)),
    "two_below": ((8, 2, 2), (33, 70, 30), (3., 3., 3.), 97, 127, 0.55, _rows(48, off=4.)),
    "two_full": ((8, 2, 2), (30, 73, 35), (3., 2., 3.), 96, 128, 0.60, _rows(48)),
    "two_half_empty": ((8, 2, 2), (33, 20, 30), (3., 3., 3.), 97, 128, 0.60, _rows(48)),
    "three_above_two": ((8, 3, 2), (33, 90, 30), (3., 3., 3.), 97, 129, 0.55, _rows(48)),
    "three_full": ((8, 3, 2), (35, 100, 30), (3., 3., 2.5), 97, 192, 0.55, _rows(48, off=4.)),
    "three_empty_groups": ((8, 3, 2), (33, 9, 30), (3., 3., 3.), 97, 191, 0.55, _rows(48)),
    "three_two_bands": ((8, 3, 2), (30, 150, 33), (2., 2., 2.), 98, 257, 0.50, _rows(48)),
    "large_steps": ((8, 3, 3), (33, 130, 30), (3., 3., 3.), 97, 190, 0.66, _rows(48)),
    "large_steps_empty_groups": ((8, 3, 3), (33, 11, 30), (3., 3., 3.), 97, 192, 0.66, _rows(48, off=4.)),
    "four_below": ((8, 4, 3), (33, 120, 30), (3., 3., 3.), 97, 255, 0.55, _rows(48)),
    "four_full": ((8, 4, 3), (30, 160, 35), (3., 3., 3.), 96, 256, 0.66, _rows(48)),
    "four_empty_groups": ((8, 4, 3), (33, 12, 30), (3., 3., 3.), 97, 256, 0.55, _rows(48)),
    "four_second_band": ((8, 4, 3), (33, 230, 30), (2., 2., 2.), 97, 449, 0.55, _rows(48)),
    "diagonals": ((8, 4, 3), (33, 120, 33), (3., 3., 3.), 97, 256, 0.55, _rows(48, start=45., step=90.)),
    "near_diagonals": ((8, 2, 2), (33, 70, 30), (3., 3., 3.), 97, 128, 0.55, _rows(48, start=44.9, step=90.)),
}


def _images(name):
    shape, vsize, vsp, nu, nv, step, rows = CASES[name]
    dv = step * vsp[1] * SDD / SID
    du = 1.5 * SDD / SID * max(vsize[0] * vsp[0], vsize[2] * vsp[2]) / nu
    ssp = (du, dv, 1.)
    vorig = tuple(-(k - 1) * s / 2. + (0. if "diagonals" in name else 0.3) for k, s in zip(vsize, vsp))
    return shape, rows, (nu, nv, len(rows)), (-(nu - 1) * du / 2., -(nv - 1) * dv / 2., 0.), ssp, vsize, vorig, vsp


def _descriptor(size, origin, spacing):
    from rtk_amd import _lib
    d = _lib.Image()
    d.size[:], d.origin[:], d.spacing[:] = size, origin, spacing
    return d


def _shape(rows, stack, vol):
    """The library's choice for images given as (size, origin, spacing)."""
    import rtk_amd
    from rtk_amd import _lib
    g, got = hip_geometry(rtk_amd, rows), _lib.int3((-1,) * 3)
    _lib.check(_lib.lib().rtkhip_forward_project_shape(g.handle, ctypes.byref(_descriptor(*stack)),
                                                       ctypes.byref(_descriptor(*vol)), got))
    return tuple(got)


@pytest.mark.parametrize("name", list(CASES))
def test_shape_chosen(name):
    shape, rows, ssize, sorig, ssp, vsize, vorig, vsp = _images(name)
    assert _shape(rows, (ssize, sorig, ssp), (vsize, vorig, vsp)) == shape


def test_other_geometries_go_ray_by_ray():
    _, rows, ssize, sorig, ssp, *vol = _images("four_full")
    tilted = rows.copy()
    tilted[:, 5] = 1.
    assert _shape(tilted, (ssize, sorig, ssp), vol) == (0, 0, 0)
    assert _shape(rows, (ssize, sorig, (ssp[0], 1.2 * ssp[1], 1.)), vol) == (0, 0, 0)  # steps above 0.714
    assert _shape(rows, (ssize, sorig, (ssp[0], 0.6 * ssp[1], 1.)), vol) == (0, 0, 0)  # below 0.4
    # a flat volume whose y-fastest copy would be 38 times its size
    flat, sp = (1024, 5, 1024), (0.1, 3., 0.1)
    assert _shape(rows, (ssize, sorig, ssp), (flat, tuple(-(k - 1) * s / 2. for k, s in zip(flat, sp)), sp)) == (0, 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_columns_match_the_oracle(oracle, hip, name):
    """Against the per-ray projector elementwise: a height is off by at most 6e-5 voxel (three
    FP32 roundings of up to 0.7 x 449), a sample by that times the volume's largest step of 1.
    Against the float oracle the projector's bar, relative L2 <= 1e-5."""
    _, rows, ssize, sorig, ssp, vsize, vorig, vsp = _images(name)
    rng = np.random.default_rng(111)
    vol = rng.random(vsize[::-1], dtype=np.float32)
    p0 = rng.normal(size=ssize[::-1]).astype(np.float32)
    f = hip.HipForwardProjectionImageFilter()
    f.SetInput(0, to_device(hip, p0, sorig, ssp))
    f.SetInput(1, to_device(hip, vol, vorig, vsp))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    out = f.GetOutput().numpy()
    f.Update(count_samples=True)
    per_ray = f.GetOutput().numpy()
    samples, length = max(vsize[0], vsize[2]) + 1, 1.5 * max(vsp)
    assert np.abs(out - per_ray).max() <= 6e-5 * samples * length
    ref = oracle.joseph(rows, oracle.image(ssize, sorig, ssp), p0, oracle.image(vsize, vorig, vsp), vol)
    assert np.abs(ref - p0).max() > 10.
    assert rel_l2(out - p0, ref - p0) <= 1e-5
