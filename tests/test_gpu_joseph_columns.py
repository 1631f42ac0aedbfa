"""The column forward projector (untilted geometries) against the per-ray projector, which
the same call takes when it counts samples, and against the float oracle.  Both sum the
same samples in FP32: relative L2 <= 1e-6 between them (a few hundred roundings of 6e-8,
uncorrelated), 1e-5 to the oracle, the projector's bar."""
import numpy as np
import pytest

from helpers import hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu


def _rows(n, start=3., sid=700., sdd=1100., off=0.):
    return np.array([[sid, sdd, start + i * 360. / n, off * (-1) ** i, 0.6 * off, 0., 0., 0.4 * off, 0.]
                     for i in range(n)])


# (volume, voxel mm, detector, pixel mm, rows): row counts around the 64-row groups and
# their multiples, column counts around a workgroup's 4 and 8, steps between rows from 0.45
# to 3 voxels (runs of 64 to 256 heights), volumes flatter and taller than a run, spacings
# that differ, views on the diagonals (workgroups that mix axes, columns on the tie),
# rays that enter and leave through the top and bottom faces
CASES = {
    "one_row": ((40, 36, 32), (3., 3., 3.), (33, 1), (5., 5.), _rows(6)),
    "rows_63": ((40, 36, 32), (3., 3., 3.), (31, 63), (5., 2.5), _rows(6, off=4.)),
    "rows_65": ((40, 36, 32), (3., 3., 3.), (8, 65), (16., 2.2), _rows(6, off=4.)),
    "rows_200": ((64, 61, 67), (2., 2., 2.), (9, 200), (14., 1.4), _rows(5)),
    "rows_330": ((90, 120, 70), (1.5, 1.5, 1.5), (17, 330), (11., 1.05), _rows(4)),
    "large_steps": ((64, 200, 50), (2., 0.5, 2.), (40, 100), (4., 1.6), _rows(7)),
    "flat": ((61, 7, 53), (2., 9., 2.), (70, 40), (2.9, 2.9), _rows(6)),
    "tall": ((33, 280, 35), (3., 1., 3.), (37, 290), (4., 1.3), _rows(5)),
    "diagonals": ((48, 40, 44), (2.5, 2.5, 2.5), (96, 80), (2., 2.), _rows(8, start=0.)),
    "diagonal_ties": ((41, 33, 41), (3., 3., 3.), (65, 41), (3., 4.), _rows(8, start=45.)),
    "steep": ((40, 60, 40), (3., 3., 3.), (45, 150), (4.5, 3.), _rows(6, sid=200., sdd=420.)),
    "many_waves": ((30, 28, 26), (4., 4., 4.), (100, 96), (2., 2.), _rows(90)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_columns_match_the_per_ray_projector(oracle, hip, name):
    vsize, vsp, (nu, nv), (du, dv), rows = CASES[name]
    n = len(rows)
    vorig = tuple(-(k - 1) * s / 2. + 0.3 for k, s in zip(vsize, vsp))
    sorig = (-(nu - 1) * du / 2., -(nv - 1) * dv / 2., 0.)
    rng = np.random.default_rng(31)
    vol = rng.random(vsize[::-1]).astype(np.float32)
    p0 = rng.normal(size=(n, nv, nu)).astype(np.float32)
    f = hip.HipForwardProjectionImageFilter()
    f.SetInput(0, to_device(hip, p0, sorig, (du, dv, 1.)))
    f.SetInput(1, to_device(hip, vol, vorig, vsp))
    f.SetGeometry(hip_geometry(hip, rows))
    f.Update()
    out = f.GetOutput().numpy()
    f.Update(count_samples=True)
    per_ray = f.GetOutput().numpy()
    scale = np.linalg.norm((per_ray - p0).astype(np.float64))
    assert scale > 0.
    e = np.linalg.norm(out.astype(np.float64) - per_ray) / scale
    assert e <= 1e-6, f"{name}: rel L2 to the per-ray projector {e:.3g}"
    ref = oracle.joseph(rows, oracle.image((nu, nv, n), sorig, (du, dv, 1.)), p0, oracle.image(vsize, vorig, vsp), vol)
    e = rel_l2(out - p0, ref - p0)
    assert e <= 1e-5, f"{name}: rel L2 to the oracle {e:.3g}"
    # in place, and a second volume through the same plan
    f.SetInPlace(True)
    f.SetInput(1, to_device(hip, vol[::-1].copy(), vorig, vsp))
    f.Update()
    again = f.GetOutput().numpy()
    ref = oracle.joseph(rows, oracle.image((nu, nv, n), sorig, (du, dv, 1.)), p0, oracle.image(vsize, vorig, vsp),
                        vol[::-1].copy())
    assert rel_l2(again - p0, ref - p0) <= 1e-5
