"""The matched backprojector of scans whose central column lies exactly on a diagonal of the
volume: the column is gathered like any other, so a call repeats bit for bit."""
import numpy as np
import pytest

from helpers import hip_geometry, rel_l2, to_device

pytestmark = pytest.mark.gpu


def test_diagonal_columns_repeat_bit_for_bit(oracle, hip):
    rows = np.array([[700., 1100., 45. + 90. * i, 0., 0., 0., 0., 0., 0.] for i in range(4)])
    n, sp, nd, dsp = 64, 3., 129, 2.8
    vorig, sorig = (-(n - 1) * sp / 2.,) * 3, (-(nd - 1) * dsp / 2.,) * 2 + (0.,)
    p = np.random.default_rng(71).normal(size=(4, nd, nd)).astype(np.float32)
    v0 = np.zeros((n,) * 3, np.float32)
    outs = []
    for _ in range(6):
        f = hip.HipJosephBackProjectionImageFilter()
        f.SetInput(0, to_device(hip, v0, vorig, (sp,) * 3))
        f.SetInput(1, to_device(hip, p, sorig, (dsp, dsp, 1.)))
        f.SetGeometry(hip_geometry(hip, rows))
        f.Update()
        outs.append(f.GetOutput().numpy())
    assert all(np.array_equal(outs[0], o) for o in outs[1:])
    ref = oracle.joseph_back(rows, oracle.image((n,) * 3, vorig, (sp,) * 3), v0,
                             oracle.image((nd, nd, 4), sorig, (dsp, dsp, 1.)), p)
    assert rel_l2(outs[0], ref) <= 1e-5
