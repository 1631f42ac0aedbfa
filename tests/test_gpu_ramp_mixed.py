"""The mixed-radix ramp filter at the edges of its row groups (several pairs of rows per
workgroup): row counts around a group, every radix, lengths with and without the twiddles in
LDS and with one pair of rows per workgroup; in place.  Bar: 1e-5 relative L2 to the oracle,
the filter's."""
import numpy as np
import pytest

from helpers import rel_l2, to_device

pytestmark = pytest.mark.gpu


# padded lengths: 301 -> 605 = 5 11^2; 169 -> 338 = 2 13^2; 343 -> 686 = 2 7^3; 243 -> 486 =
# 2 3^5; 1001 -> 2002 = 2 7 11 13; 1750 -> 3500 = 2^2 5^3 7; 5 -> 10 = 2 5; 2 -> 4
@pytest.mark.parametrize("nu", [301, 169, 343, 243, 1001, 1750, 5, 3])
@pytest.mark.parametrize("nv,n", [(1, 1), (2, 1), (7, 1), (8, 3), (17, 2)])
def test_row_groups(oracle, hip, nu, nv, n):
    org, sp = (-(nu - 1) * 0.35, -(nv - 1) * 0.4, 0.), (0.7, 0.8, 1.)
    p = (1 + 0.2 * np.random.default_rng(nu + nv).normal(size=(n, nv, nu))).astype(np.float32)
    ref = oracle.ramp(oracle.image((nu, nv, n), org, sp), p, gpf=13, hann=0.9)
    for in_place in (False, True):
        f = hip.HipFFTRampImageFilter()
        f.SetInput(to_device(hip, p, org, sp))
        f.SetInPlace(in_place)
        f.SetHannCutFrequency(0.9)
        f.Update()
        e = rel_l2(f.GetOutput().numpy(), ref)
        assert e <= 1e-5, f"{nu} x {nv} x {n}, in place {in_place}: {e:.3g}"
