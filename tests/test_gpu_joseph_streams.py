"""Matched backprojections of different volume sizes one after the other on a stream of their
own, with no wait between them: each call works with its own sizes, whatever the stream still
has to do for the call before."""
import numpy as np
import pytest
import torch

from helpers import circular_rows, hip_geometry, to_device

pytestmark = pytest.mark.gpu

# more outer columns first, then fewer (the same buffers serve both), then more again
SIZES = [(96, 80, 90), (33, 70, 30), (5, 64, 40), (96, 80, 90)]


def _filters(hip):
    rows = circular_rows(60, 700., 1100., start=3.)
    rng = np.random.default_rng(91)
    p = rng.normal(size=(len(rows), 120, 140)).astype(np.float32)
    stack = to_device(hip, p, (-139 * 1.4, -119 * 1.4, 0.), (2.8, 2.8, 1.))
    out = []
    for size in SIZES:
        f = hip.HipJosephBackProjectionImageFilter()
        f.SetInput(0, hip.ConstantImageSource(size, (3.,) * 3, tuple(-(k - 1) * 1.5 for k in size), 0.))
        f.SetInput(1, stack)
        f.SetGeometry(hip_geometry(hip, rows))
        out.append(f)
    return out


def test_sizes_back_to_back_on_a_stream(hip):
    filters = _filters(hip)
    ref = []
    for f in filters:
        f.Update()
        ref.append(f.GetOutput().numpy())
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(stream):
            outs = []
            for f in filters:
                f.Update()
                outs.append(f.GetOutput())
        stream.synchronize()
        assert all(np.array_equal(o.numpy(), r) for o, r in zip(outs, ref))
