"""An activation of the warm-start network's last layer that overflowed to infinity gives its 27
outputs an infinity of the weights' signs, and no output a NaN."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# the voxel inside the volume, at its corner, in the second 16 x 16 column
@pytest.mark.parametrize("shape,at", [((1, 9, 9, 9), (4, 4, 4)), ((1, 5, 6, 7), (0, 0, 0)), ((2, 6, 20, 33), (3, 17, 31))])
def test_infinite_activation(hip, shape, at):
    from oracle import cnn_ref
    from rtk_amd.warmstart import WarmStartCNN
    C, T, channel = cnn_ref.C, cnn_ref.T, 5
    rng = np.random.default_rng(7)
    # layer 1 takes the input to one channel, layers 2 - 4 keep it, layer 5 takes it past FP32's range
    d = {"w1": np.zeros((T, C)), "b1": np.zeros(C), "b6": np.zeros(1)}
    d["w1"][T // 2, channel] = 1.
    for l in range(2, 6):
        d[f"w{l}"], d[f"b{l}"] = np.zeros((T, C, C)), np.zeros(C)
        d[f"w{l}"][T // 2] = np.eye(C)
    d["w5"][T // 2, channel, channel] = 4.
    d["w6"] = (rng.choice([-1., 1.], (T, C)) * rng.uniform(0.1, 1., (T, C))).astype(np.float32).astype(float)
    x = np.zeros(shape, np.float32)
    x[(-1,) + at] = 2. ** 127
    y = WarmStartCNN(params=cnn_ref.pack(d), scale=1.).forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = x.copy()
    for t, (dx, dy, dz) in cnn_ref._taps():
        v = (at[0] - dz, at[1] - dy, at[2] - dx)
        if all(0 <= q < n for q, n in zip(v, shape[1:])):
            ref[(-1,) + v] = np.copysign(np.inf, d["w6"][t, channel])
    assert np.array_equal(y, ref)
