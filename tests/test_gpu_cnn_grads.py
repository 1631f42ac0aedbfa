"""Weight gradients of the warm-start network on inputs whose arithmetic is exact: small
integers in every activation, weight and gradient, so BF16 storage and FP32 sums lose
nothing and the GPU's gradients equal the FP64 oracle's in any order of summation."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _integer_params(rng):
    """One weight +-1 per output channel (a permutation of the channels at random taps), so
    activations and data gradients stay within a few units; three per channel in the last
    layer."""
    from oracle import cnn_ref
    C, T = cnn_ref.C, cnn_ref.T
    d = {"w1": np.zeros((T, C)), "b1": rng.integers(0, 2, C)}
    d["w1"][rng.integers(0, T, C), np.arange(C)] = rng.choice([1., 1., -1.], C)
    for l in range(2, 6):
        w = np.zeros((T, C, C))
        w[rng.integers(0, T, C), np.arange(C), rng.permutation(C)] = rng.choice([1., 1., 1., -1.], C)
        d[f"w{l}"], d[f"b{l}"] = w, rng.integers(0, 2, C)
    d["w6"] = np.zeros((T, C))
    for _ in range(3):
        d["w6"][rng.integers(0, T, C), np.arange(C)] = rng.choice([1., -1.], C)
    d["b6"] = np.ones(1)
    return cnn_ref.pack(d)


# below, at and across the 16 x 4 x 4 tile; batches; more tiles than workgroups (512)
@pytest.mark.parametrize("shape", [(1, 1, 1, 2), (1, 4, 4, 16), (2, 5, 6, 17), (1, 9, 3, 34), (3, 3, 8, 15),
                                   (1, 1, 1, 16 * 520 + 2)])
def test_gradients_are_exact_on_integers(hip, shape):
    from oracle import cnn_ref
    from rtk_amd.warmstart import WarmStartCNN
    rng = np.random.default_rng(sum(shape))
    p = _integer_params(rng)
    x = rng.integers(0, 4, shape).astype(np.float32)
    net = WarmStartCNN(params=p, scale=1.)
    xd = torch.from_numpy(x).cuda()
    y = net.forward(xd).cpu().numpy()
    yr, _ = cnn_ref.forward(p, x.astype(np.float64), 1.)
    assert np.array_equal(y, yr)
    # 2 (y - t) / N is a whole number for an even number of voxels N
    t = (y - rng.integers(-2, 3, shape) * (y.size / 2)).astype(np.float32)
    loss, _ = net.loss_and_grads(xd, torch.from_numpy(t).cuda())
    lr, gr = cnn_ref.loss_and_grad(p, x.astype(np.float64), t.astype(np.float64), 1.)
    assert loss == pytest.approx(lr, rel=1e-12)
    assert np.any(gr != 0.)
    assert np.array_equal(net.grads(), gr)


# the 16 x 8 x 4 tile of the 32 -> 32 layers: one row under, at and over it, and over twice
@pytest.mark.parametrize("shape", [(2, 4, 7, 15), (1, 5, 8, 16), (1, 3, 9, 18), (1, 4, 17, 32)])
def test_layers_are_exact_on_integers(hip, shape):
    test_gradients_are_exact_on_integers(hip, shape)


# layer 6 from three BF16 terms per weight: one voxel, partial and several 16 x 16 columns, several
# z runs of a workgroup; a5 is exact (layers 2 - 5 pass their input on), so y's error is that of an
# FP32 sum: at most n 2^-24 of the sum of magnitudes, n < 3 * 864 + 40
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 9, 15, 16), (1, 5, 17, 18), (1, 13, 33, 31)])
def test_last_layer_to_float_rounding(hip, shape):
    from oracle import cnn_ref
    from rtk_amd.warmstart import WarmStartCNN
    C, T = cnn_ref.C, cnn_ref.T
    rng = np.random.default_rng(sum(shape))
    d = {"w1": np.zeros((T, C)), "b1": np.zeros(C), "b6": np.array([0.25])}
    d["w1"][T // 2] = rng.choice([1., -1., 0.5, -0.25], C)
    for l in range(2, 6):
        d[f"w{l}"], d[f"b{l}"] = np.zeros((T, C, C)), np.zeros(C)
        d[f"w{l}"][T // 2] = np.eye(C)
    d["w6"] = (rng.standard_normal((T, C)) * 10. ** rng.uniform(-3, 1, (T, C))).astype(np.float32).astype(float)
    x = torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).bfloat16().float()
    p = cnn_ref.pack(d)
    y = WarmStartCNN(params=p, scale=1.).forward(x.cuda()).cpu().numpy()
    yr, _ = cnn_ref.forward(p, x.numpy().astype(np.float64), 1.)
    mags = dict(d, w6=np.abs(d["w6"]))
    bound = 2600 * 2. ** -24 * (cnn_ref.forward(cnn_ref.pack(mags), x.numpy().astype(np.float64), 1.)[0]
                                + 2 * np.abs(x.numpy()))
    assert np.all(np.abs(y - yr) <= bound)
