"""The proposal network's kernels at the edges of their tiles: 32-sample tiles, four waves of them per
workgroup, 256 training workgroups (32,768 samples in the first round), and feature pointers that
are aligned to four bytes only. Tolerances as in the network's other tests: logits at 1e-2 of their
scale and 1e-3 in the median (BF16 roundings that fall on the other side of a midpoint), gradients
at 5e-5 of the sum of their terms' magnitudes."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu


def _placed(gsn, array, skip):
    """A buffer with the array `skip` elements past its start, and the array's address."""
    buffer = gsn.DeviceBuffer.from_numpy(np.concatenate([np.zeros(skip, array.dtype), array.ravel()]))
    return buffer, buffer.ptr.value + skip * array.itemsize


def _problem(n):
    rng = np.random.default_rng(n)
    features = (rng.standard_normal((n, mlp.IN)) * rng.uniform(0.2, 3.0, mlp.IN)).astype(np.float32)
    return features, rng.integers(0, 3, n).astype(np.int32), mlp.init_params(n)


@pytest.mark.parametrize("n,skip", [(127, 0), (128, 1), (129, 3), (4097, 1), (32_769, 0), (131_073, 0)])
def test_forward(gsn, context, n, skip):
    features, _, params = _problem(n)
    net = gsn.ProposalNetwork(context, params)
    logits, to = _placed(gsn, np.full((n, 3), 7.0, np.float32), skip)
    x, address = _placed(gsn, features, skip)
    net.forward(address, n, to)
    context.synchronize()
    out = logits.numpy()
    np.testing.assert_array_equal(out[:skip], 0.0)
    expected = mlp.forward(features, params)["logits"]
    error = np.abs(out[skip:].reshape(n, 3) - expected)
    scale = np.abs(expected).max()
    assert error.max() <= 1e-2 * scale and np.median(error) <= 1e-3 * scale


@pytest.mark.parametrize("n,skip", [(2, 0), (32, 1), (33, 0), (129, 3), (32_767, 0), (32_769, 1)])
def test_gradients(gsn, context, n, skip):
    features, labels, params = _problem(n)
    net = gsn.ProposalNetwork(context, params)
    gradients = gsn.DeviceBuffer((mlp.PARAMETERS,), np.float32)
    x, address = _placed(gsn, features, skip)
    net.train_step(address, gsn.DeviceBuffer.from_numpy(labels), n, 0.0, None, gradients, want_loss=True)
    _, expected, magnitude = mlp.loss_and_gradients(features, labels, params, None, magnitudes=True)
    assert np.all(np.abs(gradients.numpy() - expected) <= 5e-5 * magnitude + 1e-12)
