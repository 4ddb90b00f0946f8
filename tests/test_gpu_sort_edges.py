"""The radix sort on either side of the 128 tiles (524,288 pairs) up to which a pass's scatter forms its
digits' starts itself, against NumPy's stable argsort: every digit width the library uses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8193, 524_287, 524_288, 524_289, 528_385])
@pytest.mark.parametrize("bits", [13, 30, 32])
def test_sort(gsn, context, n, bits):
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(np.uint32)
    keys[rng.random(n) < 0.3] = keys[0]
    values = np.arange(n, dtype=np.uint32)
    k, v = gsn.DeviceBuffer.from_numpy(keys), gsn.DeviceBuffer.from_numpy(values)
    keys_out, values_out = gsn.DeviceBuffer((n,), np.uint32), gsn.DeviceBuffer((n,), np.uint32)
    gsn.call("gsn_selftest_sort_pairs", context.handle, k.ptr, v.ptr, n, bits, keys_out.ptr, values_out.ptr)
    context.synchronize()
    order = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(keys_out.numpy(), keys[order])
    np.testing.assert_array_equal(values_out.numpy(), values[order])
