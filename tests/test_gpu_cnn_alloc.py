"""A network handle after a call whose work buffers do not fit the GPU: the call
fails, the buffers of the call before are gone, and the next call takes new ones."""
import ctypes

import numpy as np
import pytest

from allium_amd import _lib, cnn

pytestmark = pytest.mark.gpu


def test_small_call_after_a_failed_allocation():
    rng = np.random.default_rng(3)
    net = cnn.FluxCorrector(1)
    x = rng.normal(size=(2, 5, 6, 7, 3)).astype(np.float32)
    t = rng.normal(size=(2, 5, 6, 7)).astype(np.float32)
    out, (loss, grad) = net.forward(x), net.gradient(x, t)
    d = cnn.DeviceArray32(x)
    lib = _lib.load()
    # 2^50 voxels: the first buffer of 2^54 bytes is refused before anything is launched
    for call in (lambda: lib.allium_cnn_forward_device(net.handle, 1, 1 << 15, 1 << 20, 1 << 15, d.ptr, d.ptr, None),
                 lambda: lib.allium_cnn_train_step_device(net.handle, 1, 1 << 15, 1 << 20, 1 << 15, d.ptr, d.ptr,
                                                          ctypes.c_float(1e-3), None)):
        assert call() == -4
        # no larger than the first call, and larger: neither may meet freed buffers or the old error
        np.testing.assert_array_equal(net.forward(x[:1]), out[:1])
        np.testing.assert_array_equal(net.forward(x), out)
        loss2, grad2 = net.gradient(x, t)
        assert loss2 == loss
        np.testing.assert_array_equal(grad2, grad)
