"""Forward passes whose outputs overwrite their inputs: the outputs of inputs
left alone, bit for bit, on the device (ofx_mlp_forward_noalloc, every
workgroup shape of the one-kernel form, and the layered form) and on the host
(enough samples for the piped form)."""
import ctypes

import numpy as np
import pytest

from oracle.mlp_oracle import NIN
from tests.test_zz_no_alloc import D2H, H2D, hip_runtime

pytestmark = pytest.mark.gpu
NOUT = 5


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("n", [1, 17, 4096, 5000, 8192])
def test_device_buffers(n, variant):
    from oneflow_amd.mlp import Mlp, _lib
    L, net = _lib(), Mlp(seed=11)
    net.set_forward_variant(variant)
    hip = hip_runtime()
    x = np.random.default_rng(n).normal(0, 1, (n, NIN)).astype(np.float32)
    want = net.forward(x)
    d = ctypes.c_void_p()
    pad, f = NOUT * n, 4  # floats before and after the inputs
    assert hip.hipMalloc(ctypes.byref(d), (2 * pad + NIN * n) * f) == 0
    xd = d.value + pad * f
    for shift in (0, -pad, -pad + 1, -1, 1, (NIN - NOUT) * n, NIN * n - 1, NIN * n):  # outputs' first float from the inputs'
        y = np.full((n, NOUT), np.nan, np.float32)
        assert hip.hipMemcpy(xd, x.ctypes.data, x.nbytes, H2D) == 0
        assert L.ofx_mlp_forward_noalloc(net.h, xd, n, xd + shift * f, None) == 0, L.ofx_last_error().decode()
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemcpy(y.ctypes.data, xd + shift * f, y.nbytes, D2H) == 0
        assert np.array_equal(y, want), shift
    assert hip.hipFree(d) == 0
    net.close()


@pytest.mark.parametrize("n", [262144, 500001])
def test_host_buffers(n):
    from oneflow_amd.mlp import Mlp, _fp, _lib
    L, net = _lib(), Mlp(seed=11)
    x = np.random.default_rng(n).normal(0, 1, NIN * n).astype(np.float32)
    want = net.forward(x.reshape(n, NIN)).ravel()
    pad = NOUT * n
    for shift in (0, -pad + 1, 4 * n, NIN * n - 1):
        buf = np.zeros(2 * pad + NIN * n, np.float32)
        buf[pad: pad + NIN * n] = x
        y = buf[pad + shift: pad + shift + pad]
        assert L.ofx_mlp_forward(net.h, _fp(buf[pad:]), n, _fp(y)) == 0, L.ofx_last_error().decode()
        assert np.array_equal(y, want), shift
    net.close()
