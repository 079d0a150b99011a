"""ofx_mlp_forward_noalloc on a caller's stream as the first call on a new
network (seeded weights): its weight copies are complete when ofx_mlp_create
returns, so the outputs are ofx_mlp_forward's, bit for bit."""
import ctypes

import numpy as np
import pytest

from oracle.mlp_oracle import NIN
from tests.test_zz_no_alloc import D2H, H2D, hip_runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 700, 8192])
def test_first_call_on_another_stream(n):
    from oneflow_amd.mlp import Mlp, _lib
    L = _lib()
    first = Mlp(seed=1)  # the library and its runtime are up before the buffers are made
    hip = hip_runtime()
    x = np.random.default_rng(n).normal(0, 1, (n, NIN)).astype(np.float32)
    y = np.full((n, 5), np.nan, np.float32)
    xd, yd, st = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(xd), x.nbytes) == 0
    assert hip.hipMalloc(ctypes.byref(yd), y.nbytes) == 0
    assert hip.hipStreamCreate(ctypes.byref(st)) == 0
    assert hip.hipMemcpy(xd, x.ctypes.data, x.nbytes, H2D) == 0
    net = Mlp(seed=11)
    assert L.ofx_mlp_forward_noalloc(net.h, xd, n, yd, st) == 0, L.ofx_last_error().decode()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemcpy(y.ctypes.data, yd, y.nbytes, D2H) == 0
    assert np.array_equal(y, net.forward(x)) and np.isfinite(y).all() and np.abs(y).max() > 0
    assert hip.hipStreamDestroy(st) == 0
    assert hip.hipFree(xd) == 0 and hip.hipFree(yd) == 0
    net.close()
    first.close()
