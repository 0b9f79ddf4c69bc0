"""Static steps that ask for no speed leave the library's workspace alone: one that does ask, on
another stream, gets its own."""
import ctypes

import numpy as np
import pytest
import torch

import pmfmhd as M
from pmfmhd._lib import lib
from test_gpu_parity import smooth_state
from test_zz_no_alloc import _buffers, _ptrs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_speed_beside_a_step_without_one(integrator, dtype):
    """The other stream's flow is thirty times as fast, so one of its partials among those of the
    call that asks would show in the speed. Expected: the call's own speed when it runs alone."""
    L, dims = lib(), (64, 60, 48)
    s = M.allocate_state(dims, 1.0 / 64, dtype=dtype)
    slow = smooth_state(dims, seed=1).astype(dtype)
    fast = slow.copy()
    fast[1:4] += 30 * slow[0]
    fast[4] += 0.5 * ((fast[1:4] ** 2).sum(0) - (slow[1:4] ** 2).sum(0)) / slow[0]
    ins = [_buffers(list(slow)), _buffers(list(fast))]
    outs = [_buffers([np.zeros(s.ncells, dtype)] * 9) for _ in range(2)]
    speeds = M.DeviceBuffer(8 * 64)
    streams = [torch.cuda.Stream() for _ in range(2)]

    def call(k, smax):
        rc = L.pmf_step_into_static(ctypes.byref(s._p), _ptrs(ins[k]), _ptrs(outs[k]), None, 1e-4, 40.0, 0.95,
                                    integrator, ctypes.c_void_p(streams[k].cuda_stream), smax)
        assert rc == 0, L.pmf_last_error().decode()

    call(0, ctypes.c_void_p(speeds.ptr))
    torch.cuda.synchronize()
    alone = speeds.download(np.float64, 1)[0]
    assert 1 < alone < 10
    for i in range(64):
        call(1, None)
        call(0, ctypes.c_void_p(speeds.ptr + 8 * i))
        call(1, None)
    torch.cuda.synchronize()
    assert np.all(speeds.download(np.float64, 64) == alone)
