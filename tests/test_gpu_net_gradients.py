"""The weight gradients' bricks (32 x 4 x 4 voxels, one or several per
workgroup) on ragged grids, against the numpy restatement in FP64."""
import ctypes

import numpy as np
import pytest

import cnn_reference as cnn
import hipmem
from test_gpu_net import GRAD_RTOL, Net, flatten, make_problem, to_device_layout, unflatten

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(32, 1, 3), (64, 5, 9), (96, 7, 18), (64, 62, 66)])
def test_weight_gradients_on_ragged_grids(pcf, shape):
    """The bound of the bf16 gradients at one size holds at the others; the
    last grid has 544 bricks, two per workgroup."""
    lib = pcf._abi.load_library()
    x, target, params = make_problem(shape, 6)
    net = Net(lib, shape, True)
    net.set_params(flatten(params))
    xin, tin = to_device_layout(x), to_device_layout(target)
    dx = hipmem.DeviceArray(xin.shape, dtype=np.float32).upload(xin)
    dt = hipmem.DeviceArray(tin.shape, dtype=np.float32).upload(tin)
    g = np.empty(net.n, dtype=np.float32)
    loss = ctypes.c_double(0.0)
    assert lib.pcf_net_gradients(net.h, ctypes.c_void_p(dx.ptr), ctypes.c_void_p(dt.ptr),
                                 g.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), ctypes.byref(loss)) == 0
    _, want = cnn.loss_and_grads(unflatten(flatten(params)), x, target)
    for n, ((gw, gb), (ww, wb)) in enumerate(zip(unflatten(g), want)):
        for a, b in ((gw, ww), (gb, wb)):
            err = float(np.linalg.norm(a - b)) / max(float(np.linalg.norm(b)), 1e-30)
            print(shape, "layer", n, "grad rel err", err)
            assert err <= GRAD_RTOL, (n, err)
    net.close()
