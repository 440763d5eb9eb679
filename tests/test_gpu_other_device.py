"""An application whose stream belongs to another device than the operator is refused or
right: its kernels never run on a device that does not hold the operator's memory."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_stream_of_another_device(g, gpu):
    import torch
    from galerkinsparsegrids_jl_amd import _lib
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two devices")
    op = g.transport_matrix(2, 3, 5, [0.3, -0.7])
    x = torch.tensor(np.random.default_rng(0).standard_normal(op.len), device="cuda:0")
    ref, y = op @ x, torch.zeros_like(x)
    torch.cuda.synchronize(0)
    for stream in (0, torch.cuda.Stream(device="cuda:1").cuda_stream):
        print(f"[gpu] stream of another device {stream}", flush=True)
        with torch.cuda.device(1):
            rc = _lib.lib().gsg_op_apply_device(op._h, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), op.len,
                                                C.c_void_p(stream))
            torch.cuda.synchronize(1)
        torch.cuda.synchronize(0)
        assert rc < 0 or torch.equal(y, ref)
    op.close()
