"""FP32 applications whose result overwrites the input: the operator reads the rounded copy of
the input, so y = A x in place equals y = A x beside it, bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ops(g):
    import scipy.sparse as sp
    m = 60000  # rows that gather from all over the vector
    A = sp.random(m, m, 40 / m, format="csc", random_state=np.random.default_rng(0))
    yield "csc", g.csc_matrix(A, precision="fp32")
    yield "transport", g.transport_matrix(3, 3, 6, [0.3, -0.7, 0.5], precision="fp32")
    yield "wave", g.wave_matrix(2, 3, 6, precision="fp32")


def test_in_place_equals_out_of_place(g, gpu):
    import torch
    from galerkinsparsegrids_jl_amd import _lib
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for name, op in _ops(g):
        for shift in (0, 5, -5):  # the result starts at the input, after it and before it
            print(f"[gpu] in place {name} {shift}", flush=True)
            buf = torch.tensor(np.random.default_rng(1).standard_normal(op.len + 10), device=gpu)
            x, y = buf[5:5 + op.len], buf[5 + shift:5 + shift + op.len]
            ref = (op @ x.clone()).cpu().numpy()
            _lib.check(_lib.lib().gsg_op_apply_device(op._h, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), op.len, s))
            np.testing.assert_array_equal(y.cpu().numpy(), ref)
        op.close()
