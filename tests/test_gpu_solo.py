"""Small RK4 solves run resident in one workgroup: the same sums as the stage launches.

Each grid is integrated by the resident kernel and, with the stage kernel of its tuned
variant forced, stage by stage; the states are equal bit for bit (both take entries in
list order, modes in order, directions in order).  FP64 also against the oracle's RK4 at
1e-12, the tolerance of every FP64 path.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one-cell-group remainders, both lane maps, blocks in LDS and not, every k, D = 1 and 6
GRIDS = [(1, 1, 3), (1, 5, 7), (2, 2, 5), (2, 3, 5), (2, 3, 6), (2, 4, 3), (2, 5, 4), (3, 1, 4), (3, 2, 5), (3, 3, 3),
         (3, 4, 2), (4, 2, 3), (4, 3, 2), (5, 2, 2), (6, 2, 1)]


def _op(g, kind, D, k, n, prec):
    a = [0.7, -0.3, 0.5, 0.2, 0.9, -0.4][:D]
    if kind == "wave":
        return g.wave_matrix(D, k, n, precision=prec)
    if kind == "deriv":
        return g.D_matrix(D, D, k, n, precision=prec)
    return g.transport_matrix(D, k, n, a, precision=prec)


@pytest.mark.parametrize("kind", ["transport", "wave", "deriv"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_resident_equals_stages(g, O, gpu, monkeypatch, kind, prec):
    from galerkinsparsegrids_jl_amd import _lib
    for D, k, n in GRIDS:
        print(f"[gpu] resident {kind} {prec} D={D} k={k} n={n}", flush=True)
        rng = np.random.default_rng(D * 100 + k * 10 + n)
        op = _op(g, kind, D, k, n, prec)
        y0 = rng.standard_normal(op.len)
        dt = 0.02 * 2.0 ** -n
        steps = 5
        y = op.rk4(y0, dt, steps)
        var = _lib.lib().gsg_tune_get(D, k, n, _lib.PREC[prec])
        monkeypatch.setenv("GSG_KERNEL", "plan" if var == 1 else "tile")
        ref = _op(g, kind, D, k, n, prec)
        monkeypatch.delenv("GSG_KERNEL")
        np.testing.assert_array_equal(y, ref.rk4(y0, dt, steps))
        if prec == "fp64" and kind != "deriv":
            a = [0.7, -0.3, 0.5, 0.2, 0.9, -0.4][:D] if kind == "transport" else None
            yo = O.System(kind, D, k, n, a=a).rk4(y0, dt, steps)
            assert np.linalg.norm(y - yo) < 1e-12 * np.linalg.norm(yo)
        op.close()
        ref.close()


def test_resident_many_steps_snapshots_and_device(g, gpu):
    """More steps than one launch holds, snapshots, the device call and the call without
    allocation give the same states."""
    import torch
    from galerkinsparsegrids_jl_amd import _lib
    D, k, n, steps = 2, 3, 4, 600
    op = g.wave_matrix(D, k, n)
    y0 = np.random.default_rng(0).standard_normal(op.len)
    dt = 0.02 * 2.0 ** -n
    y, snaps = op.rk4(y0, dt, steps, save_every=250)
    assert snaps.shape[0] == 2
    np.testing.assert_array_equal(op.rk4(snaps[1], dt, 100), y)
    t = torch.tensor(y0, device="cuda")
    op.rk4(t, dt, steps)
    np.testing.assert_array_equal(t.cpu().numpy(), y)
    t = torch.tensor(y0, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib().gsg_op_rk4_device_noalloc(op._h, C.c_void_p(t.data_ptr()), op.len, dt, steps, C.c_void_p(s)))
    np.testing.assert_array_equal(t.cpu().numpy(), y)


def test_resident_batch_of_uneven_sizes(g, gpu):
    """A batch whose resident solves share launches with larger ones of their shape, some
    finishing earlier: each equals its solve alone."""
    for prec in ("fp64", "fp32"):
        b = g.Batch(prec)
        ref = []
        for i, (kind, D, k, n, steps) in enumerate([("transport", 2, 3, 3, 7), ("transport", 2, 3, 5, 20),
                                                    ("wave", 2, 2, 4, 9), ("transport", 2, 3, 8, 12),
                                                    ("wave", 3, 3, 2, 20), ("transport", 3, 2, 3, 1)]):
            N = g.get_size(D, k, n) * (2 if kind == "wave" else 1)
            y0 = np.random.default_rng(i).standard_normal(N)
            a = [0.3, -0.8, 0.5][:D] if kind == "transport" else None
            dt = 0.02 * 2.0 ** -n
            b.add(kind, D, k, n, y0, dt, steps, a=a)
            op = g.wave_matrix(D, k, n, precision=prec) if kind == "wave" else g.transport_matrix(D, k, n, a, precision=prec)
            ref.append(op.rk4(y0, dt, steps))
            op.close()
        b.run()
        for i, r in enumerate(ref):
            np.testing.assert_array_equal(b.get(i), r)
        b.close()
