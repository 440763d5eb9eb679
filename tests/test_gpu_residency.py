"""FP32 solves that change between the resident kernel and the stage launches.

A served solve runs resident while little else runs and in stage launches beside a large
one, and changes whenever the server rebuilds its batch.  The stage launches read the
first stage's input from the float copy of the state that the step before left, so the
resident kernel has to leave one too.  Both give the same sums, so each result equals the
solve run alone bit for bit."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = [("transport", 2, 3, 5), ("wave", 3, 2, 4), ("wave", 2, 3, 4)]
LARGE = ("transport", 4, 4, 8)  # 2.7 M coefficients: the small solves run in stage launches beside it


def _input(g, kind, D, k, n, seed):
    rng = np.random.default_rng(seed)
    a = [0.7, -0.3, 0.5, 0.2][:D]
    return a, rng.standard_normal(g.get_size(D, k, n) * (2 if kind == "wave" else 1)), 0.02 * 2.0 ** -n


def _alone(g, kind, D, k, n, a, y0, dt, steps):
    op = g.wave_matrix(D, k, n, precision="fp32") if kind == "wave" else g.transport_matrix(D, k, n, a, precision="fp32")
    y = op.rk4(y0, dt, steps)
    op.close()
    return y


def _until(srv, rid, status):
    end = time.time() + 60
    while srv.poll(rid) != status:
        assert time.time() < end
        time.sleep(0.001)


def test_server_solves_leave_and_enter_residency(g, gpu):
    steps = 40000
    print("[gpu] residency: the large solve alone", flush=True)
    al, yl, dtl = _input(g, *LARGE, 1)
    large = _alone(g, *LARGE, al, yl, dtl, 5)
    small = [(s,) + _input(g, *s, 10 + i) for i, s in enumerate(SMALL)]
    with g.Server(precision="fp32") as srv:
        ids = [srv.submit(*s, y0, dt, steps, a=a if s[0] == "transport" else None) for s, a, y0, dt in small]
        for i in ids:
            _until(srv, i, "running")
        time.sleep(0.02)  # some ticks resident
        for rep in range(2):  # beside the large solve, and resident again after it
            print(f"[gpu] residency: large solve {rep}", flush=True)
            y, _ = srv.wait(srv.submit(*LARGE, yl, dtl, 5, a=al))
            np.testing.assert_array_equal(y, large)
            assert all(srv.poll(i) == "running" for i in ids)
        got = [srv.wait(i)[0] for i in ids]
    for (s, a, y0, dt), y in zip(small, got):
        print(f"[gpu] residency: {s} alone", flush=True)
        np.testing.assert_array_equal(y, _alone(g, *s, a, y0, dt, steps))
