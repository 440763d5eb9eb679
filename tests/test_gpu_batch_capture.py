"""Uneven batches long enough to capture their steps: eager phases, captured ones, a rebuild
when finished solves hold a quarter of the batch, and phases too short to capture after it.
Each solve equals its run alone, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOLVES = [("transport", 3, 3, 5, 90), ("transport", 2, 3, 8, 41), ("wave", 3, 2, 5, 64), ("transport", 4, 3, 3, 33),
          ("wave", 2, 4, 5, 1), ("transport", 3, 4, 4, 40)]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("parts", [(200,), (20, 3, 200), (1, 40, 1, 1, 200)])
def test_uneven_batch_equals_alone(g, gpu, prec, parts):
    print(f"[gpu] uneven captured batch {prec} {parts}", flush=True)
    b = g.Batch(prec)
    ref = []
    for i, (kind, D, k, n, steps) in enumerate(SOLVES):
        y0 = np.random.default_rng(i).standard_normal(g.get_size(D, k, n) * (2 if kind == "wave" else 1))
        a = [0.3, -0.8, 0.5, 0.1][:D] if kind == "transport" else None
        dt = 0.02 * 2.0 ** -n
        b.add(kind, D, k, n, y0, dt, steps, a=a)
        op = g.wave_matrix(D, k, n, precision=prec) if kind == "wave" else g.transport_matrix(D, k, n, a, precision=prec)
        ref.append(op.rk4(y0, dt, steps))
        op.close()
    for p in parts:
        b.step(p)
    for i, r in enumerate(ref):
        np.testing.assert_array_equal(b.get(i), r)
    b.close()
